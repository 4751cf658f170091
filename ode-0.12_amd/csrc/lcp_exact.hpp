// lcp_exact.hpp -- the LCP of one island solved exactly on the device
// (dWorldStep): A = J M^-1 J^T + cfm/h, b = rhs, bounds lo/hi, friction rows
// bounded by their normal row.  The answer is the one dSolveLCP defines
// (lcp.cpp:784-1100): the LCP of the rows without a findex with the friction
// impulses at zero, then every friction row's bounds fixed at
// +-|hi * lambda_normal| (0 when the normal impulse is 0) and the LCP of all
// rows solved with those bounds.  With cfm > 0 each of the two
// box-constrained LCPs has one solution; it is found by block principal
// pivoting (Judice & Pires) with a single-index fallback (Murty), on a
// Cholesky factorisation of the free rows computed by the whole workgroup.
//
// What bounds it: the factorisations of a pivoting round are a few hundred
// dependent steps of little work each, so everything they touch is kept in
// the LDS pool when an island fits, the triangular solves run in one
// wavefront without barriers, and a column costs two barriers.
//
// Included by step_kernels.hip inside namespace odemi, after its workgroup
// helpers (Shared, block_sum, block_max).
#pragma once

// Placement of an island's workspace: everything in the LDS pool; all but the
// matrix; all in global memory.
enum { LCP_IN_LDS = 0, LCP_A_GLOBAL = 1, LCP_IN_GLOBAL = 2 };

// One island's workspace: A[m*m], L[m*ld], diag[m], then x, r, lo, hi, b (m
// each) and the int arrays st, fr (m each); the rows' J and inv(M) J^T (12
// floats each) and bodies.  ld is odd, so that a column's elements fall on
// different LDS banks.
struct LcpWs {
  float *A, *L, *diag, *x, *r, *lo, *hi, *b, *J, *iMJ;
  int *st, *fr, *b1, *b2;
  int ld;
};

__device__ inline int lcp_ld(int m) { return m | 1; }
__device__ inline long long lcp_vec_bytes(int m) { return 4LL * m * (10 + 24); }
__device__ inline long long lcp_factor_bytes(int m) { return 4LL * m * lcp_ld(m); }
__device__ inline long long lcp_matrix_bytes(int m) { return 4LL * m * m; }

// ws: the world's workspace in global memory (lcp_ws_floats of its M >= m rows)
template <int PLACE>
__device__ inline LcpWs lcp_place(float *ws, char *lds, int m) {
  LcpWs W;
  W.ld = PLACE == LCP_IN_GLOBAL ? m : lcp_ld(m);
  W.x = PLACE == LCP_IN_GLOBAL ? ws + 2 * (size_t)m * m : (float *)lds;
  W.r = W.x + m; W.lo = W.r + m; W.hi = W.lo + m; W.b = W.hi + m; W.diag = W.b + m;
  W.st = (int *)(W.diag + m); W.fr = W.st + m; W.b1 = W.fr + m; W.b2 = W.b1 + m;
  W.J = (float *)(W.b2 + m); W.iMJ = W.J + 12 * m;
  W.L = PLACE == LCP_IN_GLOBAL ? ws + (size_t)m * m : W.iMJ + 12 * m;
  W.A = PLACE == LCP_IN_LDS ? W.L + (size_t)m * W.ld : ws;
  return W;
}

// st: 0 free, 1 at lo, 2 at hi, 3 outside the problem (held at 0)
enum { LS_FREE = 0, LS_LO = 1, LS_HI = 2, LS_OUT = 3 };

// x_F solving A_FF x_F = b_F - A_F,fixed x_fixed for the n free rows listed
// in W.fr; false when A_FF is not positive definite.  All lanes call it.
template <int PLACE>
__device__ inline bool lcp_free_solve(const LcpWs &W, const float *b, int m, int n, Shared &sh) {
  const int nt = blockDim.x, t = threadIdx.x, ld = W.ld;
  float *L = W.L;
  for (int a = t; a < n; a += nt) {
    const int i = W.fr[a];
    float v = b[i];
    for (int j = 0; j < m; j++)
      if (W.st[j] == LS_LO || W.st[j] == LS_HI) v -= W.A[(size_t)i * m + j] * W.x[j];
    W.r[a] = v;
  }
  // lanes as rows of 16 columns
  const int tj = t & 15, ti = t >> 4, ni = nt >> 4;
  for (int a = ti; a < n; a += ni) {
    const size_t row = (size_t)W.fr[a] * m;
    for (int c = tj; c <= a; c += 16) L[(size_t)a * ld + c] = W.A[row + W.fr[c]];
  }
  __syncthreads();
  // right-looking Cholesky, one column per round; the diagonal goes to diag
  // (the column's own is read by all lanes until the next barrier)
  for (int k = 0; k < n; k++) {
    const float d = L[(size_t)k * ld + k];
    if (!(d > 0.f)) return false;   // the same in every lane
    const float dk = sqrtf(d);
    if (t == 0) W.diag[k] = dk;
    for (int i = k + 1 + t; i < n; i += nt) L[(size_t)i * ld + k] /= dk;
    __syncthreads();
    for (int i = k + 1 + ti; i < n; i += ni) {   // trailing triangle
      const float lik = L[(size_t)i * ld + k];
#pragma unroll 4
      for (int j = k + 1 + tj; j <= i; j += 16) L[(size_t)i * ld + j] -= lik * L[(size_t)j * ld + k];
    }
    __syncthreads();
  }
  // L y = r, then L^T x = y: one wavefront, whose LDS accesses are in order
  auto step = [] {
    if (PLACE == LCP_IN_GLOBAL) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  if (t < 64) {
    for (int k = 0; k < n; k++) {
      const float rk = W.r[k] / W.diag[k];
      if (t == 0) W.r[k] = rk;
      for (int i = k + 1 + t; i < n; i += 64) W.r[i] -= L[(size_t)i * ld + k] * rk;
      step();
    }
    for (int k = n - 1; k >= 0; k--) {
      const float rk = W.r[k] / W.diag[k];
      if (t == 0) W.r[k] = rk;
      for (int i = t; i < k; i += 64) W.r[i] -= L[(size_t)k * ld + i] * rk;
      step();
    }
    for (int a = t; a < n; a += 64) W.x[W.fr[a]] = W.r[a];
  }
  __syncthreads();
  return true;
}

// The box-constrained LCP over the rows with st != LS_OUT (their start
// partition in st).  Returns the pivoting rounds, or -1 at the cap or on a
// matrix that is not positive definite.  All lanes call it.
template <int PLACE>
__device__ inline int lcp_blcp(const LcpWs &W, const float *b, int m, float bscale, Shared &sh) {
  const int nt = blockDim.x, t = threadIdx.x;
  int best = m + 1, backup = 3;
  const float tw = 1e-5f * (1.f + bscale);
  for (int round = 0; round < 8 * m + 16; round++) {
    // fixed rows at their bound, rows outside at 0; the free list
    int n = 0;
    for (int i0 = 0; i0 < m; i0 += nt) {
      const int i = i0 + t, s = i < m ? W.st[i] : LS_OUT;
      if (i < m) {
        if (s == LS_LO) W.x[i] = W.lo[i];
        else if (s == LS_HI) W.x[i] = W.hi[i];
        else if (s == LS_OUT) W.x[i] = 0.f;
      }
      int tot;
      const int off = block_excl_scan(s == LS_FREE ? 1 : 0, tot, sh);
      if (s == LS_FREE) W.fr[n + off] = i;
      n += tot;
    }
    __syncthreads();
    if (!lcp_free_solve<PLACE>(W, b, m, n, sh)) return -1;
    // infeasible rows: free ones outside their bounds, bound ones whose w
    // pushes away from the bound
    int nbad = 0, last = -1;
    for (int i = t; i < m; i += nt) {
      const int s = W.st[i];
      bool bad = false;
      if (s == LS_FREE) {
        const float tx = 1e-6f * (1.f + fabsf(W.x[i]));
        bad = W.x[i] < W.lo[i] - tx || W.x[i] > W.hi[i] + tx;
      } else if (s != LS_OUT) {
        float w = -b[i];
        for (int j = 0; j < m; j++)
          if (W.st[j] != LS_OUT) w += W.A[(size_t)i * m + j] * W.x[j];
        bad = (s == LS_LO && w < -tw) || (s == LS_HI && w > tw);
      }
      if (bad) { nbad++; last = i > last ? i : last; }
      W.r[i] = bad ? 1.f : 0.f;   // the free solve's scratch is free again
    }
    const int cnt = block_sum(nbad, sh);
    if (cnt == 0) return round;
    const int lastbad = (int)block_max((float)last, sh);
    // all infeasible rows change sides while their number falls (and for a
    // few rounds after), else only the last one
    bool all;
    if (cnt < best) { best = cnt; backup = 3; all = true; }
    else if (backup > 0) { backup--; all = true; }
    else all = false;
    for (int i = t; i < m; i += nt) {
      if (W.r[i] == 0.f || (!all && i != lastbad)) continue;
      const int s = W.st[i];
      if (s == LS_FREE) W.st[i] = W.x[i] < W.lo[i] ? LS_LO : LS_HI;
      else W.st[i] = LS_FREE;
    }
    __syncthreads();
  }
  return -1;
}

// One island, its m rows from r0 on: lambda into the rows, fc of its bodies
// into bt.  False when the solve did not finish (the impulses are then the
// clamped last iterate).
template <int PLACE>
__device__ __attribute__((noinline)) bool lcp_exact_island(Row *rows, float *bt, float *ws, LdsChar *pool, int r0,
                                                           int m, int nb, Shared &sh) {
  r0 = uniform(r0);
  rows = uniform_global(rows) + r0;
  bt = uniform_global(bt);
  nb = uniform(nb);
  ws = uniform_global(ws);
  m = uniform(m);
  const LcpWs W = lcp_place<PLACE>(ws, (char *)uniform(pool), m);
  const int nt = blockDim.x, t = threadIdx.x;
  for (int e = t; e < 12 * m; e += nt) {
    const int i = e / 12, k = e - 12 * i;
    W.J[e] = rows[i].J[k];
    W.iMJ[e] = rows[i].iMJ[k];
  }
  float bmax = 0.f;
  bool fric = false;
  for (int i = t; i < m; i += nt) {
    const Row &R = rows[i];
    W.b1[i] = R.b1;
    W.b2[i] = R.b2;
    W.lo[i] = R.lo;
    W.hi[i] = R.hi;
    // rows held at lo = hi (= 0) and, first, the friction rows stay out
    W.st[i] = (R.findex >= 0 || R.lo == R.hi) ? LS_OUT : LS_FREE;
    W.x[i] = 0.f;
    W.b[i] = R.rhs;
    W.diag[i] = R.cfm;
    bmax = fmaxf(bmax, fabsf(R.rhs));
    fric |= R.findex >= 0;
  }
  bmax = block_max(bmax, sh);
  const int any_fric = block_sum(fric ? 1 : 0, sh);
  // A_ij = J_i . M^-1 J_j^T over the bodies the rows share, + cfm/h (in diag
  // until the first factorisation)
  for (int i = t >> 4; i < m; i += nt >> 4)
    for (int j = t & 15; j < m; j += 16) {
      float s = 0.f;
      for (int si = 0; si < 2; si++) {
        const int bi = si ? W.b2[i] : W.b1[i];
        if (bi < 0) continue;
        for (int sj = 0; sj < 2; sj++)
          if ((sj ? W.b2[j] : W.b1[j]) == bi)
            for (int q = 0; q < 6; q++) s += W.J[12 * i + 6 * si + q] * W.iMJ[12 * j + 6 * sj + q];
      }
      W.A[(size_t)i * m + j] = s + (i == j ? W.diag[i] : 0.f);
    }
  __syncthreads();
  int rounds = lcp_blcp<PLACE>(W, W.b, m, bmax, sh);
  if (rounds >= 0 && any_fric) {
    for (int i = t; i < m; i += nt) {
      const Row &R = rows[i];
      if (R.findex < 0) continue;
      const float xn = W.x[R.findex - r0];
      if (xn == 0.f) {
        W.lo[i] = W.hi[i] = 0.f;
        W.st[i] = LS_OUT;
      } else {
        W.hi[i] = fabsf(R.hi * xn);
        W.lo[i] = -W.hi[i];
        W.st[i] = LS_FREE;
      }
    }
    __syncthreads();
    rounds = lcp_blcp<PLACE>(W, W.b, m, bmax, sh);
  }
  for (int i = t; i < m; i += nt) rows[i].lambda = W.x[i] = fminf(fmaxf(W.x[i], W.lo[i]), W.hi[i]);
  __syncthreads();
  // the rows of each body in order (a body's rows are all in this island)
  for (int e = t; e < 6 * nb; e += nt) {
    const int b = e / 6, q = e - 6 * b;
    float f = 0.f;
    bool any = false;
#pragma unroll 4
    for (int r = 0; r < m; r++) {
      const bool one = W.b1[r] == b;
      if (one || W.b2[r] == b) {
        f += W.iMJ[12 * r + (one ? 0 : 6) + q] * W.x[r];
        any = true;
      }
    }
    if (any) bt[32 * b + 9 + q] = f;
  }
  __syncthreads();
  return rounds >= 0;
}

// Every island of the world (isl: [cons0, ncons, row0, nrows, seed] per
// island) solved exactly; lambda into the rows, fc = M^-1 J^T lambda per body
// into bt.  An island larger than the workspace, or a solve that does not
// finish, sets OVF_LCP; its impulses are then zero or the clamped last iterate.
__device__ void lcp_exact_world(const DevBatch &B, int w, Row *rows, float *bt, const int *isl, int ngroups, int nb,
                                Shared &sh) {
  const int nt = blockDim.x, t = threadIdx.x, M = B.lcp_ws_rows;
  float *ws = B.lcp_ws + (size_t)w * B.lcp_ws_stride;
  LdsChar *pool = (LdsChar *)od_pool;
  bool fail = false;
  for (int b = t; b < nb; b += nt)
    for (int q = 0; q < 6; q++) bt[32 * b + 9 + q] = 0.f;
  __syncthreads();
  for (int k = 0; k < ngroups; k++) {
    const int r0 = isl[5 * k + 2], m = isl[5 * k + 3];
    if (m <= 0) continue;
    if (m > M) {
      for (int i = t; i < m; i += nt) rows[r0 + i].lambda = 0.f;
      fail = true;
      continue;
    }
    const long long v = lcp_vec_bytes(m), f = lcp_factor_bytes(m), a = lcp_matrix_bytes(m);
    bool ok;
    if (v + f + a <= B.lds_bytes) ok = lcp_exact_island<LCP_IN_LDS>(rows, bt, ws, pool, r0, m, nb, sh);
    else if (v + f <= B.lds_bytes) ok = lcp_exact_island<LCP_A_GLOBAL>(rows, bt, ws, pool, r0, m, nb, sh);
    else ok = lcp_exact_island<LCP_IN_GLOBAL>(rows, bt, ws, pool, r0, m, nb, sh);
    fail |= !ok;
  }
  if (fail && t == 0) raise_overflow(B, w, OVF_LCP);
  __syncthreads();
}
