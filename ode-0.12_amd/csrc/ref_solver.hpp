// ref_solver.hpp -- SOR_LCP in the reference's row order
// (ode/src/quickstep.cpp:406-582), relaxed by the whole workgroup.
//
// A row reads and writes the constraint forces of its two bodies and its own
// impulse (a friction row also reads its normal row's impulse, a row of the
// same bodies).  So the sequence only orders rows that share a body: with
//   level(row) = 1 + max(level of the previous row of body 1, of body 2)
// (previous in the sweep's order) the rows of one level share no body and
// relax at once, and every body still sees its rows in the sequence's order:
// the same operations on the same operands, bit for bit.  Islands share no
// body, so one set of levels covers them all.
//
// What bounds it: a level is one dependent pass of about 70 instructions with
// an LDS round trip, so a sweep costs its number of levels, which a shuffled
// order keeps near the largest number of rows on one body: 43 levels of 0.27
// us for a stack of 10 boxes (120 rows), about 200 for a pile of 1500 bodies
// (11 889 rows).  One lane per island in sequence, the kernel before this,
// took 0.44 us (rows in LDS) to 1.3 us (in global memory) a row: the solve of
// the stack went from 1.06 to 0.27 ms, that of the pile from 304 to 3.5 ms.
//
// Every 8 sweeps the order is shuffled; shuffle and levels are built by all
// lanes as well:
//  - the draws of step i of an island start from the generator state skipped
//    ahead by i - 1 draws;
//  - "for i: swap(o[i], o[sw_i])", sw_i <= i, finds o[i] untouched by the
//    steps before it, so step i puts the element i at sw_i and moves what was
//    there to position i.  An element placed at p by step i is moved next by
//    the first later step that draws p (to that step's own position), and
//    from a position j by the first later step that draws j: chains of
//    logarithmic length, followed by every element on its own;
//  - each row finds its successor on either body among that body's rows; the
//    levels come from a breadth-first pass that releases a row when its
//    predecessors are placed.
//
// Included by step_kernels.hip inside namespace odemi, after its workgroup
// helpers.
#pragma once

// One side (body) of a row: two lanes relax a row, one per body, and exchange
// their halves of J fc.  A shuffle is followed by writing the sides in the
// levels' order, so that a level's are read side by side, without an index.
struct alignas(16) RefSide {
  float J[6], iMJ[6];
  float rhs, cfm, lo, hi, ad;
  int lam, lf, f;   // where the impulse, the normal row's impulse and the body's fc are
};
// lf of a row without a friction index, and of a lane that writes nothing
enum { REF_NO_FRICTION = -1, REF_IDLE = -2 };

// Placement of the working set: everything in the LDS pool; the (read-only)
// sides in global memory; sides and schedule in global memory (both are read
// ahead of their level); everything in the world's scratch.
enum { REF_IN_LDS = 0, REF_ROWS_GLOBAL = 1, REF_SCHED_GLOBAL = 2, REF_IN_GLOBAL = 3 };

// Worlds up to this many rows place their levels with one wavefront, and relax
// them with it where few levels are wider than it.  It saves the barriers of
// worlds of few rows: against all wavefronts throughout, a pass of a stack of
// 10 (120 rows) takes 370 for 395 us, of 24 (282 rows) 442 for 473, of a pile
// of 30 bodies (186 rows) 616 for 664; 333 worlds of 360 rows, a world of 633
// and worlds above the limit the same within 1 %; 333 worlds of 656 rows 1.66
// for 1.60 ms (1.71 if they were relaxed by one wavefront whatever the levels'
// width).  A limit of 256 rows costs the stack of 24 its gain, one of 4096
// changes nothing beyond 2 %.
constexpr int REF_SOLO_ROWS = 1024;

// Bytes of the solve's working set: 6 fc floats per body and for no body
// (which stay zero), and the impulses (state); the order with its levels
// (schedule); the sides in the levels' order.
__device__ inline long long ref_state_bytes(int nrows, int nb) {
  return (24LL * (nb + 1) + 4LL * nrows + 15) & ~15LL;
}
__device__ inline long long ref_sched_bytes(int nrows, int nb) { return (4LL * (9LL * nrows + 1 + nb) + 15) & ~15LL; }
__device__ inline long long ref_sides_bytes(int nrows) { return 2LL * (long long)sizeof(RefSide) * nrows; }

// The order and its levels, in LDS or in the world's scratch.  While an
// order is shuffled s1, s2, pos, deg and lv hold the draws, the heads and
// links of the lists of steps by drawn position, the first later step that
// draws each position, and the new order.
struct RefSched {
  int *o, *lv, *ls;    // the order; rows by level; first of each level
  int *ba, *bs;        // rows of each body (bs: end of its part of ba)
  int *s1, *s2;        // a row's successor on body 1 and body 2, or -1
  int *pos, *deg;      // position in the order; predecessors not yet placed
  int state;           // where the state is (ref_at)
  __device__ RefSched(int *p, int m, int state_at) {
    state = state_at;
    o = p; lv = o + m; ls = lv + m; ba = ls + m + 1; s1 = ba + 2 * m; s2 = s1 + m; pos = s2 + m; deg = pos + m;
    bs = deg + m;
  }
};

// island of position x: the last whose first row is at most x
__device__ inline int ref_island_of(const int *isl, int ngroups, int x) {
  int lo = 0, hi = ngroups - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (isl[5 * mid + 2] <= x) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Rows of each body, and the order before the first shuffle: an island's rows
// without a friction index from its head, the others from its tail.
__device__ inline void ref_sched_init(const RefSched &W, const Row *R, const int *isl, int m, int ngroups, int nb,
                                      Shared &sh) {
  const int nt = blockDim.x, t = threadIdx.x;
  for (int b = t; b < nb; b += nt) W.bs[b] = 0;
  __syncthreads();
  for (int r = t; r < m; r += nt) {
    atomicAdd(&W.bs[R[r].b1], 1);
    if (R[r].b2 >= 0) atomicAdd(&W.bs[R[r].b2], 1);
  }
  __syncthreads();
  {
    const int per = (nb + nt - 1) / nt, d0 = min(t * per, nb), d1 = min(d0 + per, nb);
    int loc = 0;
    for (int d = d0; d < d1; d++) loc += W.bs[d];
    int tot;
    int off = block_excl_scan(loc, tot, sh);
    for (int d = d0; d < d1; d++) { const int cnt = W.bs[d]; W.bs[d] = off; off += cnt; }
  }
  const int per = (m + nt - 1) / nt, x0 = min(t * per, m), x1 = min(x0 + per, m);
  {
    int loc = 0;
    for (int r = x0; r < x1; r++) loc += R[r].findex == -1;
    int tot;
    int off = block_excl_scan(loc, tot, sh);   // its barriers also order bs
    for (int r = x0; r < x1; r++) { W.pos[r] = off; off += R[r].findex == -1; }
  }
  __syncthreads();
  for (int r = t; r < m; r += nt) {
    W.ba[atomicAdd(&W.bs[R[r].b1], 1)] = r;
    if (R[r].b2 >= 0) W.ba[atomicAdd(&W.bs[R[r].b2], 1)] = r;
  }
  if (x0 < x1) {
    int k = ref_island_of(isl, ngroups, x0), r0 = isl[5 * k + 2], mk = isl[5 * k + 3], n0 = W.pos[r0];
    for (int r = x0; r < x1; r++) {
      while (r >= r0 + mk) { k++; r0 = isl[5 * k + 2]; mk = isl[5 * k + 3]; n0 = r < r0 + mk ? W.pos[r0] : 0; }
      const int n = W.pos[r] - n0;   // rows without a friction index before r in its island
      if (R[r].findex == -1) W.o[r0 + n] = r;
      else W.o[r0 + mk - 1 - (r - r0 - n)] = r;
    }
  }
  __syncthreads();
}

// the order's `nth` shuffle (each island makes rows - 1 draws per shuffle)
__device__ inline void ref_shuffle(const RefSched &W, const int *isl, int m, int ngroups, int nth) {
  const int nt = blockDim.x, t = threadIdx.x;
  int *sw = W.s1, *head = W.s2, *nxt = W.pos, *first = W.deg, *o2 = W.lv;
  for (int x = t; x < m; x += nt) head[x] = -1;
  __syncthreads();
  const int per = (m + nt - 1) / nt, x0 = min(t * per, m), x1 = min(x0 + per, m);
  if (x0 < x1) {
    int k = ref_island_of(isl, ngroups, x0), r0 = isl[5 * k + 2], mk = isl[5 * k + 3];
    unsigned seed = lcg_skip((unsigned)isl[5 * k + 4],
                             (unsigned long long)nth * (mk - 1) + (x0 > r0 ? x0 - r0 - 1 : 0));
    for (int x = x0; x < x1; x++) {
      if (x >= r0 + mk) {
        do { k++; r0 = isl[5 * k + 2]; mk = isl[5 * k + 3]; } while (x >= r0 + mk);
        seed = lcg_skip((unsigned)isl[5 * k + 4], (unsigned long long)nth * (mk - 1));
      }
      if (x == r0) {
        sw[x] = x;   // the first position draws nothing
      } else {
        const int p = r0 + lcg_below(seed, x - r0 + 1);
        sw[x] = p;
        nxt[x] = atomicExch(&head[p], x);
      }
    }
  }
  __syncthreads();
  for (int x = t; x < m; x += nt) {
    int f = m;
    for (int j = head[x]; j >= 0; j = nxt[j])
      if (j > x && j < f) f = j;
    first[x] = f;
  }
  __syncthreads();
  for (int x = t; x < m; x += nt) {
    const int p = sw[x];
    int f = m, fin = p;
    for (int j = head[p]; j >= 0; j = nxt[j])
      if (j > x && j < f) f = j;
    while (f < m) { fin = f; f = first[f]; }
    o2[fin] = W.o[x];
  }
  __syncthreads();
  for (int x = t; x < m; x += nt) W.o[x] = o2[x];
  __syncthreads();
}

// the row of body b (its rows at ba[lo, hi)) that follows position p, or -1;
// has_prev: some row of the body precedes p
__device__ inline int ref_successor(const RefSched &W, int b, int p, int &has_prev) {
  const int lo = b > 0 ? W.bs[b - 1] : 0, hi = W.bs[b];
  int best = 0x7fffffff, row = -1, prev = 0;
  for (int k = lo; k < hi; k += 4) {
    int q[4], pq[4];
#pragma unroll
    for (int u = 0; u < 4; u++) q[u] = W.ba[min(k + u, hi - 1)];
#pragma unroll
    for (int u = 0; u < 4; u++) pq[u] = W.pos[q[u]];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      prev |= pq[u] < p;
      if (pq[u] > p && pq[u] < best) { best = pq[u]; row = q[u]; }
    }
  }
  has_prev = prev;
  return row;
}

// the levels of the current order; returns their number.  solo: one wavefront
// is to relax them.
__device__ inline int ref_levels(const RefSched &W, const Row *R, int m, bool &solo, Shared &sh) {
  const int nt = blockDim.x, t = threadIdx.x;
  for (int x = t; x < m; x += nt) W.pos[W.o[x]] = x;
  if (t < 3) sh.lcount[t] = 0;
  __syncthreads();
  for (int r = t; r < m; r += nt) {
    const int p = W.pos[r], b2 = R[r].b2;
    int d1, d2 = 0, n2 = -1;
    W.s1[r] = ref_successor(W, R[r].b1, p, d1);
    if (b2 >= 0) n2 = ref_successor(W, b2, p, d2);
    W.s2[r] = n2;
    W.deg[r] = d1 + d2;
    if (d1 + d2 == 0) W.lv[atomicAdd(&sh.lcount[2], 1)] = r;
  }
  __syncthreads();
  int b = 0, e = sh.lcount[2], d = 0;
  if (t == 0) W.ls[0] = 0;
  if (m <= REF_SOLO_ROWS) {
    // few rows: the first wavefront places all levels, the others wait once
    // (no barriers between levels; places from ballots)
    if (t < 64) {
      int passes = 0;
      while (b < e) {
        if (t == 0) W.ls[d + 1] = e;
        passes += (e - b + 31) >> 5;
        int n = e;
        for (int x0 = b; x0 < e; x0 += 64) {
          const int x = x0 + t, r = x < e ? W.lv[x] : 0;
          const int n1 = x < e ? W.s1[r] : -1, n2 = x < e ? W.s2[r] : -1;
          const bool p1 = n1 >= 0 && atomicSub(&W.deg[n1], 1) == 1;
          const bool p2 = n2 >= 0 && atomicSub(&W.deg[n2], 1) == 1;
          const unsigned long long m1 = __ballot(p1), m2 = __ballot(p2), lt = (1ULL << t) - 1;
          if (p1) W.lv[n + __popcll(m1 & lt)] = n1;
          n += __popcll(m1);
          if (p2) W.lv[n + __popcll(m2 & lt)] = n2;
          n += __popcll(m2);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        b = e;
        e = n;
        d++;
      }
      if (t == 0) { sh.lcount[0] = d; sh.lcount[1] = passes; }
    }
    __syncthreads();
    // one wavefront relaxes the levels if few of them are wider than it (up
    // to a quarter more passes than levels; the limit above has both sides)
    d = sh.lcount[0];
    solo = sh.lcount[1] <= d + (d >> 2);
    __syncthreads();
    return d;
  }
  solo = false;
  while (b < e) {
    // the next level is counted in lcount[d % 3]; the counter after it is
    // cleared here, two barriers after its last reader
    const int c = d % 3, c1 = c == 2 ? 0 : c + 1;
    if (t == 0) { W.ls[d + 1] = e; sh.lcount[c1] = 0; }
    for (int x = b + t; x < e; x += nt) {
      const int r = W.lv[x], n1 = W.s1[r], n2 = W.s2[r];
      if (n1 >= 0 && atomicSub(&W.deg[n1], 1) == 1) W.lv[e + atomicAdd(&sh.lcount[c], 1)] = n1;
      if (n2 >= 0 && atomicSub(&W.deg[n2], 1) == 1) W.lv[e + atomicAdd(&sh.lcount[c], 1)] = n2;
    }
    __syncthreads();
    b = e;
    e += sh.lcount[c];
    d++;
  }
  __syncthreads();
  return d;
}

// A place of the state as an int: an LDS address, or a byte offset into the
// world's scratch.
template <int PLACE>
__device__ inline float *ref_at(char *base, int where) {
  if constexpr (PLACE == REF_IN_GLOBAL) return (float *)(base + where);
  else return (float *)(LdsFloat *)(unsigned long long)(unsigned)where;
}

// the sides of all rows in the levels' order
template <int PLACE>
__device__ inline void ref_sides(const RefSched &W, const Row *rows, RefSide *sides, int m, int nb, int F, int LAM) {
  for (int x = threadIdx.x; x < 2 * m; x += blockDim.x) {
    const int side = x & 1, r = W.lv[x >> 1];
    const Row &R = rows[r];
    RefSide q;
    for (int k = 0; k < 6; k++) { q.J[k] = R.J[6 * side + k]; q.iMJ[k] = R.iMJ[6 * side + k]; }
    q.rhs = R.rhs; q.cfm = R.cfm; q.lo = R.lo; q.hi = R.hi; q.ad = R.ad;
    const int b = side ? R.b2 : R.b1;
    q.lam = LAM + 4 * r;
    q.lf = b < 0 ? REF_IDLE : (R.findex >= 0 ? LAM + 4 * R.findex : REF_NO_FRICTION);
    q.f = F + 24 * (b >= 0 ? b : nb);
    if (b < 0)
      for (int k = 0; k < 6; k++) q.J[k] = 0.f;
    sides[x] = q;
  }
}

// The sweeps over the levels, lanes 2 k and 2 k + 1 for the two bodies of a
// level's k-th row.  A level's sides are loaded DEPTH levels before it, its
// end one or two before that; a level wider than the lanes goes on in steps
// of them.  SOLO: one wavefront does it all and needs no barriers (its LDS
// accesses are in order).
template <int PLACE, bool SOLO>
__device__ inline void ref_sweeps(const RefSched &W, const RefSide *sides, char *base, int D, int total) {
  constexpr int DEPTH = PLACE == REF_IN_LDS ? 1 : 2, NB = DEPTH + 1;
  const int t = threadIdx.x, step = SOLO ? 32 : blockDim.x >> 1, k0 = t >> 1;
  const RefSide *mine = sides + t;
  // quickstep.cpp:484-582 (J and b scaled by ad there), the sums in its order
  auto relax = [&](const RefSide &q, auto &&ahead) {
    float *f = ref_at<PLACE>(base, q.f), *lam = ref_at<PLACE>(base, q.lam);
    const float old = *lam, lf = *ref_at<PLACE>(base, max(q.lf, 0));
    float v[6];
    for (int k = 0; k < 6; k++) v[k] = f[k];
    ahead();
    float s = q.J[0] * v[0] + q.J[1] * v[1] + q.J[2] * v[2] + q.J[3] * v[3] + q.J[4] * v[4] + q.J[5] * v[5];
    // body 1's half plus body 2's (zero where there is none)
    s += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(s), 0xB1, 0xf, 0xf, true));
    float delta = q.ad * (q.rhs - old * q.cfm - s);
    const bool fr = q.lf >= 0;
    const float hf = fabsf(q.hi * lf), hi = fr ? hf : q.hi, lo = fr ? -hf : q.lo;
    float nl = old + delta;
    const bool below = nl < lo, above = !below && nl > hi;
    nl = below ? lo : (above ? hi : nl);
    delta = below || above ? nl - old : delta;
    if (q.lf != REF_IDLE) {
      *lam = nl;
      for (int k = 0; k < 6; k++) f[k] = v[k] + delta * q.iMJ[k];
    }
  };
  // ends of the levels to come, in the order of the sweeps
  int dn = 0;
  auto next_end = [&] {
    const int e = W.ls[dn + 1];
    dn = dn + 1 == D ? 0 : dn + 1;
    return e;
  };
  int e1 = next_end(), e2 = next_end();
  int dl = 0, last = 0;   // the level loaded next, end of the one before it
  RefSide q[NB];
  int sq[NB], eq[NB];
#pragma unroll
  for (int u = 0; u < NB; u++) { q[u].lam = q[u].f = W.state; q[u].lf = REF_IDLE; }
  auto load = [&](RefSide &qn, int &s, int &e) {
    e = __builtin_amdgcn_readfirstlane(e1);
    s = dl == 0 ? 0 : last;
    last = e;
    dl = dl + 1 == D ? 0 : dl + 1;
    e1 = e2;
    e2 = next_end();
    if (s + k0 < e) qn = mine[2 * (size_t)s];
    else qn.lf = REF_IDLE;
  };
#pragma unroll
  for (int u = 0; u < DEPTH; u++) load(q[u], sq[u], eq[u]);
  for (int n = 0; n < total; n += NB) {
#pragma unroll
    for (int u = 0; u < NB; u++) {
      if (n + u >= total) break;
      constexpr int ahead_by = DEPTH;
      const int un = (u + ahead_by) % NB;
      relax(q[u], [&] { load(q[un], sq[un], eq[un]); });
      for (int x = sq[u] + step; x < eq[u]; x += step) {
        RefSide w;
        if (x + k0 < eq[u]) w = mine[2 * (size_t)x];
        else { w.lam = w.f = W.state; w.lf = REF_IDLE; }
        relax(w, [] {});
      }
      if (SOLO) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      else if (PLACE == REF_IN_GLOBAL) __syncthreads();
      else lds_barrier();
    }
  }
}

// isl: [cons0, ncons, row0, nrows, seed] per island, rows ascending; gws:
// the world's scratch for ref_state_bytes + ref_sched_bytes + ref_sides_bytes.
template <int PLACE>
__device__ __attribute__((noinline)) void sor_reference(Row *rows, float *bt, const int *isl, char *gws, LdsChar *pool,
                                                        int nrows, int ngroups, int nb, int iters, Shared &sh) {
  rows = uniform_global(rows);
  bt = uniform_global(bt);
  isl = uniform_global(isl);
  gws = uniform_global(gws);
  pool = uniform(pool);
  nrows = uniform(nrows);
  ngroups = uniform(ngroups);
  nb = uniform(nb);
  iters = uniform(iters);
  const int nt = blockDim.x, t = threadIdx.x, m = nrows;
  char *const lds = (char *)pool;
  const long long b0 = ref_state_bytes(m, nb), b1 = b0 + ref_sched_bytes(m, nb);
  float *F = PLACE == REF_IN_GLOBAL ? (float *)gws : (float *)lds;
  float *LAM = F + 6 * (nb + 1);
  RefSide *sides = PLACE == REF_IN_LDS ? (RefSide *)(lds + b1) : (RefSide *)(gws + b1);
  // the state's place as ref_at takes it
  const int at = PLACE == REF_IN_GLOBAL ? 0 : (int)(unsigned long long)pool;
  const RefSched W(PLACE >= REF_SCHED_GLOBAL ? (int *)(gws + b0) : (int *)(lds + b0), m, at);
  for (int i = t; i < m; i += nt) LAM[i] = 0.f;
  for (int i = t; i < 6 * (nb + 1); i += nt) F[i] = 0.f;
  __syncthreads();
  if (m > 0 && iters > 0) {
    ref_sched_init(W, rows, isl, m, ngroups, nb, sh);
    for (int it = 0; it < iters; it += 8) {
      ref_shuffle(W, isl, m, ngroups, it >> 3);
      bool solo;
      const int D = uniform(ref_levels(W, rows, m, solo, sh));
      ref_sides<PLACE>(W, rows, sides, m, nb, at, at + 24 * (nb + 1));
      __syncthreads();
      const int total = D * min(8, iters - it);
      if (uniform(solo)) {
        if (t < 64) ref_sweeps<PLACE, true>(W, sides, gws, D, total);
      } else {
        ref_sweeps<PLACE, false>(W, sides, gws, D, total);
      }
      __syncthreads();
    }
  }
  // the integration reads the fc of all bodies
  for (int i = t; i < m; i += nt) rows[i].lambda = LAM[i];
  for (int b = t; b < nb; b += nt)
    for (int k = 0; k < 6; k++) bt[32 * b + 9 + k] = F[6 * b + k];
  __syncthreads();
}
