// step_kernels.hip -- the ODE 0.12 step path on MI355X, one workgroup per
// world.
//
//   collide:  geom AABBs -> uniform-grid broadphase (cell keys, bitonic sort,
//             run scan with a home-cell rule) -> narrowphase, one pair per lane
//   step:     body preprocessing -> constraint rows (contact, ball, hinge,
//             hinge2) -> SOR-LCP -> velocity update -> integration
//
// The SOR-LCP runs in one of two orders:
//   ORDER_REFERENCE  islands found by the reference's depth-first walk, rows in
//                    island/joint order, non-friction rows first and friction
//                    rows reversed at the tail, shuffled every 8 iterations by
//                    the reference's LCG (each island's RNG state is obtained by
//                    skip-ahead so islands relax in parallel); candidate pairs
//                    are sorted into the reference hash space's callback order.
//   ORDER_COLORED    constraints coloured so that one colour shares no body;
//                    a colour's constraints relax in parallel, one per lane.
//
// Reference: ode/src/collision_space.cpp:420-583 (hash space),
// ode/src/quickstep.cpp:342-1025 (SOR-LCP, dxQuickStepper),
// ode/src/util.cpp:255-568 (integrator, islands).
#include <hip/hip_runtime.h>

#include "colliders.hpp"
#include "devmath.hpp"
#include "joints_dev.hpp"
#include "layout.hpp"

namespace odemi {

constexpr int WG = 512;            // most lanes of a workgroup
constexpr int COLOUR_WIDTH = 256;  // most constraints of a colour
constexpr int MAX_COLORS_LDS = 256;   // colour buckets counted in LDS

struct Shared {
  int wsum[WG / 64];
  float wmax[WG / 64];
  int ival[16];
  float fval[8];
  int ccount[MAX_COLORS_LDS + 1];
  int ccur[MAX_COLORS_LDS];
  int lcount[4];   // rows of a level (ref_levels)
};

// dynamic LDS pool of the workgroup (size DevBatch::lds_bytes): sort keys,
// colouring state and the coloured solver's working set, one after another
extern __shared__ __align__(16) unsigned char od_pool[];

// optional per-phase wall-clock ticks (thread 0)
struct PhaseClock {
  unsigned long long *dst;
  unsigned long long t;
  __device__ void start(const DevBatch &B, int w) {
    dst = B.prof ? B.prof + (size_t)w * PH_N : nullptr;
    if (dst && threadIdx.x == 0) t = wall_clock64();
  }
  __device__ void lap(int ph) {
    if (dst && threadIdx.x == 0) {
      unsigned long long n = wall_clock64();
      dst[ph] += n - t;
      t = n;
    }
  }
};

// Raises an overflow flag of world w; called by thread 0, the counters' only
// writer.  Not an atomic OR: dSpaceCollide's counters are pinned host memory,
// and the bus carries add, swap and compare-and-swap only.
__device__ inline void raise_overflow(const DevBatch &B, int w, int flag) {
  B.counters[w * CNT_N + CNT_OVERFLOW] |= flag;
}

// ------------------------------------------------------------------ block helpers

__device__ inline int block_excl_scan(int v, int &total, Shared &sh) {
  int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int x = v;
  for (int o = 1; o < 64; o <<= 1) {
    int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) sh.wsum[wid] = x;
  __syncthreads();
  int nw = (blockDim.x + 63) >> 6, off = 0, tot = 0;
  for (int k = 0; k < nw; k++) {
    int s = sh.wsum[k];
    if (k < wid) off += s;
    tot += s;
  }
  __syncthreads();
  total = tot;
  return off + x - v;
}

__device__ inline float block_max(float v, Shared &sh) {
  int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  if (lane == 0) sh.wmax[wid] = v;
  __syncthreads();
  int nw = (blockDim.x + 63) >> 6;
  float m = sh.wmax[0];
  for (int k = 1; k < nw; k++) m = fmaxf(m, sh.wmax[k]);
  __syncthreads();
  return m;
}

__device__ inline float block_fsum(float v, Shared &sh) {
  int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (lane == 0) sh.wmax[wid] = v;
  __syncthreads();
  int nw = (blockDim.x + 63) >> 6;
  float m = 0.f;
  for (int k = 0; k < nw; k++) m += sh.wmax[k];
  __syncthreads();
  return m;
}

__device__ inline int block_sum(int v, Shared &sh) {
  int t;
  block_excl_scan(v, t, sh);
  return t;
}

// Ascending bitonic sort of n (power of two) u64 keys; in LDS when it fits.
// A stage is bound by the latency of its compare-exchanges, so a lane takes
// four pairs at a time, their loads before their stores, and every lane of a
// stage has a pair (a walk over all n keys leaves half of them idle).
__device__ inline void bitonic_stages(unsigned long long *k, int n) {
  const int nt = blockDim.x, half = n >> 1;
  for (int size = 2; size <= n; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int p0 = threadIdx.x; p0 < half; p0 += 4 * nt) {
        int lo[4];
        unsigned long long x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int p = min(p0 + u * nt, half - 1);
          lo[u] = 2 * p - (p & (stride - 1));
          x[u] = k[lo[u]];
          y[u] = k[lo[u] + stride];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const bool asc = (lo[u] & size) == 0;
          if (p0 + u * nt < half && (x[u] > y[u]) == asc) {
            k[lo[u]] = y[u];
            k[lo[u] + stride] = x[u];
          }
        }
      }
      __syncthreads();
    }
  }
}

__device__ inline void bitonic_sort(unsigned long long *a, int n, Shared &sh, int lds_bytes) {
  if ((long long)n * 8 > lds_bytes) {
    bitonic_stages(a, n);
    return;
  }
  unsigned long long *pool = (unsigned long long *)od_pool;
  for (int i = threadIdx.x; i < n; i += blockDim.x) pool[i] = a[i];
  __syncthreads();
  bitonic_stages(pool, n);
  for (int i = threadIdx.x; i < n; i += blockDim.x) a[i] = pool[i];
  __syncthreads();
}

// LDS bytes the block radix sort needs for a workgroup of nt lanes: digit
// bases (256) and per-wavefront digit counts of one tile
__host__ __device__ inline int radix_lds_bytes(int nt) { return 4 * (256 + 256 * ((nt + 63) / 64)); }

// Workgroup barrier that orders LDS accesses only: global loads and stores
// in flight stay in flight (a full __syncthreads waits for them).  For
// phases whose cross-lane exchange is in LDS and whose global writes are
// read only after a later full barrier.
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Ascending LSD radix sort of n u64 keys in global memory by one workgroup,
// by bits [lo_bit, 64) in 8-bit digits (lo_bit a multiple of 8); tmp holds n
// keys.  A digit that is zero in every key is skipped (a stable pass over
// one digit value is the identity).  Each pass counts digits (LDS atomics),
// scans the 256 counts (block scan) and scatters tile by tile, stably: the
// rank of a key among the equal digits of its wavefront comes from eight
// ballots, the wavefronts of a tile are ordered through per-wavefront counts
// in LDS.  Keys equal in the sorted bits keep their input order.  The result
// is in keys.
__device__ inline void block_radix_sort(unsigned long long *keys, unsigned long long *tmp, int n, int lo_bit,
                                        Shared &sh) {
  const int nt = blockDim.x, nw = (nt + 63) >> 6;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int *base = (int *)od_pool;      // 256 digit bases
  int *wc = base + 256;            // per wavefront: 256 digit counts of the current tile
  unsigned long long any = 0;
  for (int i = threadIdx.x; i < n; i += nt) any |= keys[i];
  // bits present in some key (OR over the workgroup, 32 bits at a time)
  unsigned lo = (unsigned)any, hi = (unsigned)(any >> 32);
  for (int o = 32; o > 0; o >>= 1) { lo |= __shfl_xor(lo, o, 64); hi |= __shfl_xor(hi, o, 64); }
  if (lane == 0) { sh.ival[0] = 0; sh.ival[1] = 0; }
  __syncthreads();
  if (lane == 0) { atomicOr(&sh.ival[0], (int)lo); atomicOr(&sh.ival[1], (int)hi); }
  __syncthreads();
  const unsigned long long all = ((unsigned long long)(unsigned)sh.ival[1] << 32) | (unsigned)sh.ival[0];
  __syncthreads();
  unsigned long long *src = keys, *dst = tmp;
  for (int shift = lo_bit; shift < 64; shift += 8) {
    if (((all >> shift) & 255) == 0) continue;
    for (int d = threadIdx.x; d < 256; d += nt) base[d] = 0;
    for (int d = threadIdx.x; d < 256 * nw; d += nt) wc[d] = 0;
    __syncthreads();
    // digit counts, four keys per lane in flight at a time
    for (int i0 = threadIdx.x; i0 < n; i0 += 4 * nt) {
      unsigned long long k4[4];
      for (int u = 0; u < 4; u++) k4[u] = (i0 + u * nt < n) ? src[i0 + u * nt] : 0ULL;
      for (int u = 0; u < 4; u++)
        if (i0 + u * nt < n) atomicAdd(&base[(int)((k4[u] >> shift) & 255)], 1);
    }
    __syncthreads();
    {
      // exclusive scan of the digit counts, a run of digits per lane
      const int per = (256 + nt - 1) / nt, d0 = threadIdx.x * per;
      const int d1 = d0 + per < 256 ? d0 + per : 256;
      int loc = 0;
      for (int d = d0; d < d1; d++) loc += base[d];
      int tot;
      int off = block_excl_scan(loc, tot, sh);
      for (int d = d0; d < d1; d++) { const int cnt = base[d]; base[d] = off; off += cnt; }
    }
    __syncthreads();
    // tiles of nt keys; the next tile's key is loaded before this tile's
    // LDS-only barriers, the scattered stores are waited for once per pass
    unsigned long long knext = threadIdx.x < n ? src[threadIdx.x] : 0ULL;
    for (int t0 = 0; t0 < n; t0 += nt) {
      const int i = t0 + threadIdx.x;
      const bool valid = i < n;
      const unsigned long long k = knext;
      knext = (i + nt < n) ? src[i + nt] : 0ULL;
      const int d = (int)((k >> shift) & 255);
      unsigned long long peers = __ballot(valid);
      for (int b = 0; b < 8; b++) {
        const unsigned long long m = __ballot(valid && ((d >> b) & 1));
        peers &= ((d >> b) & 1) ? m : ~m;
      }
      const unsigned long long lt = (lane == 0) ? 0ULL : (~0ULL >> (64 - lane));
      const int rank = __popcll(peers & lt);
      const int cnt = __popcll(peers);
      if (valid && rank == cnt - 1) wc[wid * 256 + d] = cnt;
      lds_barrier();
      if (valid) {
        int off = base[d] + rank;
        for (int w = 0; w < wid; w++) off += wc[w * 256 + d];
        dst[off] = k;
      }
      lds_barrier();
      for (int dd = threadIdx.x; dd < 256; dd += nt) {
        int tot = 0;
        for (int w = 0; w < nw; w++) { tot += wc[w * 256 + dd]; wc[w * 256 + dd] = 0; }
        base[dd] += tot;
      }
      lds_barrier();
    }
    __syncthreads();   // this pass's stores before the next pass reads them
    unsigned long long *t = src; src = dst; dst = t;
  }
  if (src != keys) {
    for (int i = threadIdx.x; i < n; i += nt) keys[i] = src[i];
    __syncthreads();
  }
}

__device__ inline int pow2_at_least(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

// ------------------------------------------------------------------ world context

struct Ctx {
  int w;
  WorldInfo W;
  ScratchLayout L;
  char *S;
  mutable PhaseClock clk;
  template <class T> __device__ T *at(long long off) const { return (T *)(S + off); }
};

__device__ inline GeomView load_geom(const DevBatch &B, const Ctx &c, int g) {
  int gg = c.W.g0 + g;
  GeomView v;
  v.type = B.gtype[gg];
  v.prm = B.gparam[gg];
  int b = B.gbody[gg];
  if (b >= 0) {
    int gb = c.W.b0 + b;
    v.p = xyz(B.pos[gb]);
    v.R = load_mat(B.R + 3 * (size_t)gb);
  } else {
    v.p = xyz(B.gpos[gg]);
    v.R = load_mat(B.gR + 3 * (size_t)gg);
  }
  return v;
}

__device__ inline bool aabb_overlap(const float *a, const float *b) {
  return !(a[0] > b[1] || a[1] < b[0] || a[2] > b[3] || a[3] < b[2] || a[4] > b[5] || a[5] < b[4]);
}

// collideAABBs filters (collision_space_internal.h:48-82)
__device__ inline bool pair_passes(const DevBatch &B, const Ctx &c, int g1, int g2, const float *aabb) {
  int b1 = B.gbody[c.W.g0 + g1], b2 = B.gbody[c.W.g0 + g2];
  if (b1 == b2 && b1 >= 0) return false;
  unsigned c1 = B.gcat[c.W.g0 + g1], c2 = B.gcat[c.W.g0 + g2];
  unsigned k1 = B.gcol[c.W.g0 + g1], k2 = B.gcol[c.W.g0 + g2];
  if (((c1 & k2) || (c2 & k1)) == 0) return false;
  return aabb_overlap(aabb + 6 * g1, aabb + 6 * g2);
}

// the reference's near-callback filter: skip bodies joined by a permanent joint
__device__ inline bool connected(const DevBatch &B, const Ctx &c, int b1, int b2) {
  if (b1 < 0 || b2 < 0 || !B.adj_start) return false;
  int s = B.adj_start[c.W.b0 + b1], e = B.adj_start[c.W.b0 + b1 + 1];
  for (int k = s; k < e; k++)
    if (B.adj_other[k] == b2) return true;
  return false;
}

__device__ inline unsigned cell_hash(int x, int y, int z) {
  return ((unsigned)x * 73856093u) ^ ((unsigned)y * 19349663u) ^ ((unsigned)z * 83492791u);
}

// ------------------------------------------------------------------ collide

// AABBs, big-geom flags, reference hash levels and discrete bounds
// (collision_space.cpp:331-351, 444-476).
__device__ void phase_aabb(const DevBatch &B, const Ctx &c, const WorldParams &P, Shared &sh) {
  float *aabb = c.at<float>(c.L.aabb);
  int *gbig = c.at<int>(c.L.gbig);
  int *glevel = c.at<int>(c.L.glevel);
  int *gdb = c.at<int>(c.L.gdb);
  for (int g = threadIdx.x; g < c.W.ng; g += blockDim.x) {
    GeomView v = load_geom(B, c, g);
    float a[6];
    geom_aabb(v, a);
    for (int k = 0; k < 6; k++) aabb[6 * g + k] = a[k];
    bool inf = false;
    for (int k = 0; k < 6; k++) inf |= isinf(a[k]);
    int lvl = 0x7fffffff;
    if (!inf) {
      float q = fmaxf(a[1] - a[0], fmaxf(a[3] - a[2], a[5] - a[4]));
      int e;
      frexpf(q, &e);
      lvl = e < P.hash_min ? P.hash_min : e;
    }
    bool big = inf || lvl > P.hash_max;
    gbig[g] = big ? 1 : 0;
    glevel[g] = lvl;
    if (!big) {
      float cell = ldexpf(1.f, lvl);
      for (int k = 0; k < 6; k++) gdb[6 * g + k] = (int)floorf(a[k] / cell);
    }
  }
  __syncthreads();
}

// reference hash index of every non-big geom (position in the space list
// among non-big geoms) and the big-geom list in reverse space order.
__device__ void phase_ref_index(const DevBatch &B, const Ctx &c, Shared &sh) {
  int *gbig = c.at<int>(c.L.gbig);
  int *gidx = c.at<int>(c.L.gidx);
  int *inv = c.at<int>(c.L.order);   // rank -> geom, then big list
  const int ng = c.W.ng;
  for (int g = threadIdx.x; g < ng; g += blockDim.x) inv[B.grank[c.W.g0 + g]] = g;
  __syncthreads();
  // in space-list order (block scans): non-big geoms get consecutive hash
  // indices; big geoms note their position among the big ones (-2 - pos)
  int n = 0, nbig = 0;
  for (int r0 = 0; r0 < ng; r0 += blockDim.x) {
    const int r = r0 + threadIdx.x;
    const int g = r < ng ? inv[r] : -1;
    const int isb = (g >= 0 && gbig[g]) ? 1 : 0;
    const int nonb = (g >= 0 && !isb) ? 1 : 0;
    int t1, t2;
    const int o1 = block_excl_scan(nonb, t1, sh);
    const int o2 = block_excl_scan(isb, t2, sh);
    if (nonb) gidx[g] = n + o1;
    if (isb) gidx[g] = -2 - (nbig + o2);
    n += t1;
    nbig += t2;
  }
  __syncthreads();
  // big geoms in reverse space order: big rank k = nbig - 1 - pos
  int *big = inv + ng;
  for (int g = threadIdx.x; g < ng; g += blockDim.x) {
    const int v = gidx[g];
    if (v <= -2) {
      const int k = nbig - 1 - (-2 - v);
      big[k] = g;
      gbig[g] = 1 + k;   // 1 + big rank
      gidx[g] = -1;
    }
  }
  if (threadIdx.x == 0) {
    sh.ival[0] = n;
    sh.ival[1] = nbig;
  }
  __syncthreads();
}

// key placing pair (a,b) of non-big geoms at the reference's first encounter
// in the hash-space traversal; also returns the emitted orientation.
__device__ inline unsigned long long ref_pair_key(const Ctx &c, int a, int b, int n, int &g1, int &g2) {
  const int *gidx = c.at<int>(c.L.gidx);
  const int *glevel = c.at<int>(c.L.glevel);
  const int *gdb = c.at<int>(c.L.gdb);
  int X = gidx[a] > gidx[b] ? a : b;    // larger index: earlier in the traversal
  int Y = X == a ? b : a;
  int outer, part;
  if (glevel[Y] >= glevel[X]) { outer = X; part = Y; }
  else { outer = Y; part = X; }
  int L = glevel[part];
  int sh = L - glevel[outer];
  int d[3];
  for (int k = 0; k < 3; k++) {
    int o0 = gdb[6 * outer + 2 * k] >> sh;
    int p0 = gdb[6 * part + 2 * k];
    int c0 = o0 > p0 ? o0 : p0;
    d[k] = c0 - o0;
  }
  g1 = outer;
  g2 = part;
  unsigned long long rank = (unsigned long long)(n - 1 - gidx[outer]);
  return (rank << 40) | ((unsigned long long)(sh & 31) << 35) | ((unsigned long long)(d[0] & 1) << 34) |
         ((unsigned long long)(d[1] & 1) << 33) | ((unsigned long long)(d[2] & 1) << 32) |
         (unsigned long long)gidx[part];
}

// Uniform-grid broadphase.  Each non-big geom enters the (at most 8) cells
// its AABB covers; entries are sorted by cell key; a pair is reported from the
// run of its home cell (the low corner of the two cell ranges' overlap), so
// every overlapping pair appears exactly once.  Big geoms (unbounded AABBs)
// are tested against everything.  Returns the pair count.
__device__ int phase_broadphase(const DevBatch &B, const Ctx &c, const WorldParams &P, Shared &sh, bool ref) {
  const float *aabb = c.at<float>(c.L.aabb);
  const int *gbig = c.at<int>(c.L.gbig);
  unsigned long long *cells = c.at<unsigned long long>(c.L.cells);
  int *ecount = c.at<int>(c.L.ecount);
  PairRec *pairs = c.at<PairRec>(c.L.pairs);
  unsigned long long *pkeys = c.at<unsigned long long>(c.L.pkeys);
  const int ng = c.W.ng;
  int nref = 0;
  if (ref) {
    phase_ref_index(B, c, sh);
    nref = sh.ival[0];
  }
  // cell size from the largest extent
  float ext = 0.f;
  for (int g = threadIdx.x; g < ng; g += blockDim.x) {
    if (gbig[g]) continue;
    const float *a = aabb + 6 * g;
    ext = fmaxf(ext, fmaxf(a[1] - a[0], fmaxf(a[3] - a[2], a[5] - a[4])));
  }
  ext = block_max(ext, sh);
  float cell = fmaxf(ext * P.cell_scale * 1.0001f, 1e-6f);
  float inv = 1.f / cell;
  // cell entries: key = hash << 32 | geom << 3 | subcell
  int base = 0;
  for (int start = 0; start < ng; start += blockDim.x) {
    int g = start + threadIdx.x;
    int cnt = 0, lo[3] = {0, 0, 0}, span[3] = {1, 1, 1};
    if (g < ng && !gbig[g]) {
      const float *a = aabb + 6 * g;
      for (int k = 0; k < 3; k++) {
        lo[k] = (int)floorf(a[2 * k] * inv);
        int hi = (int)floorf(a[2 * k + 1] * inv);
        span[k] = hi > lo[k] ? 2 : 1;
      }
      cnt = span[0] * span[1] * span[2];
    }
    int tot;
    int off = block_excl_scan(cnt, tot, sh);
    if (cnt) {
      int e = base + off;
      for (int dz = 0; dz < span[2]; dz++)
        for (int dy = 0; dy < span[1]; dy++)
          for (int dx = 0; dx < span[0]; dx++) {
            unsigned h = cell_hash(lo[0] + dx, lo[1] + dy, lo[2] + dz);
            cells[e++] = ((unsigned long long)h << 32) | ((unsigned long long)g << 3) | (unsigned)(dx | dy << 1 | dz << 2);
          }
    }
    base += tot;
  }
  const int ne = base;
  const int np2 = pow2_at_least(ne < 2 ? 2 : ne);
  if ((long long)np2 * 8 > B.lds_bytes && B.lds_bytes >= radix_lds_bytes(blockDim.x) && ne <= c.W.pcap) {
    // too many keys for the LDS pool: radix sort in global memory (pkeys,
    // pcap entries written only by the pair scan below, holds the second
    // buffer), by the cell hash only: the pair scan needs the entries of a
    // cell together, and the pairs it finds are sorted by their own keys
    // below, so the order inside a cell does not reach the result
    __syncthreads();
    block_radix_sort(cells, pkeys, ne, 32, sh);
  } else {
    for (int i = ne + threadIdx.x; i < np2; i += blockDim.x) cells[i] = ~0ULL;
    __syncthreads();
    bitonic_sort(cells, np2, sh, B.lds_bytes);
  }
  // pair scan: one lane per cell entry walks the rest of its cell's run.
  // A pair is found once, from the entry of the pair's home cell (the low
  // corner of the two cell ranges' overlap) that comes first in the run.
  auto pair_key = [&](int gi, int gj) -> unsigned long long {
    if (ref) {
      int a, b;
      return ref_pair_key(c, gi, gj, nref, a, b);
    }
    return gi < gj ? ((unsigned long long)gi << 32) | (unsigned)gj : ((unsigned long long)gj << 32) | (unsigned)gi;
  };
  auto visit = [&](int i, auto &&emit) {
    const unsigned long long ei = cells[i];
    const unsigned hi = (unsigned)(ei >> 32);
    const int gi = (int)((ei & 0xffffffffu) >> 3), si = (int)(ei & 7);
    const int G = c.W.g0;
    float ai[6];
    for (int k = 0; k < 6; k++) ai[k] = aabb[6 * gi + k];
    const int bi = B.gbody[G + gi];
    const unsigned ci = B.gcat[G + gi], ki = B.gcol[G + gi];
    int li[3];
    for (int k = 0; k < 3; k++) li[k] = (int)floorf(ai[2 * k] * inv) + ((si >> k) & 1);
    for (int j = i + 1; j < ne; j++) {
      const unsigned long long ej = cells[j];
      if ((unsigned)(ej >> 32) != hi) break;
      const int gj = (int)((ej & 0xffffffffu) >> 3), sj = (int)(ej & 7);
      if (gj == gi) continue;
      float aj[6];
      for (int k = 0; k < 6; k++) aj[k] = aabb[6 * gj + k];
      const int bj = B.gbody[G + gj];
      const unsigned cj = B.gcat[G + gj], kj = B.gcol[G + gj];
      bool same = true, home = true;
      for (int k = 0; k < 3; k++) {
        int ljk0 = (int)floorf(aj[2 * k] * inv);
        int lj = ljk0 + ((sj >> k) & 1);
        int lik0 = li[k] - ((si >> k) & 1);
        int hc = lik0 > ljk0 ? lik0 : ljk0;
        same &= lj == li[k];
        home &= hc == li[k];
      }
      if (!same || !home) continue;
      // collideAABBs filters (collision_space_internal.h:54-71)
      if (bi == bj && bi >= 0) continue;
      if (((ci & kj) || (cj & ki)) == 0) continue;
      if (!aabb_overlap(ai, aj)) continue;
      emit(gi, gj);
    }
  };
  // every pair takes the next slot of a workgroup counter: the keys are
  // sorted below, so the slot order does not reach the result
  if (threadIdx.x == 0) sh.ival[2] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < ne; i += blockDim.x)
    visit(i, [&](int gi, int gj) {
      const int o = atomicAdd(&sh.ival[2], 1);
      if (o < c.W.pcap) pkeys[o] = pair_key(gi, gj);
    });
  __syncthreads();
  int npairs = sh.ival[2];
  __syncthreads();
  if (npairs > c.W.pcap) {
    // more pairs than slots: scan again in entry order (counting pass, then
    // writing pass) so that the pairs kept are the same on every run
    npairs = 0;
    for (int start = 0; start < ne; start += blockDim.x) {
      const int i = start + threadIdx.x;
      int cnt = 0;
      if (i < ne) visit(i, [&](int, int) { cnt++; });
      int tot;
      const int off = block_excl_scan(cnt, tot, sh);
      if (i < ne && cnt) {
        int o = npairs + off;
        visit(i, [&](int gi, int gj) {
          if (o < c.W.pcap) pkeys[o] = pair_key(gi, gj);
          o++;
        });
      }
      npairs += tot;
    }
  }
  // big geoms against the rest, then big against big; the big geoms first
  // listed in ascending index order (ecount is free scratch here)
  int *blist = ecount;
  int nbig = 0;
  for (int start = 0; start < ng; start += blockDim.x) {
    int g = start + threadIdx.x;
    int isb = (g < ng && gbig[g]) ? 1 : 0;
    int tot;
    int off = block_excl_scan(isb, tot, sh);
    if (isb) blist[nbig + off] = g;
    nbig += tot;
  }
  __syncthreads();
  for (int start = 0; start < ng; start += blockDim.x) {
    int g = start + threadIdx.x;
    int cnt = 0;
    if (g < ng)
      for (int t = 0; t < nbig; t++) {
        const int b = blist[t];
        if (b == g) continue;
        if (gbig[g] && !(b > g)) continue;  // big-big once
        if (pair_passes(B, c, g, b, aabb)) cnt++;
      }
    int tot;
    int off = block_excl_scan(cnt, tot, sh);
    if (cnt) {
      int o = npairs + off;
      for (int t = 0; t < nbig; t++) {
        const int b = blist[t];
        if (b == g) continue;
        if (gbig[g] && !(b > g)) continue;
        if (!pair_passes(B, c, g, b, aabb)) continue;
        if (o < c.W.pcap) {
          if (ref) {
            const int *gidx = c.at<int>(c.L.gidx);
            int bb = gbig[b] - 1;
            if (!gbig[g]) {
              pkeys[o] = (1ULL << 63) | ((unsigned long long)(nref - 1 - gidx[g]) << 32) | (unsigned)bb;
            } else {
              int ga = gbig[g] - 1;
              int r1 = ga < bb ? ga : bb, r2 = ga < bb ? bb : ga;
              pkeys[o] = (3ULL << 62) | ((unsigned long long)r1 << 24) | (unsigned)r2;
            }
          } else {
            pkeys[o] = g < b ? ((unsigned long long)g << 32) | (unsigned)b
                             : ((unsigned long long)b << 32) | (unsigned)g;
          }
        }
        o++;
      }
    }
    npairs += tot;
  }
  if (npairs > c.W.pcap) {
    if (threadIdx.x == 0) raise_overflow(B, c.w, OVF_PAIRS);
    npairs = c.W.pcap;
  }
  {
    // sort the keys: in reference mode into the callback order, in coloured
    // mode into (g1, g2) order with g1 < g2, so that the contact order (and
    // with it the colouring) does not depend on the grid
    int np = pow2_at_least(npairs < 2 ? 2 : npairs);
    if (np > c.W.pcap) np = c.W.pcap;  // pcap is a power of two
    if ((long long)np * 8 > B.lds_bytes && B.lds_bytes >= radix_lds_bytes(blockDim.x)) {
      // radix sort in global memory; the pair records (written after the
      // sort) hold the second buffer
      __syncthreads();
      block_radix_sort(pkeys, (unsigned long long *)pairs, npairs, 0, sh);
    } else {
      for (int i = npairs + threadIdx.x; i < np; i += blockDim.x) pkeys[i] = ~0ULL;
      __syncthreads();
      bitonic_sort(pkeys, np, sh, B.lds_bytes);
    }
  }
  if (!ref) {
    for (int i = threadIdx.x; i < npairs; i += blockDim.x) {
      unsigned long long k = pkeys[i];
      pairs[i].g1 = (int)(k >> 32);
      pairs[i].g2 = (int)(k & 0xffffffffu);
      pairs[i].key = k;
    }
  } else {
    const int *gidx = c.at<int>(c.L.gidx);
    // inverse maps: hash index -> geom, big rank -> geom
    int *inv = c.at<int>(c.L.order);
    int *byidx = c.at<int>(c.L.island);
    for (int g = threadIdx.x; g < ng; g += blockDim.x)
      if (gidx[g] >= 0) byidx[gidx[g]] = g;
    __syncthreads();
    const int *big = inv + ng;
    for (int i = threadIdx.x; i < npairs; i += blockDim.x) {
      unsigned long long k = pkeys[i];
      int a, b;
      if ((k >> 62) == 3ULL) { a = big[(k >> 24) & 0xffffff]; b = big[k & 0xffffff]; }
      else if (k >> 63) { a = byidx[nref - 1 - (int)((k >> 32) & 0x3fffffff)]; b = big[k & 0xffffffff]; }
      else { a = byidx[nref - 1 - (int)(k >> 40)]; b = byidx[k & 0xffffffff]; }
      pairs[i].g1 = a;
      pairs[i].g2 = b;
      pairs[i].key = k;
    }
  }
  __syncthreads();
  return npairs;
}

__device__ inline void store_contacts(const DevBatch &B, const Ctx &c, int g1, int g2, const CPoint *pts, int n,
                                      ContactRec *dst, int room) {
  int b1 = B.gbody[c.W.g0 + g1], b2 = B.gbody[c.W.g0 + g2];
  int flags = 0;
  if (b1 < 0) { b1 = b2; b2 = -1; flags = JF_REVERSE; }
  for (int i = 0; i < n && i < room; i++) {
    ContactRec &r = dst[i];
    r.pos[0] = pts[i].pos.x; r.pos[1] = pts[i].pos.y; r.pos[2] = pts[i].pos.z;
    r.depth = pts[i].depth;
    r.normal[0] = pts[i].n.x; r.normal[1] = pts[i].n.y; r.normal[2] = pts[i].n.z;
    r.g1 = g1; r.g2 = g2; r.b1 = b1; r.b2 = b2; r.flags = flags | (i << 8);
  }
}

// narrowphase over the pair list, one pair per lane; contacts keep pair order.
__device__ int phase_narrowphase(const DevBatch &B, const Ctx &c, const WorldParams &P, int npairs, Shared &sh,
                                 int maxc, bool apply_policy) {
  const PairRec *pairs = c.at<PairRec>(c.L.pairs);
  int *pcount = c.at<int>(c.L.pcount);
  ContactRec *con = c.at<ContactRec>(c.L.contacts);
  int nk = 0;
  if (maxc > MAX_SLOTS) maxc = MAX_SLOTS;
  for (int start = 0; start < npairs; start += blockDim.x) {
    int i = start + threadIdx.x;
    CPoint pts[MAX_SLOTS];
    int n = 0;
    if (i < npairs) {
      int g1 = pairs[i].g1, g2 = pairs[i].g2;
      bool skip = false;
      if (apply_policy && P.skip_connected) {
        int b1 = B.gbody[c.W.g0 + g1], b2 = B.gbody[c.W.g0 + g2];
        skip = connected(B, c, b1, b2);
      }
      if (!skip) {
        GeomView a = load_geom(B, c, g1), b = load_geom(B, c, g2);
        n = collide_pair(a, b, maxc, pts);
      }
      pcount[i] = n;
    }
    int tot;
    int off = block_excl_scan(n, tot, sh);
    if (n) {
      int o = nk + off;
      int room = c.W.kcap - o;
      if (room > 0) store_contacts(B, c, pairs[i].g1, pairs[i].g2, pts, n, con + o, room);
    }
    nk += tot;
  }
  if (nk > c.W.kcap) {
    if (threadIdx.x == 0) raise_overflow(B, c.w, OVF_CONTACTS);
    nk = c.W.kcap;
  }
  __syncthreads();
  return nk;
}

// ------------------------------------------------------------------ step

struct StepIn {
  int nk;               // contacts
  bool from_host;       // contacts are ContactIn records of the host
  int seq_base;         // attach sequence of the first fused contact
};

__device__ inline Surf world_surface(const WorldParams &P) {
  Surf s;
  s.mode = P.surf_mode; s.mu = P.mu; s.mu2 = P.mu2; s.bounce = P.bounce; s.bounce_vel = P.bounce_vel;
  s.soft_erp = P.soft_erp; s.soft_cfm = P.soft_cfm; s.motion1 = P.motion1; s.motion2 = P.motion2;
  s.motionN = P.motionN; s.slip1 = P.slip1; s.slip2 = P.slip2; s.fdir1 = mk3(0.f, 0.f, 0.f);
  return s;
}

__device__ inline Surf host_surface(const ContactIn &ci) {
  Surf s;
  s.mode = ci.mode; s.mu = ci.mu; s.mu2 = ci.mu2; s.bounce = ci.bounce; s.bounce_vel = ci.bounce_vel;
  s.soft_erp = ci.soft_erp; s.soft_cfm = ci.soft_cfm; s.motion1 = ci.motion1; s.motion2 = ci.motion2;
  s.motionN = ci.motionN; s.slip1 = ci.slip1; s.slip2 = ci.slip2;
  s.fdir1 = mk3(ci.fdir1[0], ci.fdir1[1], ci.fdir1[2]);
  return s;
}

#include "colouring.hpp"
#include "ref_solver.hpp"

// |lambda - clamp(lambda - d, lo, hi)| evaluated without the cancellation of
// lambda - (lambda - d): |d| when the step stays inside the bounds, else the
// distance from lambda to the bound it crosses
__device__ inline float proj_residual(float lambda, float d, float lo, float hi) {
  const float p = lambda - d;
  if (p < lo) return fabsf(lambda - lo);
  if (p > hi) return fabsf(hi - lambda);
  return fabsf(d);
}

// complementarity residual of one row: |lambda - clamp(lambda - (A lambda - b)/A_ii)|
__device__ inline float row_residual(const Row *rows, int r, const float *fc) {
  const Row &R = rows[r];
  const float *f1 = fc + 32 * R.b1 + 9;
  float s = 0.f, d = 0.f;
  for (int k = 0; k < 6; k++) { s += R.J[k] * f1[k]; d += R.J[k] * R.iMJ[k]; }
  if (R.b2 >= 0) {
    const float *f2 = fc + 32 * R.b2 + 9;
    for (int k = 0; k < 6; k++) { s += R.J[6 + k] * f2[k]; d += R.J[6 + k] * R.iMJ[6 + k]; }
  }
  float Aii = d + R.cfm;
  float y = s + R.cfm * R.lambda - R.rhs;
  float lo = R.lo, hi = R.hi;
  if (R.findex >= 0) { hi = fabsf(R.hi * rows[R.findex].lambda); lo = -hi; }
  return proj_residual(R.lambda, y / Aii, lo, hi);
}

// Coloured SOR-LCP.  The working set -- per-body fc; the constraints sorted
// by colour with their rows stored contiguously in that order -- is copied
// into the LDS pool as far as it fits, else stays in the world's scratch.
// One lane relaxes all rows of one constraint with both bodies' fc in
// registers; the constraints of a colour share no body, so a colour is one
// parallel pass.  Each row follows the reference's update
// (quickstep.cpp:484-582) on the inverse masses and the angular parts of
// inv(M) J^T (every supported row has J_lin2 = -J_lin1).
constexpr int SOR_MAX_ROWS = 6;   // rows of one constraint (contact 3, ball 3, hinge 6, hinge2 6)

// J_1 . f1 (+ J_2 . f2) of one row (J_l2 = -J_l1), summed in the order written
__device__ inline float sor_dot(const SRow &r, const float *f1, bool two, const float *f2) {
  const float s = r.l[0] * f1[0] + r.l[1] * f1[1] + r.l[2] * f1[2] + r.a1[0] * f1[3] + r.a1[1] * f1[4] + r.a1[2] * f1[5];
  const float s2 =
      -r.l[0] * f2[0] - r.l[1] * f2[1] - r.l[2] * f2[2] + r.a2[0] * f2[3] + r.a2[1] * f2[4] + r.a2[2] * f2[5];
  return two ? s + s2 : s;
}

// largest complementarity residual |lambda - clamp(lambda - (A lambda - b)_i / A_ii)|
// over the rows of one constraint of the coloured solver (A_ii = w / ad)
__device__ inline float sor_cons_residual(const float *fc, const SRow *sr, const float *slam, const SCons q,
                                          float sor_w) {
  float f1[6], f2[6];
  const bool two = q.b2 >= 0;
  for (int k = 0; k < 6; k++) { f1[k] = fc[6 * q.b1 + k]; f2[k] = fc[6 * max(q.b2, 0) + k]; }
  float r = 0.f, lam0 = 0.f;
  for (int k = 0; k < q.m; k++) {
    const SRow w = sr[q.row0 + k];
    const float lam = slam[q.row0 + k];
    if (k == 0) lam0 = lam;
    const float y = sor_dot(w, f1, two, f2) + w.cfm * lam - w.rhs;
    float lo = w.lo, hi = w.hi;
    if (w.findex >= 0) {
      hi = fabsf(w.hi * lam0);
      lo = -hi;
    }
    r = fmaxf(r, proj_residual(lam, y * (w.ad / sor_w), lo, hi));
  }
  return r;
}

// fc += delta * inv(M) J^T of one row for both bodies of its constraint (f2
// of a constraint with one body is not used)
__device__ inline void sor_push(const SRow &r, float delta, float *f1, float *f2) {
  const float d1 = delta * r.im1, d2 = delta * r.im2;
  for (int k = 0; k < 3; k++) {
    f1[k] += d1 * r.l[k];
    f1[3 + k] += delta * r.t1[k];
    f2[k] -= d2 * r.l[k];
    f2[3 + k] += delta * r.t2[k];
  }
}

// One row (quickstep.cpp:484-582): its new impulse; f1, f2 follow.  lam0: the
// impulse of the constraint's first row; tol_mode: fc follows the stored
// impulse.  Free of branches, so that the two bodies' chains overlap.
__device__ inline float sor_relax_row(const SRow &r, float old, float lam0, bool two, float *f1, float *f2,
                                      bool tol_mode) {
  const float s = sor_dot(r, f1, two, f2);
  float delta = r.ad * (r.rhs - old * r.cfm - s);
  const bool fr = r.findex >= 0;
  const float hf = fabsf(r.hi * lam0), hi = fr ? hf : r.hi, lo = fr ? -hf : r.lo;
  float nl = old + delta;
  const bool below = nl < lo, above = !below && nl > hi;
  nl = below ? lo : (above ? hi : nl);
  delta = tol_mode || below || above ? nl - old : delta;
  sor_push(r, delta, f1, f2);
  return nl;
}

// Starting impulses of one constraint's rows from the warm-start records of
// the previous step: a contact by its key (records sorted by key, binary
// search), a permanent joint by index when its row count is unchanged.
__device__ inline void warm_lookup(const WorldParams &P, const Cons &q, const ContactRec *con, const WarmRec *wrec,
                                   int nprev, const float *wjnt, float *wl) {
  if (q.kind == JT_CONTACT) {
    const ContactRec &cr = con[q.src];
    const unsigned long long key = contact_key(cr.g1, cr.g2, cr.flags >> 8);
    int lo = 0, hi = nprev;
    while (lo < hi) {
      int mid = (lo + hi) >> 1;
      if (wrec[mid].key < key) lo = mid + 1;
      else hi = mid;
    }
    if (lo < nprev && wrec[lo].key == key)
      for (int k = 0; k < q.m && k < 3; k++) wl[k] = P.warm * wrec[lo].lam[k];
  } else {
    const float *jw = wjnt + 8 * q.src;
    if (__float_as_int(jw[6]) == q.m)
      for (int k = 0; k < q.m && k < 6; k++) wl[k] = P.warm * jw[k];
  }
}

// The coloured solver's working set: the rows (read-only during the sweeps),
// the bodies' fc, constraints in colour order, colour starts, the row impulses
// and (accelerated mode) the conjugate-gradient state: per row lambda before
// the sweep and the direction, per body fc before the sweep and the
// direction's fc (last, so that a pool can hold all but it).  Built in the
// world's scratch; copied to the LDS pool for the sweeps when it fits there
// (same layout).
struct SorSet {
  SRow *sr;
  float *fc;
  SCons *sc;
  int *sstart;
  float *slam;
  float2 *ld;
  float *fp, *fdir;
};

__device__ inline SorSet sor_set(char *base, SRow *sr, int nb, int nrows, int nact, int ngroups) {
  SorSet S;
  S.sr = sr;
  S.fc = (float *)base;
  S.sc = (SCons *)(base + ((24LL * nb + 15) & ~15LL));
  S.sstart = (int *)(S.sc + nact);
  S.slam = (float *)((char *)S.sstart + ((4LL * (ngroups + 1LL) + 15) & ~15LL));
  S.ld = (float2 *)((char *)S.slam + ((4LL * nrows + 15) & ~15LL));
  S.fp = (float *)((char *)S.ld + ((8LL * nrows + 15) & ~15LL));
  S.fdir = S.fp + 6 * nb;
  return S;
}

__device__ inline SorSet sor_global(const Ctx &c, int nrows, int nact, int ngroups) {
  SRow *sr = c.at<SRow>(c.L.sor);
  return sor_set((char *)(sr + nrows), sr, c.W.nb, nrows, nact, ngroups);
}

// per-world values handed from the solver's set-up to the sweeps and on to
// the integration (split launches), in the world's misc block
enum { MISC_SOR_ROWS = 8, MISC_SOR_GROUPS = 9, MISC_SOR_RESIDUAL = 10, MISC_SOR_READY = 11 };

// inverse inertia (world, symmetric: its upper triangle) times a
__device__ inline void sor_turn(const float *t, const float *a, float *o) {
  o[0] = t[0] * a[0] + t[1] * a[1] + t[2] * a[2];
  o[1] = t[1] * a[0] + t[4] * a[1] + t[5] * a[2];
  o[2] = t[2] * a[0] + t[5] * a[1] + t[8] * a[2];
}

// Set-up: the working set in the world's scratch, in colour order, with the
// starting impulses (zero, or the warm start from the previous step).
__device__ void sor_prepare(const DevBatch &B, const Ctx &c, const WorldParams &P, const Cons *cons, const Row *rows,
                            const float *bt, const int *corder, const int *cstart, int nrows, int ngroups,
                            bool host_contacts, Shared &sh) {
  const int nb = c.W.nb;
  const int nact = cstart[ngroups];   // constraints with rows, in colour order
  const bool warm_on = P.warm != 0.f && !host_contacts && B.warm_n != nullptr;
  const int nprev = warm_on ? B.warm_n[c.w] : -1;
  const bool warm = warm_on && nprev >= 0;
  const WarmRec *wrec = warm_on ? (const WarmRec *)(B.warm + c.W.warm) : nullptr;
  const float *wjnt = warm_on ? (const float *)(B.warm + c.W.warm + od_align(24LL * c.W.kcap)) : nullptr;
  const ContactRec *con = c.at<ContactRec>(c.L.contacts);
  const int nt = blockDim.x;
  const SorSet S = sor_global(c, nrows, nact, ngroups);
  for (int e = threadIdx.x; e < 6 * nb; e += nt) S.fc[e] = 0.f;
  for (int k = threadIdx.x; k <= ngroups; k += nt) S.sstart[k] = cstart[k];
  int rbase = 0;
  for (int x0 = 0; x0 < nact; x0 += nt) {
    int x = x0 + threadIdx.x;
    const Cons *q = x < nact ? &cons[corder[x]] : nullptr;
    int m = q ? q->m : 0;
    int tot;
    int off = block_excl_scan(m, tot, sh);
    if (q) {
      SCons o;
      o.row0 = rbase + off; o.m = m; o.b1 = q->b1; o.b2 = q->b2;
      S.sc[x] = o;
      float wl[SOR_MAX_ROWS] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      if (warm) warm_lookup(P, *q, con, wrec, nprev, wjnt, wl);
      const int b2 = max(o.b2, 0);
      const float *t1 = bt + 32 * o.b1, *t2 = bt + 32 * b2;
      const float im1 = B.invMass[c.W.b0 + o.b1], im2 = B.invMass[c.W.b0 + b2];
      for (int k = 0; k < m; k++) {
        const Row &R = rows[q->row0 + k];
        SRow w;
        for (int j = 0; j < 3; j++) {
          w.l[j] = R.J[j]; w.a1[j] = R.J[3 + j]; w.a2[j] = R.J[9 + j];
        }
        sor_turn(t1, w.a1, w.t1);
        sor_turn(t2, w.a2, w.t2);
        w.rhs = R.rhs; w.cfm = R.cfm; w.ad = R.ad; w.lo = R.lo; w.hi = R.hi;
        w.im1 = im1; w.im2 = im2; w.pad = 0.f;
        w.findex = R.findex >= 0 ? 0 : -1;
        S.sr[o.row0 + k] = w;
        S.slam[o.row0 + k] = k < SOR_MAX_ROWS ? wl[k] : 0.f;
      }
    }
    rbase += tot;
  }
  __syncthreads();
}

// Placement of the coloured solver's working set during the sweeps: all in
// global scratch, all in the LDS pool, everything but the (read-only) rows
// in the pool, everything but the rows and the bodies' conjugate-gradient
// state (read and written once per sweep, by one coalesced pass) in the
// pool, or also the rows' conjugate-gradient state in global scratch (inside
// the colour chain a relaxation only stores to it), or the fc alone in the
// pool (large worlds: it is all that one relaxation hands to another).
enum {
  SOR_IN_GLOBAL = 0, SOR_IN_LDS = 1, SOR_ROWS_GLOBAL = 2, SOR_ROWS_ACC_GLOBAL = 3, SOR_ROWS_CG_GLOBAL = 4,
  SOR_FC_LDS = 5
};

// The sweeps.  The working set (rows included, or all but the rows) is
// copied to the LDS pool first and back at the end; the placement is a
// template argument so that every access compiles to LDS (or global)
// instructions rather than generic flat ones.  Writes the iteration count
// and leaves the last residual in the world's misc block.
//
// One pass relaxes up to blockDim.x constraints of a colour, one per lane,
// with the fc of both bodies in registers.  Its chain (read fc, three rows of
// two dot products and a clamp each, write fc, barrier) and its number of
// instructions bound a sweep, the 0.8 TB/s of rows do not.  So a relaxation
// has no branches inside a row and reads inv(M) J^T instead of multiplying it
// out (96 bytes a row for 64, and no inertia in LDS); a row's successor is
// loaded as soon as the row is done, which hides its latency behind one pass
// without a second set of registers; and the barrier between colours orders
// LDS only (the loads stay in flight) unless the fc are in global memory.
// Two sets of rows in turn, loaded a pass ahead, spilled: 40 % slower than
// this.  2048 uneven worlds, 64 lanes each: 20.7 -> 16.1 us a sweep of 816
// rows at 20 sweeps, 150 -> 95 ms a step at a tolerance of 1e-4.
template <bool TOL, int PLACE>
__device__ __attribute__((noinline)) void sor_solve(char *gsor, int *cnt, int *misc, const WorldParams *Pg,
                                                    LdsChar *pool, int nb, int nrows, int ngroups, int nact, bool warm,
                                                    Shared &sh) {
  constexpr bool IN_POOL = PLACE != SOR_IN_GLOBAL && PLACE != SOR_FC_LDS;
  constexpr bool ROWS_LDS = PLACE == SOR_IN_LDS;
  gsor = uniform_global(gsor);
  cnt = uniform_global(cnt);
  misc = uniform_global(misc);
  pool = uniform(pool);
  nb = uniform(nb);
  nrows = uniform(nrows);
  ngroups = uniform(ngroups);
  nact = uniform(nact);
  warm = uniform(warm);
  const WorldParams &P = *uniform_global(Pg);
  const float tol = uniform(P.tol), sor_w = uniform(P.sor_w);
  const bool use_tol = TOL && tol > 0.f;
  const bool accel = use_tol && uniform(P.accel) != 0;
  const int nt = blockDim.x;
  SRow *const grow = (SRow *)gsor;
  const SorSet G = sor_set((char *)(grow + nrows), grow, nb, nrows, nact, ngroups);
  char *const lds = (char *)pool;
  const SorSet S = ROWS_LDS  ? sor_set((char *)((SRow *)lds + nrows), (SRow *)lds, nb, nrows, nact, ngroups)
                   : IN_POOL ? sor_set(lds, G.sr, nb, nrows, nact, ngroups)
                             : G;
  SRow *__restrict__ sr = ROWS_LDS ? S.sr : G.sr;
  float *__restrict__ fc = PLACE == SOR_FC_LDS ? (float *)lds : S.fc;
  SCons *__restrict__ sc = S.sc;
  int *__restrict__ sstart = S.sstart;
  float *__restrict__ slam = S.slam;
  float *__restrict__ fp = PLACE >= SOR_ROWS_ACC_GLOBAL ? G.fp : S.fp;
  float *__restrict__ fdir = PLACE >= SOR_ROWS_ACC_GLOBAL ? G.fdir : S.fdir;
  float2 *__restrict__ ld = PLACE >= SOR_ROWS_CG_GLOBAL ? G.ld : S.ld;
  if (IN_POOL) {
    if (ROWS_LDS)
      for (int e = threadIdx.x; e < 6 * nrows; e += nt) ((float4 *)sr)[e] = ((const float4 *)G.sr)[e];
    for (int x = threadIdx.x; x < nact; x += nt) sc[x] = G.sc[x];
    for (int k = threadIdx.x; k <= ngroups; k += nt) sstart[k] = G.sstart[k];
    for (int r = threadIdx.x; r < nrows; r += nt) slam[r] = G.slam[r];
  }
  if (PLACE != SOR_IN_GLOBAL)
    for (int e = threadIdx.x; e < 6 * nb; e += nt) fc[e] = 0.f;
  if (accel) {
    for (int e = threadIdx.x; e < 6 * nb; e += nt) fdir[e] = fp[e] = 0.f;
    for (int r = threadIdx.x; r < nrows; r += nt) ld[r] = make_float2(0.f, 0.f);
  }
  __syncthreads();
  if (warm) {
    // fc = inv(M) J^T lambda of the starting impulses, colour by colour
    // (a colour's constraints share no body)
    for (int g = 0; g < ngroups; g++) {
      const int x1 = sstart[g + 1];
      for (int x = sstart[g] + threadIdx.x; x < x1; x += nt) {
        const SCons q = sc[x];
        const bool two = q.b2 >= 0;
        float f1[6], f2[6], *F1 = fc + 6 * q.b1, *F2 = fc + 6 * max(q.b2, 0);
        for (int k = 0; k < 6; k++) { f1[k] = F1[k]; f2[k] = F2[k]; }
        for (int k = 0; k < q.m && k < SOR_MAX_ROWS; k++) {
          const float lam = slam[q.row0 + k];
          if (lam != 0.f) sor_push(sr[q.row0 + k], lam, f1, f2);
        }
        for (int k = 0; k < 6; k++) F1[k] = f1[k];
        if (two)
          for (int k = 0; k < 6; k++) F2[k] = f2[k];
      }
      __syncthreads();
    }
  }
  // The passes of a sweep, in order and over again: [x0, x1) of a colour,
  // whether the pass ends its colour and the sweep.  The end of the next
  // colour is read a pass before it is needed.
  struct Pass {
    int x0;
    bool colour_end, sweep_end;
  };
  int px0 = 0, px1 = 0, pg = ngroups - 1;   // the pass given out last and its colour; start as before colour 0
  int pend = ngroups > 0 ? sstart[1] : 0;   // end of the colour after pg
  auto next_pass = [&](SCons &q) -> Pass {
    if (px0 + nt < px1) {
      px0 += nt;
    } else {
      pg = pg + 1 == ngroups ? 0 : pg + 1;
      px0 = pg == 0 ? 0 : px1;
      px1 = __builtin_amdgcn_readfirstlane(pend);
      pend = sstart[(pg + 1 == ngroups ? 0 : pg + 1) + 1];
    }
    const int x = px0 + (int)threadIdx.x;
    q = sc[min(x, nact - 1)];
    if (x >= px1) q.m = 0;
    Pass v;
    v.x0 = px0;
    v.colour_end = px0 + nt >= px1;
    v.sweep_end = v.colour_end && pg == ngroups - 1;
    return v;
  };
  // The lane's three rows in hand and their impulses.  As soon as a row is
  // relaxed the one that takes its place is loaded: the third row after it in
  // a joint of more than three, else the next pass's.  (A lane without a
  // constraint, or with fewer rows, loads a row that exists: one path for all
  // lanes.)
  SRow r[3];
  float lam[3];
  auto first_row = [&](const SCons &c, int j) { return c.row0 + max(0, min(j, c.m - 1)); };
  SCons q, qn;    // the lane's constraint in this pass and in the next
  Pass pc, pn;
  if (nact > 0) {
    pc = next_pass(q);
#pragma unroll
    for (int j = 0; j < 3; j++) { r[j] = sr[first_row(q, j)]; lam[j] = slam[first_row(q, j)]; }
    pn = next_pass(qn);
  }
  auto reload_lam = [&] {
    if (nact > 0)
#pragma unroll
      for (int j = 0; j < 3; j++) lam[j] = slam[first_row(q, j)];
  };
  // relaxes the pass; true at the sweep's end
  auto pass = [&]() -> bool {
    const bool on = q.m > 0, two = on && q.b2 >= 0;
    float f1[6], f2[6], *F1 = fc + 6 * q.b1, *F2 = fc + 6 * max(q.b2, 0);
    for (int k = 0; k < 6; k++) { f1[k] = F1[k]; f2[k] = F2[k]; }
    const Pass nx = pn;
    SCons q2;
    pn = next_pass(q2);
    float lam0 = 0.f;
#pragma unroll
    for (int j = 0; j < 3; j++) {
      const int i = q.row0 + j;
      if (j < q.m) {
        if (accel) ld[i].x = lam[j];
        lam[j] = sor_relax_row(r[j], lam[j], lam0, two, f1, f2, use_tol);
        slam[i] = lam[j];
        if (j == 0) lam0 = lam[j];
      }
      const int n = 3 + j < q.m ? i + 3 : first_row(qn, j);
      r[j] = sr[n];
      lam[j] = slam[n];
    }
    for (int k0 = 3; k0 < q.m; k0 += 3) {
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const int i = q.row0 + k0 + j;
        if (k0 + j < q.m) {
          if (accel) ld[i].x = lam[j];
          slam[i] = sor_relax_row(r[j], lam[j], lam0, two, f1, f2, use_tol);
          const int n = k0 + 3 + j < q.m ? i + 3 : first_row(qn, j);
          r[j] = sr[n];
          lam[j] = slam[n];
        }
      }
    }
    if (on)
      for (int k = 0; k < 6; k++) F1[k] = f1[k];
    if (two)
      for (int k = 0; k < 6; k++) F2[k] = f2[k];
    const Pass done = pc;
    pc = nx;
    q = qn;
    qn = q2;
    if (done.colour_end) {
      // the end of a sweep hands on impulses and directions too
      if (PLACE == SOR_IN_GLOBAL || done.sweep_end) __syncthreads();
      else lds_barrier();
    }
    return done.sweep_end;
  };
  // fixed iteration count, or (tol > 0) iterate until the LCP residual of
  // the world is at most tol, checked every check_every iterations, up to
  // max_iterations; accelerated: between sweeps a nonsmooth nonlinear
  // conjugate-gradient step (Silcowitz, Niebe, Erleben 2010): with
  // d = lambda_after - lambda_before, beta = |d|^2/|d_prev|^2 (0 if > 1),
  // lambda += beta p_prev (applied before the next sweep, so the solver
  // always ends on a projected sweep), p = d + beta p_prev; fc follows
  // through M^-1 J^T p
  const int maxit = uniform(use_tol ? P.max_iterations : P.iterations);
  const int every = uniform(use_tol ? (P.check_every > 0 ? P.check_every : 1) : (maxit > 0 ? maxit : 1));
  float rr_prev = 0.f, res_prev = INFINITY;
  bool acc = accel;        // CG steps still on for this solve
  float res_last = 0.f;    // residual at the last check
  int it = 0;
  while (it < maxit) {
    const int n = every < maxit - it ? every : maxit - it;
    for (int rep = 0; rep < n; rep++) {
      if (acc && rep == 0) {
        // the pending momentum beta p_prev of the previous sweep (kept in
        // ld.x for the rows and fp for the bodies), then fc before this
        // sweep; inside a block of sweeps between two checks this is folded
        // into the previous sweep's CG update below
        for (int r = threadIdx.x; r < nrows; r += nt)
          if (ld[r].x != 0.f) slam[r] += ld[r].x;
        for (int e = threadIdx.x; e < 6 * nb; e += nt) fp[e] = fc[e] += fp[e];   // one fc component per lane
        __syncthreads();
        reload_lam();
      }
      if (nact > 0)
        while (!pass()) {}
      if (acc) {
        // d = this sweep's change; beta = |d|^2 / |d_prev|^2 (restart when
        // > 1); the momentum beta p_prev is applied before the next sweep
        float loc = 0.f;
#pragma unroll 4
        for (int r = threadIdx.x; r < nrows; r += nt) {
          float d = slam[r] - ld[r].x;
          loc += d * d;
        }
        const float rr = uniform(block_fsum(loc, sh));
        float beta = (rr_prev > 0.f) ? rr / rr_prev : 0.f;
        if (!(beta <= 1.f)) beta = 0.f;
        // the next sweep of this block takes the momentum now (the same
        // operations as the pending-momentum step above); the last sweep
        // before a check leaves it pending, so the check sees the sweep's
        // own result
        const bool now = rep + 1 < n;
#pragma unroll 4
        for (int r = threadIdx.x; r < nrows; r += nt) {
          const float2 o = ld[r];
          const float lam = slam[r], d = lam - o.x;
          const float pend = beta * o.y;                             // momentum along the previous direction
          ld[r] = make_float2(now ? o.x : pend, d + pend);           // and the new direction
          if (now) slam[r] = pend != 0.f ? lam + pend : lam;
        }
        for (int e = threadIdx.x; e < 6 * nb; e += nt) {   // one fc component per lane
          const float f = fc[e], pend = beta * fdir[e];
          fdir[e] = (f - fp[e]) + pend;
          fp[e] = now ? f + pend : pend;
          if (now) fc[e] = f + pend;
        }
        rr_prev = rr;
        __syncthreads();
        reload_lam();
      }
    }
    it += n;
    if (use_tol) {
      float r = 0.f;
      for (int x = threadIdx.x; x < nact; x += nt) r = fmaxf(r, sor_cons_residual(fc, sr, slam, sc[x], sor_w));
      r = uniform(block_max(r, sh));
      res_last = r;
      if (r <= tol) break;
      if (acc && !(r <= res_prev)) {
        // the residual rose since the last check: restart the CG steps, and
        // stop them for the rest of the solve when the residual is still far
        // (> 1000 tol) from the tolerance
        for (int q = threadIdx.x; q < nrows; q += nt) ld[q] = make_float2(0.f, 0.f);
        for (int e = threadIdx.x; e < 6 * nb; e += nt) fdir[e] = fp[e] = 0.f;
        rr_prev = 0.f;
        if (r > 1000.f * tol) acc = false;
        __syncthreads();
      }
      res_prev = r;
    }
  }
  if (threadIdx.x == 0) {
    cnt[CNT_ITERS] = it;
    misc[MISC_SOR_RESIDUAL] = __float_as_int(use_tol ? res_last : 0.f);
    if (use_tol) {
      if (!(res_last <= tol)) cnt[CNT_UNCONV] += 1;
      // non-negative floats order like their bit patterns
      const int rb = __float_as_int(res_last == res_last ? res_last : INFINITY);
      if (rb > cnt[CNT_RESMAX]) cnt[CNT_RESMAX] = rb;
    }
  }
  if (PLACE != SOR_IN_GLOBAL) {
    __syncthreads();
    for (int e = threadIdx.x; e < 6 * nb; e += nt) G.fc[e] = fc[e];
  }
  if (IN_POOL)
    for (int r = threadIdx.x; r < nrows; r += nt) G.slam[r] = slam[r];
  __syncthreads();
}

// the placement with as much as fits in `lds` bytes of the pool
template <bool TOL>
__device__ inline void sor_solve_any(const DevBatch &B, const Ctx &c, const WorldParams &P, int nrows, int ngroups,
                                     int nact, bool host_contacts, int lds, Shared &sh) {
  const int nb = c.W.nb;
  const bool accel = TOL && P.tol > 0.f && P.accel != 0;
  const bool warm = P.warm != 0.f && !host_contacts && B.warm_n != nullptr && B.warm_n[c.w] >= 0;
  char *gsor = c.at<char>(c.L.sor);
  int *cnt = B.counters + c.w * CNT_N, *misc = c.at<int>(c.L.misc);
  LdsChar *pool = (LdsChar *)od_pool;
  if (sor_lds_bytes(nb, nrows, nact, ngroups, accel) <= lds)
    sor_solve<TOL, SOR_IN_LDS>(gsor, cnt, misc, &P, pool, nb, nrows, ngroups, nact, warm, sh);
  else if (sor_lds_bytes_rows_global(nb, nrows, nact, ngroups, accel) <= lds)
    sor_solve<TOL, SOR_ROWS_GLOBAL>(gsor, cnt, misc, &P, pool, nb, nrows, ngroups, nact, warm, sh);
  else if (accel && sor_lds_bytes_rows_acc_global(nb, nrows, nact, ngroups, accel) <= lds)
    sor_solve<TOL, SOR_ROWS_ACC_GLOBAL>(gsor, cnt, misc, &P, pool, nb, nrows, ngroups, nact, warm, sh);
  else if (accel && sor_lds_bytes_rows_cg_global(nb, nrows, nact, ngroups) <= lds)
    sor_solve<TOL, SOR_ROWS_CG_GLOBAL>(gsor, cnt, misc, &P, pool, nb, nrows, ngroups, nact, warm, sh);
  else if (24LL * nb <= lds)
    sor_solve<TOL, SOR_FC_LDS>(gsor, cnt, misc, &P, pool, nb, nrows, ngroups, nact, warm, sh);
  else
    sor_solve<TOL, SOR_IN_GLOBAL>(gsor, cnt, misc, &P, pool, nb, nrows, ngroups, nact, warm, sh);
}

// After the sweeps: impulses back to the rows (constraint order), fc to the
// per-body scratch, and the warm-start records of the next step.
__device__ void sor_finish(const DevBatch &B, const Ctx &c, const WorldParams &P, const Cons *cons, Row *rows,
                           float *bt, const int *corder, int nrows, int nact, int ngroups, int nk, int ncons,
                           bool host_contacts) {
  const int nb = c.W.nb;
  const int nt = blockDim.x;
  const SorSet G = sor_global(c, nrows, nact, ngroups);
  const bool warm_on = P.warm != 0.f && !host_contacts && B.warm_n != nullptr;
  WarmRec *wrec = warm_on ? (WarmRec *)(B.warm + c.W.warm) : nullptr;
  float *wjnt = warm_on ? (float *)(B.warm + c.W.warm + od_align(24LL * c.W.kcap)) : nullptr;
  const ContactRec *con = c.at<ContactRec>(c.L.contacts);
  const float res_last = __int_as_float(c.at<int>(c.L.misc)[MISC_SOR_RESIDUAL]);
  for (int x = threadIdx.x; x < nact; x += nt) {
    const Cons &q = cons[corder[x]];
    const SCons o = G.sc[x];
    for (int k = 0; k < o.m; k++) rows[q.row0 + k].lambda = G.slam[o.row0 + k];
  }
  for (int b = threadIdx.x; b < nb; b += nt)
    for (int k = 0; k < 6; k++) bt[32 * b + 9 + k] = G.fc[6 * b + k];
  __syncthreads();
  const bool use_tol = P.tol > 0.f;
  if (warm_on && use_tol && !(res_last <= 100.f * P.tol)) {
    // a solve that ended at the cap far from the tolerance (residual > 100
    // tol) is no starting point: the next solve starts from zero
    if (threadIdx.x == 0) B.warm_n[c.w] = -1;
    __syncthreads();
  } else if (warm_on) {
    // this step's impulses, the next step's starting point; contacts are in
    // pair order, so the records come out sorted by key
    for (int i = threadIdx.x; i < nk; i += nt) {
      const Cons &q = cons[i];
      const ContactRec &cr = con[q.src];
      WarmRec r;
      r.key = contact_key(cr.g1, cr.g2, cr.flags >> 8);
      for (int k = 0; k < 3; k++) r.lam[k] = k < q.m ? rows[q.row0 + k].lambda : 0.f;
      r.pad = 0;
      wrec[i] = r;
    }
    for (int i = nk + threadIdx.x; i < ncons; i += nt) {
      const Cons &q = cons[i];
      float *jw = wjnt + 8 * q.src;
      for (int k = 0; k < 6; k++) jw[k] = k < q.m ? rows[q.row0 + k].lambda : 0.f;
      jw[6] = __int_as_float(q.m);
      jw[7] = 0.f;
    }
    if (threadIdx.x == 0) B.warm_n[c.w] = nk;
    __syncthreads();
  }
}

// the coloured solver in one kernel: set-up, sweeps, write-back
template <bool TOL>
__device__ void sor_colored(const DevBatch &B, const Ctx &c, const WorldParams &P, const Cons *cons, Row *rows,
                            float *bt, const int *corder, const int *cstart, int nrows, int ngroups, int nk,
                            int ncons, bool host_contacts, Shared &sh) {
  const int nact = cstart[ngroups];
  sor_prepare(B, c, P, cons, rows, bt, corder, cstart, nrows, ngroups, host_contacts, sh);
  sor_solve_any<TOL>(B, c, P, nrows, ngroups, nact, host_contacts, B.lds_bytes, sh);
  sor_finish(B, c, P, cons, rows, bt, corder, nrows, nact, ngroups, nk, ncons, host_contacts);
}

#include "ref_order.hpp"
#include "lcp_exact.hpp"

// inv(M) J^T, rhs, cfm and ad of a row whose rhs holds c.  t1, t2: its
// bodies' temporaries (t2 null: one body): world inverse inertia 0..8, v/h +
// inv(M) f_ext 15..20.
__device__ inline void finish_row(Row &R, const float *t1, const float *t2, float im1, float im2, float hinv,
                                  float sor_w) {
  float s = 0.f;
  for (int k = 0; k < 6; k++) s += R.J[k] * t1[15 + k];
  float d = 0.f;
  for (int k = 0; k < 3; k++) R.iMJ[k] = im1 * R.J[k];
  for (int k = 0; k < 3; k++) R.iMJ[3 + k] = t1[3 * k] * R.J[3] + t1[3 * k + 1] * R.J[4] + t1[3 * k + 2] * R.J[5];
  for (int k = 0; k < 6; k++) d += R.iMJ[k] * R.J[k];
  if (t2) {
    for (int k = 0; k < 6; k++) s += R.J[6 + k] * t2[15 + k];
    for (int k = 0; k < 3; k++) R.iMJ[6 + k] = im2 * R.J[6 + k];
    for (int k = 0; k < 3; k++) R.iMJ[9 + k] = t2[3 * k] * R.J[9] + t2[3 * k + 1] * R.J[10] + t2[3 * k + 2] * R.J[11];
    for (int k = 6; k < 12; k++) d += R.iMJ[k] * R.J[k];
  } else {
    for (int k = 6; k < 12; k++) R.iMJ[k] = 0.f;
  }
  R.rhs = R.rhs * hinv - s;
  R.cfm = R.cfm * hinv;
  R.ad = sor_w / (d + R.cfm);
  R.lambda = 0.f;
}

__device__ inline void store_row(Row *dst, const Row &R) {
  static_assert(sizeof(Row) % 16 == 0, "rows are written 16 bytes at a time");
  __builtin_memcpy(__builtin_assume_aligned(dst, 16), &R, sizeof(Row));
}

// STAGE 0: the whole step; 1: up to the coloured solver's set-up (the sweeps
// and the rest run in later kernels); 2: after the sweeps (write-back,
// velocities, integration)
template <bool TOL, int STAGE>
__device__ __attribute__((always_inline)) void phase_step(const DevBatch &B, const Ctx &c, WorldParams &P,
                                                          const StepIn &in, Shared &sh, bool ref) {
  const int nb = c.W.nb, nj = c.W.nj, nk = in.nk;
  const float h = P.dt, hinv = 1.f / P.dt;
  float *bt = c.at<float>(c.L.btmp);   // per body: invIw 0..8, fc 9..14, tmp 15..20, extra torque 21..23
  Cons *cons = c.at<Cons>(c.L.cons);
  Row *rows = c.at<Row>(c.L.rows);
  const ContactRec *con = c.at<ContactRec>(c.L.contacts);
  int *misc = c.at<int>(c.L.misc);
  const int ncons = nk + nj;
  int *corder = c.at<int>(c.L.order);          // constraint order (island order when ref)
  int *isl = c.at<int>(c.L.island);            // ref: [cons0, ncons, row0, nrows, seed] per island
  int *color = c.at<int>(c.L.color);           // ref: body tags, then constraint tags and Info2 erp
  int nrows = 0, ngroups = 0;
  if (STAGE == 2) {
    if (misc[MISC_SOR_READY] == 0) return;     // the step left the world unchanged
    nrows = misc[MISC_SOR_ROWS];
    ngroups = misc[MISC_SOR_GROUPS];
    const int nact = isl[ngroups];
    const bool accel = TOL && P.tol > 0.f && P.accel != 0;
    if (sor_lds_bytes(nb, nrows, nact, ngroups, accel) > B.sor_lds_bytes) {
      // not solved by the sweep kernel (its LDS pool is too small)
      sor_solve_any<TOL>(B, c, P, nrows, ngroups, nact, in.from_host, 0, sh);
      c.clk.lap(PH_SOR);
    }
    sor_finish(B, c, P, cons, rows, bt, corder, nrows, nact, ngroups, nk, ncons, in.from_host);
  } else {
  // --- bodies: world inverse inertia, gyroscopic torque, gravity
  //     (quickstep.cpp:609-665)
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    int gb = c.W.b0 + b;
    Mat3 R = load_mat(B.R + 3 * (size_t)gb);
    Mat3 iI = rotate_tensor(R, load_mat(B.invI + 3 * (size_t)gb));
    float *t = bt + 32 * b;
    t[0] = iI.r0.x; t[1] = iI.r0.y; t[2] = iI.r0.z;
    t[3] = iI.r1.x; t[4] = iI.r1.y; t[5] = iI.r1.z;
    t[6] = iI.r2.x; t[7] = iI.r2.y; t[8] = iI.r2.z;
    for (int k = 9; k < 24; k++) t[k] = 0.f;
    float3 w = xyz(B.avel[gb]);
    float4 ta = B.tacc[gb];
    Mat3 Iw = rotate_tensor(R, load_mat(B.I + 3 * (size_t)gb));
    float3 gyro = cross(w, Iw.mul(w));
    ta.x -= gyro.x; ta.y -= gyro.y; ta.z -= gyro.z;
    B.tacc[gb] = ta;
    float4 fa = B.facc[gb];
    float m = B.mass[gb];
    if (P.gravity[0] != 0.f) fa.x += m * P.gravity[0];
    if (P.gravity[1] != 0.f) fa.y += m * P.gravity[1];
    if (P.gravity[2] != 0.f) fa.z += m * P.gravity[2];
    B.facc[gb] = fa;
  }
  // --- constraints: contacts (k < nk) then permanent joints
  for (int i = threadIdx.x; i < ncons; i += blockDim.x) {
    Cons &q = cons[i];
    if (i < nk) {
      q.kind = JT_CONTACT;
      q.src = i;
      if (in.from_host) {
        const ContactIn &ci = B.cin[B.cin_start[c.w] + i];
        q.b1 = ci.b1; q.b2 = ci.b2; q.seq = ci.seq; q.fb = ci.fb;
      } else {
        q.b1 = con[i].b1; q.b2 = con[i].b2; q.seq = in.seq_base + i; q.fb = -1;
      }
    } else {
      const JointDev &j = B.joints[c.W.j0 + i - nk];
      q.kind = j.type; q.src = i - nk; q.b1 = j.b1; q.b2 = j.b2; q.seq = j.seq; q.fb = j.fb;
    }
    q.m = 0;
    q.row0 = 0;
  }
  __syncthreads();
  // --- getInfo1 (quickstep.cpp:670-688); joints update their limit state
  for (int i = threadIdx.x; i < ncons; i += blockDim.x) {
    Cons &q = cons[i];
    int m = 0;
    if (q.b1 >= 0) {
      if (q.kind == JT_CONTACT) {
        Surf s = in.from_host ? host_surface(B.cin[B.cin_start[c.w] + i]) : world_surface(P);
        m = contact_info1(s);
      } else {
        JointDev &j = B.joints[c.W.j0 + q.src];
        BodyPose s1 = load_pose(B, c.W.b0 + q.b1);
        BodyPose s2;
        if (q.b2 >= 0) s2 = load_pose(B, c.W.b0 + q.b2);
        if (!(j.type == JT_HINGE2 && q.b2 < 0)) m = joint_info1(j, s1, q.b2 >= 0 ? &s2 : nullptr);
      }
    }
    q.m = m;
  }
  __syncthreads();
  c.clk.lap(PH_BODIES);
  // --- constraint order, row offsets, groups
  if (ref && nb < 65535 && ncons < 65535 && ref_order_lds_bytes(nb, ncons) <= B.lds_bytes) {
    ref_order_lds(cons, B.joints + c.W.j0, B.invMass + c.W.b0, &P, nb, nk, ncons, in.from_host, corder, isl,
                  (float *)(color + nb), misc, (LdsChar *)od_pool, sh);
    nrows = misc[0];
    ngroups = misc[1];
  } else if (ref) {
    if (threadIdx.x == 0) {
      // adjacency, newest attach first: body joint lists prepend (ode.cpp:1382-1389)
      int *adjs = c.at<int>(c.L.adjs);
      int *adj = c.at<int>(c.L.adj);
      for (int b = 0; b <= nb; b++) adjs[b] = 0;
      for (int i = 0; i < ncons; i++) {
        if (cons[i].m <= 0 && cons[i].kind != JT_CONTACT) continue;
        if (cons[i].b1 < 0) continue;
        adjs[cons[i].b1 + 1]++;
        if (cons[i].b2 >= 0) adjs[cons[i].b2 + 1]++;
      }
      for (int b = 0; b < nb; b++) adjs[b + 1] += adjs[b];
      // visit constraints in descending attach sequence: contacts carry
      // increasing sequence numbers in order; joints are merged in by seq
      int *jord = color;   // joints sorted by seq (insertion sort, few joints)
      int nj2 = 0;
      for (int i = nk; i < ncons; i++) {
        if (cons[i].b1 < 0) continue;
        int s = cons[i].seq, p = nj2++;
        while (p > 0 && cons[jord[p - 1]].seq > s) { jord[p] = jord[p - 1]; p--; }
        jord[p] = i;
      }
      int *fill = isl;     // per-body fill cursor (scratch reuse)
      for (int b = 0; b < nb; b++) fill[b] = adjs[b];
      int ci = nk - 1, jj = nj2 - 1;
      while (ci >= 0 || jj >= 0) {
        int pick;
        if (jj < 0) pick = ci--;
        else if (ci < 0) pick = jord[jj--];
        else if (cons[ci].seq > cons[jord[jj]].seq) pick = ci--;
        else pick = jord[jj--];
        const Cons &q = cons[pick];
        if (q.b1 < 0) continue;
        adj[fill[q.b1]++] = pick;
        if (q.b2 >= 0) adj[fill[q.b2]++] = pick;
      }
      // islands: depth-first walk from bodies in world-list order, newest
      // body first (util.cpp:420-487)
      int *tag = color;           // body tags, then constraint tags
      int *ctag = color + nb;
      for (int b = 0; b < nb; b++) tag[b] = 0;
      for (int i = 0; i < ncons; i++) ctag[i] = 0;
      int *border = corder + ncons;  // body visit order
      int *stack = isl + 5 * (nb + 1);  // island table first, then the stack
      int nic = 0, nib = 0, nisl = 0;
      for (int bb = nb - 1; bb >= 0; bb--) {
        if (tag[bb]) continue;
        tag[bb] = 1;
        int c0 = nic;
        border[nib++] = bb;
        int sp = 0, b = bb;
        while (true) {
          for (int k = adjs[b]; k < adjs[b + 1]; k++) {
            int qi = adj[k];
            if (ctag[qi]) continue;
            const Cons &q = cons[qi];
            bool enabled = B.invMass[c.W.b0 + q.b1] > 0.f || (q.b2 >= 0 && B.invMass[c.W.b0 + q.b2] > 0.f);
            if (!enabled) { ctag[qi] = 2; continue; }
            ctag[qi] = 1;
            corder[nic++] = qi;
            int other = (q.b1 == b) ? q.b2 : q.b1;
            if (other >= 0 && tag[other] <= 0) {
              tag[other] = 1;
              stack[sp++] = other;
            }
          }
          if (sp == 0) break;
          b = stack[--sp];
          border[nib++] = b;
        }
        isl[5 * nisl + 0] = c0;
        isl[5 * nisl + 1] = nic - c0;
        nisl++;
      }
      for (int i = 0; i < ncons; i++)
        if (ctag[i] != 1) cons[i].m = 0;
      // rows in island order; the RNG state of every island by skip-ahead:
      // an island with m rows makes ceil(iterations/8) * (m-1) draws
      // (quickstep.cpp:473-482)
      unsigned seed = P.seed;
      unsigned long long shuffles = (unsigned long long)((P.iterations + 7) / 8);
      int r = 0;
      float erp = P.erp;
      for (int k = 0; k < nisl; k++) {
        int c0 = isl[5 * k], cn = isl[5 * k + 1];
        int r0 = r;
        erp = P.erp;   // Info2 erp is reset per island (quickstep.cpp:777-779)
        for (int x = 0; x < cn; x++) {
          Cons &q = cons[corder[c0 + x]];
          q.row0 = r;
          r += q.m;
          // a ball joint sets the Info2 erp seen by the joints after it
          if (q.kind == JT_BALL) erp = B.joints[c.W.j0 + q.src].erp;
          ((float *)ctag)[corder[c0 + x]] = erp;
        }
        int m = r - r0;
        isl[5 * k + 2] = r0;
        isl[5 * k + 3] = m;
        isl[5 * k + 4] = (int)seed;
        if (m > 0 && m - 1 > 0) seed = lcg_skip(seed, shuffles * (unsigned long long)(m - 1));
      }
      P.seed = seed;
      misc[0] = r;
      misc[1] = nisl;
      misc[2] = nic;
      misc[3] = nib;
    }
    __syncthreads();
    nrows = misc[0];
    ngroups = misc[1];
  } else {
    // natural order; rows by a block scan
    int r0 = 0;
    for (int start = 0; start < ncons; start += blockDim.x) {
      int i = start + threadIdx.x;
      int m = (i < ncons) ? cons[i].m : 0;
      int tot;
      int off = block_excl_scan(m, tot, sh);
      if (i < ncons) { cons[i].row0 = r0 + off; corder[i] = i; }
      r0 += tot;
    }
    nrows = r0;
    int *bmax = c.at<int>(c.L.adjs), *lists = c.at<int>(c.L.sor);
    LdsChar *pool = (LdsChar *)od_pool;
    const long long cb = col_bodies_bytes(nb);
    if (cb + col_lists_bytes(ncons) <= B.lds_bytes)
      ngroups = colour_constraints<COL_IN_LDS>(cons, bt, bmax, lists, pool, nb, ncons, corder, isl, sh);
    else if (cb <= B.lds_bytes)
      ngroups = colour_constraints<COL_BODIES_LDS>(cons, bt, bmax, lists, pool, nb, ncons, corder, isl, sh);
    else
      ngroups = colour_constraints<COL_IN_GLOBAL>(cons, bt, bmax, lists, pool, nb, ncons, corder, isl, sh);
    ngroups = uniform(ngroups);
  }
  c.clk.lap(PH_ORDER);
  if (nrows > c.W.rcap) {
    // not enough row storage: leave the world unchanged for this step (and
    // start the next solve from zero)
    if (threadIdx.x == 0) {
      raise_overflow(B, c.w, OVF_ROWS);
      if (B.warm_n) B.warm_n[c.w] = -1;
      if (STAGE == 1) misc[MISC_SOR_READY] = 0;
    }
    __syncthreads();
    return;
  }
  // --- getInfo2 (quickstep.cpp:764-830) and rhs = c/h - J (v/h + inv(M)
  //     f_ext), cfm /= h (832-857), one constraint per lane.  The joints come
  //     first: a motor pushing against its limit adds to f_ext.  A contact's
  //     rows are built and finished in registers and written once, 16 bytes
  //     at a time: written word by word, read back and written again they
  //     cost a pass of 64 cache lines per word (4096 uneven worlds: 2047 ->
  //     1391 workgroup-ms in 4 steps).
  const float *erp_of = ref ? (const float *)(color + nb) : nullptr;
  for (int i = nk + threadIdx.x; i < ncons; i += blockDim.x) {
    Cons &q = cons[i];
    if (q.m <= 0) continue;
    Row *r = rows + q.row0;
    for (int k = 0; k < q.m; k++) {
      row_clear(r[k], P.cfm);
      r[k].b1 = q.b1;
      r[k].b2 = q.b2;
    }
    BodyPose s1 = load_pose(B, c.W.b0 + q.b1);
    BodyPose s2;
    if (q.b2 >= 0) s2 = load_pose(B, c.W.b0 + q.b2);
    const BodyPose *p2 = q.b2 >= 0 ? &s2 : nullptr;
    JointDev &j = B.joints[c.W.j0 + q.src];
    float3 e1 = mk3(0.f, 0.f, 0.f), e2 = mk3(0.f, 0.f, 0.f);
    float e = erp_of ? erp_of[i] : P.erp;
    joint_info2(j, r, s1, p2, hinv, e, e1, e2);
    float *t1 = bt + 32 * q.b1 + 21;
    if (e1.x != 0.f || e1.y != 0.f || e1.z != 0.f) {
      // a motor pushing against its limit: torque applied below in order
      atomicAdd(&t1[0], e1.x); atomicAdd(&t1[1], e1.y); atomicAdd(&t1[2], e1.z);
      if (q.b2 >= 0) {
        float *t2 = bt + 32 * q.b2 + 21;
        atomicAdd(&t2[0], e2.x); atomicAdd(&t2[1], e2.y); atomicAdd(&t2[2], e2.z);
      }
    }
    for (int k = 0; k < q.m; k++)
      if (r[k].findex >= 0) r[k].findex += q.row0;
  }
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    int gb = c.W.b0 + b;
    float *t = bt + 32 * b;
    float4 ta = B.tacc[gb];
    ta.x += t[21]; ta.y += t[22]; ta.z += t[23];
    B.tacc[gb] = ta;
    float im = B.invMass[gb];
    float4 fa = B.facc[gb];
    float3 v = xyz(B.lvel[gb]), w = xyz(B.avel[gb]);
    t[15] = fa.x * im + v.x * hinv;
    t[16] = fa.y * im + v.y * hinv;
    t[17] = fa.z * im + v.z * hinv;
    float3 it = mk3(t[0] * ta.x + t[1] * ta.y + t[2] * ta.z, t[3] * ta.x + t[4] * ta.y + t[5] * ta.z,
                    t[6] * ta.x + t[7] * ta.y + t[8] * ta.z);
    t[18] = it.x + w.x * hinv;
    t[19] = it.y + w.y * hinv;
    t[20] = it.z + w.z * hinv;
  }
  __syncthreads();
  for (int x = threadIdx.x; x < SOR_MAX_ROWS * nj; x += blockDim.x) {
    const int i = nk + x / SOR_MAX_ROWS, k = x % SOR_MAX_ROWS;
    if (k >= cons[i].m) continue;
    Row *dst = rows + cons[i].row0 + k;
    Row R = *dst;
    finish_row(R, bt + 32 * R.b1, R.b2 >= 0 ? bt + 32 * R.b2 : nullptr, B.invMass[c.W.b0 + R.b1],
               R.b2 >= 0 ? B.invMass[c.W.b0 + R.b2] : 0.f, hinv, P.sor_w);
    store_row(dst, R);
  }
  for (int i = threadIdx.x; i < nk; i += blockDim.x) {
    const Cons q = cons[i];
    if (q.m <= 0) continue;
    Row r[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      row_clear(r[k], P.cfm);
      r[k].b1 = q.b1;
      r[k].b2 = q.b2;
    }
    const BodyPose s1 = load_pose(B, c.W.b0 + q.b1);
    BodyPose s2;
    if (q.b2 >= 0) s2 = load_pose(B, c.W.b0 + q.b2);
    float3 cpos, cn;
    float cd;
    bool rev;
    Surf s;
    if (in.from_host) {
      const ContactIn &ci = B.cin[B.cin_start[c.w] + q.src];
      cpos = mk3(ci.pos[0], ci.pos[1], ci.pos[2]);
      cn = mk3(ci.normal[0], ci.normal[1], ci.normal[2]);
      cd = ci.depth;
      rev = (ci.flags & JF_REVERSE) != 0;
      s = host_surface(ci);
    } else {
      const ContactRec &cr = con[q.src];
      cpos = mk3(cr.pos[0], cr.pos[1], cr.pos[2]);
      cn = mk3(cr.normal[0], cr.normal[1], cr.normal[2]);
      cd = cr.depth;
      rev = (cr.flags & JF_REVERSE) != 0;
      s = world_surface(P);
    }
    contact_info2(r, contact_info1(s), s, cpos, cn, cd, rev, s1, q.b2 >= 0 ? &s2 : nullptr, hinv,
                  erp_of ? erp_of[i] : P.erp, P.min_depth, P.max_vel);
    const float *t1 = bt + 32 * q.b1, *t2 = q.b2 >= 0 ? bt + 32 * q.b2 : nullptr;
    const float im1 = B.invMass[c.W.b0 + q.b1], im2 = q.b2 >= 0 ? B.invMass[c.W.b0 + q.b2] : 0.f;
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (k < q.m) {
        if (r[k].findex >= 0) r[k].findex += q.row0;
        finish_row(r[k], t1, t2, im1, im2, hinv, P.sor_w);
        store_row(rows + q.row0 + k, r[k]);
      }
  }
  __syncthreads();
  c.clk.lap(PH_ROWS);
  // --- SOR-LCP
  const int iters = P.iterations;
  if (ref) {
    // the placement with as much as fits in the LDS pool
    char *gws = c.at<char>(c.L.sor);
    const long long st = ref_state_bytes(nrows, nb), sched = ref_sched_bytes(nrows, nb);
    if (P.exact && B.lcp_ws)
      lcp_exact_world(B, c.w, rows, bt, isl, ngroups, nb, sh);
    else if (st + sched + ref_sides_bytes(nrows) <= B.lds_bytes)
      sor_reference<REF_IN_LDS>(rows, bt, isl, gws, (LdsChar *)od_pool, nrows, ngroups, nb, iters, sh);
    else if (st + sched <= B.lds_bytes)
      sor_reference<REF_ROWS_GLOBAL>(rows, bt, isl, gws, (LdsChar *)od_pool, nrows, ngroups, nb, iters, sh);
    else if (st <= B.lds_bytes)
      sor_reference<REF_SCHED_GLOBAL>(rows, bt, isl, gws, (LdsChar *)od_pool, nrows, ngroups, nb, iters, sh);
    else
      sor_reference<REF_IN_GLOBAL>(rows, bt, isl, gws, (LdsChar *)od_pool, nrows, ngroups, nb, iters, sh);
    if (threadIdx.x == 0) B.counters[c.w * CNT_N + CNT_ITERS] = iters;
  } else if (STAGE == 1) {
    // the sweeps run in their own kernel
    sor_prepare(B, c, P, cons, rows, bt, corder, isl, nrows, ngroups, in.from_host, sh);
    if (threadIdx.x == 0) {
      misc[MISC_SOR_ROWS] = nrows;
      misc[MISC_SOR_GROUPS] = ngroups;
      misc[MISC_SOR_READY] = 1;
    }
    __syncthreads();
    return;
  } else {
    sor_colored<TOL>(B, c, P, cons, rows, bt, corder, isl, nrows, ngroups, nk, ncons, in.from_host, sh);
  }
  }
  c.clk.lap(PH_SOR);
  // --- residual (optional), feedback
  if (B.track_residual) {
    float mr = 0.f;
    for (int i = threadIdx.x; i < nrows; i += blockDim.x) mr = fmaxf(mr, row_residual(rows, i, bt));
    mr = block_max(mr, sh);
    if (threadIdx.x == 0) B.residual[c.w] = mr;
  }
  if (B.feedback) {
    for (int i = threadIdx.x; i < ncons; i += blockDim.x) {
      const Cons &q = cons[i];
      if (q.fb < 0 || q.m <= 0) continue;
      float d[12];
      for (int k = 0; k < 12; k++) d[k] = 0.f;
      for (int r = 0; r < q.m; r++) {
        const Row &R = rows[q.row0 + r];
        for (int k = 0; k < 12; k++) d[k] += R.J[k] * R.lambda;
      }
      float *o = B.feedback + 12 * (size_t)q.fb;
      for (int k = 0; k < 6; k++) o[k] = d[k];
      if (q.b2 >= 0)
        for (int k = 0; k < 6; k++) o[6 + k] = d[6 + k];
    }
  }
  // --- velocity update, integration (quickstep.cpp:905-1021, util.cpp:255-360)
  if (threadIdx.x == 0) sh.ival[13] = 0;
  __syncthreads();
  for (int b = threadIdx.x; b < nb; b += blockDim.x) {
    int gb = c.W.b0 + b;
    float *t = bt + 32 * b;
    float3 v = xyz(B.lvel[gb]), w = xyz(B.avel[gb]);
    v = v + h * mk3(t[9], t[10], t[11]);
    w = w + h * mk3(t[12], t[13], t[14]);
    float im = B.invMass[gb] * h;
    float4 fa = B.facc[gb], ta = B.tacc[gb];
    v = v + im * xyz(fa);
    float3 th = h * xyz(ta);
    w = w + mk3(t[0] * th.x + t[1] * th.y + t[2] * th.z, t[3] * th.x + t[4] * th.y + t[5] * th.z,
                t[6] * th.x + t[7] * th.y + t[8] * th.z);
    float3 p = xyz(B.pos[gb]) + h * v;
    float4 q = B.q[gb];
    float4 dq = make_float4(0.5f * (-w.x * q.y - w.y * q.z - w.z * q.w), 0.5f * (w.x * q.x + w.y * q.w - w.z * q.z),
                            0.5f * (-w.x * q.w + w.y * q.x + w.z * q.y), 0.5f * (w.x * q.z - w.y * q.y + w.z * q.x));
    q = make_float4(q.x + h * dq.x, q.y + h * dq.y, q.z + h * dq.z, q.w + h * dq.w);
    q = quat_normalize(q);
    B.pos[gb] = f4(p);
    B.q[gb] = q;
    store_mat(B.R + 3 * (size_t)gb, quat_to_mat(q));
    B.lvel[gb] = f4(v);
    B.avel[gb] = f4(w);
    B.facc[gb] = make_float4(0.f, 0.f, 0.f, 0.f);
    B.tacc[gb] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (!(isfinite(p.x) && isfinite(p.y) && isfinite(p.z) && isfinite(q.x) && isfinite(v.x) && isfinite(v.y) &&
          isfinite(v.z) && isfinite(w.x) && isfinite(w.y) && isfinite(w.z)))
      sh.ival[13] = 1;
  }
  // --- space list after dGeomMoved of every stepped body: moved geoms move
  //     to the front in reverse move order (collision_space.cpp:47-75, 209-213)
  if (ref) {
    // in parallel: old rank -> geom; the moved geoms in move order (bodies
    // in island visit order, each body's geoms newest first) take ranks
    // M-1..0; the others follow in their old relative order
    const int nib = misc[3];
    const int *border = corder + ncons;
    int *old = isl + 5 * (ngroups + 1);
    const int ng = c.W.ng;
    int *inv = old;                     // old rank -> geom
    int *moved = old + ng;
    int *flag = moved + ng;
    for (int g = threadIdx.x; g < ng; g += blockDim.x) {
      inv[B.grank[c.W.g0 + g]] = g;
      flag[g] = 0;
    }
    __syncthreads();
    int M = 0;
    for (int x0 = 0; x0 < nib; x0 += blockDim.x) {
      const int x = x0 + threadIdx.x;
      int k0 = 0, cnt = 0;
      if (x < nib) {
        const int gb = c.W.b0 + border[x];
        k0 = B.bgeom_start[gb];
        cnt = B.bgeom_start[gb + 1] - k0;
      }
      int tot;
      const int off = block_excl_scan(cnt, tot, sh);
      for (int j = 0; j < cnt; j++) moved[M + off + j] = B.bgeom[k0 + j];
      M += tot;
    }
    __syncthreads();
    for (int x = threadIdx.x; x < M; x += blockDim.x) {
      B.grank[c.W.g0 + moved[x]] = M - 1 - x;
      flag[moved[x]] = 1;
    }
    __syncthreads();
    int r = M;
    for (int k0 = 0; k0 < ng; k0 += blockDim.x) {
      const int k = k0 + threadIdx.x;
      const int g = k < ng ? inv[k] : -1;
      const int keep = (g >= 0 && !flag[g]) ? 1 : 0;
      int tot;
      const int off = block_excl_scan(keep, tot, sh);
      if (keep) B.grank[c.W.g0 + g] = r + off;
      r += tot;
    }
  }
  if (threadIdx.x == 0) {
    B.counters[c.w * CNT_N + CNT_ROWS] = nrows;
    B.counters[c.w * CNT_N + CNT_GROUPS] = ngroups;
  }
  __syncthreads();
  // a world whose state became non-finite is frozen (and reported) from now on
  if (threadIdx.x == 0 && sh.ival[13]) {
    P.dead = 1;
    raise_overflow(B, c.w, OVF_NONFINITE);
  }
  c.clk.lap(PH_INTEGRATE);
}

// joint controls (steer stops, wheel torques) at the start of a step
__device__ void phase_controls(const DevBatch &B, const Ctx &c) {
  if (!B.ctrl) return;
  if (threadIdx.x == 0) {
    for (int i = 0; i < c.W.nj; i++) {
      JointDev &j = B.joints[c.W.j0 + i];
      float4 u = B.ctrl[c.W.j0 + i];
      if (!isnan(u.x)) j.lm1.lostop = u.x;
      if (!isnan(u.y)) j.lm1.histop = u.y;
      if (j.type == JT_HINGE2 && (u.z != 0.f || u.w != 0.f) && j.b1 >= 0 && j.b2 >= 0) {
        // dJointAddHinge2Torques (hinge2.cpp:393-410)
        int g1 = c.W.b0 + j.b1, g2 = c.W.b0 + j.b2;
        float3 a1 = load_mat(B.R + 3 * (size_t)g1).mul(mk3(j.axis1[0], j.axis1[1], j.axis1[2]));
        float3 a2 = load_mat(B.R + 3 * (size_t)g2).mul(mk3(j.axis2[0], j.axis2[1], j.axis2[2]));
        float3 t = u.z * a1 + u.w * a2;
        float4 t1 = B.tacc[g1], t2 = B.tacc[g2];
        t1.x += t.x; t1.y += t.y; t1.z += t.z;
        t2.x -= t.x; t2.y -= t.y; t2.z -= t.z;
        B.tacc[g1] = t1;
        B.tacc[g2] = t2;
      }
    }
  }
  __syncthreads();
}

// ------------------------------------------------------------------ kernels

// Kernel modes (bit set): COLLIDE runs AABBs, broadphase and narrowphase;
// STEP runs the quickstep.  API_OUT hands pairs and contacts of one world to
// the host (dSpaceCollide); HOST_CONTACTS steps with contact joints the host
// created (dWorldQuickStep).  Batch steps run COLLIDE|STEP in one kernel, or
// COLLIDE then STEP as two kernels with the contact count passed through
// the world's counters.
// TOL: the coloured solver honours the world's residual tolerance (its own
// instantiation, so the iterate-to-tolerance step is a separate kernel).
enum { MF_COLLIDE = 1, MF_STEP = 2, MF_API_OUT = 4, MF_HOST_CONTACTS = 8, MF_TOL = 16, MF_PRE = 32, MF_POST = 64 };
enum {
  MODE_BATCH_COLLIDE = MF_COLLIDE,
  MODE_BATCH_STEP = MF_STEP,
  MODE_FUSED = MF_COLLIDE | MF_STEP,
  MODE_API_COLLIDE = MF_COLLIDE | MF_API_OUT,
  MODE_API_STEP = MF_STEP | MF_HOST_CONTACTS,
  MODE_BATCH_STEP_TOL = MF_STEP | MF_TOL,
  MODE_FUSED_TOL = MF_COLLIDE | MF_STEP | MF_TOL,
  MODE_FUSED_PRE = MF_COLLIDE | MF_STEP | MF_TOL | MF_PRE,   // collide and step up to the solver set-up
  MODE_POST = MF_STEP | MF_TOL | MF_POST,                    // the step after the sweeps
  KM_SOR = 1000                                               // the sweeps (sor_kernel)
};

template <int MODE>
__device__ __attribute__((always_inline)) void run_world(const DevBatch &B, int w, Shared &sh, int api_maxc) {
  Ctx c;
  c.w = w;
  c.W = B.wi[w];
  c.L = scratch_layout(c.W.nb, c.W.ng, c.W.nj, c.W.pcap, c.W.kcap, c.W.rcap);
  c.S = B.scratch + c.W.scratch;
  c.clk.start(B, w);
  WorldParams &P = B.wp[w];
  const bool ref = B.order_mode == ORDER_REFERENCE;
  constexpr bool api = (MODE & (MF_API_OUT | MF_HOST_CONTACTS)) != 0;
  if (!api && P.dead) {
    // frozen after its state became non-finite
    if (threadIdx.x == 0) B.counters[w * CNT_N + CNT_OVERFLOW] = OVF_NONFINITE;
    return;
  }
  // the first kernel of a step clears the overflow flags
  if (((MODE & MF_COLLIDE) || api) && threadIdx.x == 0) B.counters[w * CNT_N + CNT_OVERFLOW] = 0;
  if ((MODE & MF_COLLIDE) && !api) phase_controls(B, c);
  int nk = 0;
  if (MODE & MF_COLLIDE) {
    phase_aabb(B, c, P, sh);
    c.clk.lap(PH_AABB);
    int np = phase_broadphase(B, c, P, sh, ref);
    c.clk.lap(PH_BROAD);
    int maxc = api ? api_maxc : P.max_contacts;
    nk = phase_narrowphase(B, c, P, np, sh, maxc, !api);
    c.clk.lap(PH_NARROW);
    if (threadIdx.x == 0) {
      B.counters[w * CNT_N + CNT_PAIRS] = np;
      B.counters[w * CNT_N + CNT_CONTACTS] = nk;
    }
    if (MODE & MF_API_OUT) {
      // hand pairs and contacts to the host (one world per launch)
      const PairRec *pr = c.at<PairRec>(c.L.pairs);
      const int *pc = c.at<int>(c.L.pcount);
      const ContactRec *cr = c.at<ContactRec>(c.L.contacts);
      for (int i = threadIdx.x; i < np; i += blockDim.x) {
        B.pairs_out[i] = pr[i];
        B.pcount_out[i] = pc[i];
      }
      for (int i = threadIdx.x; i < nk; i += blockDim.x) B.contacts_out[i] = cr[i];
    }
  }
  if (MODE & MF_STEP) {
    StepIn in;
    in.from_host = (MODE & MF_HOST_CONTACTS) != 0;
    if (in.from_host) in.nk = B.cin_count[w];
    else if (MODE & MF_COLLIDE) in.nk = nk;
    else in.nk = B.counters[w * CNT_N + CNT_CONTACTS];
    in.seq_base = 1 << 20;
    if (in.from_host && in.nk > c.W.kcap) {
      if (threadIdx.x == 0) raise_overflow(B, w, OVF_CONTACTS);
      in.nk = c.W.kcap;
    }
    phase_step<(MODE & MF_TOL) != 0, (MODE & MF_PRE) ? 1 : ((MODE & MF_POST) ? 2 : 0)>(B, c, P, in, sh, ref);
  }
  __syncthreads();
}

// Two wavefronts per SIMD: the phases of a step are chains of dependent
// accesses, and without the bound the kernel takes 284 registers, which leaves
// each SIMD one wavefront (a CU one workgroup of 256).  Measured (20 sweeps):
// 8192 cars 19.5 -> 10.7 ms, 300 mixed worlds 1.92 -> 1.42 ms, 333 uneven
// worlds 2.05 -> 1.46 ms.  Four (128 registers) spill in the solvers: 15 %
// slower on the uneven worlds.
template <int MODE>
__global__ __launch_bounds__(WG, 2) void world_kernel(DevBatch B, int first_world, int persistent, int api_maxc) {
  __shared__ Shared sh;
  if (!persistent) {
    int w = first_world + blockIdx.x;
    if (w < B.nworlds) run_world<MODE>(B, B.world_order ? B.world_order[w] : w, sh, api_maxc);
    return;
  }
  // persistent: workgroups pull worlds (largest first) from a queue
  while (true) {
    if (threadIdx.x == 0) sh.ival[15] = atomicAdd(B.work_counter, 1);
    __syncthreads();
    int k = sh.ival[15];
    __syncthreads();
    if (k >= B.nworlds) break;
    run_world<MODE>(B, B.world_order ? B.world_order[k] : k, sh, api_maxc);
  }
}

// The coloured solver's sweeps of every world (between MODE_FUSED_PRE and
// MODE_POST): a lean kernel, so that many workgroups fit on a CU.
template <bool TOL>
__device__ void sor_world(const DevBatch &B, int w, Shared &sh) {
  const WorldParams &P = B.wp[w];
  if (P.dead) return;
  Ctx c;
  c.w = w;
  c.W = B.wi[w];
  c.L = scratch_layout(c.W.nb, c.W.ng, c.W.nj, c.W.pcap, c.W.kcap, c.W.rcap);
  c.S = B.scratch + c.W.scratch;
  const int *misc = c.at<int>(c.L.misc);
  if (misc[MISC_SOR_READY] == 0) return;
  const int nrows = misc[MISC_SOR_ROWS], ngroups = misc[MISC_SOR_GROUPS];
  const int nact = c.at<int>(c.L.island)[ngroups];
  const bool accel = TOL && P.tol > 0.f && P.accel != 0;
  // a world whose working set does not fit the pool is solved by the
  // integration kernel, in global scratch
  if (sor_lds_bytes(c.W.nb, nrows, nact, ngroups, accel) > B.lds_bytes) return;
  c.clk.start(B, w);
  sor_solve_any<TOL>(B, c, P, nrows, ngroups, nact, false, B.lds_bytes, sh);
  c.clk.lap(PH_SOR);
}

template <bool TOL>
__global__ __launch_bounds__(WG, 2) void sor_kernel(DevBatch B, int first_world, int persistent) {
  __shared__ Shared sh;
  if (!persistent) {
    int w = first_world + blockIdx.x;
    if (w < B.nworlds) sor_world<TOL>(B, B.world_order ? B.world_order[w] : w, sh);
    return;
  }
  while (true) {
    if (threadIdx.x == 0) sh.ival[15] = atomicAdd(B.work_counter, 1);
    __syncthreads();
    int k = sh.ival[15];
    __syncthreads();
    if (k >= B.nworlds) break;
    sor_world<TOL>(B, B.world_order ? B.world_order[k] : k, sh);
  }
}

__global__ void reset_counter_kernel(int *ctr) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *ctr = 0;
}

// Processing order of the persistent queue by expected cost, most expensive
// first, ties in the static order (largest first, `rank`).  The estimate of
// a world (est, kept per world) is the larger of its last step's rows times
// solver sweeps and 3/4 of its previous estimate: a tolerance solve that
// ended at the sweep cap far from the tolerance starts the next one cold,
// which may then converge quickly, so a world's cost alternates and the
// last step alone predicts the next one badly; plus bodies and geoms,
// which is all the first step has.  One workgroup; a bitonic sort of
// n <= 8192 64-bit keys (cost << 32 | position from the end of the static
// order) in the dynamic LDS (8 bytes per key, n rounded up to a power of two).
__global__ __launch_bounds__(1024) void order_worlds_kernel(DevBatch B, const int *rank, float *est, int n) {
  extern __shared__ unsigned long long okey[];
  int N = 1;
  while (N < n) N <<= 1;
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
    unsigned long long k = 0;   // padding sorts last
    if (i < n) {
      const int w = rank[i];
      const int *cnt = B.counters + (size_t)w * CNT_N;
      const float work = (float)max(cnt[CNT_ROWS], 0) * (float)max(cnt[CNT_ITERS], 1);
      const float e = fmaxf(work, 0.75f * est[w]);
      est[w] = e;
      const float c = e + (float)(B.wi[w].nb + B.wi[w].ng);
      const unsigned long long cost = c < 4.0e9f ? (unsigned long long)c : 0xffffffffull;
      k = (cost << 32) | (unsigned long long)(unsigned)(N - 1 - i);
    }
    okey[i] = k;
  }
  // descending bitonic sort
  for (int size = 2; size <= N; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      __syncthreads();
      for (int i = threadIdx.x; i < (N >> 1); i += blockDim.x) {
        const int lo = 2 * i - (i & (stride - 1)), hi = lo + stride;
        const bool desc = (lo & size) == 0;
        const unsigned long long a = okey[lo], b = okey[hi];
        if ((a < b) == desc) {
          okey[lo] = b;
          okey[hi] = a;
        }
      }
    }
  __syncthreads();
  int *order = const_cast<int *>(B.world_order);
  for (int k = threadIdx.x; k < n; k += blockDim.x) order[k] = rank[N - 1 - (int)(okey[k] & 0xffffffffull)];
}

hipError_t launch_order_worlds(const DevBatch &B, const int *rank, float *est, hipStream_t st) {
  const int n = B.nworlds;
  if (n < 2) return hipSuccess;
  if (n > 8192) return hipErrorInvalidValue;
  int N = 1;
  while (N < n) N <<= 1;
  order_worlds_kernel<<<1, 1024, sizeof(unsigned long long) * (size_t)N, st>>>(B, rank, est, n);
  return hipGetLastError();
}

// one dCollide call on the device (ODE API path outside a cached batch)
__global__ void collide_one_kernel(GeomView a, GeomView b, int maxc, CPoint *out, int *n) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    CPoint pts[MAX_SLOTS];
    int k = collide_pair(a, b, maxc > MAX_SLOTS ? MAX_SLOTS : maxc, pts);
    for (int i = 0; i < k; i++) out[i] = pts[i];
    *n = k;
  }
}

// the narrowphase of a list of geom pairs, one pair per lane (the
// geom-geom pairs dSpaceCollide2 reports): out holds MAX_SLOTS contacts per
// pair, n the count of each
__global__ void collide_list_kernel(const GeomView *a, const GeomView *b, int npairs, int maxc, CPoint *out,
                                    int *n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npairs) return;
  CPoint pts[MAX_SLOTS];
  const int k = collide_pair(a[i], b[i], maxc > MAX_SLOTS ? MAX_SLOTS : maxc, pts);
  for (int j = 0; j < k; j++) out[(size_t)MAX_SLOTS * i + j] = pts[j];
  n[i] = k;
}

// body-frame setup: inverse inertia is computed on the host; here the
// rotation matrices are derived from the quaternions
__global__ void init_rot_kernel(DevBatch B, int nbodies) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < nbodies) store_mat(B.R + 3 * (size_t)b, quat_to_mat(B.q[b]));
}

}  // namespace odemi

// ------------------------------------------------------------------ launch API
namespace odemi {

int world_kernel_static_lds() { return (int)sizeof(Shared); }

template <int MODE>
static const void *world_kernel_fn() { return (const void *)world_kernel<MODE>; }

static const void *kernel_of(int mode) {
  switch (mode) {
    case MODE_BATCH_COLLIDE: return world_kernel_fn<MODE_BATCH_COLLIDE>();
    case MODE_BATCH_STEP: return world_kernel_fn<MODE_BATCH_STEP>();
    case MODE_FUSED: return world_kernel_fn<MODE_FUSED>();
    case MODE_API_COLLIDE: return world_kernel_fn<MODE_API_COLLIDE>();
    case MODE_API_STEP: return world_kernel_fn<MODE_API_STEP>();
    case MODE_BATCH_STEP_TOL: return world_kernel_fn<MODE_BATCH_STEP_TOL>();
    case MODE_FUSED_TOL: return world_kernel_fn<MODE_FUSED_TOL>();
    case MODE_FUSED_PRE: return world_kernel_fn<MODE_FUSED_PRE>();
    case MODE_POST: return world_kernel_fn<MODE_POST>();
    case KM_SOR: return (const void *)sor_kernel<true>;
    default: return nullptr;
  }
}

hipError_t allow_world_kernel_lds(int bytes) {
  const int modes[] = {MODE_BATCH_COLLIDE, MODE_BATCH_STEP, MODE_FUSED, MODE_API_COLLIDE, MODE_API_STEP,
                       MODE_BATCH_STEP_TOL, MODE_FUSED_TOL, MODE_FUSED_PRE, MODE_POST, KM_SOR};
  for (int m : modes) {
    hipError_t e = hipFuncSetAttribute(kernel_of(m), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

int world_kernel_occupancy(int mode, int wg, int lds_bytes) {
  int n = 0;
  const void *f = kernel_of(mode);
  if (!f) return 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, f, wg, (size_t)lds_bytes) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return n;
}

// queue: which of the batch's work counters a persistent launch pulls from
// (kernels of one step use different counters)
hipError_t launch_world_kernel(int mode, const DevBatch &B0, int first_world, int nworlds_launch, int grid,
                               int wg, int api_maxc, hipStream_t st, int queue) {
  int persistent = grid > 0 ? 1 : 0;
  int blocks = persistent ? grid : nworlds_launch;
  if (blocks <= 0) return hipSuccess;
  if (wg > WG || wg < 64 || (wg & 63)) return hipErrorInvalidValue;
  if (B0.lds_bytes < 0 || (B0.lds_bytes & 15)) return hipErrorInvalidValue;
  if (queue < 0 || queue >= WORK_QUEUES) return hipErrorInvalidValue;
  DevBatch B = B0;
  if (persistent) {
    B.work_counter += 16 * queue;
    reset_counter_kernel<<<1, 64, 0, st>>>(B.work_counter);
  }
  size_t lds = (size_t)B.lds_bytes;
  switch (mode) {
    case MODE_BATCH_COLLIDE:
      world_kernel<MODE_BATCH_COLLIDE><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc);
      break;
    case MODE_BATCH_STEP:
      world_kernel<MODE_BATCH_STEP><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc);
      break;
    case MODE_FUSED: world_kernel<MODE_FUSED><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc); break;
    case MODE_API_COLLIDE:
      world_kernel<MODE_API_COLLIDE><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc);
      break;
    case MODE_API_STEP:
      world_kernel<MODE_API_STEP><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc);
      break;
    case MODE_BATCH_STEP_TOL:
      world_kernel<MODE_BATCH_STEP_TOL><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc);
      break;
    case MODE_FUSED_TOL:
      world_kernel<MODE_FUSED_TOL><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc);
      break;
    case MODE_FUSED_PRE:
      world_kernel<MODE_FUSED_PRE><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc);
      break;
    case MODE_POST: world_kernel<MODE_POST><<<blocks, wg, lds, st>>>(B, first_world, persistent, api_maxc); break;
    case KM_SOR: sor_kernel<true><<<blocks, wg, lds, st>>>(B, first_world, persistent); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_collide_list(const GeomView *a, const GeomView *b, int npairs, int maxc, CPoint *out, int *n,
                               hipStream_t st) {
  if (npairs <= 0) return hipSuccess;
  collide_list_kernel<<<(npairs + 63) / 64, 64, 0, st>>>(a, b, npairs, maxc, out, n);
  return hipGetLastError();
}

hipError_t launch_collide_one(const GeomView &a, const GeomView &b, int maxc, CPoint *out, int *n, hipStream_t st) {
  collide_one_kernel<<<1, 64, 0, st>>>(a, b, maxc, out, n);
  return hipGetLastError();
}

hipError_t launch_init_rot(const DevBatch &B, int nbodies, hipStream_t st) {
  if (nbodies <= 0) return hipSuccess;
  init_rot_kernel<<<(nbodies + 255) / 256, 256, 0, st>>>(B, nbodies);
  return hipGetLastError();
}

}  // namespace odemi
