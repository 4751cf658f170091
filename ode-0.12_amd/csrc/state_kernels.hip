// state_kernels.hip -- the host's view of the state: 13 floats per body (pos
// 3, q 4, lvel 3, avel 3), written from and into the device's float4 arrays.
//
// A copy between device and pageable host memory costs 20 to 30 us whatever
// its size, and the host rearranging 13 of 16 floats per body costs more than
// moving them.  So one kernel reads or writes pinned host memory itself, and
// the host copies that to or from the caller's array: no copy on the device
// queue at all, where there were four.
#include <hip/hip_runtime.h>

#include "devmath.hpp"
#include "layout.hpp"

namespace odemi {

// float k (0..12) of body i
__device__ inline float state_float(const float4 *x, const float4 *q, const float4 *v, const float4 *w, int i, int k) {
  if (k < 3) return ((const float *)(x + i))[k];
  if (k < 7) return ((const float *)(q + i))[k - 3];
  return k < 10 ? ((const float *)(v + i))[k - 7] : ((const float *)(w + i))[k - 10];
}

__global__ void pack_state_kernel(const float4 *x, const float4 *q, const float4 *v, const float4 *w, int n,
                                  float *out) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 13LL * n) return;
  const int i = (int)(e / 13);
  out[e] = state_float(x, q, v, w, i, (int)(e - 13LL * i));
}

// R: the bodies' rotations from their quaternions (null: gradients, which
// have none)
__global__ void unpack_state_kernel(const float *in, int n, float4 *x, float4 *q, float4 *v, float4 *w, float4 *R) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float *r = in + 13 * (size_t)i;
  const float4 qi = make_float4(r[3], r[4], r[5], r[6]);
  x[i] = make_float4(r[0], r[1], r[2], 0.f);
  q[i] = qi;
  v[i] = make_float4(r[7], r[8], r[9], 0.f);
  w[i] = make_float4(r[10], r[11], r[12], 0.f);
  if (R) store_mat(R + 3 * (size_t)i, quat_to_mat(qi));
}

// after a new state: frozen worlds revive, and the previous impulses belong
// to the old one (the next solve starts from zero)
__global__ void revive_kernel(WorldParams *wp, int *warm_n, int nworlds) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= nworlds) return;
  wp[w].dead = 0;
  warm_n[w] = -1;
}

// what the ODE API reads after a step of its world: counters (CNT_N ints),
// generator state, geom ranks (ng ints), then the state
__global__ void api_gather_kernel(DevBatch B, int nb, int ng, int *out) {
  const int n = CNT_N + 1 + ng;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n + 13 * nb; e += gridDim.x * blockDim.x) {
    if (e < CNT_N) out[e] = B.counters[e];
    else if (e == CNT_N) out[e] = (int)B.wp[0].seed;
    else if (e < n) out[e] = B.grank[e - CNT_N - 1];
    else {
      const int i = (e - n) / 13;
      out[e] = __float_as_int(state_float(B.pos, B.q, B.lvel, B.avel, i, e - n - 13 * i));
    }
  }
}

hipError_t launch_pack_state(const float4 *const a[4], int n, float *out, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  pack_state_kernel<<<(unsigned)((13LL * n + 255) / 256), 256, 0, st>>>(a[0], a[1], a[2], a[3], n, out);
  return hipGetLastError();
}

hipError_t launch_unpack_state(const float *in, int n, float4 *const a[4], float4 *R, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  unpack_state_kernel<<<(n + 255) / 256, 256, 0, st>>>(in, n, a[0], a[1], a[2], a[3], R);
  return hipGetLastError();
}

hipError_t launch_revive(WorldParams *wp, int *warm_n, int nworlds, hipStream_t st) {
  if (nworlds <= 0) return hipSuccess;
  revive_kernel<<<(nworlds + 255) / 256, 256, 0, st>>>(wp, warm_n, nworlds);
  return hipGetLastError();
}

hipError_t launch_api_gather(const DevBatch &B, int nb, int ng, int *out, hipStream_t st) {
  const int n = CNT_N + 1 + ng + 13 * nb;
  const int blocks = (n + 255) / 256;
  api_gather_kernel<<<blocks < 256 ? blocks : 256, 256, 0, st>>>(B, nb, ng, out);
  return hipGetLastError();
}

}  // namespace odemi
