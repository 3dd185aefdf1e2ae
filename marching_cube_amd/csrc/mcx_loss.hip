// mcx_loss.hip -- a Chamfer-style vertex loss over a batch of meshes (no
// counterpart in the reference; the loss of the differentiable fusion pass).
//
// Vertices of volume b are [vbase[b], vbase[b+1]) of one concatenated float3
// array; volume b has M target points.  Per vertex: its nearest target t*
// (squared distance from explicit differences, fma(dz, dz, fma(dy, dy,
// dx * dx)), the first index of the minimum), its loss |p - t*|^2 and its gradient
// 2 (p - t*).  Per volume: the sum of its vertices' losses in a fixed order
// (each thread of a workgroup sums a fixed stride, then a fixed tree), so
// the result does not depend on scheduling.
#include <hip/hip_runtime.h>

#include "mcx_internal.h"

namespace mcx {
namespace {

constexpr int kMaxTargets = 1024;  // targets staged in LDS per workgroup

// Volume of vertex v: the last b with vbase[b] <= v (vbase ascending).
__device__ __forceinline__ int volume_of_vertex(const int64_t* vbase, int nvol, int64_t v) {
  int lo = 0, hi = nvol - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (vbase[mid] <= v) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// The first nearest of M targets (at(m): target m) to p, and its distance squared.
template <class At>
__device__ __forceinline__ float nearest(const float (&p)[3], int M, At at, int* j) {
  float best = __builtin_inff();
  *j = 0;
#pragma unroll 4
  for (int m = 0; m < M; ++m) {
    const float4 t = at(m);
    const float dx = p[0] - t.x, dy = p[1] - t.y, dz = p[2] - t.z;
    const float d2 = __fmaf_rn(dz, dz, __fmaf_rn(dy, dy, dx * dx));
    if (d2 < best) {
      best = d2;
      *j = m;
    }
  }
  return best;
}

// One thread per vertex row (rows past the total or past cap: gradient 0; a wave
// of only such rows looks at no target: 2 M rows without a vertex, 1024 targets,
// 9 us, and 348 where it did).  The targets of the volume of the workgroup's first
// vertex are staged in LDS, one 16-byte read of all lanes for each; a wave with a
// vertex of another volume (a workgroup spanning a boundary) reads targets from
// memory.  Bound by the arithmetic (9 instructions a row and target) and by what
// a row reads and writes.  Loss and sum: 64 volumes, 0.9 M rows, 64 targets 24 us
// (98 with three reads a target through a pointer that could be either, as with
// two rows a thread); 4 volumes, 30,000 rows 9.2 us, 300, 0.1 M rows, 1024 targets
// 49 (12.1 and 89 with two rows, on half the waves).
__global__ __launch_bounds__(256) void chamfer_vertex_kernel(const float* pos,
                                                             const int64_t* vbase, int nvol,
                                                             const float* targets, int M,
                                                             int64_t cap, float* gpos,
                                                             float* vloss) {
  __shared__ float4 s_t[kMaxTargets];
  __shared__ int s_b0;
  const int64_t v0 = (int64_t)blockIdx.x * 256;
  const int64_t total = vbase[nvol];
  if (threadIdx.x == 0) s_b0 = v0 < total ? volume_of_vertex(vbase, nvol, v0) : 0;
  __syncthreads();
  const int b0 = s_b0;
  if (v0 < total) {
    const float* t = targets + (int64_t)b0 * M * 3;
    for (int i = threadIdx.x; i < M; i += 256)
      s_t[i] = make_float4(t[3 * i], t[3 * i + 1], t[3 * i + 2], 0.0f);
  }
  __syncthreads();
  const int64_t live = min(total, cap), v = v0 + threadIdx.x;
  const bool row = v < live;
  float p[3] = {0.0f, 0.0f, 0.0f}, best = 0.0f;
  int j = 0, b = b0;
  if (__any(row)) {
    if (row) {
      p[0] = pos[3 * v];
      p[1] = pos[3 * v + 1];
      p[2] = pos[3 * v + 2];
    }
    if (__all(!row || v < vbase[b0 + 1])) {
      best = nearest(p, M, [&](int m) { return s_t[m]; }, &j);
    } else {
      if (row) b = volume_of_vertex(vbase, nvol, v);
      const float* t = targets + (int64_t)b * M * 3;
      best = nearest(
          p, M, [&](int m) { return make_float4(t[3 * m], t[3 * m + 1], t[3 * m + 2], 0.0f); }, &j);
    }
  }
  if (v >= cap) return;
  float g[3] = {0.0f, 0.0f, 0.0f};
  if (row) {
    const float* t = targets + ((int64_t)b * M + j) * 3;
#pragma unroll
    for (int c = 0; c < 3; ++c) g[c] = 2.0f * (p[c] - t[c]);
    vloss[v] = best;
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) gpos[3 * v + c] = g[c];
}

// One workgroup per volume: the sum of its vertex losses (vertices below cap).
// A thread's sum is serial; its loads go out eight at a time, ahead of it (the
// same batch: 68 us with one at a time, now 15).
__global__ __launch_bounds__(256) void chamfer_sum_kernel(const float* vloss,
                                                          const int64_t* vbase, int64_t cap,
                                                          float* loss) {
  __shared__ float s_sum[256];
  const int b = blockIdx.x;
  const int64_t lo = vbase[b], hi = min(vbase[b + 1], cap);
  float acc = 0.0f;
  int64_t v = lo + threadIdx.x;
  for (; v + 7 * 256 < hi; v += 8 * 256) {
    float x[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) x[k] = vloss[v + k * 256];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc += x[k];
  }
  for (; v < hi; v += 256) acc += vloss[v];
  s_sum[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s_sum[threadIdx.x] += s_sum[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[b] = s_sum[0];
}

}  // namespace
}  // namespace mcx

using namespace mcx;

extern "C" size_t mcx_chamfer_workspace_size(int64_t cap) {
  return cap > 0 ? (size_t)cap * sizeof(float) : 0;
}

extern "C" int mcx_chamfer_batched(const float* d_pos, const int64_t* d_vbase, int nvol,
                                   const float* d_targets, int M, int64_t cap, float* d_loss,
                                   float* d_grad_pos, void* d_ws, size_t ws_bytes,
                                   void* stream) {
  if (!d_pos || !d_vbase || nvol < 1 || !d_targets || M < 1 || cap < 1 || !d_loss ||
      !d_grad_pos)
    return MCX_ERR_ARG;
  if (M > kMaxTargets) return MCX_ERR_UNSUPPORTED;
  if (!d_ws || ws_bytes < mcx_chamfer_workspace_size(cap)) return MCX_ERR_WORKSPACE;
  hipStream_t s = as_stream(stream);
  float* vloss = static_cast<float*>(d_ws);
  if (cap > kMaxLaunchBlocks * 256) return MCX_ERR_UNSUPPORTED;
  const int64_t blocks = (cap + 255) / 256;
  hipLaunchKernelGGL(chamfer_vertex_kernel, dim3((unsigned)blocks), dim3(256), 0, s, d_pos,
                     d_vbase, nvol, d_targets, M, cap, d_grad_pos, vloss);
  MCX_HIP(hipGetLastError());
  hipLaunchKernelGGL(chamfer_sum_kernel, dim3((unsigned)nvol), dim3(256), 0, s, vloss, d_vbase,
                     cap, d_loss);
  MCX_HIP(hipGetLastError());
  return MCX_OK;
}
