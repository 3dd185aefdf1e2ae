// mcx_normals.hip -- per-vertex surface normals for gfx950.
//
// Replaces d_voxel_extract_surface_normals / _d_voxel_extract_surface_normal
// (cu_kinect_fusion_v1.cu:3146-3238): p_f = ver_pos / grid_s (without the
// +0.5 shift, as the reference, :3241), p_i = (int)p_f, the 2x2x2 corner
// tsdf values at p_i; the normal is zero if any of them is +-32766
// (CU_VOXEL_MAX_TSDF); else the x/y/z differences of bilinear interpolations
// over the two opposite faces (:3201-3218), normalised when the norm exceeds
// FLT_EPSILON (float3_unit, cu_vector_functions.h:258-264).  Where p_i + 1
// leaves the volume (the reference reads out of bounds) the normal is zero.
// One thread per vertex; positions are read with a stride so vertex_voxel
// records (7 words) and packed float3 arrays (3 words) both work.  Its eight
// corners are four pairs along x, one 64-bit load each, and its 14 divisions
// and square root take the exact short forms where their arguments allow it
// (else IEEE, the same bits): 2.1 M vertex records of a fused volume take 21.6
// us, of which 16 are their bytes at the copy rate, and took 24.5 with eight
// loads and IEEE forms throughout.
#include <algorithm>
#include <float.h>
#include <hip/hip_runtime.h>

#include "mcx_internal.h"

namespace mcx {
namespace {

__device__ __forceinline__ float bilinear(float v0, float v1, float v2, float v3, float x, float y) {
  const float a = 1.0f - x, b = 1.0f - y;
  return v0 * a * b + v1 * x * b + v2 * a * y + v3 * x * y;
}

typedef uint32_t u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));  // 4-byte aligned

constexpr float kFormMin = 0x1p-60f, kFormMax = 0x1p60f;  // what div_rn takes

// In range for div_rn and not zero (a quotient of -0 keeps its sign in IEEE).
__device__ __forceinline__ bool form_ok(float a) {
  return fabsf(a) >= kFormMin && fabsf(a) <= kFormMax;
}

__global__ __launch_bounds__(256) void normals_kernel(const uint32_t* __restrict__ vol, int X, int Y,
                                                      int Z, float h, const float* __restrict__ pos,
                                                      int64_t stride, int64_t n, float* out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float pf[3], t[3];
  int pi[3];
  const float p0 = pos[i * stride], p1 = pos[i * stride + 1], p2 = pos[i * stride + 2];
  if (form_ok(h) && form_ok(p0) && form_ok(p1) && form_ok(p2)) {
    const float r = recip_rn(h);
    pf[0] = div_rn(p0, h, r);
    pf[1] = div_rn(p1, h, r);
    pf[2] = div_rn(p2, h, r);
  } else {
    pf[0] = p0 / h;
    pf[1] = p1 / h;
    pf[2] = p2 / h;
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    pi[d] = (int)pf[d];
    t[d] = pf[d] - (float)pi[d];
  }
  float nx = 0.f, ny = 0.f, nz = 0.f;
  const bool inb = pf[0] >= 0.f && pf[1] >= 0.f && pf[2] >= 0.f && pi[0] + 1 < X && pi[1] + 1 < Y &&
                   pi[2] + 1 < Z;
  if (inb) {
    const int64_t XY = (int64_t)X * Y;
    const uint32_t* c = vol + (((int64_t)pi[2] * Y + pi[1]) * X + pi[0]);
    const u32x2a4 w00 = *reinterpret_cast<const u32x2a4*>(c);
    const u32x2a4 w10 = *reinterpret_cast<const u32x2a4*>(c + X);
    const u32x2a4 w01 = *reinterpret_cast<const u32x2a4*>(c + XY);
    const u32x2a4 w11 = *reinterpret_cast<const u32x2a4*>(c + XY + X);
    const uint32_t all[8] = {w00.x, w00.y, w10.x, w10.y, w01.x, w01.y, w11.x, w11.y};
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int16_t v = (int16_t)(all[k] & 0xffffu);
      bad = bad || v == 32766 || v == -32766;
    }
    if (!bad) {
      auto f = [](uint32_t w) { return tsdf_unit((int16_t)(w & 0xffffu)); };
      // reference slots: 0 V000, 1 V100, 2 V010, 3 V001, 4 V101, 5 V011, 6 V110, 7 V111
      const float s0 = f(w00.x), s1 = f(w00.y), s2 = f(w10.x), s3 = f(w01.x);
      const float s4 = f(w01.y), s5 = f(w11.x), s6 = f(w10.y), s7 = f(w11.y);
      nx = bilinear(s1, s6, s4, s7, t[1], t[2]) - bilinear(s0, s2, s3, s5, t[1], t[2]);
      ny = bilinear(s2, s6, s5, s7, t[0], t[2]) - bilinear(s0, s1, s3, s4, t[0], t[2]);
      nz = bilinear(s3, s4, s5, s7, t[0], t[1]) - bilinear(s0, s1, s2, s6, t[0], t[1]);
      const float sq = nx * nx + ny * ny + nz * nz;
      // below 2^-50 the norm is under 2^-25, and FLT_EPSILON is 2^-23
      if (sq >= 0x1p-50f) {
        const float nn = sqrt_rn(sq);
        if (nn > FLT_EPSILON) {
          if (form_ok(nx) && form_ok(ny) && form_ok(nz)) {
            const float r = recip_rn(nn);
            nx = div_rn(nx, nn, r);
            ny = div_rn(ny, nn, r);
            nz = div_rn(nz, nn, r);
          } else {
            nx = nx / nn;
            ny = ny / nn;
            nz = nz / nn;
          }
        }
      }
    }
  }
  out[3 * i + 0] = nx;
  out[3 * i + 1] = ny;
  out[3 * i + 2] = nz;
}

}  // namespace
}  // namespace mcx

using namespace mcx;

extern "C" int mcx_normals(const void* d_vol, int X, int Y, int Z, float h, const float* d_pos,
                           int64_t stride_floats, int64_t n, float* d_normals, void* stream) {
  if (!d_vol || X < 1 || Y < 1 || Z < 1 || n < 0 || stride_floats < 3) return MCX_ERR_ARG;
  if (n == 0) return MCX_OK;
  if (!d_pos || !d_normals) return MCX_ERR_ARG;
  // a thread per vertex, in launches of at most kMaxLaunchBlocks workgroups
  const int64_t per = kMaxLaunchBlocks * 256;
  for (int64_t v0 = 0; v0 < n; v0 += per) {
    const int64_t nn = std::min(per, n - v0);
    hipLaunchKernelGGL(normals_kernel, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0,
                       as_stream(stream), static_cast<const uint32_t*>(d_vol), X, Y, Z, h,
                       d_pos + v0 * stride_floats, stride_floats, nn, d_normals + v0 * 3);
    MCX_HIP(hipGetLastError());
  }
  return MCX_OK;
}
