// mcx_raycast.hip -- depth and normal maps ray-marched through a packed short2
// TSDF volume (gfx950).
//
// Replaces _cu_voxel_extract_depth_and_normal_map (cu_kinect_fusion_v1.cu:972-986)
// and its kernel d_voxel_extract_depth_and_normal_map (:786-970) with the
// samplers d_voxel_extract_trilinear_interpolated_sdf (:551-659) and
// _d_voxel_extract_surface_normal (:697-776).  Per pixel:
//   ray   = unit(IM (x, y, 1)), IM = (K R^T)^-1 (host, cofactors / det),
//           zero components replaced by 1e-15;
//   t range from the six planes at 1 and size-1 (t_min = 1 when one plane is
//           crossed); march t += 1, or 0.25 inside the band |sdf| < 1 (one
//           step back on entering it), samples outside [0, size-1) skipped;
//   hit   sdf1 in [0, 1) then sdf in (-1, 0): t2 = t1 - dt sdf1 / (sdf - sdf1),
//           z-depth |ray t2| / |(K^-1 (x, y, 1))| * h, normal R^T unit(grad);
//   back face  sdf1 in (-1, 0] then sdf in [0, 1): the ray ends, no hit.
// The trilinear sample returns +-1 at the first corner (V000 V100 V010 V001
// V101 V011 V110 V111) holding +-32766; the normal is 0 if any corner does.
// Two guards the reference lacks end every ray: t past the last parameter at
// which the ray can lie in the volume grown by one voxel (all later samples
// would be skipped), and 2^20 steps.
//
// Layout: LANES lanes take a ray and its next LANES samples at once; a wave
// holds 64 / LANES pixels, an XCD the waves of 16 x 16 pixels in a row.  Each
// sample reads its eight corner words as four x-neighbour pairs (one 64-bit load
// each).  With a ray to a lane the march is as slow as its slowest waves: a ray
// along a surface takes hundreds of fine steps, some 1500 cycles each, one after
// the other (640x480 rays through 512^3: 1.28 ms, of which most waves ran 0.3).
// Eight samples a step cut that chain, also where the samples are only free
// space (four lanes 0.49 ms, sixteen 0.50), and patches per XCD cut the L2 misses
// to an eighth (0.475 -> 0.458 ms).  What bounds it then is the vector cache: 34
// accesses a load, 0.98 M a CU in 1.05 M cycles.  Where the rays fill the chip by
// themselves, samples past a ray's end are only waste: ray_lanes.  A map of the
// bricks without a surface, built in every call by a pass over the volume, needs
// memory that the entry point is not given and left 0.42 ms.
// Bit-exact with the CPU oracle: every fused multiply-add is explicit and the
// build disables contraction.
#include <hip/hip_runtime.h>

#include <float.h>

#include <algorithm>

#include "mcx_internal.h"

namespace mcx {
namespace {

constexpr int kMaxTsdf = 32766;
constexpr int kRayMaxSteps = 1 << 20;
// Workgroups go round the 8 XCDs; an XCD's are the tiles of patches of kPatch x
// kPatch pixels, one after the other, so that its L2 holds what they share.
constexpr int kPatch = 16;
// LANES lanes take a ray; a wave's rays are a tile of W x H pixels.
template <int LANES>
struct Tile {
  static constexpr int kW = LANES == 8 ? 2 : 8, kH = 64 / LANES / kW;
  static constexpr int kPatchX = kPatch / kW;               // tiles in a patch's row
  static constexpr int kInPatch = kPatchX * (kPatch / kH);  // tiles of a patch
};

struct RaycastArgs {
  const int16_t* vol16;  // tsdf halves: word i's tsdf at vol16[2 i]
  float* depth;
  float* normal;  // 3 floats per pixel, may be null
  int X, Y, Z, W, H;
  int patches_x;      // patches in a row
  int first_patch;    // this launch's first one
  float h;
  float im[9];  // (K R^T)^-1, row-major
  float R[9];   // camera-to-world rotation, row-major
  float cc[3];  // camera centre in grid units
  float fx, fy, cx, cy;
};

__device__ __forceinline__ float lerpf(float a, float b, float t) { return fmaf(t, b - a, a); }

// s / 32766 correctly rounded for every 16-bit s: one multiply by the
// rounded reciprocal and one fused correction step (checked exhaustively
// against IEEE division over [-32767, 32767]).
__device__ __forceinline__ float unpack_tsdf(int s) {
  constexpr float r = 1.0f / 32766.0f;
  const float x = (float)s;
  const float q = x * r;
  const float e = fmaf(-q, 32766.0f, x);
  return fmaf(e, r, q);
}

// two consecutive voxel words (4-byte aligned, which the vector memory path
// accepts for a 64-bit load)
typedef uint32_t u32x2a4 __attribute__((ext_vector_type(2), aligned(4), may_alias));

// Corner tsdf values in the reference's order V000 V100 V010 V001 V101 V011
// V110 V111 for the cell whose lower corner is word `base`: the words of
// (x, x + 1) in the rows (y, z), (y + 1, z), (y, z + 1), (y + 1, z + 1).
__device__ __forceinline__ void load_corners(const int16_t* __restrict__ v16, int64_t base,
                                             int64_t X, int64_t XY, int* s) {
  const uint32_t* w = reinterpret_cast<const uint32_t*>(v16) + base;
  auto pair = [](const uint32_t* q) { return *reinterpret_cast<const u32x2a4*>(q); };
  const u32x2a4 a = pair(w);           // V000 V100
  const u32x2a4 b = pair(w + X);       // V010 V110
  const u32x2a4 c = pair(w + XY);      // V001 V101
  const u32x2a4 d = pair(w + XY + X);  // V011 V111
  s[0] = (int16_t)a[0];
  s[1] = (int16_t)a[1];
  s[2] = (int16_t)b[0];
  s[3] = (int16_t)c[0];
  s[4] = (int16_t)c[1];
  s[5] = (int16_t)d[0];
  s[6] = (int16_t)b[1];
  s[7] = (int16_t)d[1];
}

// Sides of a cell: +1 where every corner is at least kMaxTsdf (its samples
// are 1 or more: outside the band, which is all the march asks of them), -1
// where every corner is at most -kMaxTsdf, else 0.
__device__ __forceinline__ int cell_side(const int* s) {
  const int lo = min(min(min(s[0], s[1]), min(s[2], s[3])), min(min(s[4], s[5]), min(s[6], s[7])));
  const int hi = max(max(max(s[0], s[1]), max(s[2], s[3])), max(max(s[4], s[5]), max(s[6], s[7])));
  return lo >= kMaxTsdf ? 1 : hi <= -kMaxTsdf ? -1 : 0;
}

// The trilinear sample of the corners s of a cell, (tx, ty, tz) into it.
__device__ __forceinline__ float sample_sdf(const int* s, float tx, float ty, float tz) {
  float stop = 0.0f;  // the first corner's at +-kMaxTsdf
#pragma unroll
  for (int k = 7; k >= 0; --k) stop = s[k] == kMaxTsdf ? 1.0f : s[k] == -kMaxTsdf ? -1.0f : stop;
  if (stop != 0.0f) return stop;
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) v[k] = unpack_tsdf(s[k]);
  const float c00 = lerpf(v[0], v[1], tx);
  const float c10 = lerpf(v[2], v[6], tx);
  const float c01 = lerpf(v[3], v[4], tx);
  const float c11 = lerpf(v[5], v[7], tx);
  return lerpf(lerpf(c00, c10, ty), lerpf(c01, c11, ty), tz);
}

__device__ void surface_normal(const RaycastArgs& A, int64_t XY, float px, float py, float pz,
                               float* n) {
  const int ix = min(max((int)px, 0), A.X - 2);
  const int iy = min(max((int)py, 0), A.Y - 2);
  const int iz = min(max((int)pz, 0), A.Z - 2);
  const float tx = px - (float)ix, ty = py - (float)iy, tz = pz - (float)iz;
  int s[8];
  load_corners(A.vol16, (int64_t)iz * XY + (int64_t)iy * A.X + ix, A.X, XY, s);
  n[0] = n[1] = n[2] = 0.0f;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (s[k] == kMaxTsdf || s[k] == -kMaxTsdf) return;
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) v[k] = unpack_tsdf(s[k]);
  const float x0 = lerpf(lerpf(v[0], v[2], ty), lerpf(v[3], v[5], ty), tz);
  const float x1 = lerpf(lerpf(v[1], v[6], ty), lerpf(v[4], v[7], ty), tz);
  const float y0 = lerpf(lerpf(v[0], v[1], tx), lerpf(v[3], v[4], tx), tz);
  const float y1 = lerpf(lerpf(v[2], v[6], tx), lerpf(v[5], v[7], tx), tz);
  const float z0 = lerpf(lerpf(v[0], v[1], tx), lerpf(v[2], v[6], tx), ty);
  const float z1 = lerpf(lerpf(v[3], v[4], tx), lerpf(v[5], v[7], tx), ty);
  float gx = x1 - x0, gy = y1 - y0, gz = z1 - z0;
  const float norm = sqrtf(fmaf(gz, gz, fmaf(gy, gy, gx * gx)));
  if (norm > FLT_EPSILON || norm < -FLT_EPSILON) {
    gx = gx / norm;
    gy = gy / norm;
    gz = gz / norm;
  }
  n[0] = gx;
  n[1] = gy;
  n[2] = gz;
}

// The value of lane `from` (0 to LANES - 1) of this lane's group.
template <int LANES>
__device__ __forceinline__ float group_get(float v, int from) {
  return __shfl(v, from, LANES);
}
// This group's bits of a condition over the wave.
template <int LANES>
__device__ __forceinline__ uint32_t group_bits(bool c) {
  const int first = threadIdx.x & (64 - LANES);
  return (uint32_t)(__ballot(c) >> first) & ((1u << LANES) - 1u);
}

template <int LANES>
__global__ __launch_bounds__(64) void raycast_kernel(RaycastArgs A) {
  using T = Tile<LANES>;
  const int j = threadIdx.x & (LANES - 1), ray = threadIdx.x / LANES;
  const int b = blockIdx.x >> 3, tile = b % T::kInPatch;
  const int patch = A.first_patch + b / T::kInPatch * 8 + (blockIdx.x & 7);
  const int py = patch / A.patches_x, px = patch - py * A.patches_x;
  const int x = px * kPatch + tile % T::kPatchX * T::kW + ray % T::kW;
  const int y = py * kPatch + tile / T::kPatchX * T::kH + ray / T::kW;
  const bool live = x < A.W && y < A.H;
  const float xf = (float)x, yf = (float)y;
  float r[3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
    r[i] = fmaf(A.im[3 * i + 1], yf, fmaf(A.im[3 * i + 0], xf, A.im[3 * i + 2]));
  const float rn = sqrtf(fmaf(r[2], r[2], fmaf(r[1], r[1], r[0] * r[0])));
  if (rn > FLT_EPSILON || rn < -FLT_EPSILON) {
#pragma unroll
    for (int i = 0; i < 3; ++i) r[i] = r[i] / rn;
  }
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (r[i] == 0.0f) r[i] = 1e-15f;
  const float mx[3] = {(float)A.X - 1.0f, (float)A.Y - 1.0f, (float)A.Z - 1.0f};
  const float margin = 1.0f;
  float t_min = FLT_MAX, t_max = 0.0f;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int b = a == 0 ? 1 : 0, c = a == 2 ? 1 : 2;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const float t = ((side ? mx[a] : margin) - A.cc[a]) / r[a];
      if (t > 0.0f) {
        const float u = fmaf(r[b], t, A.cc[b]), v = fmaf(r[c], t, A.cc[c]);
        if (u > margin && u < mx[b] && v > margin && v < mx[c]) {
          t_min = fminf(t_min, t);
          t_max = fmaxf(t_max, t);
        }
      }
    }
  }
  const float dt_max = 1.0f, dt_min = 0.25f;
  bool marching = live && !(t_min == FLT_MAX && t_max == 0.0f);
  if (t_min == t_max) t_min = dt_max * margin;
  float t_far = FLT_MAX;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float e = ((r[a] > 0.0f ? mx[a] + 1.0f : -1.0f) - A.cc[a]) / r[a];
    t_far = fminf(t_far, e);
  }
  t_far = t_far + fabsf(t_far) * 0x1p-20f + 1.0f;
  const int64_t XY = (int64_t)A.X * A.Y;

  // The march, LANES samples at a time: lane j takes the j-th next one.  The
  // samples are those of a step-by-step march up to the first event (the end,
  // a hit, a back face, a change between coarse and fine steps); what was
  // sampled past an event is dropped.  State, the same in a group's lanes:
  float t = t_min, dt = dt_max;      // the next sample, the step
  float t1 = 0.0f, sdf1 = 1.0f;      // the last sample
  bool fine = false, hit = false;
  int steps = 0;
  float hit_t = 0.0f;
  while (__any(marching)) {
    float ts = t, last = t;          // this lane's sample, the group's last one
#pragma unroll
    for (int i = 1; i < LANES; ++i) {
      last = last + dt;
      ts = j >= i ? last : ts;
    }
    const float px = fmaf(r[0], ts, A.cc[0]), py = fmaf(r[1], ts, A.cc[1]),
                pz = fmaf(r[2], ts, A.cc[2]);
    const bool stop = !(ts < t_max) || ts > t_far || steps + j >= kRayMaxSteps;
    const bool in = !stop && marching && !(px < 0.0f || py < 0.0f || pz < 0.0f || px >= mx[0] ||
                                           py >= mx[1] || pz >= mx[2]);
    const int ix = in ? (int)px : 0, iy = in ? (int)py : 0, iz = in ? (int)pz : 0;
    int side = 0;  // +-1: the sample lies outside the band
    float sdf = 1.0f;
    if (in) {
      int s[8];
      load_corners(A.vol16, (int64_t)iz * XY + (int64_t)iy * A.X + ix, A.X, XY, s);
      side = cell_side(s);
      sdf = side ? (float)side : sample_sdf(s, px - (float)ix, py - (float)iy, pz - (float)iz);
    }
    // all lanes in free or unseen space, taking coarse steps: on
    if (__all(!marching || (in && side != 0 && !fine))) {
      steps += LANES;
      sdf1 = group_get<LANES>(sdf, LANES - 1);
      t = last + dt;
      continue;
    }
    // the sample before this lane's (samples outside the volume do not count,
    // and lie before all or after all of the others)
    const float before = __shfl_up(sdf, 1, LANES), t_before = __shfl_up(ts, 1, LANES);
    const uint32_t ins = group_bits<LANES>(in);
    const bool carried = j == 0 || !(ins >> (j - 1) & 1u);
    const float prev = carried ? sdf1 : before, t_prev = carried ? t1 : t_before;
    const bool band = sdf > -1.0f && sdf < 1.0f;
    const bool crossed = sdf < 0.0f && sdf > -1.0f && prev >= 0.0f && prev < 1.0f;
    const bool back = prev <= 0.0f && prev > -1.0f && sdf >= 0.0f && sdf < 1.0f;
    const uint32_t events = group_bits<LANES>(stop || (in && (crossed || back || band != fine)));
    if (!marching) continue;
    if (!events) {
      steps += LANES;
      if (ins) {
        const int l = 31 - __builtin_clz(ins);
        sdf1 = group_get<LANES>(sdf, l);
        t1 = group_get<LANES>(ts, l);
      }
      t = last + dt;
      continue;
    }
    const int e = __builtin_ctz(events);
    steps += e + 1;
    const bool ends = stop || crossed || back;
    if (j == e && crossed && !stop) {
      hit = true;
      hit_t = t_prev - dt * prev / (sdf - prev);
    }
    const bool ended = __shfl((int)ends, e, LANES);
    const float te = group_get<LANES>(ts, e), sdfe = group_get<LANES>(sdf, e), preve = group_get<LANES>(prev, e),
                t_preve = group_get<LANES>(t_prev, e);
    if (ended) {
      marching = false;
      continue;
    }
    fine = !fine;
    if (fine) {  // into the band: back to the sample before, which stays the last
      t = te - dt;
      dt = dt_min;
      sdf1 = preve;
      t1 = t_preve;
    } else {
      dt = dt_max;
      sdf1 = sdfe;
      t1 = te;
      t = te;
    }
    t += dt;
  }
  const uint32_t hits = group_bits<LANES>(hit);
  if (!live || !(hits ? hit : j == 0)) return;
  float out_d = 0.0f, out_n[3] = {0.0f, 0.0f, 0.0f};
  if (hit) {
    const float nx = r[0] * hit_t, ny = r[1] * hit_t, nz = r[2] * hit_t;
    const float ax = (xf - A.cx) / A.fx, ay = (yf - A.cy) / A.fy;
    const float len = sqrtf(fmaf(nz, nz, fmaf(ny, ny, nx * nx)));
    out_d = len / sqrtf(fmaf(ay, ay, ax * ax) + 1.0f) * A.h;
    float n[3];
    surface_normal(A, XY, nx + A.cc[0], ny + A.cc[1], nz + A.cc[2], n);
    out_n[0] = fmaf(A.R[6], n[2], fmaf(A.R[3], n[1], A.R[0] * n[0]));
    out_n[1] = fmaf(A.R[7], n[2], fmaf(A.R[4], n[1], A.R[1] * n[0]));
    out_n[2] = fmaf(A.R[8], n[2], fmaf(A.R[5], n[1], A.R[2] * n[0]));
  }
  const int64_t pix = (int64_t)y * A.W + x;
  A.depth[pix] = out_d;
  if (A.normal) {
    A.normal[3 * pix + 0] = out_n[0];
    A.normal[3 * pix + 1] = out_n[1];
    A.normal[3 * pix + 2] = out_n[2];
  }
}

// IM = (K R^T)^-1 by cofactors over the determinant (float33_inv,
// cu_vector_functions.h:555-571); false when |det| < FLT_EPSILON.
bool camera_inverse(const float* intr, const float* R, float* im) {
  const float fx = intr[0], fy = intr[1], cx = intr[2], cy = intr[3];
  float M[3][3];
  for (int j = 0; j < 3; ++j) {
    M[0][j] = fx * R[3 * j + 0] + cx * R[3 * j + 2];
    M[1][j] = fy * R[3 * j + 1] + cy * R[3 * j + 2];
    M[2][j] = R[3 * j + 2];
  }
  float C[3][3];
  C[0][0] = M[1][1] * M[2][2] - M[1][2] * M[2][1];
  C[0][1] = M[1][2] * M[2][0] - M[1][0] * M[2][2];
  C[0][2] = M[1][0] * M[2][1] - M[1][1] * M[2][0];
  C[1][0] = M[0][2] * M[2][1] - M[0][1] * M[2][2];
  C[1][1] = M[0][0] * M[2][2] - M[0][2] * M[2][0];
  C[1][2] = M[0][1] * M[2][0] - M[0][0] * M[2][1];
  C[2][0] = M[0][1] * M[1][2] - M[0][2] * M[1][1];
  C[2][1] = M[0][2] * M[1][0] - M[0][0] * M[1][2];
  C[2][2] = M[0][0] * M[1][1] - M[0][1] * M[1][0];
  const float det = M[0][0] * C[0][0] + M[0][1] * C[0][1] + M[0][2] * C[0][2];
  if (det > -FLT_EPSILON && det < FLT_EPSILON) return false;
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) im[3 * i + j] = C[j][i] / det;
  return true;
}

// Lanes of a ray.  One fills every SIMD with a wave for each 2^16 rays; with 14
// waves the next ones hide the slowest, whatever the volume; from 4 on two lanes
// do, the longer the volume's marches the later; else the chip would idle behind
// the slow rays.  Eight, two and one lanes, us, through a fused scene and through
// one without a surface: 640x480, 64^3 147, 123, 171 and 88, 65, 59; 160^3 211, 210,
// 260 and 199, 169, 167; 256^3 290, 313, 409 and 315, 283, 311; 512^3 573, 738,
// 1022 and 738, 914, 1360.  1024x768, 512^3 1273, 1196, 1658 and 1585, 1498, 2053.
// 1280x720, 64^3 388, 251, 258 and 244, 170, 136; 512^3 1481, 1288, 1484 and 1871,
// 1655, 1864.  1920x1080, 512^3 3236, 2498, 2459 and 4161, 3301, 3227.  480x360,
// 96^3 109, 127, 180 and 75, 61, 68.
int ray_lanes(int64_t rays, int side) {
  if (rays >= (int64_t)14 << 16) return 1;
  return rays >= (int64_t)4 << 16 && (int64_t)side << 16 <= 40 * rays ? 2 : 8;
}

// All patches, in launches of at most 2^25 waves.
template <int LANES>
int launch_rays(RaycastArgs A, int64_t patches, hipStream_t s) {
  constexpr int kTiles = Tile<LANES>::kInPatch;
  constexpr int64_t kMost = ((int64_t)1 << 25) / kTiles;
  for (int64_t p = 0; p < patches; p += kMost) {
    A.first_patch = (int)p;
    const int64_t n = (std::min(kMost, patches - p) + 7) / 8 * 8 * kTiles;
    hipLaunchKernelGGL(raycast_kernel<LANES>, dim3((unsigned)n), dim3(64), 0, s, A);
    MCX_HIP(hipGetLastError());
  }
  return MCX_OK;
}

}  // namespace
}  // namespace mcx

using namespace mcx;

extern "C" int mcx_raycast(const void* d_vol, int X, int Y, int Z, float h, float origin,
                           const float* intr, const float* pose, int W, int H, float* d_depth,
                           float* d_normals, void* stream) {
  if (!d_vol || !intr || !pose || !d_depth) return MCX_ERR_ARG;
  if (X < 2 || Y < 2 || Z < 2 || W < 1 || H < 1 || !(h > 0.0f)) return MCX_ERR_ARG;
  if ((int64_t)W * H >= ((int64_t)1 << 40)) return MCX_ERR_ARG;
  RaycastArgs A;
  if (!camera_inverse(intr, pose, A.im)) return MCX_ERR_ARG;
  A.vol16 = static_cast<const int16_t*>(d_vol);
  A.depth = d_depth;
  A.normal = d_normals;
  A.X = X;
  A.Y = Y;
  A.Z = Z;
  A.W = W;
  A.H = H;
  A.h = h;
  for (int i = 0; i < 9; ++i) A.R[i] = pose[i];
  for (int a = 0; a < 3; ++a) A.cc[a] = pose[9 + a] / h - origin;
  A.fx = intr[0];
  A.fy = intr[1];
  A.cx = intr[2];
  A.cy = intr[3];
  if ((H + 15) / 16 > 65535) return MCX_ERR_ARG;  // the entry point's limit of rows
  A.patches_x = (W + kPatch - 1) / kPatch;
  const int64_t patches = (int64_t)A.patches_x * ((H + kPatch - 1) / kPatch);
  if (patches >= ((int64_t)1 << 31)) return MCX_ERR_ARG;
  const int lanes = ray_lanes((int64_t)W * H, std::max(X, std::max(Y, Z)));
  if (lanes == 1) return launch_rays<1>(A, patches, as_stream(stream));
  if (lanes == 2) return launch_rays<2>(A, patches, as_stream(stream));
  return launch_rays<8>(A, patches, as_stream(stream));
}
