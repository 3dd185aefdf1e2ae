// mcx_integrate.hip -- TSDF volume init and projective integration for gfx950.
//
// Replaces the reference's dead KinectFusion kernels
//   d_voxel_initialize / cu_voxel_new      cu_kinect_fusion_v1.cu:364-398
//   d_voxel_volumetric_depth_scaling       :416-425
//   d_voxel_volumetric_integration         :427-532
//   _cu_voxel_volumetric_integration       :534-549
// The reference gives each thread one (y, z) row and walks x inside the
// thread, so a wave strides the volume by 4*X bytes (uncoalesced), and it
// sweeps the whole volume once per frame.  Here a wave, a workgroup of its
// own, owns bricks of 8 x 8 x 4 voxels (a lane one x, y and four z), four
// neighbouring waves a row of x (32 consecutive voxels: whole 128-byte
// lines), and K frames are fused per sweep: the voxel is read once, updated
// for every frame in order in registers, and written once, so a sweep costs
// 8 B/voxel plus the depth reads instead of 8 B/voxel/frame.
//
// Per voxel and frame (bit-for-bit the oracle's update_voxel):
//   p = ((i + 0.5) h) per axis; q = R^T (p - t)          (camera-to-world pose)
//   skip q.z < FLT_MIN; u = rint(fx q.x / q.z + cx), v likewise (round half even)
//   skip u,v outside [0, W-2) x [0, H-2)                 (reference :449)
//   zval = depth * scale * sqrt(((u-cx)/fx)^2 + ((v-cy)/fy)^2 + 1)  (ray distance)
//   skip zval <= FLT_MIN (dropout); sdf = zval - |q|; skip sdf < -trunc_neg
//   tsdf = sdf > 0 ? min(sdf / trunc, 1) : sdf / trunc_neg (:455-463, min_t
//   and max_t of the volume; one truncation gives clamp(sdf / trunc, -1, 1));
//   running average with integer weights capped at max_w; tsdf stored as
//   trunc(t * 32767) clamped to +-32767.
// A wave first tests 64 (brick, frame) pairs at a time, one a lane
// (test_brick), and passes over those that no voxel can observe: out of the
// frame's view, or behind everything the frame measured there.  The per-voxel
// arithmetic and its results are those of every voxel taken by itself.
#include <float.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mcx_internal.h"
#include "mcx_region_order.h"

namespace mcx {
namespace {

constexpr int kFramesPerPass = 512;  // frames of one sweep; calls of more are several

__global__ __launch_bounds__(256) void init_kernel(uint32_t* vol, int64_t n) {
  const uint32_t v = (uint32_t)(uint16_t)(int16_t)-32766;  // (-CU_VOXEL_MAX_TSDF, 0)
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) vol[i] = v;
}

struct IntegrateParams {
  uint32_t* vol;
  int X, Y, Z;
  float h, trunc;        // trunc: the positive side (max_t)
  float trunc_neg;       // the negative side (min_t) of the packed integration
  float rtrunc, rtrunc_neg;  // their reciprocals
  int max_w;
  float fx, fy, cx, cy;
  const float* poses;      // [K][12] device
  const void* depth;       // [K][H][W] device, uint16 or float
  const float* rayfac;     // [H][W]
  const float2* tiles;     // per tiled frame: [TY][TX] tiles, then [TY1][TX1] large tiles,
                           // each (largest, smallest) ray distance
  float depth_scale;
  int W, H, K;
  int TX, TY, TX1, TY1;    // tiles of kTile x kTile pixels; of 4 x 4 tiles
  int tiled;               // frames [0, tiled) have a tile table
  int framed;              // sides of at most 2^22 pixels (test_brick)
  int plain;               // camera, scale and truncation within the fast forms' ranges
  FastDiv divX, divY;      // workgroups along x and y of the volume
  int64_t first_block, end_block;  // this launch's regions
  int log2_run;            // regions in a row of one XCD
};

// Ray-length factor sqrt(((u-cx)/fx)^2 + ((v-cy)/fy)^2 + 1) of a pixel
// (d_voxel_volumetric_depth_scaling, :416-425), shared by all frames.
__device__ __forceinline__ float ray_factor(int u, int v, float fx, float fy, float cx, float cy) {
  const float ax = ((float)u - cx) / fx, ay = ((float)v - cy) / fy;
  return sqrtf(__fmaf_rn(ay, ay, ax * ax) + 1.0f);
}

// Largest and smallest measured ray distance (depth * scale * factor, the
// voxels' own operations; pixels without a measurement do not count) of every
// 8 x 8 pixels, and of every 32 x 32, of the window [0, W-2) x [0, H-2) that
// voxels can observe: (0, inf) where a tile holds none.  A wave takes eight
// tiles of a tile row, a lane eight pixels of one image row, and the four
// waves of a workgroup four tile rows (two large tiles), for every
// gridDim.z-th frame; the ray factors are computed once per lane and written
// for the integration by the waves of blockIdx.z = 0, 16 bytes a store where W
// allows it (one 3840x2160 frame: 25.1 us with 4-byte stores, now 16.6).  Tiles
// of 8 pixels: an 8 x 8 x 4 brick of a 512^3 scan covers about 14 pixels, so 3 x 3
// tiles.
constexpr int kTile = 8, kTiles1 = 4;  // pixels a tile, tiles a large tile (each way)
template <typename DT>
__global__ __launch_bounds__(256) void frame_tiles_kernel(const DT* __restrict__ depth,
                                                          float scale, int W, int H, int frames,
                                                          float fx, float fy, float cx, float cy,
                                                          float* rayfac, int TX, int TY, int TX1,
                                                          int TY1, int first_row, int vec,
                                                          float2* tiles) {
  __shared__ float2 s_quad[2][4][2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row1 = first_row + blockIdx.y;
  const int tx = blockIdx.x * 8 + (lane & 7), ty = row1 * kTiles1 + wave;
  const int u0 = tx * kTile, v = ty * kTile + (lane >> 3);
  float rf[kTile];
#pragma unroll
  for (int i = 0; i < kTile; ++i) rf[i] = ray_factor(u0 + i, v, fx, fy, cx, cy);
  if (blockIdx.z == 0 && v < H && u0 < W) {
    float* const to = rayfac + (int64_t)v * W + u0;
    if (vec & 2) {
#pragma unroll
      for (int i = 0; i < kTile; i += 4)
        *reinterpret_cast<float4*>(to + i) = make_float4(rf[i], rf[i + 1], rf[i + 2], rf[i + 3]);
    } else {
#pragma unroll
      for (int i = 0; i < kTile; ++i)
        if (u0 + i < W) to[i] = rf[i];
    }
  }
  int buf = 0;
  for (int k = blockIdx.z; k < frames; k += gridDim.z, buf ^= 1) {
    const DT* row = depth + (int64_t)k * W * H + (int64_t)v * W + u0;
    DT d[kTile];
    if (vec & 1) {  // W a multiple of 8 and 16-byte aligned frames: whole 16-byte words
      constexpr int NQ = kTile * (int)sizeof(DT) / 16;
      uint4 q[NQ] = {};
      if (v < H && u0 < W)
        for (int i = 0; i < NQ; ++i) q[i] = reinterpret_cast<const uint4*>(row)[i];
      __builtin_memcpy(d, q, sizeof(d));
    } else {
#pragma unroll
      for (int i = 0; i < kTile; ++i) d[i] = v < H && u0 + i < W ? row[i] : (DT)0;
    }
    float hi = 0.0f, lo = INFINITY;
#pragma unroll
    for (int i = 0; i < kTile; ++i) {
      const float z = v < H - 2 && u0 + i < W - 2 ? ((float)d[i] * scale) * rf[i] : 0.0f;
      if (z > FLT_MIN) {
        hi = fmaxf(hi, z);
        lo = fminf(lo, z);
      }
    }
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) {
      hi = fmaxf(hi, __shfl_xor(hi, o));
      lo = fminf(lo, __shfl_xor(lo, o));
    }
    float2* const T = tiles + (int64_t)k * (TX * TY + TX1 * TY1);
    if (lane < 8 && tx < TX && ty < TY) T[ty * TX + tx] = make_float2(hi, lo);
#pragma unroll
    for (int o = 1; o < kTiles1; o <<= 1) {
      hi = fmaxf(hi, __shfl_xor(hi, o));
      lo = fminf(lo, __shfl_xor(lo, o));
    }
    // two buffers: a wave may be one frame ahead of the two lanes that read
    if (lane == 0 || lane == 4) s_quad[buf][wave][lane >> 2] = make_float2(hi, lo);
    __syncthreads();
    if (threadIdx.x < 2) {
      for (int w = 0; w < 4; ++w) {
        hi = fmaxf(w ? hi : 0.0f, s_quad[buf][w][threadIdx.x].x);
        lo = fminf(w ? lo : INFINITY, s_quad[buf][w][threadIdx.x].y);
      }
      const int tx1 = blockIdx.x * 2 + threadIdx.x;
      if (tx1 < TX1) T[TX * TY + row1 * TX1 + tx1] = make_float2(hi, lo);
    }
  }
}

// Depth value and ray factor of pixel pix of frame k, as buffer loads from
// uniform per-frame bases with 32-bit offsets (no 64-bit address arithmetic
// per voxel and frame); a pixel of kNoPixel lies past the buffer and reads 0,
// no measurement.  Word 3 of a raw 32-bit-element buffer resource on gfx950.
constexpr int kRawBufferWord3 = 0x00020000;
constexpr uint32_t kNoPixel = 0x20000000u;  // times 4 bytes: past every frame of < 2^31 bytes
template <typename DT>
__device__ __forceinline__ float frame_depth(const IntegrateParams& P, int k, uint32_t pix) {
  const int64_t wh = (int64_t)P.W * P.H;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<DT*>(static_cast<const DT*>(P.depth) + (int64_t)k * wh), (short)0,
      (int)(wh * (int64_t)sizeof(DT)), kRawBufferWord3);
  if constexpr (sizeof(DT) == 2)
    return (float)(DT)__builtin_amdgcn_raw_buffer_load_b16(rs, pix * 2u, 0, 0);
  else
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, pix * 4u, 0, 0));
}
__device__ __forceinline__ float frame_rayfac(const IntegrateParams& P, uint32_t pix) {
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(P.rayfac), (short)0, (int)((int64_t)P.W * P.H * 4), kRawBufferWord3);
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, pix * 4u, 0, 0));
}

// ---- bricks ---------------------------------------------------------------
// A wave's 8 x 8 x NZ voxels (NZ = 4, or 1 in small volumes):
// compact, so that its image is a few tiles (256 voxels in a row of x, the
// former split, cover a line of some 300 pixels) and one test serves 256
// voxels; a lane's NZ voxels share x, y and so two of the three products of
// each row of R^T (p - t).  VALU-issue bound before and after: the observations
// that are left out are the gain.  640x480 frames into 512^3: one frame a call
// 405 -> 127 us, 300 frames 84.1 -> 19.4 ms; 64 volumes of 64-192 a side with
// 16 frames each (a far wall: little is hidden) 5.2 -> 4.5 ms.
constexpr int kBrick = 8, kBrickZ = 4;
constexpr int kRegionX = 4 * kBrick;  // a workgroup's four bricks lie side by side in x

// What a brick has to do with a frame: kSkip, no voxel can observe it; else
// kFast, the brick is well in front of the camera (the quick exact arithmetic
// applies); with it kInside, every voxel is seen at a pixel of the window, and
// kFree, every measured pixel in sight lies at least trunc in front of every
// voxel (observations are +1 or none).  One lane decides for one brick and
// frame, 64 of them at once (eight lanes per frame, one box corner each, took
// eight times the instructions, half of a 300-frame sweep's: 15.8 -> 12.6 ms).
//   The box of voxel centres maps to a parallelepiped around the centre's
// q = R^T (p - t), with half extents e = |R^T| (half sides) per component.
// Out of view: wholly behind the camera, or in front of it (every point deeper
// than 1 cm) and past one edge of the pixel window; a point's image differs
// from the centre's by |qx / qz - cx / cz| <= (ex + |cx / cz| ez) / (cz - ez)
// times fx, likewise v.
//   Behind what was measured: the largest ray distance z measured in that
// rectangle of pixels (the tiles that meet it) and a lower bound q of the
// voxels' distances give sdf <= z - q (the subtraction rounds monotonically),
// and nothing is updated where that is below -trunc_neg, or where nothing was
// measured at all.  q is the least value of q(p) . n over the box, n the
// direction of its centre (|n| = 1, so |q(p)| >= q(p) . n, linear in p).
//   kFree is the same argument from the other side: the least distance
// measured against the centre's plus the half diagonal of e.
// Margins, in sum = (|dx| + |dy| + |dz| + |p| + half sides) * m, m the largest
// |entry| of R (any matrix is a pose; at least 1): a voxel's fp32 q, and the
// box's, differ from the exact one by at most 2.4e-7 sum per component (the
// coordinates, the subtraction, the fma chain), the quotients by the hardware
// reciprocals from the exact ones by 2.4e-7 of themselves, and |q| <= sum: d =
// 8e-7 sum widens e for all of it.  The rectangle is wider by one pixel, half
// of it for the rounding to the nearest pixel and half for that of u (2^-24 of
// up to 2^22; wider frames are not tested).  Distances differ by less than
// 1.6e-6 sum, taken as 4e-6.  So every voxel of a skipped frame would have
// taken its q.z, window, dropout or -trunc_neg skip.  (d = 4e-7 and m = 1 left
// out updates at sdf = -trunc_neg under matrices of scale 100 and more.)
// Rectangles of up to 4 x 4 tiles are read from the table of 8-pixel tiles,
// larger ones from the 32-pixel tiles; beyond that nothing is known of the
// depth.
constexpr int kSkip = 1, kFast = 2, kInside = 4, kFree = 8;
template <int NZ>
__device__ int test_brick(const IntegrateParams& P, int x0, int y0, int z0, int k) {
  const float* R = P.poses + 12 * k;
  // box of voxel centres
  const float wx = (float)(min(kBrick, P.X - x0) - 1), wy = (float)(min(kBrick, P.Y - y0) - 1),
              wz = (float)(min(NZ, P.Z - z0) - 1);
  const float hx = 0.5f * wx * P.h, hy = 0.5f * wy * P.h, hz = 0.5f * wz * P.h;
  const float px = ((float)x0 + 0.5f + 0.5f * wx) * P.h, py = ((float)y0 + 0.5f + 0.5f * wy) * P.h,
              pz = ((float)z0 + 0.5f + 0.5f * wz) * P.h;
  const float r0 = R[0], r1 = R[1], r2 = R[2], r3 = R[3], r4 = R[4], r5 = R[5], r6 = R[6],
              r7 = R[7], r8 = R[8];
  const float dx = px - R[9], dy = py - R[10], dz = pz - R[11];
  const float m = fmaxf(fmaxf(fmaxf(fmaxf(1.0f, fabsf(r0)), fmaxf(fabsf(r1), fabsf(r2))),
                              fmaxf(fmaxf(fabsf(r3), fabsf(r4)), fmaxf(fabsf(r5), fabsf(r6)))),
                        fmaxf(fabsf(r7), fabsf(r8)));
  const float sum =
      (fabsf(dx) + fabsf(dy) + fabsf(dz) + (px + hx) + (py + hy) + (pz + hz)) * m;
  const float d = 8e-7f * sum;
  const float qx = __fmaf_rn(r6, dz, __fmaf_rn(r3, dy, r0 * dx));
  const float qy = __fmaf_rn(r7, dz, __fmaf_rn(r4, dy, r1 * dx));
  const float qz = __fmaf_rn(r8, dz, __fmaf_rn(r5, dy, r2 * dx));
  const float ex = __fmaf_rn(fabsf(r6), hz, __fmaf_rn(fabsf(r3), hy, __fmaf_rn(fabsf(r0), hx, d)));
  const float ey = __fmaf_rn(fabsf(r7), hz, __fmaf_rn(fabsf(r4), hy, __fmaf_rn(fabsf(r1), hx, d)));
  const float ez = __fmaf_rn(fabsf(r8), hz, __fmaf_rn(fabsf(r5), hy, __fmaf_rn(fabsf(r2), hx, d)));
  if (qz + ez < -fmaxf(1e-4f, 4.0f * d)) return kSkip;
  const float zlo = qz - ez;
  if (!(zlo > 0.01f) || !P.framed) return 0;
  const float rz = __builtin_amdgcn_rcpf(qz), rl = __builtin_amdgcn_rcpf(zlo);
  const float tx = qx * rz, ty = qy * rz;
  const float u = __fmaf_rn(P.fx, tx, P.cx), v = __fmaf_rn(P.fy, ty, P.cy);
  const float du = __fmaf_rn(fabsf(P.fx) * 1.00001f, __fmaf_rn(fabsf(tx), ez, ex) * rl, 1.0f);
  const float dv = __fmaf_rn(fabsf(P.fy) * 1.00001f, __fmaf_rn(fabsf(ty), ez, ey) * rl, 1.0f);
  const float wu = (float)(P.W - 3), wv = (float)(P.H - 3);  // the window's last pixel
  float u0 = u - du, u1 = u + du, v0 = v - dv, v1 = v + dv;
  if (u1 < 0.0f || u0 > wu || v1 < 0.0f || v0 > wv) return kSkip;
  int cls = 0;
  if (P.plain && sum < 0x1p30f) {
    cls = kFast;
    if (u0 >= 0.0f && u1 <= wu && v0 >= 0.0f && v1 <= wv && wx == (float)(kBrick - 1) &&
        wy == (float)(kBrick - 1) && wz == (float)(NZ - 1))
      cls |= kInside;
  }
  if (k >= P.tiled) return cls;
  u0 = fmaxf(u0, 0.0f);
  v0 = fmaxf(v0, 0.0f);
  u1 = fminf(u1, wu);
  v1 = fminf(v1, wv);
  if (!(u0 <= u1 && v0 <= v1)) return cls;  // (NaN) not decided here
  const float2* T = P.tiles + (int64_t)k * (P.TX * P.TY + P.TX1 * P.TY1);
  int a0 = (int)u0 / kTile, a1 = (int)u1 / kTile, b0 = (int)v0 / kTile, b1 = (int)v1 / kTile;
  int stride = P.TX;
  if (a1 - a0 > 3 || b1 - b0 > 3) {
    a0 /= 4;
    a1 /= 4;
    b0 /= 4;
    b1 /= 4;
    T += P.TX * P.TY;
    stride = P.TX1;
    if (a1 - a0 > 3 || b1 - b0 > 3) return cls;
  }
  // two rows of four tiles (the last ones again where there are fewer) in
  // flight together: a loop over single tiles waits for each
  float most = 0.0f, least = INFINITY;
  for (int b = b0; b <= b1; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float2 t = T[b * stride + min(a0 + i, a1)];
      most = fmaxf(most, t.x);
      least = fminf(least, t.y);
    }
  const float n2 = __fmaf_rn(qz, qz, __fmaf_rn(qy, qy, qx * qx));
  const float rn = __builtin_amdgcn_rsqf(n2), dist = n2 * rn;
  const float sx = fabsf(__fmaf_rn(qz, r2, __fmaf_rn(qy, r1, qx * r0)));
  const float sy = fabsf(__fmaf_rn(qz, r5, __fmaf_rn(qy, r4, qx * r3)));
  const float sz = fabsf(__fmaf_rn(qz, r8, __fmaf_rn(qy, r7, qx * r6)));
  const float margin = 4e-6f * sum;
  const float near = dist - __fmaf_rn(sz, hz, __fmaf_rn(sy, hy, sx * hx)) * rn - margin;
  if (most == 0.0f || most - near < -P.trunc_neg) return kSkip;
  const float far =
      dist + __builtin_amdgcn_sqrtf(__fmaf_rn(ez, ez, __fmaf_rn(ey, ey, ex * ex))) + margin;
  if ((cls & kFast) && least - far >= P.trunc) cls |= kFree;
  return cls;
}

// A brick: its first voxel and this lane's column of NZ.
template <int NZ>
struct Brick {
  int x0, y0, z0;
  int nz;          // planes of the volume in it, 1 to NZ
  bool inside;     // the lane's column lies in the volume
  float px, py;    // the column's voxel centre
  __device__ __forceinline__ Brick(const IntegrateParams& P, int bx, int by, int bz)
      : x0(bx), y0(by), z0(bz) {
    const int lane = threadIdx.x & 63, x = x0 + (lane & 7), y = y0 + (lane >> 3);
    nz = min(NZ, P.Z - z0);
    inside = x < P.X && y < P.Y;
    px = ((float)x + 0.5f) * P.h;
    py = ((float)y + 0.5f) * P.h;
  }
  __device__ __forceinline__ float pz(const IntegrateParams& P, int j) const {
    return ((float)(z0 + j) + 0.5f) * P.h;
  }
  // index of the lane's first voxel (the next ones are a plane further each)
  __device__ __forceinline__ int64_t first(const IntegrateParams& P) const {
    const int lane = threadIdx.x & 63;
    return ((int64_t)z0 * P.Y + (y0 + (lane >> 3))) * P.X + (x0 + (lane & 7));
  }
};

// A wave is a workgroup: the four waves of a region end at different times,
// and a workgroup of four would hold the places of those that ended (3.1 waves
// ran per SIMD where five fit; one frame into 512^3 111 -> 81 us, 300 frames
// 12.6 -> 11.2 ms).  This workgroup's region (-1: past the launch's last) and
// which of the region's waves it is.
__device__ __forceinline__ int64_t region_of(const IntegrateParams& P, int* wave) {
  *wave = wave_of_block(blockIdx.x);
  return region_of_block(blockIdx.x, P.first_block, P.end_block, P.log2_run);
}

// A wave's first brick of region `blk` >= 0 of a volume; false past the
// volume's edge.  Regions are numbered x first, or (BLOCKS) in blocks.
template <bool BLOCKS>
__device__ __forceinline__ bool brick_origin(const IntegrateParams& P, uint32_t blk, int wave,
                                             int zstep, int* x0, int* y0, int* z0) {
  RegionAt at;
  if (BLOCKS) {
    at = blocked_region(blk, P.divX.d, P.divY.d, (uint32_t)((P.Z + zstep - 1) / zstep));
  } else {
    const uint32_t row = P.divX.div(blk);
    at.z = P.divY.div(row);
    at.x = blk - row * P.divX.d;
    at.y = row - at.z * P.divY.d;
  }
  *x0 = __builtin_amdgcn_readfirstlane((int)at.x) * kRegionX + wave * kBrick;
  *y0 = __builtin_amdgcn_readfirstlane((int)at.y) * kBrick;
  *z0 = __builtin_amdgcn_readfirstlane((int)at.z) * zstep;
  return *x0 < P.X;
}

// The frames that bricks may observe.  A wave's 64 lanes test `lanes` frames
// (a power of two, at least K up to 64) of 64 / lanes bricks above one another
// at once; with more than 64 frames, 64 frames of one brick at a time.  Every
// lane of the wave takes part.
template <int NZ>
struct Frames {
  const IntegrateParams& P;
  int x0, y0, z0;          // the first of the bricks tested together
  int log2_lanes, shift;   // lanes per brick; this brick's first lane
  bool tested;
  int cls;                 // this lane's class (read from its lane at the frame's turn)
  uint64_t act;

  __device__ __forceinline__ Frames(const IntegrateParams& p, int bx, int by, int bz)
      : P(p), x0(bx), y0(by), z0(bz), shift(0), tested(false), cls(kSkip), act(0) {
    log2_lanes = P.K > 32 ? 6 : P.K > 1 ? 32 - __builtin_clz((unsigned)(P.K - 1)) : 0;
  }
  __device__ __forceinline__ int bricks() const { return 64 >> log2_lanes; }
  __device__ __forceinline__ void test(int kb) {
    const int lane = threadIdx.x & 63, k = kb + (lane & ((1 << log2_lanes) - 1));
    const int z = z0 + (lane >> log2_lanes) * NZ;
    cls = k < P.K && z < P.Z ? test_brick<NZ>(P, x0, y0, z, k) : kSkip;
    act = __ballot(!(cls & kSkip));
    tested = true;
  }
  // f(k, class) for every frame k that some voxel of the brick may observe, in
  // order.
  template <typename F>
  __device__ __forceinline__ void each(F&& f) {
    for (int kb = 0; kb < P.K; kb += 64) {
      if (!tested || P.K > 64) test(kb);
      uint64_t m = act >> shift;
      if (log2_lanes < 6) m &= (1ull << (1 << log2_lanes)) - 1;
      while (m) {
        const int b = __builtin_ctzll(m);
        m &= m - 1;
        f(kb + b, __builtin_amdgcn_readlane(cls, b + shift));
      }
    }
  }
};

// body(brick, frames) for the wave's `count` bricks above one another from
// (x0, y0, z0) on.
template <int NZ, typename F>
__device__ __forceinline__ void for_bricks(const IntegrateParams& P, int x0, int y0, int z0,
                                           int count, F&& body) {
  Frames<NZ> fr(P, x0, y0, z0);
  const int together = fr.bricks();
  for (int b = 0; b < count; ++b) {
    const int z = z0 + b * NZ;
    if (z >= P.Z) break;
    if (b % together == 0) {  // (a power of two)
      fr.z0 = z;
      fr.tested = false;
    }
    if (!fr.tested && P.K <= 64) fr.test(0);
    fr.shift = (b % together) << fr.log2_lanes;
    body(Brick<NZ>(P, x0, y0, z), fr);
  }
}

// Poses are read with a uniform index through the constant address space
// (scalar loads: the wave's registers hold no pose).
typedef const float __attribute__((address_space(4))) cfloat;

// Frame k's view of a brick: per voxel the pixel it is seen at (kNoPixel:
// none) and its distance from the camera.
template <int NZ>
struct View {
  uint32_t pix[NZ];
  float qn[NZ];
};

// The rows of R^T (p - t) over a lane's column: R^T's products with the x and
// y offsets are the column's, the third is each voxel's.
struct ColumnRows {
  float ax, ay, az, r6, r7, r8, tz;
  template <int NZ>
  __device__ __forceinline__ ColumnRows(const IntegrateParams& P, const Brick<NZ>& B, int k) {
    cfloat* R = (cfloat*)(uintptr_t)(P.poses + 12 * k);
    const float dx = B.px - R[9], dy = B.py - R[10];
    ax = __fmaf_rn(R[3], dy, R[0] * dx);
    ay = __fmaf_rn(R[4], dy, R[1] * dx);
    az = __fmaf_rn(R[5], dy, R[2] * dx);
    r6 = R[6];
    r7 = R[7];
    r8 = R[8];
    tz = R[11];
  }
};

template <int NZ>
__device__ __forceinline__ View<NZ> view_brick(const IntegrateParams& P, const Brick<NZ>& B,
                                               int k) {
  const ColumnRows C(P, B, k);
  View<NZ> V;
#pragma unroll
  for (int j = 0; j < NZ; ++j) {
    const float dz = B.pz(P, j) - C.tz;
    const float qx = __fmaf_rn(C.r6, dz, C.ax), qy = __fmaf_rn(C.r7, dz, C.ay),
                qz = __fmaf_rn(C.r8, dz, C.az);
    V.pix[j] = kNoPixel;
    V.qn[j] = 0.0f;
    if (!B.inside || j >= B.nz || qz < FLT_MIN) continue;
    const float u = __fmaf_rn(P.fx, qx / qz, P.cx);
    const float v = __fmaf_rn(P.fy, qy / qz, P.cy);
    if (!(fabsf(u) < 1e9f) || !(fabsf(v) < 1e9f)) continue;
    const int ui = (int)rintf(u), vi = (int)rintf(v);
    if (ui < 0 || vi < 0 || ui >= P.W - 2 || vi >= P.H - 2) continue;
    V.pix[j] = (uint32_t)(vi * P.W + ui);
    V.qn[j] = sqrtf(__fmaf_rn(qz, qz, __fmaf_rn(qy, qy, qx * qx)));
  }
  return V;
}

// The same for a kFast frame: one reciprocal serves both quotients, quotients
// and root by the short exact forms (an offset |qx| below 2^-60, past their
// range, leaves u at cx's nearest pixel either way), and u rounds to the
// nearest even integer by adding 1.5 * 2^23, so that its low bits hold it: the
// pixel index is one 24-bit multiply-add and a constant.  Pixel numbers
// outside [0, 2^22) leave the float's bits beyond every window (the sum is
// monotonic, a NaN's bits are larger still).  With kFree's shorter path:
// one 640x480 frame into 512^3 127 -> 110 us, 300 frames 19.4 -> 15.8 ms, 64
// volumes with a far wall (mostly kFree) 4.5 -> 2.6 ms.
constexpr float kRoundInt = 12582912.0f;  // 1.5 * 2^23
constexpr uint32_t kRoundIntBits = 0x4B400000u;
template <bool INSIDE, bool DISTANCE, int NZ>
__device__ __forceinline__ View<NZ> view_fast(const IntegrateParams& P, const Brick<NZ>& B, int k) {
  const ColumnRows C(P, B, k);
  const uint32_t base = (kRoundIntBits & 0xffffffu) * (uint32_t)P.W + kRoundIntBits;
  View<NZ> V;
#pragma unroll
  for (int j = 0; j < NZ; ++j) {
    const float dz = B.pz(P, j) - C.tz;
    const float qx = __fmaf_rn(C.r6, dz, C.ax), qy = __fmaf_rn(C.r7, dz, C.ay),
                qz = __fmaf_rn(C.r8, dz, C.az);
    const float r = recip_rn(qz);
    const uint32_t u = __float_as_uint(__fmaf_rn(P.fx, div_rn(qx, qz, r), P.cx) + kRoundInt);
    const uint32_t v = __float_as_uint(__fmaf_rn(P.fy, div_rn(qy, qz, r), P.cy) + kRoundInt);
    V.pix[j] = __umul24(v, (uint32_t)P.W) + u - base;
    if (!INSIDE &&
        !(B.inside && j < B.nz && u - kRoundIntBits < (uint32_t)(P.W - 2) &&
          v - kRoundIntBits < (uint32_t)(P.H - 2)))
      V.pix[j] = kNoPixel;
    V.qn[j] = DISTANCE ? sqrt_rn(__fmaf_rn(qz, qz, __fmaf_rn(qy, qy, qx * qx))) : 0.0f;
  }
  return V;
}

// f(fast, j, sdf, rayfac, pix) for the voxels j of the lane's column that
// frame k updates (zval > FLT_MIN, sdf >= -trunc_neg), fast telling whether
// the quick forms hold; g(j) where the observation is known to be +1 (kFree):
// there a pixel with depth * scale > FLT_MIN is a measurement (the ray factor
// is at least 1, and a product that small would not lie trunc in front of
// anything), so neither the ray factor nor the distance is needed.  The loads
// of all the column's voxels are in flight together.
template <typename DT, int NZ, typename F, typename G>
__device__ __forceinline__ void observe_brick(const IntegrateParams& P, const Brick<NZ>& B, int k,
                                              int cls, F&& f, G&& g) {
  float dm[NZ], rf[NZ];
  if (cls & kFree) {
    const View<NZ> V =
        cls & kInside ? view_fast<true, false>(P, B, k) : view_fast<false, false>(P, B, k);
#pragma unroll
    for (int j = 0; j < NZ; ++j) dm[j] = frame_depth<DT>(P, k, V.pix[j]);
#pragma unroll
    for (int j = 0; j < NZ; ++j)
      if (dm[j] * P.depth_scale > FLT_MIN) g(j);
    return;
  }
  const auto observe = [&](auto fast, const View<NZ>& V) {
#pragma unroll
    for (int j = 0; j < NZ; ++j) {
      dm[j] = frame_depth<DT>(P, k, V.pix[j]);
      rf[j] = frame_rayfac(P, V.pix[j]);
    }
#pragma unroll
    for (int j = 0; j < NZ; ++j) {
      const float zval = (dm[j] * P.depth_scale) * rf[j];
      if (!(zval > FLT_MIN)) continue;
      const float sdf = zval - V.qn[j];
      if (!(sdf >= -P.trunc_neg)) continue;
      f(fast, j, sdf, rf[j], V.pix[j]);
    }
  };
  if (cls & kFast)
    observe(std::true_type{},
            cls & kInside ? view_fast<true, true>(P, B, k) : view_fast<false, true>(P, B, k));
  else
    observe(std::false_type{}, view_brick(P, B, k));
}

// One packed update (the oracle's update_voxel after its lookups): the new
// (tsdf, weight) word from the current one and the observation t.
// A voxel at +1 observed at +1 (free space seen again) stays at +1 with no
// division: told = 32767 / 32767 = 1, fma(1, wi, 1) = wi + 1 and
// (wi + 1) / (wi + 1) = 1 exactly (integers below 2^24), 1 * 32767 = 32767.
// FAST: |tsdf| is 0 or at least 2^-91 (a kFast frame's), within div_rn's range.
template <bool FAST>
__device__ __forceinline__ uint32_t packed_update(uint32_t cur, float tsdf, int max_w) {
  const int16_t ti = (int16_t)(cur & 0xffffu);
  const int wi = (int)(cur >> 16);
  const int wnew = wi + 1 < max_w ? wi + 1 : max_w;
  if (ti == 32767 && tsdf == 1.0f) return 0x7fffu | ((uint32_t)wnew << 16);
  const float told = tsdf_fraction(ti);  // ti / 32767, correctly rounded
  const float num = __fmaf_rn(told, (float)wi, tsdf), den = (float)(wi + 1);
  const float tnew = FAST ? div_rn(num, den, recip_rn(den)) : num / den;
  int fixedp = (int)(tnew * 32767.0f);
  fixedp = fixedp > 32767 ? 32767 : (fixedp < -32767 ? -32767 : fixedp);
  return (uint32_t)(uint16_t)(int16_t)fixedp | ((uint32_t)wnew << 16);
}

// The truncated observation of a signed distance: sdf / max_t in front of the
// surface (at most 1), sdf / min_t behind it (at least -1 once sdf >= -min_t
// was tested): one division by the selected distance.  At sdf >= max_t (> 0,
// checked by every entry point) the quotient is at least 1 before rounding,
// so at least 1 after it (rounding is monotonic): 1 without the division.
// FAST: sdf is 0 or at least 2^-31 (a kFast frame's distances are a centimetre
// or more), and the reciprocals are correctly rounded: the same quotient.
template <bool FAST>
__device__ __forceinline__ float truncated(const IntegrateParams& P, float sdf) {
  if (sdf >= P.trunc) return 1.0f;
  const bool front = sdf > 0.0f;
  const float t = front ? P.trunc : P.trunc_neg;
  return fminf(FAST ? div_rn(sdf, t, front ? P.rtrunc : P.rtrunc_neg) : sdf / t, 1.0f);
}

// Packed short2 update of a wave's bricks by frames [0, K) (the oracle's
// update_voxel).  A brick is read when its first frame comes up and a voxel is
// written only if some frame updated it: outside every frustum and behind
// every surface it costs no memory traffic.
template <typename DT, int NZ>
__global__ __launch_bounds__(64) void integrate_kernel(IntegrateParams P, int bricks) {
  int wave, x0, y0, z0;
  const int64_t blk = region_of(P, &wave);
  if (blk < 0 || !brick_origin<true>(P, (uint32_t)blk, wave, NZ * bricks, &x0, &y0, &z0))
    return;
  const int64_t XY = (int64_t)P.X * P.Y;
  for_bricks<NZ>(P, x0, y0, z0, bricks, [&](const Brick<NZ>& B, Frames<NZ>& F) {
    uint32_t* const v = P.vol + B.first(P);
    uint32_t cur[NZ] = {};
    uint32_t changed = 0;
    bool have = false;
    F.each([&](int k, int cls) {
      if (!have) {
        have = true;
#pragma unroll
        for (int j = 0; j < NZ; ++j)
          if (B.inside && j < B.nz) cur[j] = v[j * XY];
      }
      observe_brick<DT>(
          P, B, k, cls,
          [&](auto fast, int j, float sdf, float, uint32_t) {
            cur[j] = packed_update<fast.value>(cur[j], truncated<fast.value>(P, sdf), P.max_w);
            changed |= 1u << j;
          },
          [&](int j) {
            cur[j] = packed_update<true>(cur[j], 1.0f, P.max_w);
            changed |= 1u << j;
          });
    });
#pragma unroll
    for (int j = 0; j < NZ; ++j)
      if (changed & (1u << j)) v[j * XY] = cur[j];
  });
}

// One frame (the reference's per-frame call): a wave tests `bricks` bricks
// above one another (up to eight, one lane each) and passes through those that
// can observe the frame, the voxels loaded beside the depth.
template <typename DT>
__global__ __launch_bounds__(64) void integrate1_kernel(IntegrateParams P, int bricks) {
  int wave, x0, y0, z0;
  const int64_t blk = region_of(P, &wave);
  if (blk < 0 || !brick_origin<false>(P, (uint32_t)blk, wave, kBrickZ * bricks, &x0, &y0, &z0))
    return;
  const int64_t XY = (int64_t)P.X * P.Y;
  const int lane = threadIdx.x & 63, zt = z0 + lane * kBrickZ;
  const int cls =
      lane < bricks && zt < P.Z ? test_brick<kBrickZ>(P, x0, y0, zt, 0) : kSkip;
  uint64_t act = __ballot(!(cls & kSkip));
  while (act) {
    const int b = __builtin_ctzll(act);
    const Brick<kBrickZ> B(P, x0, y0, z0 + b * kBrickZ);
    act &= act - 1;
    uint32_t* const v = P.vol + B.first(P);
    uint32_t cur[kBrickZ];
#pragma unroll
    for (int j = 0; j < kBrickZ; ++j) cur[j] = B.inside && j < B.nz ? v[j * XY] : 0u;
    observe_brick<DT>(
        P, B, 0, __builtin_amdgcn_readlane(cls, b),
        [&](auto fast, int j, float sdf, float, uint32_t) {
          v[j * XY] = packed_update<fast.value>(cur[j], truncated<fast.value>(P, sdf), P.max_w);
        },
        [&](int j) { v[j * XY] = packed_update<true>(cur[j], 1.0f, P.max_w); });
  }
}


// ---- fp32 TSDF volumes (differentiable form; no counterpart in the reference)
// tsdf (fp32) and weight (int32) in separate [z][y][x] arrays; the same
// observation as above, stored unpacked:
//   f <- fma(f, w, t) / (w + 1),  w <- min(w + 1, max_w),  t = clamp(sdf / trunc, -1, 1).
// The observation t of a signed distance (>= -trunc).
template <bool FAST>
__device__ __forceinline__ float truncated_f32(const IntegrateParams& P, float sdf) {
  if (sdf >= P.trunc) return 1.0f;  // sdf / trunc >= 1 before rounding, so after it
  return fminf(fmaxf(FAST ? div_rn(sdf, P.trunc, P.rtrunc) : sdf / P.trunc, -1.0f), 1.0f);
}

// One fp32 update.  f = 1 observed at 1 stays 1: fma(1, w, 1) = w + 1 =
// (float)(w + 1) exactly for 0 <= w < 2^24 (a weight read from the caller's
// volume may lie outside), and the quotient of equal values is 1.  The
// caller's f and w may be anything: outside div_rn's range the division is
// IEEE's.
__device__ __forceinline__ void update_f32(float& f, int& w, float t, int max_w) {
  const bool usual = (uint32_t)w < (1u << 24);
  if (!(f == 1.0f && t == 1.0f && usual)) {
    const float num = __fmaf_rn(f, (float)w, t), den = (float)(w + 1);
    float q = div_rn(num, den, recip_rn(den));
    const bool odd =
        !usual || !((fabsf(num) >= 0x1p-60f && fabsf(num) <= 0x1p60f) || num == 0.0f);
    if (__any(odd)) q = odd ? num / den : q;
    f = q;
  }
  w = w + 1 < max_w ? w + 1 : max_w;
}

// d(observation)/d(depth value): zero where t is clamped.
__device__ __forceinline__ float observation_slope(const IntegrateParams& P, float sdf, float rf) {
  if (sdf >= P.trunc) return 0.0f;
  const float ts = sdf / P.trunc;
  return ts > -1.0f && ts < 1.0f ? P.depth_scale * rf / P.trunc : 0.0f;
}

// fp32 update of a brick by frames [0, K), from (f, w) as given.  Returns the
// voxels (bits j) that some frame updated.
template <int NZ, typename LOAD>
__device__ __forceinline__ uint32_t integrate_tsdf_brick(const IntegrateParams& P,
                                                         const Brick<NZ>& B, Frames<NZ>& F,
                                                         float (&f)[NZ], int (&w)[NZ],
                                                         LOAD&& load) {
  uint32_t changed = 0;
  bool have = false;
  F.each([&](int k, int cls) {
    if (!have) {
      have = true;
      load();
    }
    observe_brick<float>(
        P, B, k, cls,
        [&](auto fast, int j, float sdf, float, uint32_t) {
          changed |= 1u << j;
          update_f32(f[j], w[j], truncated_f32<fast.value>(P, sdf), P.max_w);
        },
        [&](int j) {
          changed |= 1u << j;
          update_f32(f[j], w[j], 1.0f, P.max_w);
        });
  });
  return changed;
}

// The brick's voxels are read when the first frame that may observe it comes
// up; only updated voxels are written.
template <int NZ>
__device__ __forceinline__ void integrate_tsdf_stored(const IntegrateParams& P,
                                                      const Brick<NZ>& B, Frames<NZ>& F,
                                                      float* tsdf, int32_t* wvol) {
  const int64_t i = B.first(P), XY = (int64_t)P.X * P.Y;
  float f[NZ] = {};
  int w[NZ] = {};
  const uint32_t changed = integrate_tsdf_brick(P, B, F, f, w, [&]() {
#pragma unroll
    for (int j = 0; j < NZ; ++j)
      if (B.inside && j < B.nz) {
        f[j] = tsdf[i + j * XY];
        w[j] = wvol[i + j * XY];
      }
  });
#pragma unroll
  for (int j = 0; j < NZ; ++j)
    if (changed & (1u << j)) {
      tsdf[i + j * XY] = f[j];
      wvol[i + j * XY] = w[j];
    }
}

template <int NZ>
__global__ __launch_bounds__(64) void integrate_tsdf_kernel(IntegrateParams P, int bricks,
                                                             float* tsdf, int32_t* wvol) {
  int wave, x0, y0, z0;
  const int64_t blk = region_of(P, &wave);
  if (blk < 0 || !brick_origin<true>(P, (uint32_t)blk, wave, NZ * bricks, &x0, &y0, &z0))
    return;
  for_bricks<NZ>(P, x0, y0, z0, bricks, [&](const Brick<NZ>& B, Frames<NZ>& F) {
    integrate_tsdf_stored(P, B, F, tsdf, wvol);
  });
}

constexpr int kMaxabsSpan = 4096;  // floats a workgroup reads at once

// Deterministic max of |g| over n floats: per-block max, then an integer
// atomicMax on the bit pattern (order-preserving for non-negative floats),
// only where it can raise the maximum: most blocks see a larger one already
// (the plain read is a filter: a stale value only lets an atomic through).
// 16 floats a thread and pass: the atomics on one address are what it costs
// (0.88 M floats, a block for each 256: 41 us; now 6.7).
__global__ __launch_bounds__(256) void maxabs_kernel(const float* g, int64_t n, uint32_t* out) {
  __shared__ uint32_t s_m[4];
  uint32_t m = 0;
  for (int64_t i0 = (int64_t)blockIdx.x * kMaxabsSpan; i0 < n;
       i0 += (int64_t)gridDim.x * kMaxabsSpan) {
    uint32_t x[kMaxabsSpan / 256];
#pragma unroll
    for (int k = 0; k < kMaxabsSpan / 256; ++k) {
      const int64_t i = i0 + k * 256 + threadIdx.x;
      x[k] = i < n ? __float_as_uint(g[i]) & 0x7fffffffu : 0u;
    }
#pragma unroll
    for (int k = 0; k < kMaxabsSpan / 256; ++k) m = max(m, x[k]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    m = max(max(s_m[0], s_m[1]), max(s_m[2], s_m[3]));
    if (m > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, m);
  }
}

// Fixed-point scale of the depth-gradient accumulators: contributions are
// bounded by max|g| * max(dt/dd); at most 2^20 of them reach one pixel, so
// scale * bound * 2^20 <= 2^62 keeps every int64 sum exact.
__device__ __forceinline__ double grad_scale(uint32_t maxg_bits, float max_dtdd) {
  const double bound = (double)__uint_as_float(maxg_bits) * (double)max_dtdd;
  return bound > 0.0 ? 4398046511104.0 / bound : 1.0;  // 2^42 / bound
}

// Backward of the fp32 update of a brick for the K frames of one call:
// recompute its observations; a voxel's observation i (weight before it wb_i =
// min(w0 + i, max_w)) has df/dt_i = 1/(wb_i + 1) * prod over later
// observations j of wb_j / (wb_j + 1) (closed form: the uncapped part
// telescopes, the capped part is a power of max_w / (max_w + 1)); the
// contribution g * df/dt_i * dt_i/dd goes to the observed pixel of acc (K
// frames of W x H) as an int64 fixed-point atomic add (integer sums do not
// depend on the order).  Bricks without a gradient (most: only the corners of
// active cubes carry one) are left after reading it, and lanes without one look
// at no pixel: with a gradient on one voxel in 37, 16 frames of 320x240 of eight
// 40^3 volumes each 151 -> 104 us (110 with a wave for 64 voxels of a row whose
// lanes left by themselves), of 64 128^3 volumes 3275 -> 2438.
template <int NZ>
__device__ __forceinline__ void backward_brick(const IntegrateParams& P, const Brick<NZ>& B,
                                               const float* __restrict__ g,
                                               const int32_t* __restrict__ w0vol,
                                               const uint32_t* maxg, float max_dtdd,
                                               unsigned long long* acc) {
  const int64_t i = B.first(P), XY = (int64_t)P.X * P.Y;
  float gi[NZ];
#pragma unroll
  for (int j = 0; j < NZ; ++j) gi[j] = B.inside && j < B.nz ? g[i + j * XY] : 0.0f;
  bool any = false;
#pragma unroll
  for (int j = 0; j < NZ; ++j) any |= gi[j] != 0.0f;
  if (!__any(any)) return;
  Brick<NZ> A = B;  // with the lanes that carry a gradient
  A.inside = any;
  const int drop = __all(any) ? 0 : kInside;
  const double scale = grad_scale(*maxg, max_dtdd);
  const int M = P.max_w;
  int nobs[NZ] = {}, o[NZ] = {}, w0[NZ] = {};
  if (w0vol) {
#pragma unroll
    for (int j = 0; j < NZ; ++j)
      if (gi[j] != 0.0f) w0[j] = w0vol[i + j * XY];
  }
  Frames<NZ> F(P, B.x0, B.y0, B.z0);
  F.each([&](int k, int cls) {
    observe_brick<float>(
        P, A, k, cls & ~drop, [&](auto, int j, float, float, uint32_t) { ++nobs[j]; },
        [&](int j) { ++nobs[j]; });
  });
  const double cap_a = (double)M / (double)(M + 1);
  F.each([&](int k, int cls) {
    const auto add = [&](auto, int j, float sdf, float rf, uint32_t pix) {
      const int oi = o[j]++;
      if (gi[j] == 0.0f) return;
      const float dtdd = observation_slope(P, sdf, rf);
      if (dtdd == 0.0f) return;
      const int w = w0[j], n = nobs[j];
      const int jc = M - w > 0 ? M - w : 0;  // first observation that sees the cap
      const int wb = w + oi < M ? w + oi : M;
      double c = 1.0 / (double)(wb + 1);
      const int last_unc = (n - 1 < jc - 1) ? n - 1 : jc - 1;  // last uncapped index
      if (oi + 1 <= last_unc) c *= (double)(w + oi + 1) / (double)(w + last_unc + 1);
      const int first_cap = oi + 1 > jc ? oi + 1 : jc;
      const int ncap = n - first_cap;
      if (ncap > 0) {
        // cap_a^ncap by squaring (a library pow inlined here costs the kernel
        // registers on every path, capped or not)
        double pw = 1.0, base = cap_a;
        for (int e = ncap; e; e >>= 1) {
          if (e & 1) pw *= base;
          base *= base;
        }
        c *= pw;
      }
      const double contrib = (double)gi[j] * c * (double)dtdd;
      if (contrib != 0.0) {
        const long long q = llrint(contrib * scale);
        atomicAdd(acc + (int64_t)k * P.W * P.H + pix, (unsigned long long)q);
      }
    };
    // where t is known to be +1 the slope is 0: the observation only counts
    observe_brick<float>(P, A, k, cls & ~drop, add, [&](int j) { ++o[j]; });
  });
}

template <int NZ>
__global__ __launch_bounds__(64) void integrate_tsdf_backward_kernel(
    IntegrateParams P, const float* __restrict__ g, const int32_t* __restrict__ w0vol,
    const uint32_t* maxg, float max_dtdd, unsigned long long* acc) {
  int wave, x0, y0, z0;
  const int64_t blk = region_of(P, &wave);
  if (blk < 0 || !brick_origin<true>(P, (uint32_t)blk, wave, NZ, &x0, &y0, &z0)) return;
  backward_brick(P, Brick<NZ>(P, x0, y0, z0), g, w0vol, maxg, max_dtdd, acc);
}

// ---- batches of fp32 volumes (the per-volume layout of a batch plan:
// concatenated per-voxel arrays, K frames of W x H and K poses per volume,
// one set of intrinsics); a workgroup takes four bricks of one volume.
struct BatchIntegrateParams {
  IntegrateParams base;  // intrinsics, truncation, frames; depth / poses of volume 0
  const BatchVol* bvol;
  int nvol;
  int from_init;         // start every voxel from (init_value, 0) without reading it
  float init_value;
  int bricks;            // bricks above one another in a workgroup
  int tiled_vol;         // volumes [tiled_vol, tiled_vol + base.tiled / K) have tile tables
};

// This workgroup's volume (binary search over the block ranges), its launch
// parameters and this wave's brick; false past the volume's edge.
template <int NZ>
__device__ __forceinline__ bool batch_setup(const BatchIntegrateParams& B, IntegrateParams& P,
                                            int64_t* vox_begin, int* vol, int* x0, int* y0,
                                            int* z0) {
  int wave;
  const int64_t blk = region_of(B.base, &wave);
  if (blk < 0) return false;
  const int vi = __builtin_amdgcn_readfirstlane(
      batch_volume_of<&BatchVol::blk_begin>(B.bvol, B.nvol, blk));
  const BatchVol& V = B.bvol[vi];
  P = B.base;
  P.X = V.X;
  P.Y = V.Y;
  P.Z = V.Z;
  P.h = V.h;
  P.divX = V.divX;
  P.divY = V.divY;
  P.depth = static_cast<const float*>(B.base.depth) + (int64_t)vi * P.K * P.W * P.H;
  P.poses = B.base.poses + (int64_t)vi * P.K * 12;
  P.tiled = vi >= B.tiled_vol ? max(0, min(P.K, P.tiled - (vi - B.tiled_vol) * P.K)) : 0;
  P.tiles = B.base.tiles + (int64_t)(vi - B.tiled_vol) * P.K * (P.TX * P.TY + P.TX1 * P.TY1);
  *vox_begin = V.vox_begin;
  *vol = vi;
  return brick_origin<true>(P, (uint32_t)(blk - V.blk_begin), wave, NZ * B.bricks, x0, y0, z0);
}

template <int NZ>
__global__ __launch_bounds__(64) void integrate_tsdf_batched_kernel(BatchIntegrateParams B,
                                                                     float* tsdf, int32_t* wvol) {
  IntegrateParams P;
  int64_t vb;
  int vi, x0, y0, z0;
  if (!batch_setup<NZ>(B, P, &vb, &vi, &x0, &y0, &z0)) return;
  for_bricks<NZ>(P, x0, y0, z0, B.bricks, [&](const Brick<NZ>& K, Frames<NZ>& F) {
    if (!B.from_init) {
      integrate_tsdf_stored(P, K, F, tsdf + vb, wvol + vb);
      return;
    }
    // every voxel is written: the start value where no frame observes it
    float f[NZ];
    int w[NZ] = {};
#pragma unroll
    for (int j = 0; j < NZ; ++j) f[j] = B.init_value;
    integrate_tsdf_brick(P, K, F, f, w, []() {});
    const int64_t i = vb + K.first(P), XY = (int64_t)P.X * P.Y;
#pragma unroll
    for (int j = 0; j < NZ; ++j)
      if (K.inside && j < K.nz) {
        tsdf[i + j * XY] = f[j];
        wvol[i + j * XY] = w[j];
      }
  });
}

template <int NZ>
__global__ __launch_bounds__(64) void integrate_tsdf_backward_batched_kernel(
    BatchIntegrateParams B, const float* __restrict__ g, const int32_t* __restrict__ w0vol,
    const uint32_t* maxg, float max_dtdd, unsigned long long* acc) {
  IntegrateParams P;
  int64_t vb;
  int vi, x0, y0, z0;
  if (!batch_setup<NZ>(B, P, &vb, &vi, &x0, &y0, &z0)) return;
  for (int b = 0; b < B.bricks && z0 < P.Z; ++b, z0 += NZ)
    backward_brick(P, Brick<NZ>(P, x0, y0, z0), g + vb, w0vol ? w0vol + vb : nullptr, maxg,
                   max_dtdd, acc + (int64_t)vi * P.K * P.W * P.H);
}

// Two accumulators a thread; most are 0 (pixels that saw no active voxel) and
// need no division, unless the scale is 0 (an infinite gradient: 0 / 0).  Bound
// by its 12 bytes a pixel: 53 M pixels 145 us (178 with a division for each).
__global__ __launch_bounds__(256) void fixed_to_float_kernel(const unsigned long long* acc,
                                                             int64_t n, const uint32_t* maxg,
                                                             float max_dtdd, float* out) {
  const int64_t i = 2 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= n) return;
  const bool two = i + 1 < n;
  const long long a = (long long)acc[i], b = two ? (long long)acc[i + 1] : 0;
  float x = 0.0f, y = 0.0f;
  const bool inf = __uint_as_float(*maxg) * max_dtdd == __builtin_inff();
  if ((a | b) != 0 || inf) {
    const double scale = grad_scale(*maxg, max_dtdd);
    x = (float)((double)a / scale);
    y = (float)((double)b / scale);
  }
  out[i] = x;
  if (two) out[i + 1] = y;
}

__global__ __launch_bounds__(256) void fill_f32_i32_kernel(float* f, int32_t* w, int64_t n,
                                                           float fv, int32_t wv) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    if (f) f[i] = fv;
    if (w) w[i] = wv;
  }
}

// ---- synthetic depth frames: ray-cast spheres and axis-aligned boxes -------
__device__ __forceinline__ uint32_t hash32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}
__device__ __forceinline__ float u01(uint32_t h) { return ((h >> 8) + 0.5f) * (1.0f / 16777216.0f); }

__global__ __launch_bounds__(256) void synth_kernel(uint16_t* depth, int W, int H, int K, float fx,
                                                     float fy, float cx, float cy,
                                                     const float* poses, const float* objs,
                                                     int nobj, float sigma_m, float dropout,
                                                     uint32_t seed, float depth_unit) {
  const int64_t n = (int64_t)W * H * K;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int k = (int)(i / ((int64_t)W * H));
  const int pix = (int)(i - (int64_t)k * W * H);
  const int u = pix % W, v = pix / W;
  const float* R = poses + 12 * k;
  const float a = ((float)u - cx) / fx, b = ((float)v - cy) / fy;
  // world direction of the pixel ray with unit camera-z component
  const float dx = R[0] * a + R[1] * b + R[2];
  const float dy = R[3] * a + R[4] * b + R[5];
  const float dz = R[6] * a + R[7] * b + R[8];
  const float ox = R[9], oy = R[10], oz = R[11];
  float best = 1e30f;
  for (int j = 0; j < nobj; ++j) {
    const float* o = objs + 8 * j;
    if (o[0] < 0.5f) {  // sphere
      const float lx = ox - o[1], ly = oy - o[2], lz = oz - o[3];
      const float A = dx * dx + dy * dy + dz * dz;
      const float B = lx * dx + ly * dy + lz * dz;
      const float C = lx * lx + ly * ly + lz * lz - o[4] * o[4];
      const float disc = B * B - A * C;
      if (disc >= 0.f) {
        const float sq = sqrtf(disc);
        float s = (-B - sq) / A;
        if (s <= 1e-4f) s = (-B + sq) / A;
        if (s > 1e-4f && s < best) best = s;
      }
    } else {  // axis-aligned box
      float tmin = -1e30f, tmax = 1e30f;
      const float org[3] = {ox, oy, oz}, dir[3] = {dx, dy, dz};
      bool miss = false;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const float lo = o[1 + c] - o[4 + c], hi = o[1 + c] + o[4 + c];
        if (fabsf(dir[c]) < 1e-12f) {
          if (org[c] < lo || org[c] > hi) miss = true;
        } else {
          float t0 = (lo - org[c]) / dir[c], t1 = (hi - org[c]) / dir[c];
          if (t0 > t1) {
            const float tt = t0;
            t0 = t1;
            t1 = tt;
          }
          tmin = fmaxf(tmin, t0);
          tmax = fminf(tmax, t1);
        }
      }
      if (!miss && tmax >= tmin) {
        const float s = tmin > 1e-4f ? tmin : tmax;
        if (s > 1e-4f && s < best) best = s;
      }
    }
  }
  uint16_t out = 0;
  if (best < 1e29f) {
    const uint32_t h0 = hash32(seed ^ hash32((uint32_t)i * 2u + 1u));
    const uint32_t h1 = hash32(h0 + 0x9e3779b9u);
    const uint32_t h2 = hash32(h1 + 0x9e3779b9u);
    const float r = sqrtf(-2.0f * logf(u01(h0)));
    const float gauss = r * cosf(6.28318530718f * u01(h1));
    const float mm = rintf((best + sigma_m * gauss) / depth_unit);
    if (u01(h2) >= dropout && mm >= 1.f) out = (uint16_t)fminf(mm, 65535.f);
  }
  depth[i] = out;
}

unsigned blocks_for(int64_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace
}  // namespace mcx

using namespace mcx;

extern "C" int mcx_volume_init(void* d_vol, int X, int Y, int Z, void* stream) {
  if (!d_vol || X < 1 || Y < 1 || Z < 1) return MCX_ERR_ARG;
  const int64_t n = (int64_t)X * Y * Z;
  int64_t b = (n + 255) / 256;
  if (b > 65536) b = 65536;
  hipLaunchKernelGGL(init_kernel, dim3((unsigned)b), dim3(256), 0, as_stream(stream),
                     static_cast<uint32_t*>(d_vol), n);
  MCX_HIP(hipGetLastError());
  return MCX_OK;
}

size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

// Tile tables: bytes per frame, and of `frames` frames, but of no more than 32
// MiB hold, at least one (a 640x480 frame takes 40.8 KB, so a sweep's 512 frames
// fit; a 320x240 frame 10.2 KB: 3,276, the frames of 204 volumes of a batch with
// 16 each).
size_t tile_bytes(int W, int H) {
  const auto tiles = [&](int side) {
    return (size_t)((W + side - 1) / side) * ((H + side - 1) / side);
  };
  return (tiles(kTile) + tiles(kTile * kTiles1)) * sizeof(float2);
}
size_t tile_tables_bytes(int W, int H, int64_t frames) {
  const size_t per = tile_bytes(W, H), most = (size_t)32 << 20;
  return per * std::min((size_t)frames, std::max((size_t)1, most / std::max(per, (size_t)1)));
}

// The ray factors alone would do (they are what a call cannot run without);
// the rest holds the frames' tile tables.
size_t rayfac_bytes(int W, int H) {
  return (size_t)(W > 0 ? W : 0) * (size_t)(H > 0 ? H : 0) * sizeof(float);
}
extern "C" size_t mcx_integrate_workspace_size_frames(int W, int H, int64_t frames) {
  const size_t rf = rayfac_bytes(W, H);
  return rf && frames >= 0 ? al256(rf) + 256 + tile_tables_bytes(W, H, frames) : 0;
}

extern "C" size_t mcx_integrate_workspace_size(int W, int H) {
  return mcx_integrate_workspace_size_frames(W, H, INT64_MAX);
}

// The smaller truncation, the reciprocals, and whether everything lies where
// the quick exact forms hold (kFast): pixel numbers below 2^22, finite ray
// factors, truncations and scale within 2^-60 to 2^60.
void set_trunc_neg(IntegrateParams& P, float trunc_neg) {
  P.trunc_neg = trunc_neg;
  P.rtrunc = 1.0f / P.trunc;
  P.rtrunc_neg = 1.0f / trunc_neg;
  const auto in = [](float v, float lo, float hi) {
    return std::fabs(v) >= lo && std::fabs(v) <= hi;
  };
  P.framed = P.W <= (1 << 22) && P.H <= (1 << 22);
  P.plain = P.framed && in(P.trunc, 0x1p-60f, 0x1p60f) &&
            in(trunc_neg, 0x1p-60f, 0x1p60f) && P.depth_scale > 0.0f &&
            in(P.depth_scale, 0x1p-60f, 0x1p60f) && in(P.fx, 0x1p-20f, 0x1p20f) &&
            in(P.fy, 0x1p-20f, 0x1p20f) && in(P.cx, 0.0f, 0x1p22f) && in(P.cy, 0.0f, 0x1p22f);
}

// Checks shared by the integration entry points; fills the launch parameters
// (all but vol, K, poses, depth and the tile tables).
int prepare_integrate(IntegrateParams& P, int X, int Y, int Z, float h, float trunc, int max_w,
                      const float* intr, float depth_scale, int W, int H, int K, float* rayfac) {
  if (!intr || X < 1 || Y < 1 || Z < 1 || W < 3 || H < 3 || K < 0) return MCX_ERR_ARG;
  if (!(h > 0.f) || !(trunc > 0.f) || max_w < 1 || max_w > 65535) return MCX_ERR_ARG;
  if ((int64_t)X * Y > 0xffffffffll) return MCX_ERR_UNSUPPORTED;
  // frames are read through buffer resources of at most 2^31 - 1 bytes
  if ((int64_t)W * H * 4 >= ((int64_t)1 << 31)) return MCX_ERR_UNSUPPORTED;
  P.vol = nullptr;
  P.X = X;
  P.Y = Y;
  P.Z = Z;
  P.h = h;
  P.trunc = trunc;
  P.max_w = max_w;
  P.fx = intr[0];
  P.fy = intr[1];
  P.cx = intr[2];
  P.cy = intr[3];
  P.rayfac = rayfac;
  P.tiles = nullptr;
  P.tiled = 0;
  P.TX = (W + kTile - 1) / kTile;
  P.TY = (H + kTile - 1) / kTile;
  P.TX1 = (P.TX + kTiles1 - 1) / kTiles1;
  P.TY1 = (P.TY + kTiles1 - 1) / kTiles1;
  P.depth_scale = depth_scale;
  P.W = W;
  P.H = H;
  P.divX = FastDiv((uint32_t)((X + kRegionX - 1) / kRegionX));
  P.divY = FastDiv((uint32_t)((Y + kBrick - 1) / kBrick));
  set_trunc_neg(P, trunc);
  P.K = 0;
  P.poses = nullptr;
  P.depth = nullptr;
  P.first_block = P.end_block = 0;
  P.log2_run = 0;
  return MCX_OK;
}

// Workgroups of a volume, z planes taken zstep at a time.
int64_t regions(int X, int Y, int Z, int zstep) {
  return (int64_t)((X + kRegionX - 1) / kRegionX) * ((Y + kBrick - 1) / kBrick) *
         ((Z + zstep - 1) / zstep);
}

// The ray factors, and if wanted the tile tables of as many of `frames` frames
// (from `depth`) as [tables, end) holds; P.tiled says how many.
template <typename DT>
int frame_tiles(IntegrateParams& P, bool tables_wanted, const DT* depth, int64_t frames,
                char* tables, char* end, hipStream_t s) {
  tables = reinterpret_cast<char*>(al256(reinterpret_cast<uintptr_t>(tables)));
  const size_t per = tile_bytes(P.W, P.H);
  const int64_t room = tables < end ? (int64_t)((size_t)(end - tables) / per) : 0;
  P.tiles = reinterpret_cast<const float2*>(tables);
  P.tiled = tables_wanted ? (int)std::min(frames, room) : 0;
  const int gx = (P.TX + 7) / 8;
  // about 16 waves per SIMD in all; each takes every gz-th frame
  const int64_t plane = (int64_t)gx * P.TY1;
  const int64_t gz = std::max<int64_t>(1, std::min<int64_t>((4096 + plane - 1) / plane, P.tiled));
  int vec = 0;  // 16-byte accesses: 1 the frames', 2 the ray factors'
  if (P.W % kTile == 0) {
    vec |= (reinterpret_cast<uintptr_t>(depth) & 15u) == 0 &&
           ((int64_t)P.W * P.H * (int64_t)sizeof(DT)) % 16 == 0;
    vec |= (reinterpret_cast<uintptr_t>(P.rayfac) & 15u) == 0 ? 2 : 0;
  }
  for (int y0 = 0; y0 < P.TY1; y0 += 65535) {
    hipLaunchKernelGGL(frame_tiles_kernel<DT>,
                       dim3((unsigned)gx, (unsigned)std::min(65535, P.TY1 - y0), (unsigned)gz),
                       dim3(256), 0, s, depth, P.depth_scale, P.W, P.H, P.tiled, P.fx, P.fy, P.cx,
                       P.cy, const_cast<float*>(P.rayfac), P.TX, P.TY, P.TX1, P.TY1, y0, vec,
                       reinterpret_cast<float2*>(tables));
    MCX_HIP(hipGetLastError());
  }
  return MCX_OK;
}

// The launch over regions [b0, end), at most kMaxRegions of them.
constexpr int64_t kMaxRegions = kMaxLaunchBlocks;
dim3 region_grid(IntegrateParams& P, int64_t b0, int64_t end) {
  P.first_block = b0;
  P.end_block = std::min(end, b0 + kMaxRegions);
  return dim3((unsigned)region_workgroups(P.end_block - b0, P.log2_run));
}
// Eight regions of a block in a row for one XCD, where several frames are
// swept over regions enough for that (300 frames, 512^3: runs of 16 and 32 8.9 ms,
// of 64 10.7: the XCDs' shares of the surfaces become uneven).  One region and
// eight, 100 640x480 frames, us: 96^3 (864 regions) 311 and 323, 160^3 (4,000) 468
// and 454, 200^3 (8,750) 612 and 585, 256^3 766 and 790, 512^3 2635 and 2636; 16
// frames, 96^3 52 and 57, 200^3 105 and 100.
int region_runs(int64_t n, int K) { return K > 1 && n >= 4096 ? 3 : 0; }

// Bricks above one another that a wave takes (their frames are tested
// together): as many as its 64 lanes can test at once, up to eight, while
// that leaves 16 waves per SIMD.
int bricks_per_wave(int64_t voxels, int K) {
  int n = 1;
  while (n < 8 && n * 2 * K <= 64 && voxels >= (int64_t)16384 * 256 * n * 2) n *= 2;
  return n;
}

// Planes of a brick.  Up to 2^18 voxels four leave one wave a SIMD or fewer, each
// going through the frames alone; one plane gives four times the waves and each a
// quarter of the work a frame.  Above 2^17 that pays while the frames are few or
// stay in a CU's vector cache (2^15 pixels of 2 bytes): more waves read each
// frame.  Four planes against one, without tile tables: 32^3, 16 VGA frames 28 and
// 17 us, 300 429 and 208; 48^3 31 and 23, 452 and 308; 64^3, 16 of 320x240 25 and
// 20, 300 VGA 432 and 503, 600 of 160x120 710 and 423; 80^3, 16 VGA 46 and 55.
int brick_planes(int64_t voxels, int K, int64_t pixels) {
  if (voxels > (1 << 18)) return kBrickZ;
  return voxels <= (1 << 17) || K <= 32 || pixels <= (1 << 15) ? 1 : kBrickZ;
}

// Whether the frames' tile tables give back the reading of every frame: a frame's
// table costs its pixels, and saves part of the observations, as many as there are
// voxels (`each`: of one volume of a batch); nothing where the sweep is as short
// as the table's kernel.  With and without, us: 64^3, 4 VGA frames 16.4 and 13.3,
// 300 471 and 432; 80^3, 4 17.0 and 15.7, 16 42.7 and 46.2; 96^3, 4 of 1920x1080
// 41.9 and 35.7; 128^3, 4 VGA 23.5 and 25.8, 4 of 1920x1080 45.9 and 53.4, one of
// 3840x2160 41.6 and 39.5; 160^3, one VGA 15.0 and 16.5.
bool tables_pay(int64_t voxels, int64_t each, int K, int64_t pixels) {
  return voxels > (1 << 18) && each >= pixels && (K >= 8 || voxels >= (1 << 20));
}

template <typename DT>
int integrate_impl(void* d_vol, int X, int Y, int Z, float h, float trunc_neg, float trunc,
                   int max_w, const float* intr, const float* d_poses, const DT* d_depth,
                   float depth_scale, int W, int H, int K, void* d_ws, size_t ws_bytes,
                   void* stream) {
  if (!d_vol || !(trunc_neg > 0.f)) return MCX_ERR_ARG;
  if (K > 0 && (!d_poses || !d_depth)) return MCX_ERR_ARG;
  if (!d_ws || ws_bytes < rayfac_bytes(W, H)) return MCX_ERR_WORKSPACE;
  if (K == 0) return MCX_OK;
  hipStream_t s = as_stream(stream);
  IntegrateParams P;
  char* const ws = static_cast<char*>(d_ws);
  int rc = prepare_integrate(P, X, Y, Z, h, trunc, max_w, intr, depth_scale, W, H, K,
                             reinterpret_cast<float*>(ws));
  if (rc) return rc;
  P.vol = static_cast<uint32_t*>(d_vol);
  set_trunc_neg(P, trunc_neg);
  const int64_t voxels = (int64_t)X * Y * Z, pixels = (int64_t)W * H;
  for (int k0 = 0; k0 < K; k0 += kFramesPerPass) {
    P.K = K - k0 < kFramesPerPass ? K - k0 : kFramesPerPass;
    P.poses = d_poses + (int64_t)12 * k0;
    P.depth = d_depth + k0 * pixels;
    rc = frame_tiles(P, tables_pay(voxels, voxels, P.K, pixels), d_depth + k0 * pixels, P.K,
                     ws + rayfac_bytes(W, H), ws + ws_bytes, s);
    if (rc) return rc;
    // (integrate1_kernel has bricks of four)
    const int nz = P.K == 1 ? kBrickZ : brick_planes(voxels, P.K, pixels);
    const int bricks = bricks_per_wave(voxels, P.K);
    const int64_t nb = regions(X, Y, Z, nz * bricks);
    P.log2_run = region_runs(nb, P.K);
    for (int64_t b0 = 0; b0 < nb; b0 += kMaxRegions) {
      const dim3 grid = region_grid(P, b0, nb);
      if (P.K == 1)
        hipLaunchKernelGGL(integrate1_kernel<DT>, grid, dim3(64), 0, s, P, bricks);
      else if (nz == 1)
        hipLaunchKernelGGL((integrate_kernel<DT, 1>), grid, dim3(64), 0, s, P, bricks);
      else
        hipLaunchKernelGGL((integrate_kernel<DT, kBrickZ>), grid, dim3(64), 0, s, P, bricks);
      MCX_HIP(hipGetLastError());
    }
  }
  return MCX_OK;
}

// Largest dt/d(depth value) of any pixel in the window (the ray factor grows
// towards the corners), with a margin: the bound of the fixed-point scale.
float max_dtdd(const float* intr, float depth_scale, float trunc, int W, int H) {
  double m = 0.0;
  const int us[2] = {0, W - 3}, vs[2] = {0, H - 3};
  for (int a = 0; a < 2; ++a)
    for (int b = 0; b < 2; ++b) {
      const double ax = ((double)us[a] - intr[2]) / intr[0], ay = ((double)vs[b] - intr[3]) / intr[1];
      m = std::max(m, std::sqrt(ax * ax + ay * ay + 1.0));
    }
  return (float)(1.01 * m * (double)depth_scale / (double)trunc);
}

extern "C" int mcx_integrate(void* d_vol, int X, int Y, int Z, float h, float trunc, int max_w,
                             const float* intr, const float* d_poses, const uint16_t* d_depth,
                             float depth_scale, int W, int H, int K, void* d_ws, size_t ws_bytes,
                             void* stream) {
  return integrate_impl<uint16_t>(d_vol, X, Y, Z, h, trunc, trunc, max_w, intr, d_poses, d_depth,
                                  depth_scale, W, H, K, d_ws, ws_bytes, stream);
}

extern "C" int mcx_integrate_f32(void* d_vol, int X, int Y, int Z, float h, float trunc,
                                 int max_w, const float* intr, const float* d_poses,
                                 const float* d_depth, float depth_scale, int W, int H, int K,
                                 void* d_ws, size_t ws_bytes, void* stream) {
  return integrate_impl<float>(d_vol, X, Y, Z, h, trunc, trunc, max_w, intr, d_poses, d_depth,
                               depth_scale, W, H, K, d_ws, ws_bytes, stream);
}

extern "C" int mcx_integrate_ex(void* d_vol, int X, int Y, int Z, float h, float trunc_neg,
                                float trunc_pos, int max_w, const float* intr,
                                const float* d_poses, const void* d_depth, int depth_kind,
                                float depth_scale, int W, int H, int K, void* d_ws,
                                size_t ws_bytes, void* stream) {
  if (depth_kind == MCX_DEPTH_U16)
    return integrate_impl<uint16_t>(d_vol, X, Y, Z, h, trunc_neg, trunc_pos, max_w, intr,
                                    d_poses, static_cast<const uint16_t*>(d_depth), depth_scale,
                                    W, H, K, d_ws, ws_bytes, stream);
  if (depth_kind == MCX_DEPTH_F32)
    return integrate_impl<float>(d_vol, X, Y, Z, h, trunc_neg, trunc_pos, max_w, intr, d_poses,
                                 static_cast<const float*>(d_depth), depth_scale, W, H, K, d_ws,
                                 ws_bytes, stream);
  return MCX_ERR_ARG;
}

extern "C" int mcx_synth_depth(uint16_t* d_depth, int W, int H, int K, const float* intr,
                               const float* d_poses, const float* d_objs, int nobj,
                               float noise_sigma_m, float dropout, uint32_t seed,
                               float depth_unit_m, void* stream) {
  if (!d_depth || !intr || !d_poses || (nobj > 0 && !d_objs) || W < 1 || H < 1 || K < 1 ||
      !(depth_unit_m > 0.f))
    return MCX_ERR_ARG;
  const int64_t n = (int64_t)W * H * K;
  hipLaunchKernelGGL(synth_kernel, dim3(blocks_for(n)), dim3(256), 0, as_stream(stream), d_depth,
                     W, H, K, intr[0], intr[1], intr[2], intr[3], d_poses, d_objs, nobj,
                     noise_sigma_m, dropout, seed, depth_unit_m);
  MCX_HIP(hipGetLastError());
  return MCX_OK;
}

// ---- fp32 TSDF volumes: differentiable integration (no counterpart in the
//      reference; the forward is the same observation, stored unpacked)
extern "C" int mcx_tsdf_init(float* d_tsdf, int32_t* d_weight, int64_t n, float tsdf_value,
                             void* stream) {
  if (n < 0 || (n > 0 && !d_tsdf && !d_weight)) return MCX_ERR_ARG;
  if (n == 0) return MCX_OK;
  int64_t b = (n + 255) / 256;
  if (b > 65536) b = 65536;
  hipLaunchKernelGGL(fill_f32_i32_kernel, dim3((unsigned)b), dim3(256), 0, as_stream(stream),
                     d_tsdf, d_weight, n, tsdf_value, 0);
  MCX_HIP(hipGetLastError());
  return MCX_OK;
}

extern "C" int mcx_integrate_tsdf(float* d_tsdf, int32_t* d_weight, int X, int Y, int Z, float h,
                                  float trunc, int max_w, const float* intr,
                                  const float* d_poses, const float* d_depth, float depth_scale,
                                  int W, int H, int K, void* d_ws, size_t ws_bytes,
                                  void* stream) {
  if (!d_tsdf || !d_weight) return MCX_ERR_ARG;
  if (K > 0 && (!d_poses || !d_depth)) return MCX_ERR_ARG;
  if (!d_ws || ws_bytes < rayfac_bytes(W, H)) return MCX_ERR_WORKSPACE;
  if (K == 0) return MCX_OK;
  hipStream_t s = as_stream(stream);
  IntegrateParams P;
  char* const ws = static_cast<char*>(d_ws);
  int rc = prepare_integrate(P, X, Y, Z, h, trunc, max_w, intr, depth_scale, W, H, K,
                             reinterpret_cast<float*>(ws));
  if (rc) return rc;
  const int64_t voxels = (int64_t)X * Y * Z, pixels = (int64_t)W * H;
  for (int k0 = 0; k0 < K; k0 += kFramesPerPass) {
    P.K = K - k0 < kFramesPerPass ? K - k0 : kFramesPerPass;
    P.poses = d_poses + (int64_t)12 * k0;
    P.depth = d_depth + k0 * pixels;
    rc = frame_tiles(P, tables_pay(voxels, voxels, P.K, pixels), d_depth + k0 * pixels, P.K,
                     ws + rayfac_bytes(W, H), ws + ws_bytes, s);
    if (rc) return rc;
    const int nz = brick_planes(voxels, P.K, pixels);
    const int bricks = bricks_per_wave(voxels, P.K);
    const int64_t nb = regions(X, Y, Z, nz * bricks);
    P.log2_run = region_runs(nb, P.K);
    for (int64_t b0 = 0; b0 < nb; b0 += kMaxRegions) {
      const dim3 grid = region_grid(P, b0, nb);
      if (nz == 1)
        hipLaunchKernelGGL(integrate_tsdf_kernel<1>, grid, dim3(64), 0, s, P, bricks, d_tsdf,
                           d_weight);
      else
        hipLaunchKernelGGL(integrate_tsdf_kernel<kBrickZ>, grid, dim3(64), 0, s, P, bricks, d_tsdf,
                           d_weight);
      MCX_HIP(hipGetLastError());
    }
  }
  return MCX_OK;
}

// Ray factors, max |g| and the accumulators of `frames` frames: what the
// backward cannot run without (its workspace ends with the tile tables).
size_t backward_bytes(int W, int H, int64_t frames) {
  return al256((size_t)W * H * sizeof(float)) + 256 + (size_t)frames * W * H * 8;
}

extern "C" size_t mcx_integrate_tsdf_backward_workspace_size(int W, int H, int K) {
  if (W < 1 || H < 1 || K < 0) return 0;
  return backward_bytes(W, H, K) + 256 + tile_bytes(W, H) * K;
}

extern "C" int mcx_integrate_tsdf_backward(const float* d_grad_tsdf, const int32_t* d_weight0,
                                           int X, int Y, int Z, float h, float trunc, int max_w,
                                           const float* intr, const float* d_poses,
                                           const float* d_depth, float depth_scale, int W,
                                           int H, int K, float* d_grad_depth, void* d_ws,
                                           size_t ws_bytes, void* stream) {
  if (!d_grad_tsdf) return MCX_ERR_ARG;
  if (K > 0 && (!d_poses || !d_depth || !d_grad_depth)) return MCX_ERR_ARG;
  if (!d_ws || ws_bytes < (W < 1 || H < 1 || K < 0 ? 0 : backward_bytes(W, H, K)))
    return MCX_ERR_WORKSPACE;
  if (K == 0) return MCX_OK;
  if (K > kFramesPerPass) return MCX_ERR_UNSUPPORTED;  // one pass: weights known per voxel
  hipStream_t s = as_stream(stream);
  char* b = static_cast<char*>(d_ws);
  float* rayfac = reinterpret_cast<float*>(b);
  uint32_t* maxg = reinterpret_cast<uint32_t*>(b + al256((size_t)W * H * sizeof(float)));
  unsigned long long* acc = reinterpret_cast<unsigned long long*>(
      b + al256((size_t)W * H * sizeof(float)) + 256);
  IntegrateParams P;
  int rc = prepare_integrate(P, X, Y, Z, h, trunc, max_w, intr, depth_scale, W, H, K, rayfac);
  if (rc) return rc;
  const int64_t n = (int64_t)X * Y * Z;
  rc = frame_tiles(P, tables_pay(n, n, K, (int64_t)W * H), d_depth, K, b + backward_bytes(W, H, K),
                   b + ws_bytes, s);
  if (rc) return rc;
  const int64_t npix = (int64_t)K * W * H;
  rc = fill_bytes_zero(maxg, 256 + (size_t)npix * 8, s);  // max and accumulators
  if (rc) return rc;
  const int64_t mb = std::min<int64_t>((n + kMaxabsSpan - 1) / kMaxabsSpan, 2048);
  hipLaunchKernelGGL(maxabs_kernel, dim3((unsigned)mb), dim3(256), 0, s, d_grad_tsdf, n, maxg);
  MCX_HIP(hipGetLastError());
  const float mdt = max_dtdd(intr, depth_scale, trunc, W, H);
  P.K = K;
  P.poses = d_poses;
  P.depth = d_depth;
  // One plane a wave up to 2^22 voxels: few bricks hold a surface there, and each
  // one's frames run in series.  One and four, gradients at the surface, us: 96^3,
  // 16 frames 69 and 87; 128^3, 1 30 and 27, 4 38 and 41, 16 71 and 90; 160^3, 1 41
  // and 33, 16 88 and 94; 192^3, 1 54 and 38, 16 111 and 101; 256^3, 16 154 and 129.
  const bool small = n <= ((int64_t)1 << 22);
  const int64_t nb = regions(X, Y, Z, small ? 1 : kBrickZ);
  P.log2_run = region_runs(nb, K);
  for (int64_t b0 = 0; b0 < nb; b0 += kMaxRegions) {
    const dim3 grid = region_grid(P, b0, nb);
    if (small)
      hipLaunchKernelGGL(integrate_tsdf_backward_kernel<1>, grid, dim3(64), 0, s, P, d_grad_tsdf,
                         d_weight0, maxg, mdt, acc);
    else
      hipLaunchKernelGGL(integrate_tsdf_backward_kernel<kBrickZ>, grid, dim3(64), 0, s, P,
                         d_grad_tsdf, d_weight0, maxg, mdt, acc);
    MCX_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(fixed_to_float_kernel, dim3(blocks_for((npix + 1) / 2)), dim3(256), 0, s, acc, npix,
                     maxg, mdt, d_grad_depth);
  MCX_HIP(hipGetLastError());
  return MCX_OK;
}

// ---- batched fp32 fusion (no counterpart in the reference) ----------------
// Volumes of a batch whose K tile tables fit the workspace together (all of
// them when not even one volume's do: they then run without).
int volumes_per_turn(char* tables, char* end, int W, int H, int K, int nvol) {
  tables = reinterpret_cast<char*>(al256(reinterpret_cast<uintptr_t>(tables)));
  const int64_t fit =
      tables < end ? (int64_t)((size_t)(end - tables) / tile_bytes(W, H)) / K : 0;
  return fit < 1 ? nvol : (int)std::min<int64_t>(fit, nvol);
}

extern "C" int mcx_integrate_tsdf_batched(const mcx_batch* plan, float* d_tsdf, int32_t* d_weight,
                                          int from_init, float init_value, float trunc,
                                          int max_w, const float* intr, const float* d_poses,
                                          const float* d_depth, float depth_scale, int W, int H,
                                          int K, void* d_ws, size_t ws_bytes, void* stream) {
  if (!plan || !d_tsdf || !d_weight) return MCX_ERR_ARG;
  if (plan->elem != MCX_ELEM_F32) return MCX_ERR_ARG;
  if (K > 0 && (!d_poses || !d_depth)) return MCX_ERR_ARG;
  if (K > kFramesPerPass) return MCX_ERR_UNSUPPORTED;
  if (!d_ws || ws_bytes < rayfac_bytes(W, H)) return MCX_ERR_WORKSPACE;
  hipStream_t s = as_stream(stream);
  if (K == 0) {
    if (!from_init) return MCX_OK;
    hipLaunchKernelGGL(fill_f32_i32_kernel, dim3(blocks_for(plan->voxels) < 65536u
                                                      ? blocks_for(plan->voxels) : 65536u),
                       dim3(256), 0, s, d_tsdf, d_weight, plan->voxels, init_value, 0);
    MCX_HIP(hipGetLastError());
    return MCX_OK;
  }
  if (plan->blocks >= ((int64_t)1 << 31)) return MCX_ERR_UNSUPPORTED;
  BatchIntegrateParams B;
  int rc = prepare_integrate(B.base, 1, 1, 1, 1.0f, trunc, max_w, intr, depth_scale, W, H, K,
                             static_cast<float*>(d_ws));
  if (rc) return rc;
  B.base.K = K;
  B.base.poses = d_poses;
  B.base.depth = d_depth;
  B.bvol = plan->d_bvol;
  B.nvol = plan->nvol;
  B.bricks = plan->bricks;
  B.base.log2_run = region_runs(plan->blocks, K);
  B.from_init = from_init ? 1 : 0;
  B.init_value = init_value;
  // volumes in turn of as many as the workspace holds tile tables for
  char* const ws = static_cast<char*>(d_ws);
  const int64_t pixels = (int64_t)W * H * K;
  const bool tables = tables_pay(plan->voxels, plan->voxels / plan->nvol, K, (int64_t)W * H);
  const int turn = tables ? volumes_per_turn(ws + rayfac_bytes(W, H), ws + ws_bytes, W, H, K,
                                             plan->nvol)
                          : plan->nvol;
  for (int v0 = 0; v0 < plan->nvol; v0 += turn) {
    const int v1 = std::min(plan->nvol, v0 + turn);
    rc = frame_tiles(B.base, tables, d_depth + v0 * pixels, (int64_t)(v1 - v0) * K,
                     ws + rayfac_bytes(W, H), ws + ws_bytes, s);
    if (rc) return rc;
    B.tiled_vol = v0;
    const int64_t end = plan->blk_begin[v1];
    for (int64_t b0 = plan->blk_begin[v0]; b0 < end; b0 += kMaxRegions) {
      const dim3 grid = region_grid(B.base, b0, end);
      if (plan->brick_planes == 1)
        hipLaunchKernelGGL(integrate_tsdf_batched_kernel<1>, grid, dim3(64), 0, s, B, d_tsdf,
                           d_weight);
      else
        hipLaunchKernelGGL(integrate_tsdf_batched_kernel<kBrickZ>, grid, dim3(64), 0, s, B, d_tsdf,
                           d_weight);
      MCX_HIP(hipGetLastError());
    }
  }
  return MCX_OK;
}

extern "C" size_t mcx_integrate_tsdf_backward_batched_workspace_size(const mcx_batch* plan, int W,
                                                                     int H, int K) {
  if (!plan || W < 1 || H < 1 || K < 0) return 0;
  return backward_bytes(W, H, (int64_t)plan->nvol * K) + 256 +
         tile_bytes(W, H) * plan->nvol * K;
}

extern "C" int mcx_integrate_tsdf_backward_batched(const mcx_batch* plan,
                                                   const float* d_grad_tsdf,
                                                   const int32_t* d_weight0,
                                                   const uint32_t* d_maxabs, float trunc,
                                                   int max_w, const float* intr,
                                                   const float* d_poses, const float* d_depth,
                                                   float depth_scale, int W, int H, int K,
                                                   float* d_grad_depth, void* d_ws,
                                                   size_t ws_bytes, void* stream) {
  if (!plan || !d_grad_tsdf) return MCX_ERR_ARG;
  if (plan->elem != MCX_ELEM_F32) return MCX_ERR_ARG;
  if (K > 0 && (!d_poses || !d_depth || !d_grad_depth)) return MCX_ERR_ARG;
  if (!d_ws ||
      ws_bytes < (W < 1 || H < 1 || K < 0 ? 0 : backward_bytes(W, H, (int64_t)plan->nvol * K)))
    return MCX_ERR_WORKSPACE;
  if (K == 0) return MCX_OK;
  if (K > kFramesPerPass) return MCX_ERR_UNSUPPORTED;
  if (plan->blocks >= ((int64_t)1 << 31)) return MCX_ERR_UNSUPPORTED;
  hipStream_t s = as_stream(stream);
  char* b = static_cast<char*>(d_ws);
  float* rayfac = reinterpret_cast<float*>(b);
  uint32_t* maxg = reinterpret_cast<uint32_t*>(b + al256((size_t)W * H * sizeof(float)));
  unsigned long long* acc = reinterpret_cast<unsigned long long*>(
      b + al256((size_t)W * H * sizeof(float)) + 256);
  BatchIntegrateParams B;
  int rc = prepare_integrate(B.base, 1, 1, 1, 1.0f, trunc, max_w, intr, depth_scale, W, H, K,
                             rayfac);
  if (rc) return rc;
  rc = frame_tiles(B.base,
                   tables_pay(plan->voxels, plan->voxels / plan->nvol, K, (int64_t)W * H), d_depth,
                   (int64_t)plan->nvol * K, b + backward_bytes(W, H, (int64_t)plan->nvol * K),
                   b + ws_bytes, s);
  if (rc) return rc;
  B.tiled_vol = 0;
  const int64_t npix = (int64_t)plan->nvol * K * W * H;
  if (d_maxabs) {
    rc = fill_bytes_zero(acc, (size_t)npix * 8, s);  // the accumulators
    if (rc) return rc;
  } else {
    rc = fill_bytes_zero(maxg, 256 + (size_t)npix * 8, s);  // max and accumulators
    if (rc) return rc;
    const int64_t mb =
        std::min<int64_t>((plan->voxels + kMaxabsSpan - 1) / kMaxabsSpan, 2048);
    hipLaunchKernelGGL(maxabs_kernel, dim3((unsigned)mb), dim3(256), 0, s, d_grad_tsdf,
                       plan->voxels, maxg);
    MCX_HIP(hipGetLastError());
  }
  const uint32_t* mg = d_maxabs ? d_maxabs : maxg;
  const float mdt = max_dtdd(intr, depth_scale, trunc, W, H);
  B.base.K = K;
  B.base.poses = d_poses;
  B.base.depth = d_depth;
  B.bvol = plan->d_bvol;
  B.nvol = plan->nvol;
  B.bricks = plan->bricks;
  B.base.log2_run = region_runs(plan->blocks, K);
  B.from_init = 0;
  B.init_value = 0.0f;
  for (int64_t b0 = 0; b0 < plan->blocks; b0 += kMaxRegions) {
    const dim3 grid = region_grid(B.base, b0, plan->blocks);
    if (plan->brick_planes == 1)
      hipLaunchKernelGGL(integrate_tsdf_backward_batched_kernel<1>, grid, dim3(64), 0, s, B,
                         d_grad_tsdf, d_weight0, mg, mdt, acc);
    else
      hipLaunchKernelGGL(integrate_tsdf_backward_batched_kernel<kBrickZ>, grid, dim3(64), 0, s, B,
                         d_grad_tsdf, d_weight0, mg, mdt, acc);
    MCX_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(fixed_to_float_kernel, dim3(blocks_for((npix + 1) / 2)), dim3(256), 0, s, acc, npix,
                     mg, mdt, d_grad_depth);
  MCX_HIP(hipGetLastError());
  return MCX_OK;
}
