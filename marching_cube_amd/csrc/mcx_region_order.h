// mcx_region_order.h -- which region of a volume an integration workgroup
// takes.
//
// Plain constexpr functions (host and device in HIP, plain C++ elsewhere), so
// that the kernels and the host check tests/cpp/region_order_check.cpp run the
// same arithmetic.
//
// A region is four bricks beside one another in x; four workgroups, one wave
// each, take one.  Workgroups go round the 8 XCDs, so a region's four are those
// of every 8th workgroup (one L2 sees whole lines), and an XCD takes 2^log2_run
// regions in a row.  A grid is whole rounds of the XCDs: its last workgroups
// may lie past the last region and take none.
#pragma once

#include <stdint.h>

namespace mcx {

// The workgroups of a launch over n regions.
constexpr int64_t region_workgroups(int64_t n, int log2_run) {
  const int64_t round = (int64_t)8 << log2_run;
  return (n + round - 1) / round * round * 4;
}

// The region of workgroup `block` of a launch over regions [first, end), or -1.
constexpr int64_t region_of_block(uint32_t block, int64_t first, int64_t end, int log2_run) {
  const uint32_t r = block >> 5;
  const int64_t region = first + ((int64_t)(r >> log2_run) << (log2_run + 3)) +
                         ((block & 7) << log2_run) + (r & ((1u << log2_run) - 1));
  return region < end ? region : -1;
}
// ... and which of its four waves the workgroup is.
constexpr int wave_of_block(uint32_t block) { return (int)((block >> 3) & 3); }

// Region r < nx ny nz of a volume of nx x ny x nz regions, numbered in blocks
// of 2 x 8 x 4 regions (smaller at the far sides): waves that run together then
// see the same part of each frame, and an XCD's L2 holds it (300 frames into
// 512^3: 10.9 ms x first, where the waves of an XCD lie all over a slab, 8.8 ms
// in blocks).  An r past the last would divide by the extent 0 of a block past
// the volume.
constexpr uint32_t kBlockX = 2, kBlockY = 8, kBlockZ = 4;
struct RegionAt {
  uint32_t x, y, z;
};
constexpr RegionAt blocked_region(uint32_t r, uint32_t nx, uint32_t ny, uint32_t nz) {
  const uint32_t bz = r / (nx * ny * kBlockZ);
  r -= bz * (nx * ny * kBlockZ);
  const uint32_t hz = nz - bz * kBlockZ < kBlockZ ? nz - bz * kBlockZ : kBlockZ;
  const uint32_t by = r / (nx * kBlockY * hz);
  r -= by * (nx * kBlockY * hz);
  const uint32_t hy = ny - by * kBlockY < kBlockY ? ny - by * kBlockY : kBlockY;
  const uint32_t bx = r / (kBlockX * hy * hz);
  r -= bx * (kBlockX * hy * hz);
  const uint32_t hx = nx - bx * kBlockX < kBlockX ? nx - bx * kBlockX : kBlockX;
  const uint32_t iy = r / hx, iz = iy / hy;
  return RegionAt{bx * kBlockX + r - iy * hx, by * kBlockY + iy - iz * hy, bz * kBlockZ + iz};
}

}  // namespace mcx
