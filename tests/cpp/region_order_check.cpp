// Host check of the integration workgroups' regions (mcx_region_order.h): over
// volumes of many shapes and both run lengths, in one launch and in two, the
// grid's workgroups take every wave of every region exactly once, inside the
// volume, and those past the last region take none.  Prints how many of the
// latter would have met a block of extent 0 (a division by it) had they gone on:
// that must stay positive, or the check does not exercise the hazard.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "mcx_region_order.h"

using namespace mcx;

static void fail(const char* what, uint32_t nx, uint32_t ny, uint32_t nz, int run) {
  std::printf("%s: %u x %u x %u regions, run %d\n", what, nx, ny, nz, run);
  std::exit(1);
}

static bool empty_block(uint64_t r, uint32_t nx, uint32_t ny, uint32_t nz) {
  const uint64_t bz = r / ((uint64_t)nx * ny * kBlockZ);
  if (bz * kBlockZ >= nz) return false;  // known to lie past the volume
  r -= bz * nx * ny * kBlockZ;
  const uint64_t hz = nz - bz * kBlockZ < kBlockZ ? nz - bz * kBlockZ : kBlockZ;
  const uint64_t by = r / (nx * kBlockY * hz);
  if (by * kBlockY >= ny) return true;
  r -= by * nx * kBlockY * hz;
  const uint64_t hy = ny - by * kBlockY < kBlockY ? ny - by * kBlockY : kBlockY;
  return r / (kBlockX * hy * hz) * kBlockX >= nx;
}

int main() {
  const uint32_t sides[] = {1, 2, 3, 5, 7, 8, 9, 16, 17, 24};
  long shapes = 0, empty = 0;
  for (uint32_t nx : {1u, 2u, 3u, 6u, 16u})
    for (uint32_t ny : sides)
      for (uint32_t nz : sides)
        for (int run : {0, 3}) {
          const int64_t n = (int64_t)nx * ny * nz;
          std::vector<uint8_t> place((size_t)n), waves((size_t)n);
          for (int64_t r = 0; r < n; ++r) {
            const RegionAt a = blocked_region((uint32_t)r, nx, ny, nz);
            if (a.x >= nx || a.y >= ny || a.z >= nz) fail("outside", nx, ny, nz, run);
            place[((size_t)a.z * ny + a.y) * nx + a.x]++;
          }
          for (uint8_t p : place)
            if (p != 1) fail("not a permutation", nx, ny, nz, run);
          const int64_t half = n / 128 * 64;  // launches begin at whole rounds
          const int64_t cut[3] = {0, half, n};
          for (int l = 0; l < 2; ++l) {
            if (cut[l] == cut[l + 1]) continue;
            const int64_t g = region_workgroups(cut[l + 1] - cut[l], run);
            for (int64_t b = 0; b < g; ++b) {
              const int64_t r = region_of_block((uint32_t)b, cut[l], cut[l + 1], run);
              if (r >= 0) {
                if (r < cut[l] || r >= cut[l + 1]) fail("not this launch's", nx, ny, nz, run);
                const int bit = 1 << wave_of_block((uint32_t)b);
                if (waves[(size_t)r] & bit) fail("taken twice", nx, ny, nz, run);
                waves[(size_t)r] |= bit;
              } else if (l == 1) {
                const int64_t all = region_of_block((uint32_t)b, cut[l], INT64_MAX, run);
                if (all < n) fail("not taken", nx, ny, nz, run);
                empty += empty_block((uint64_t)all, nx, ny, nz);
              }
            }
          }
          for (uint8_t w : waves)
            if (w != 15) fail("waves missing", nx, ny, nz, run);
          ++shapes;
        }
  std::printf("ok %ld %ld\n", shapes, empty);
  return 0;
}
