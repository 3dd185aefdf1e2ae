// mcx_weld.hip -- indexed mesh from the canonical vertex list (gfx950).
//
// Replaces the reference's OBJ vertex de-duplication by printed coordinates
// ("%.4f_%.4f_%.4f" keys in a std::map, cu_kinect_fusion_v1.cu:3668-3719) with
// exact sharing by grid edge: every vertex of the extraction lies on one grid
// edge (its key: lower corner voxel * 3 + axis, written by the extraction), the
// up to 4 cubes around an edge each emit a vertex for it, and all of them
// become one vertex.  Its position is that of the first of them in the
// canonical order (the cubes interpolate the edge in different directions, so
// their fp32 positions can differ in the last bit).
//
// W1 insert  a workgroup takes 1024 vertices.  Its repeated keys are found in
//            LDS (vertices come in cube order: about every third key of a
//            block is new to it); the first of each claims the key's slot of a
//            table of vertex indices in memory (open addressing, power of two
//            >= 2V slots) with one atomicCAS, or lowers it with atomicMin, so
//            a slot ends with the first occurrence whatever the order of the
//            atomics.  Every vertex keeps its slot.
// W2 rank    rep = table[slot] = the key's first occurrence; unique vertices
//            (rep == v) get their rank in the block; per-block counts.
// W3 scan    exclusive scan of the block counts (one workgroup).
// W4 finish  triangle index = count before rep's block + rep's rank; unique
//            vertices copy their position.
// Deterministic: the table layout may vary between runs, what is read from
// it (the minimum index per key) does not.
//
// Bound by the scattered atomics of the insert: 31 us at 2.45 M vertices (a 400^3
// room), the rest of the five launches 38.  A table of keys and another of
// values, two atomics a key and per-wave repeats only, with a second probe for
// the first occurrences, took 200 us for the whole weld where this takes 69.
// Steps of one slot where groups of keys meet took 43 us for the insert there,
// and 433 for the weld of 1 M consecutive keys (now 40; shuffled 1230 and 103).
// Tried, with those steps: workgroups of 256 and 1024 threads for the insert (43
// us), a table hashed key by key (47 us), a read of the slot before the CAS (the
// same).
#include <hip/hip_runtime.h>

#include "mcx_internal.h"

namespace mcx {
namespace {

constexpr uint32_t kEmpty = 0xffffffffu;  // empty slot (V < 2^31)
constexpr int kWeldBlock = 1024;          // vertices per workgroup (256 threads x 4)
constexpr uint32_t kInsert = 512;  // threads of an insert workgroup
constexpr uint32_t kPer = kWeldBlock / kInsert;
constexpr uint32_t kLocal = 2 * kWeldBlock;  // slots of a workgroup's LDS table

__device__ __forceinline__ uint64_t mix64(uint64_t k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return k;
}

// The slots of a key.  Groups of 32 consecutive keys (the edges of 10 voxels
// along x) stay in one 128-byte line, whose place and inner order are hashed: the
// keys of a surface patch share lines, and keys a multiple of 32 apart still
// start anywhere in the table.  A key whose slot is taken goes on to the same
// place of other lines, the group's (a group that meets another moves as a whole:
// by steps of one slot, 32 dense keys walk over 32 taken ones each), and from the
// kLines-th line on to the next slots, all of the table if need be.
constexpr uint32_t kLines = 16;
struct Probe {
  uint32_t h, step, n;
};
__device__ __forceinline__ Probe first_slot(uint64_t key, uint32_t mask) {
  const uint64_t m = mix64(key >> 5);
  return Probe{(((uint32_t)m << 5) | (((uint32_t)key ^ (uint32_t)(m >> 59)) & 31u)) & mask,
               (uint32_t)(m >> 32) << 6 | 32u, 1};
}
__device__ __forceinline__ void next_slot(Probe& p, uint32_t mask) {
  p.h = (p.h + (p.n < kLines ? p.step : 1u)) & mask;
  ++p.n;
}

__global__ __launch_bounds__(kInsert) void weld_insert_kernel(const int64_t* __restrict__ ekey,
                                                          uint32_t V, uint32_t* table,
                                                          uint32_t mask, uint32_t* slot) {
  __shared__ uint64_t s_key[kWeldBlock];
  __shared__ uint32_t s_tab[kLocal];  // index in the block of a key's first vertex
  __shared__ uint32_t s_first[kWeldBlock];
  __shared__ uint32_t s_n;
  uint32_t* const s_slot = s_tab;  // once the first vertices are listed
  const uint32_t tid = threadIdx.x;
  const uint32_t base = blockIdx.x * (uint32_t)kWeldBlock;
#pragma unroll
  for (uint32_t i = tid; i < kLocal; i += kInsert) s_tab[i] = kEmpty;
  uint64_t key[kPer];
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    const uint32_t v = base + k * kInsert + tid;
    key[k] = v < V ? (uint64_t)ekey[v] : 0;
    s_key[k * kInsert + tid] = key[k];
  }
  if (tid == 0) s_n = 0;
  __syncthreads();
  uint32_t at[kPer];
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    const uint32_t l = k * kInsert + tid;
    at[k] = 0;
    if (base + l >= V) continue;
    uint32_t h = (uint32_t)mix64(key[k]) & (kLocal - 1);
    for (;;) {  // at most 1024 keys in 2048 slots: the probe ends
      const uint32_t old = atomicCAS(s_tab + h, kEmpty, l);
      if (old == kEmpty) break;
      if (s_key[old] == key[k]) {
        if (l < old) atomicMin(s_tab + h, l);
        break;
      }
      h = (h + 1) & (kLocal - 1);
    }
    at[k] = h;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    const uint32_t l = k * kInsert + tid;
    if (base + l >= V) continue;
    at[k] = s_tab[at[k]];
    if (at[k] == l) s_first[atomicAdd(&s_n, 1u)] = l;
  }
  __syncthreads();
  const uint32_t n = s_n;
  for (uint32_t i = tid; i < n; i += kInsert) {
    const uint32_t l = s_first[i], v = base + l;
    const uint64_t mine = s_key[l];
    Probe p = first_slot(mine, mask);
    for (;;) {  // at most V distinct keys in >= 2V slots: the probe ends
      const uint32_t old = atomicCAS(table + p.h, kEmpty, v);
      if (old == kEmpty) break;
      // a slot's index only changes to a lower one of the same key
      if ((uint64_t)ekey[old] == mine) {
        if (v < old) atomicMin(table + p.h, v);
        break;
      }
      next_slot(p, mask);
    }
    s_slot[l] = p.h;
  }
  __syncthreads();
#pragma unroll
  for (uint32_t k = 0; k < kPer; ++k) {
    const uint32_t v = base + k * kInsert + tid;
    if (v < V) slot[v] = s_slot[at[k]];
  }
}

// rep_of: a vertex's slot in, its key's first occurrence out.
__global__ __launch_bounds__(256) void weld_rank_kernel(uint32_t V,
                                                        const uint32_t* __restrict__ table,
                                                        uint32_t* rep_of, uint32_t* rank,
                                                        uint32_t* bsum) {
  __shared__ uint32_t s_n[16];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t base = blockIdx.x * (uint32_t)kWeldBlock;
  uint32_t s[4], r[4];
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t v = base + k * 256 + tid;
    s[k] = v < V ? rep_of[v] : 0;
  }
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) r[k] = base + k * 256 + tid < V ? table[s[k]] : kEmpty;
  uint64_t first[4];
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t v = base + k * 256 + tid;
    if (v < V) rep_of[v] = r[k];
    first[k] = __ballot(r[k] == v);  // v >= V: r is kEmpty, never v
    if (lane == 0) s_n[k * 4 + (tid >> 6)] = (uint32_t)__popcll(first[k]);
  }
  __syncthreads();
  // 16 runs of 64 consecutive vertices
  uint32_t before[4] = {0, 0, 0, 0}, all = 0;
#pragma unroll
  for (uint32_t j = 0; j < 16; ++j) {
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
      if (j < k * 4 + (tid >> 6)) before[k] += s_n[j];
    all += s_n[j];
  }
#pragma unroll
  for (uint32_t k = 0; k < 4; ++k) {
    const uint32_t v = base + k * 256 + tid;
    if (r[k] == v)
      rank[v] = before[k] + (uint32_t)__popcll(first[k] & ((1ull << lane) - 1));
  }
  if (tid == 0) bsum[blockIdx.x] = all;
}

// Exclusive scan of nb block sums in place (one workgroup of 1024 threads,
// four sums a thread: one pass up to 4 million vertices); bsum[nb] = total.
__global__ __launch_bounds__(1024) void weld_scan_kernel(uint32_t* bsum, uint32_t nb,
                                                         int64_t* d_nunique) {
  __shared__ uint32_t s_w[16];
  const uint32_t tid = threadIdx.x;
  uint32_t carry = 0;
  for (uint32_t b0 = 0; b0 < nb; b0 += 4096) {
    const uint32_t i = b0 + 4 * tid;
    uint32_t x[4], sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      x[k] = i + k < nb ? bsum[i + k] : 0u;
      sum += x[k];
    }
    const uint32_t inc = wave_incl_scan32(sum);
    if ((tid & 63) == 63) s_w[tid >> 6] = inc;
    __syncthreads();
    uint32_t pre = carry + inc - sum;
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) {
      if (k < (tid >> 6)) pre += s_w[k];
      carry += s_w[k];
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      if (i + k < nb) bsum[i + k] = pre;
      pre += x[k];
    }
    __syncthreads();
  }
  if (tid == 0) {
    bsum[nb] = carry;
    if (d_nunique) *d_nunique = carry;
  }
}

__global__ __launch_bounds__(256) void weld_finish_kernel(uint32_t V,
                                                          const uint32_t* __restrict__ rep,
                                                          const uint32_t* __restrict__ rank,
                                                          const uint32_t* __restrict__ bsum,
                                                          const float* __restrict__ pos,
                                                          int64_t stride, int32_t* idx,
                                                          float* upos) {
  const uint32_t v = blockIdx.x * 256u + threadIdx.x;
  if (v >= V) return;
  const uint32_t r = rep[v];
  const uint32_t u = bsum[r / kWeldBlock] + rank[r];
  idx[v] = (int32_t)u;
  if (r == v) {
    const float* p = pos + (int64_t)v * stride;
    float* q = upos + 3 * (int64_t)u;
    q[0] = p[0];
    q[1] = p[1];
    q[2] = p[2];
  }
}

uint64_t table_slots(int64_t V) {
  uint64_t t = 1024;
  while (t < 2 * (uint64_t)V) t <<= 1;
  return t;
}

size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

unsigned grid_for(int64_t n, int64_t per) { return (unsigned)((n + per - 1) / per); }

// Byte offsets of the workspace's arrays, the table first.
struct Layout {
  uint64_t slots;
  int64_t blocks;
  size_t rep, rank, bsum, bytes;
  explicit Layout(int64_t V)
      : slots(table_slots(V)), blocks((V + kWeldBlock - 1) / kWeldBlock), rep(al256(slots * 4)),
        rank(rep + al256((size_t)V * 4)), bsum(rank + al256((size_t)V * 4)),
        bytes(bsum + al256((size_t)(blocks + 1) * 4)) {}
};

}  // namespace
}  // namespace mcx

using namespace mcx;

extern "C" size_t mcx_weld_workspace_size(int64_t V) {
  return V < 0 ? 0 : Layout(V).bytes;
}

extern "C" int mcx_weld(const int64_t* d_edge_key, const float* d_pos, int64_t stride_floats,
                        int64_t V, float* d_upos, int32_t* d_indices, int64_t* d_nunique,
                        int64_t* h_nunique, void* d_ws, size_t ws_bytes, void* stream) {
  if (V < 0 || V >= ((int64_t)1 << 31) || stride_floats < 3) return MCX_ERR_ARG;
  hipStream_t s = as_stream(stream);
  if (V == 0) {
    if (d_nunique && fill_bytes_zero(d_nunique, sizeof(int64_t), s)) return MCX_ERR_HIP;
    if (h_nunique) {
      MCX_HIP(hipStreamSynchronize(s));
      *h_nunique = 0;
    }
    return MCX_OK;
  }
  if (!d_edge_key || !d_pos || !d_upos || !d_indices) return MCX_ERR_ARG;
  const Layout L(V);
  if (!d_ws || ws_bytes < L.bytes) return MCX_ERR_WORKSPACE;
  const int64_t nb = L.blocks;
  char* b = static_cast<char*>(d_ws);
  uint32_t* table = reinterpret_cast<uint32_t*>(b);
  uint32_t* rep = reinterpret_cast<uint32_t*>(b + L.rep);  // slots, then first occurrences
  uint32_t* rank = reinterpret_cast<uint32_t*>(b + L.rank);
  uint32_t* bsum = reinterpret_cast<uint32_t*>(b + L.bsum);
  int rc = fill_u32(table, kEmpty, (size_t)L.slots, s);
  if (rc) return rc;
  const uint32_t n = (uint32_t)V, mask = (uint32_t)(L.slots - 1);
  hipLaunchKernelGGL(weld_insert_kernel, dim3((unsigned)nb), dim3(kInsert), 0, s, d_edge_key, n, table,
                     mask, rep);
  MCX_HIP(hipGetLastError());
  hipLaunchKernelGGL(weld_rank_kernel, dim3((unsigned)nb), dim3(256), 0, s, n, table, rep, rank,
                     bsum);
  MCX_HIP(hipGetLastError());
  hipLaunchKernelGGL(weld_scan_kernel, dim3(1), dim3(1024), 0, s, bsum, (uint32_t)nb, d_nunique);
  MCX_HIP(hipGetLastError());
  hipLaunchKernelGGL(weld_finish_kernel, dim3(grid_for(V, 256)), dim3(256), 0, s, n, rep, rank,
                     bsum, d_pos, stride_floats, d_indices, d_upos);
  MCX_HIP(hipGetLastError());
  if (h_nunique) {
    uint32_t total = 0;
    MCX_HIP(hipMemcpyAsync(&total, bsum + nb, sizeof(total), hipMemcpyDeviceToHost, s));
    MCX_HIP(hipStreamSynchronize(s));
    *h_nunique = total;
  }
  return MCX_OK;
}
