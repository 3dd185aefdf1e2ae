// mcx_rle.hip -- the `.vol` run-length codec on the GPU (gfx950).
//
// Format (cu_kinect_fusion_v1.cu:1303-1447, for the 4-byte voxel
// cu_voxel_t {short tsdf; ushort w;} of structure.h:14-18): per z slice a
// uint32 byte count, then records u16 {n : 14, v : 2} covering the slice's
// voxels in [y][x] order: v = 1 a run of (+32766, w 0), v = 2 a run of
// (-32766, w 0), v = 3 (and 0 when decoding) a run of the 4-byte voxel that
// follows.  A run is a maximal stretch of equal tsdf (weights are not
// compared; the record keeps the run's first voxel), cut every 0x3fff voxels.
//
// Encode (flat over the slab's voxels, no sequential pass).  A run's bytes are
// known where the next one starts, so a block of 4096 voxels accounts for the
// runs that end in it, and blocks compose: (first and last run start, bytes of
// the runs between) of two neighbours give those of both, with the run that
// crosses from one to the other.
//   E1 runs    the state of every block;
//   scan       exclusive composition of the states (groups of 1024);
//   E2 write   the volume's second and last reading: every block writes the
//              records of the runs that end in it (a crossing run's by all
//              its threads) and, for a slice start, the slice's byte count.
// Bound by the two readings.  512^3 (a fused room, 28 MB of dump) in one call:
// E1 104 us (the copy rate), E2 190; in calls of 2^24 voxels 670 us, most of it
// eight ramps and read-backs.  With lists of run starts and of their bytes (16
// bytes of workspace a voxel, two more passes, the number of runs read back)
// it took 397 and 824.  1024 voxels a block: 720 instead of 670.
// Decode (records are 1 or 3 words, so a record boundary cannot be told
// from a word alone):
//   D0 index   each slice's payload range from the caller's offsets;
//   D1 resolve one workgroup per slice, 16 K words at a time through LDS;
//              every thread parses a 32-word chunk from each of the three
//              possible entry offsets (the first record at or after the chunk
//              start begins 0, 1 or 2 words in), giving a map entry offset ->
//              (exit offset, voxels, records); a block scan composes the maps,
//              so each chunk learns its true entry offset, voxel and record
//              positions; it re-parses and writes (first voxel, value) per
//              record and, for every 4096-voxel tile, the record covering the
//              tile's start;
//   D2 fill    one workgroup per tile stages the tile's runs in LDS, marks the
//              voxels where they start and writes every voxel by rank
//              (coalesced, balanced whatever the run lengths).
// The same dump: D1 84 us, bound by the chains of dependent record headers, D2
// 114 us, the rate that memory takes writes at; 64-word chunks parsed from
// memory one entry after the other took 196, a search for each voxel's run
// 200.  D1 with 1024 threads or 16-word chunks 99-134 us (more maps to compose
// for shorter chains), 256 threads 117-150.
// Malformed input (a run of length 0, runs past the slice, a truncated
// record, bytes left over, offsets outside the dump) is detected on the
// device and reported as MCX_ERR_FORMAT; every access stays in bounds.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mcx_internal.h"

namespace mcx {
namespace {

constexpr uint32_t kRunMax = 0x3fff;
constexpr int kMaxT = 32766;
constexpr int kSub = 1024;        // encode: voxels a workgroup reads at once (4 a thread)
constexpr int kSubs = 4;          // ... and how many times
constexpr int kEncBlk = kSub * kSubs;  // voxels of an encode block
constexpr int kBlk = 1024;        // states of a scan group
constexpr int64_t kMaxRuns = (int64_t)1 << 31;  // more are refused
constexpr int kChunkWords = 32;   // decode: words per speculative-parse chunk
constexpr int kResolve = 512;     // decode: threads (chunks) per slice and round
constexpr int kFillTile = 4096;   // decode: voxels per fill workgroup
constexpr uint32_t kNoRecord = 0xffffffffu;

__device__ __forceinline__ int tsdf_of(uint32_t v) { return (int)(int16_t)(v & 0xffffu); }
__device__ __forceinline__ bool saturated(int t) { return t == kMaxT || t == -kMaxT; }

size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

// ---------------------------------------------------------------- encode
typedef uint32_t u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));  // 4-byte aligned

// The runs of a stretch of voxels: where the first and the last start (flat
// indices; first < 0: none starts here), bytes of those that end before the
// last start, how many start, and the last one's bytes a record and lead (a
// slice's byte count before its first run).
struct Runs {
  int64_t first, last, bytes, count;
  uint32_t rec, lead;
};

__device__ __forceinline__ uint32_t records(int64_t s, int64_t e) {  // of a run [s, e)
  return ((uint32_t)(e - s) + kRunMax - 1) / kRunMax;
}

// Bytes of a's last run, which ends at e.
__device__ __forceinline__ int64_t last_bytes(const Runs& a, int64_t e) {
  return a.first < 0 ? 0 : (int64_t)records(a.last, e) * a.rec + a.lead;
}

// a, then b
__device__ __forceinline__ Runs then(const Runs& a, const Runs& b) {
  Runs o = b.first < 0 ? a : b;
  o.first = a.first < 0 ? b.first : a.first;
  o.bytes = a.bytes + b.bytes + (b.first < 0 ? 0 : last_bytes(a, b.first));
  o.count = a.count + b.count;
  return o;
}

__device__ __forceinline__ Runs no_runs() { return Runs{-1, -1, 0, 0, 0, 0}; }

__device__ __forceinline__ Runs shfl_up_runs(const Runs& a, int d) {
  Runs o;
  o.first = __shfl_up((long long)a.first, d, kWave);
  o.last = __shfl_up((long long)a.last, d, kWave);
  o.bytes = __shfl_up((long long)a.bytes, d, kWave);
  o.count = __shfl_up((long long)a.count, d, kWave);
  o.rec = __shfl_up(a.rec, d, kWave);
  o.lead = __shfl_up(a.lead, d, kWave);
  return o;
}

// Exclusive composition of 1024 states in place (kBlk a workgroup, four a
// thread); group[block] = all of them.
__global__ __launch_bounds__(256) void enc_scan_kernel(Runs* a, int64_t n, Runs* group) {
  __shared__ Runs s_w[4];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t base = (int64_t)blockIdx.x * kBlk + 4 * tid;
  Runs v[4], all = no_runs();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = base + k < n ? a[base + k] : no_runs();
    all = then(all, v[k]);
  }
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const Runs g = shfl_up_runs(all, d);
    if (lane >= d) all = then(g, all);
  }
  if (lane == 63) s_w[wv] = all;
  __syncthreads();
  Runs pre = no_runs();
  for (int k = 0; k < wv; ++k) pre = then(pre, s_w[k]);
  const Runs up = shfl_up_runs(all, 1);
  if (lane > 0) pre = then(pre, up);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (base + k < n) a[base + k] = pre;
    pre = then(pre, v[k]);
  }
  if (tid == 255) group[blockIdx.x] = pre;
}

// Levels above the first: a[i] becomes what is before it, all the way down.
__global__ __launch_bounds__(256) void enc_lift_kernel(Runs* a, int64_t n, const Runs* group) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = then(group[i / kBlk], a[i]);
}

// The four voxels of a thread and the run starts among them (bit k: the first
// voxel of the slice, or a tsdf that differs from the voxel before it).
struct Four {
  uint32_t v[4];
  uint32_t starts;
};

// sl: a slice, i0: the thread's first voxel; all lanes of a wave take part.
__device__ __forceinline__ Four four_voxels(const uint32_t* __restrict__ sl, int64_t XY,
                                            int64_t i0) {
  Four q;
  if (i0 + 4 <= XY) {
    // one 128-bit load (the slice is 4-byte aligned, which the vector memory
    // path accepts)
    const u32x4a4 v = *reinterpret_cast<const u32x4a4*>(sl + i0);
#pragma unroll
    for (int k = 0; k < 4; ++k) q.v[k] = v[k];
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k) q.v[k] = i0 + k < XY ? sl[i0 + k] : 0u;
  }
  uint32_t before = __shfl_up(q.v[3], 1, kWave);
  if ((threadIdx.x & 63) == 0 && i0 > 0 && i0 < XY) before = sl[i0 - 1];
  q.starts = 0;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const bool change = i0 + k == 0 || tsdf_of(q.v[k]) != tsdf_of(k ? q.v[k - 1] : before);
    if (change && i0 + k < XY) q.starts |= 1u << k;
  }
  return q;
}

// Bytes of a record of a run that starts with voxel v.
__device__ __forceinline__ uint32_t record_bytes(uint32_t v) {
  return saturated(tsdf_of(v)) ? 2u : 6u;
}

// Bytes of one record for each of a thread's run starts (no run inside a
// block is longer than a record: kEncBlk <= kRunMax), and the slice's lead.
__device__ __forceinline__ uint32_t four_bytes(const Four& q, int64_t i0) {
  uint32_t b = i0 == 0 ? 4u : 0u;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if (q.starts >> k & 1u) b += record_bytes(q.v[k]);
  return b;
}
static_assert(kEncBlk <= (int)kRunMax, "a run inside a block is one record");

// grid (blocks per slice, nz)
__global__ __launch_bounds__(256) void enc_runs_kernel(const uint32_t* __restrict__ vol,
                                                       int64_t XY, Runs* a) {
  // of each wave: bytes of a record for every start (and the lead) << 16 |
  // starts; first start (kEncBlk: none) and last start (-1) in the block;
  // bytes of the last one's records, and its lead in bit 8
  __shared__ uint32_t s_sum[4], s_rec[4];
  __shared__ int s_first[4], s_last[4];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t z = blockIdx.y;
  const int64_t base = (int64_t)blockIdx.x * kEncBlk;
  Four q[kSubs];
#pragma unroll
  for (int j = 0; j < kSubs; ++j) q[j] = four_voxels(vol + z * XY, XY, base + j * kSub + 4 * tid);
  uint32_t sum = 0, rec = 0;
  int first = kEncBlk, last = -1;
#pragma unroll
  for (int j = 0; j < kSubs; ++j) {
    const uint64_t any = __ballot(q[j].starts != 0);
    if (any == 0) continue;
    const int i = j * kSub + 4 * tid;
    sum += four_bytes(q[j], base + i) << 16 | (uint32_t)__popc(q[j].starts);
    const int k = 31 - __clz(q[j].starts | 1u);
    const uint32_t v = k == 0 ? q[j].v[0] : k == 1 ? q[j].v[1] : k == 2 ? q[j].v[2] : q[j].v[3];
    const int lo = __ffsll((unsigned long long)any) - 1, hi = 63 - __clzll((long long)any);
    const uint32_t r = record_bytes(v) | (base + i + k == 0 ? 4u << 8 : 0u);
    first = min(first, __builtin_amdgcn_readlane(i + __ffs(q[j].starts) - 1, lo));
    last = __builtin_amdgcn_readlane(i + k, hi);
    rec = __builtin_amdgcn_readlane(r, hi);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);  // a wave's bytes < 2^13
  if (lane == 0) {
    s_sum[wv] = sum;
    s_rec[wv] = rec;
    s_first[wv] = first;
    s_last[wv] = last;
  }
  __syncthreads();
  if (tid == 0) {
    sum = s_sum[0];
    for (int w = 1; w < 4; ++w) {
      sum += s_sum[w];
      first = min(first, s_first[w]);
      if (s_last[w] > last) {
        last = s_last[w];
        rec = s_rec[w];
      }
    }
    Runs r = no_runs();
    if (last >= 0) {
      r.first = z * XY + base + first;
      r.last = z * XY + base + last;
      r.rec = rec & 0xffu;
      r.lead = rec >> 8;
      r.bytes = (int64_t)(sum >> 16) - r.rec - r.lead;
      r.count = sum & 0xffffu;
    }
    a[z * gridDim.x + blockIdx.x] = r;
  }
}

__device__ __forceinline__ void put16(uint16_t* out16, int64_t byte_pos, uint32_t v) {
  out16[byte_pos >> 1] = (uint16_t)v;
}

// One record of n voxels, the first of them v.
__device__ __forceinline__ void put_record(uint16_t* out16, int64_t pos, uint32_t n, uint32_t v) {
  const int t = tsdf_of(v);
  const uint32_t kind = t == kMaxT ? 1u : t == -kMaxT ? 2u : 3u;
  put16(out16, pos, n | (kind << 14));
  if (kind == 3u) {
    put16(out16, pos + 2, v & 0xffffu);
    put16(out16, pos + 4, v >> 16);
  }
}

// What is before block b of the slab (group: null if there is one group).
__device__ __forceinline__ Runs before(const Runs* a, const Runs* group, int64_t b) {
  return group ? then(group[b / kBlk], a[b]) : a[b];
}

// All records of the last run of `a`, which ends at e, the last of them ending
// at byte `end`; the workgroup's threads take them in turn.
__device__ __forceinline__ void put_run(uint16_t* out16, const uint32_t* __restrict__ vol,
                                        const Runs& a, int64_t e, int64_t end) {
  const uint32_t n = records(a.last, e);
  for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
    const int64_t r = a.last + (int64_t)k * kRunMax;
    put_record(out16, end - (int64_t)(n - k) * a.rec, (uint32_t)min((int64_t)kRunMax, e - r),
               vol[r]);
  }
}

// all: the slab's state; totals: [bytes, runs]
__global__ __launch_bounds__(256) void enc_write_kernel(const uint32_t* __restrict__ vol,
                                                        int64_t XY, int64_t N, const Runs* a,
                                                        const Runs* group, const Runs* all,
                                                        uint16_t* out16, int64_t cap,
                                                        int64_t* totals, int64_t* d_total) {
  // of each run of 256 voxels: bytes, and the first start in the block
  // (kEncBlk: none)
  __shared__ uint32_t s_bytes[4 * kSubs];
  __shared__ uint32_t s_first[4 * kSubs];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t z = blockIdx.y, nblk = (int64_t)gridDim.x * gridDim.y;
  const int64_t b = z * gridDim.x + blockIdx.x;
  const int64_t base = (int64_t)blockIdx.x * kEncBlk;
  // all loads at once: a block's life is short
  Four q[kSubs];
#pragma unroll
  for (int j = 0; j < kSubs; ++j) q[j] = four_voxels(vol + z * XY, XY, base + j * kSub + 4 * tid);
  const Runs pre = before(a, group, b);
  const Runs end = *all;
  const int64_t total = end.bytes + last_bytes(end, N);
  if (b == 0 && tid == 0) {
    totals[0] = total;
    totals[1] = end.count;
    if (d_total && end.count < kMaxRuns) *d_total = total;
  }
  if (total > cap || end.count >= kMaxRuns) return;
  uint64_t any[kSubs];
  uint32_t off[kSubs];  // bytes of the run's earlier starts
#pragma unroll
  for (int j = 0; j < kSubs; ++j) {
    any[j] = __ballot(q[j].starts != 0);
    uint32_t bytes = 0, first = kEncBlk;
    off[j] = 0;
    if (any[j]) {
      const int i = j * kSub + 4 * tid;
      const uint32_t mine = four_bytes(q[j], base + i);
      const uint32_t inc = wave_incl_scan32(mine);
      off[j] = inc - mine;
      bytes = __builtin_amdgcn_readlane(inc, 63);
      first = __builtin_amdgcn_readlane(i + __ffs(q[j].starts) - 1,
                                        __ffsll((unsigned long long)any[j]) - 1);
    }
    if (lane == 0) {
      s_bytes[4 * j + wv] = bytes;
      s_first[4 * j + wv] = first;
    }
  }
  __syncthreads();
  uint32_t first = kEncBlk;
#pragma unroll
  for (int k = 4 * kSubs - 1; k >= 0; --k) first = min(first, s_first[k]);
  if (first < (uint32_t)kEncBlk) {  // uniform over the block
    // the run before the block's first, which ends here
    const int64_t begin = pre.bytes + last_bytes(pre, z * XY + base + first);
    if (pre.first >= 0) put_run(out16, vol, pre, z * XY + base + first, begin);
#pragma unroll
    for (int j = 0; j < kSubs; ++j) {
      if (any[j] == 0) continue;
      const int i = j * kSub + 4 * tid;
      // what the earlier runs of 256 take, and the next start after this one
      uint32_t skip = 0, next = kEncBlk;
#pragma unroll
      for (int k = 0; k < 4 * kSubs; ++k) {
        if (k < 4 * j + wv) skip += s_bytes[k];
        if (k > 4 * j + wv) next = min(next, s_first[k]);
      }
      // the next start after this thread's own
      const uint64_t later = lane < 63 ? any[j] >> (lane + 1) << (lane + 1) : 0;
      const uint32_t in_wave = __shfl((uint32_t)(i + __ffs(q[j].starts) - 1),
                                      later ? __ffsll((unsigned long long)later) - 1 : 0, kWave);
      if (later) next = in_wave;
      int64_t pos = begin + skip + off[j];
      if (base + i == 0) {
        int64_t stop = total;
        if (z + 1 < (int64_t)gridDim.y) {
          const Runs p = before(a, group, b + gridDim.x);
          stop = p.bytes + last_bytes(p, (z + 1) * XY);
        }
        const uint32_t size = (uint32_t)(stop - pos - 4);
        put16(out16, pos, size & 0xffffu);
        put16(out16, pos + 2, size >> 16);
        pos += 4;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (!(q[j].starts >> k & 1u)) continue;
        const uint32_t above = q[j].starts >> (k + 1);
        const uint32_t at = i + k;
        const uint32_t stop = above ? at + __ffs(above) : next;
        // the block's last run ends in a later block, which writes it
        if (stop < (uint32_t)kEncBlk) put_record(out16, pos, stop - at, q[j].v[k]);
        pos += record_bytes(q[j].v[k]);
      }
    }
  }
  if (b + 1 == nblk) put_run(out16, vol, end, N, total);
}

// ---------------------------------------------------------------- decode
struct SliceInfo {
  int64_t word_base;  // first payload word within the dump
  uint32_t words;     // payload words
  uint32_t nrec;      // records (set by the resolve kernel)
};

// Map entry offset p (0..2) -> (exit offset, voxels, records) of a chunk.
struct Fn {
  uint32_t ex;  // 2 bits per entry offset
  uint32_t v[3];
  uint32_t r[3];
};

__device__ __forceinline__ uint32_t ex_at(uint32_t ex, uint32_t p) { return (ex >> (2 * p)) & 3u; }
__device__ __forceinline__ uint32_t sel3(const uint32_t* a, uint32_t p) {
  return p == 0 ? a[0] : p == 1 ? a[1] : a[2];
}
__device__ __forceinline__ uint32_t sat_add(uint32_t a, uint32_t b) {
  const uint32_t s = a + b;
  return s < a ? 0xffffffffu : s;
}

__device__ __forceinline__ Fn fn_identity() {
  Fn f;
  f.ex = 0u | (1u << 2) | (2u << 4);
#pragma unroll
  for (int p = 0; p < 3; ++p) f.v[p] = f.r[p] = 0;
  return f;
}

// a, then b
__device__ __forceinline__ Fn compose(const Fn& a, const Fn& b) {
  Fn o;
  o.ex = 0;
#pragma unroll
  for (uint32_t p = 0; p < 3; ++p) {
    const uint32_t e = ex_at(a.ex, p);
    o.ex |= ex_at(b.ex, e) << (2 * p);
    o.v[p] = sat_add(a.v[p], sel3(b.v, e));
    o.r[p] = a.r[p] + sel3(b.r, e);
  }
  return o;
}

__device__ __forceinline__ Fn shfl_up_fn(const Fn& f, int d) {
  Fn g;
  g.ex = __shfl_up(f.ex, d, kWave);
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    g.v[p] = __shfl_up(f.v[p], d, kWave);
    g.r[p] = __shfl_up(f.r[p], d, kWave);
  }
  return g;
}

__device__ __forceinline__ uint32_t record_words(uint32_t hdr) {
  const uint32_t v = hdr >> 14;
  return v == 1u || v == 2u ? 1u : 3u;
}

__global__ __launch_bounds__(256) void dec_index_kernel(const uint16_t* __restrict__ d16,
                                                        int64_t dump_bytes, const int64_t* offs,
                                                        int nz, SliceInfo* info, uint32_t* err) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nz) return;
  const int64_t off = offs[j];
  SliceInfo si{0, 0, 0};
  if (off >= 0 && (off & 1) == 0 && off + 4 <= dump_bytes) {
    const uint32_t size = (uint32_t)d16[off >> 1] | ((uint32_t)d16[(off >> 1) + 1] << 16);
    if ((size & 1u) == 0 && size >= 2 && (int64_t)size <= dump_bytes - off - 4) {
      si.word_base = (off + 4) >> 1;
      si.words = size >> 1;
    }
  }
  if (si.words == 0) atomicOr(err, 1u);
  info[j] = si;
}

// Place of word i of a round in LDS: a dword of padding per chunk, so that the
// lanes' chunks (17 dwords apart) start in different banks.
__device__ __forceinline__ int staged(int i) { return i + 2 * (i / kChunkWords); }

__global__ __launch_bounds__(kResolve) void dec_resolve_kernel(const uint16_t* __restrict__ d16,
                                                               int64_t XY, int tps,
                                                               SliceInfo* info, uint2* rec,
                                                               uint32_t* tile_first,
                                                               uint32_t* err) {
  constexpr int kRound = kResolve * kChunkWords;  // words a workgroup resolves at once
  __shared__ Fn s_fn[kResolve / kWave];
  __shared__ uint16_t s_w[kRound + 2 * kResolve + 4];  // and the two after them
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int j = blockIdx.x;
  const SliceInfo si = info[j];
  if (si.words == 0) return;  // flagged by the index kernel
  const uint16_t* __restrict__ w = d16 + si.word_base;
  const int64_t L = si.words;
  uint2* rs = rec + si.word_base;
  uint32_t* tf = tile_first + (int64_t)j * tps;
  uint32_t cp = 0, cv = 0, cr = 0;  // carry: entry offset, voxels, records
  bool bad = false;
  for (int64_t w0 = 0; w0 < L; w0 += kRound) {
    const int n_words = (int)min((int64_t)kRound, L - w0);
    uint16_t in[kChunkWords];
#pragma unroll
    for (int k = 0; k < kChunkWords; ++k) {
      const int i = k * kResolve + tid;
      in[k] = i < n_words ? w[w0 + i] : (uint16_t)0;
    }
#pragma unroll
    for (int k = 0; k < kChunkWords; ++k) s_w[staged(k * kResolve + tid)] = in[k];
    if (tid < 2) s_w[staged(kRound + tid)] = w0 + kRound + tid < L ? w[w0 + kRound + tid] : 0;
    __syncthreads();
    const int beg = tid * kChunkWords;
    const int end = min(beg + kChunkWords, n_words);
    Fn f = fn_identity();
    if (beg < n_words) {
      // the three entry offsets side by side: three loads in flight
      int pos[3] = {beg, beg + 1, beg + 2};
      bool more = true;
      while (more) {
        more = false;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          if (pos[p] < end) {
            const uint32_t h = s_w[staged(pos[p])];
            f.v[p] = sat_add(f.v[p], h & kRunMax);
            ++f.r[p];
            pos[p] += record_words(h);
            more = true;
          }
        }
      }
      f.ex = 0;
#pragma unroll
      for (int p = 0; p < 3; ++p) f.ex |= (uint32_t)(pos[p] - end) << (2 * p);
    }
    // inclusive scan of the maps over the block
    Fn incl = f;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
      const Fn g = shfl_up_fn(incl, d);
      if (lane >= d) incl = compose(g, incl);
    }
    if (lane == 63) s_fn[wv] = incl;
    __syncthreads();
    Fn pre = fn_identity(), total = fn_identity();
    for (int k = 0; k < kResolve / kWave; ++k) {
      if (k == wv) pre = total;
      total = compose(total, s_fn[k]);
    }
    const Fn up = shfl_up_fn(incl, 1);
    const Fn excl = lane == 0 ? pre : compose(pre, up);
    if (beg < n_words) {
      // true entry state of this chunk, then its records
      int pos = beg + ex_at(excl.ex, cp);
      uint64_t v0 = (uint64_t)sat_add(cv, sel3(excl.v, cp));
      uint32_t r = cr + sel3(excl.r, cp);
      while (pos < end) {
        const uint32_t h = s_w[staged(pos)];
        const uint32_t n = h & kRunMax, v = h >> 14;
        const uint32_t len = record_words(h);
        if (n == 0 || w0 + pos + len > L || v0 + n > (uint64_t)XY) {
          bad = true;
          break;
        }
        uint32_t val;
        if (v == 1u)
          val = (uint32_t)(uint16_t)kMaxT;
        else if (v == 2u)
          val = (uint32_t)(uint16_t)(int16_t)-kMaxT;
        else
          val = (uint32_t)s_w[staged(pos + 1)] | ((uint32_t)s_w[staged(pos + 2)] << 16);
        rs[r] = make_uint2((uint32_t)v0, val);
        for (uint64_t t = (v0 + kFillTile - 1) / kFillTile; t * kFillTile < v0 + n; ++t)
          tf[t] = r;
        v0 += n;
        ++r;
        pos += len;
      }
    }
    const uint32_t np = ex_at(total.ex, cp);
    cv = sat_add(cv, sel3(total.v, cp));
    cr += sel3(total.r, cp);
    cp = np;
    __syncthreads();  // s_w and s_fn are rewritten by the next round
  }
  if (bad) atomicOr(err, 2u);
  if (tid == 0) {
    if (cp != 0 || (int64_t)cv != XY) atomicOr(err, 4u);
    info[j].nrec = cr;
  }
}

__global__ __launch_bounds__(256) void dec_fill_kernel(const SliceInfo* info, int64_t XY, int tps,
                                                       const uint2* __restrict__ rec,
                                                       const uint32_t* tile_first,
                                                       const uint32_t* err, uint32_t* out) {
  // the tile's run values in order, a bit per voxel where a run starts, and
  // the starts before each 32 voxels: a voxel's run is a rank, not a search
  __shared__ uint32_t s_val[kFillTile + 1];
  __shared__ uint32_t s_bit[kFillTile / 32];
  __shared__ uint32_t s_pre[kFillTile / 32];
  if (*err) return;  // malformed input: the call reports it, outputs are undefined
  const int tid = threadIdx.x;
  const int j = blockIdx.y, t = blockIdx.x;
  const SliceInfo si = info[j];
  const uint32_t* tf = tile_first + (int64_t)j * tps + t;
  const uint32_t r0 = tf[0];
  if (r0 == kNoRecord || r0 >= si.nrec) return;
  // up to the run that covers the next tile's first voxel (it may start there)
  const uint32_t r1 = t + 1 < tps ? min(tf[1], si.nrec - 1) : si.nrec - 1;
  const int m = (int)min(r1 - r0, (uint32_t)kFillTile) + 1;
  const uint2* rs = rec + si.word_base + r0;
  const int64_t vb = (int64_t)t * kFillTile;
  const int64_t ve = min(vb + kFillTile, XY);
  if (tid < kFillTile / 32) s_bit[tid] = tid == 0 ? 1u : 0u;  // the first run
  __syncthreads();
  for (int i = tid; i < m; i += 256) {
    const uint2 r = rs[i];
    s_val[i] = r.y;
    const uint32_t q = r.x - (uint32_t)vb;
    if (i > 0 && q < (uint32_t)kFillTile) atomicOr(&s_bit[q >> 5], 1u << (q & 31));
  }
  __syncthreads();
  if (tid < kWave) {
    const uint32_t a = __popc(s_bit[2 * tid]), b = __popc(s_bit[2 * tid + 1]);
    const uint32_t inc = wave_incl_scan32(a + b);
    s_pre[2 * tid] = inc - a - b;
    s_pre[2 * tid + 1] = inc - b;
  }
  static_assert(kFillTile / 32 == 2 * kWave, "two words of starts a lane");
  __syncthreads();
  uint32_t* o = out + (int64_t)j * XY;
#pragma unroll
  for (int k = 0; k < kFillTile / 1024; ++k) {
    const int qr = k * 1024 + 4 * tid;
    const int64_t q = vb + qr;
    if (q >= ve) break;
    const uint32_t bits = s_bit[qr >> 5], pre = s_pre[qr >> 5];
    u32x4a4 v4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t upto = 0xffffffffu >> (31 - ((qr & 31) + e));
      v4[e] = s_val[pre + __popc(bits & upto) - 1];
    }
    if (q + 3 < ve) {
      *reinterpret_cast<u32x4a4*>(o + q) = v4;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (q + e < ve) o[q + e] = v4[e];
    }
  }
}

unsigned grid_for(int64_t n, int64_t per) { return (unsigned)((n + per - 1) / per); }

}  // namespace
}  // namespace mcx

using namespace mcx;

// ------------------------------------------------------------------ C ABI
namespace {
// States of all levels of the scan over n blocks, the last level's single one
// included.
int64_t run_states(int64_t n) {
  const int64_t ng = (n + kBlk - 1) / kBlk;
  return n + (ng > 1 ? run_states(ng) : 1);
}

// a[i] becomes what is before it in its group of kBlk, the groups' prefixes
// (from the slab's start) follow a; *all = the state of everything.
int scan_runs(Runs* a, int64_t n, Runs** all, hipStream_t s) {
  const int64_t ng = (n + kBlk - 1) / kBlk;
  Runs* group = a + n;
  hipLaunchKernelGGL(enc_scan_kernel, dim3((unsigned)ng), dim3(256), 0, s, a, n, group);
  MCX_HIP(hipGetLastError());
  if (ng == 1) {
    *all = group;
    return MCX_OK;
  }
  const int rc = scan_runs(group, ng, all, s);
  if (rc) return rc;
  if (ng > kBlk) {
    hipLaunchKernelGGL(enc_lift_kernel, dim3((unsigned)((ng + 255) / 256)), dim3(256), 0, s,
                       group, ng, group + ng);
    MCX_HIP(hipGetLastError());
  }
  return MCX_OK;
}
}  // namespace

extern "C" size_t mcx_rle_encode_workspace_size(int X, int Y, int nz) {
  if (X < 1 || Y < 1 || nz < 1) return 0;
  const int64_t nblk = ((int64_t)X * Y + kEncBlk - 1) / kEncBlk * nz;
  return al256((size_t)run_states(nblk) * sizeof(Runs)) + 256;
}

extern "C" size_t mcx_rle_encode_bound(int X, int Y, int nz) {
  if (X < 1 || Y < 1 || nz < 1) return 0;
  return (size_t)nz * (4 + 6 * (size_t)X * Y);
}

extern "C" int mcx_rle_encode(const void* d_vol, int X, int Y, int Z, int z0, int nz, void* d_dump,
                              size_t dump_cap, int64_t* d_dump_bytes, int64_t* h_dump_bytes,
                              void* d_ws, size_t ws_bytes, void* stream) {
  if (!d_vol || X < 1 || Y < 1 || Z < 1 || z0 < 0 || nz < 1 || (int64_t)z0 + nz > Z)
    return MCX_ERR_ARG;
  if ((int64_t)X * Y >= ((int64_t)1 << 31)) return MCX_ERR_ARG;
  if (dump_cap > 0 && (!d_dump || (reinterpret_cast<uintptr_t>(d_dump) & 1))) return MCX_ERR_ARG;
  if (!d_ws || ws_bytes < mcx_rle_encode_workspace_size(X, Y, nz)) return MCX_ERR_WORKSPACE;
  hipStream_t s = as_stream(stream);
  const int64_t XY = (int64_t)X * Y, N = XY * nz;
  const int64_t bps = (XY + kEncBlk - 1) / kEncBlk, nblk = bps * nz;
  if (bps > 0x7fffffff || nz > 65535) return MCX_ERR_ARG;
  const uint32_t* vol = static_cast<const uint32_t*>(d_vol) + (int64_t)z0 * XY;
  int64_t* totals = static_cast<int64_t*>(d_ws);
  Runs* a = reinterpret_cast<Runs*>(static_cast<char*>(d_ws) + 256);
  const dim3 g2((unsigned)bps, (unsigned)nz);
  hipLaunchKernelGGL(enc_runs_kernel, g2, dim3(256), 0, s, vol, XY, a);
  MCX_HIP(hipGetLastError());
  Runs* all = nullptr;
  const int rc = scan_runs(a, nblk, &all, s);
  if (rc) return rc;
  const Runs* group = nblk > kBlk ? a + nblk : nullptr;  // nothing is before a single one
  hipLaunchKernelGGL(enc_write_kernel, g2, dim3(256), 0, s, vol, XY, N, a,
                     group, all, static_cast<uint16_t*>(d_dump),
                     (int64_t)dump_cap, totals, d_dump_bytes);
  MCX_HIP(hipGetLastError());
  int64_t h[2] = {0, 0};
  MCX_HIP(hipMemcpyAsync(h, totals, sizeof(h), hipMemcpyDeviceToHost, s));
  MCX_HIP(hipStreamSynchronize(s));
  const int64_t total = h[0];
  if (h[1] < nz || h[1] > N) return MCX_ERR_INTERNAL;
  if (h[1] >= kMaxRuns) return MCX_ERR_UNSUPPORTED;
  if (h_dump_bytes) *h_dump_bytes = total;
  return total > (int64_t)dump_cap ? MCX_ERR_CAPACITY : MCX_OK;
}

extern "C" size_t mcx_rle_decode_workspace_size(int64_t dump_bytes, int X, int Y, int nz) {
  if (dump_bytes < 0 || X < 1 || Y < 1 || nz < 1) return 0;
  const int64_t XY = (int64_t)X * Y;
  const int64_t tps = (XY + kFillTile - 1) / kFillTile;
  const size_t words = (size_t)(dump_bytes / 2) + 1;
  return 256 + al256((size_t)nz * sizeof(SliceInfo)) + al256((size_t)nz * 8) +
         al256((size_t)nz * tps * 4) + 2 * al256(words * 4);
}

extern "C" int mcx_rle_decode(const void* d_dump, int64_t dump_bytes,
                              const int64_t* h_slice_offsets, int nz, int X, int Y, void* d_vol,
                              void* d_ws, size_t ws_bytes, void* stream) {
  if (!d_dump || dump_bytes < 6 || !h_slice_offsets || nz < 1 || X < 1 || Y < 1 || !d_vol)
    return MCX_ERR_ARG;
  if (reinterpret_cast<uintptr_t>(d_dump) & 1) return MCX_ERR_ARG;
  const int64_t XY = (int64_t)X * Y;
  if (XY >= ((int64_t)1 << 31) || nz > 65535) return MCX_ERR_ARG;
  if (!d_ws || ws_bytes < mcx_rle_decode_workspace_size(dump_bytes, X, Y, nz))
    return MCX_ERR_WORKSPACE;
  hipStream_t s = as_stream(stream);
  const int64_t tps = (XY + kFillTile - 1) / kFillTile;
  char* b = static_cast<char*>(d_ws);
  uint32_t* err = reinterpret_cast<uint32_t*>(b);
  b += 256;
  SliceInfo* info = reinterpret_cast<SliceInfo*>(b);
  b += al256((size_t)nz * sizeof(SliceInfo));
  int64_t* offs = reinterpret_cast<int64_t*>(b);
  b += al256((size_t)nz * 8);
  uint32_t* tile_first = reinterpret_cast<uint32_t*>(b);
  b += al256((size_t)nz * tps * 4);
  uint2* rec = reinterpret_cast<uint2*>(b);  // first voxel and value of each record
  MCX_HIP(hipMemcpyAsync(offs, h_slice_offsets, (size_t)nz * 8, hipMemcpyHostToDevice, s));
  int rc = fill_u32(err, 0u, 1, s);
  if (!rc) rc = fill_u32(tile_first, kNoRecord, (size_t)nz * tps, s);
  if (rc) return rc;
  const uint16_t* d16 = static_cast<const uint16_t*>(d_dump);
  hipLaunchKernelGGL(dec_index_kernel, dim3(grid_for(nz, 256)), dim3(256), 0, s, d16, dump_bytes,
                     offs, nz, info, err);
  MCX_HIP(hipGetLastError());
  hipLaunchKernelGGL(dec_resolve_kernel, dim3((unsigned)nz), dim3(kResolve), 0, s, d16, XY,
                     (int)tps, info, rec, tile_first, err);
  MCX_HIP(hipGetLastError());
  hipLaunchKernelGGL(dec_fill_kernel, dim3((unsigned)tps, (unsigned)nz), dim3(256), 0, s, info, XY,
                     (int)tps, rec, tile_first, err, static_cast<uint32_t*>(d_vol));
  MCX_HIP(hipGetLastError());
  uint32_t herr = 0;
  MCX_HIP(hipMemcpyAsync(&herr, err, sizeof(herr), hipMemcpyDeviceToHost, s));
  MCX_HIP(hipStreamSynchronize(s));
  return herr ? MCX_ERR_FORMAT : MCX_OK;
}
