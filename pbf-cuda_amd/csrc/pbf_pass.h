// pbf_pass.h — the generic neighbour-pass kernels of the gfx950 PBF step,
// instantiated by each translation unit over its pass policies.
//
// A pass policy P defines, for one neighbour pass:
//   Args                 kernel arguments (device arrays)
//   Target, Acc          a target's own data; its running sum (<= 8 floats)
//   target(a, i, c)      load target i
//   screen(a)            the float4 array whose x, y, z the screening tests
//   kCoarse              screen on the screening coordinates (HeavyLists::coarse)
//                        instead: every pair beyond h adds exactly 0
//   load_f(a, j)         candidate data for the pair term
//   hit(t, d, c)         cheap test on the candidate's x, y, z d: false only
//                        if the pair adds exactly 0 (i itself has d == t.x)
//   near(t, d, c)        (with kNear) the same as the sign of a number: it may
//                        be positive or zero only if the pair adds exactly 0
//   add(acc, t, j, d, c, a) the pair term (the body of the reference's loop)
//   accumulate(tot, p)   tot += a chunk's partial sum
//   finish(a, t, s, c, g) store the result of target t
// Each neighbour pass is three kernels:
//   light   one work-item per target over the cell-sorted order; workgroups
//           remapped so each XCD's L2 serves runs of neighbouring particles; a
//           heavy target (pbf_device.h: kLightMax, heavy_level, kLevelShare)
//           is appended to the heavy list instead;
//   chunks  one work-item per kChunk-candidate chunk of the heavy targets;
//   combine one work-item per heavy target, adding its chunk sums in order.
// Both follow the canonical summation order of pbf_device.h.
#pragma once

#include "pbf_device.h"
#include "pbf_launch.h"
#include "pbf_team.h"

namespace pbf {
namespace {

constexpr int kBlock = 256;
// Workgroups an XCD takes in a row (xcd_runs).  One contiguous range per XCD left
// the busiest XCD with 1.2 to 1.4 times the mean work (collapsing and spread 1M
// dam, 4M under the sweeping wall).  Light kernels: runs of 128 workgroups (32K
// particles, a few x-planes, whose neighbours then share the L2) took the 4M
// frame from 16.8 to 15.8 ms and the spread 1M step from 1116 to 1080 us, the
// dense 1M step unchanged; runs of 64 cost that one 1.5%.  Chunk kernels: the
// list's order already mixes regions and a pile's chunks, all hits, lie
// together, so short runs: dense 1M step 2575 -> 2413 us with runs of 8 (64:
// 2424, 1: 2420).
constexpr int kLightRun = 128;
constexpr int kChunkRun = 8;
constexpr int kRankBuckets = 64;  // one wavefront scans them
// Blocks of 64 candidates whose hits the light kernels evaluate in one loop.
#ifndef PBF_LIGHT_GROUP
#define PBF_LIGHT_GROUP 2
#endif
constexpr int kLightGroup = PBF_LIGHT_GROUP;
inline size_t light_lds_bytes(int lb) { return (size_t)kSeqEntries * lb * sizeof(uint2); }

// Minimum wavefronts per SIMD the neighbour kernels are compiled for (caps
// their registers).
#ifndef PBF_PASS_WAVES
#define PBF_PASS_WAVES 1
#endif

inline int blocks_for(long long n) { return (int)((n + kBlock - 1) / kBlock); }

// Floats per chunk partial of pass policy P: its Acc, packed (the partial
// buffer holds kPartialWords floats per slot, the largest Acc).
template <class P>
__host__ __device__ constexpr uint32_t partial_words() {
  static_assert(sizeof(typename P::Acc) % sizeof(float) == 0, "Acc must be floats");
  static_assert(sizeof(typename P::Acc) <= kPartialWords * sizeof(float), "partial too large");
  return (uint32_t)(sizeof(typename P::Acc) / sizeof(float));
}

// ---------------------------------------------------------------------------
// The hit-mask hooks of sweep_seq for target ti with m candidates under
// policy P (MaskMode, pbf_device.h).
template <class P>
struct MaskIO {
  const HeavyLists& hl;
  uint32_t ti, m;
  __device__ __forceinline__ bool kept() const {
    return hl.masks != nullptr && m <= kMaskBlocks * kChunk;
  }
  __device__ __forceinline__ bool get(uint32_t b, uint32_t& lo, uint32_t& hi) const {
    if constexpr (MaskMode<P>::value == kMaskLoad) {
      if (kept()) {
        const uint64_t mask = hl.masks[(size_t)b * hl.mask_stride + ti];
        lo = (uint32_t)mask;
        hi = (uint32_t)(mask >> 32);
        return true;
      }
    }
    return false;
  }
  __device__ __forceinline__ void put(uint32_t b, uint32_t lo, uint32_t hi) const {
    if constexpr (MaskMode<P>::value == kMaskStore) {
      if (kept()) hl.masks[(size_t)b * hl.mask_stride + ti] = ((uint64_t)hi << 32) | lo;
    }
  }
};

// The screening test of one target for sweep_seq, eight candidates at a time.
// ScreenXyz: positions, by the policy's near() (sign bits, one shift of a bit
// pair each) or hit().
template <class P, class = void>
struct NearMode {
  static constexpr bool value = false;
};
template <class P>
struct NearMode<P, std::void_t<decltype(P::kNear)>> {
  static constexpr bool value = P::kNear;
};
template <class P>
struct ScreenXyz {
  const Float4Buf& buf;
  const typename P::Target& t;
  const StepConsts& c;
  // bits of positions u .. u + 7 (those past `last` are the caller's to mask)
  __device__ __forceinline__ uint32_t batch(SeqCursor& c1, uint32_t u, uint32_t last) const {
    uint32_t off[8];
    c1.template offsets8<4>(u, last, off);
    float3 d[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) d[k] = load_xyz_at(buf, off[k]);
    uint32_t b = 0u;
    if constexpr (NearMode<P>::value) {
#pragma unroll
      for (int k = 7; k >= 0; --k)
        b = __builtin_amdgcn_alignbit(b, __float_as_uint(P::near(t, d[k], c)), 31u);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) b |= (P::hit(t, d[k], c) ? 1u : 0u) << k;
    }
    return b;
  }
};
// ScreenCoarse (policies with kCoarse, whose pairs beyond h add nothing):
// screening coordinates, singly (light kernels) or two neighbours a load (chunk
// kernels).  A wavefront's candidates lie in ~35 cache lines however small the
// elements are, and a load costs the L1 that many accesses, so pairs halve the
// accesses: four loads for eight candidates, and one for a pair that two
// columns share, or four where a batch spans more of them.  The instructions
// for those cases cost the light kernels, whose sparse targets meet them in
// every batch, what the accesses save.
template <bool kPairs>
struct ScreenCoarse {
  const Float4Buf& buf;
  uint2 t;
  __device__ __forceinline__ uint32_t shift_in(uint32_t b, int xy, int z) const {
    return __builtin_amdgcn_alignbit(
        b, (uint32_t)screen_near(t, make_uint2((uint32_t)xy, (uint32_t)z)), 31u);
  }
  __device__ __forceinline__ uint32_t batch(SeqCursor& c1, uint32_t u, uint32_t last) const {
    uint32_t b = 0u;
    if constexpr (!kPairs) {
      uint32_t off[8];
      c1.template offsets8<3>(u, last, off);
      pbf_i32x2 d[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) d[k] = pbf_raw_buffer_load_i32x2(buf.r, (int)off[k], 0, 0);
#pragma unroll
      for (int k = 7; k >= 0; --k) b = shift_in(b, d[k].x, d[k].y);
    } else {
      uint32_t pair[4], odd[4], split;
      const bool two = c1.pairs8(u, last, pair, odd, split);
      pbf_i32x4 d[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = pbf_raw_buffer_load_i32x4(buf.r, (int)pair[k], 0, 0);
      pbf_i32x2 e[4];
      if (!two) {
#pragma unroll
        for (int k = 0; k < 4; ++k) e[k] = pbf_raw_buffer_load_i32x2(buf.r, (int)odd[k], 0, 0);
      } else if (split < 8u) {
        e[0] = pbf_raw_buffer_load_i32x2(buf.r, (int)odd[0], 0, 0);
      }
#pragma unroll
      for (int k = 3; k >= 0; --k) {
        b = shift_in(b, d[k].z, d[k].w);
        b = shift_in(b, d[k].x, d[k].y);
      }
      if (!two) {
        uint32_t o = 0u;
#pragma unroll
        for (int k = 3; k >= 0; --k) o = shift_in(o, e[k].x, e[k].y) << 1;
        b = (b & 0x55u) | (o & 0xAAu);
      } else if (split < 8u) {
        b = (b & ~(1u << split)) | (shift_in(0u, e[0].x, e[0].y) << split);
      }
    }
    return b;
  }
};
template <class P, class = void>
struct CoarseMode {
  static constexpr bool value = false;
};
template <class P>
struct CoarseMode<P, std::void_t<decltype(P::kCoarse)>> {
  static constexpr bool value = P::kCoarse;
};
// The array a pass screens (kC: its screening coordinates), and the screen of
// target ti.
template <class P, bool kC>
__device__ __forceinline__ Float4Buf screen_buf(const typename P::Args& a, const HeavyLists& hl,
                                                uint32_t n) {
  if constexpr (kC)
    return raw_buf(hl.coarse, (uint64_t)n * 8u);
  else
    return float4_buf(P::screen(a), n);
}
template <class P, bool kC, bool kPairs>
__device__ __forceinline__ auto screen_of(const Float4Buf& buf, const HeavyLists& hl, uint32_t ti,
                                          const typename P::Target& t, const StepConsts& c) {
  if constexpr (kC)
    return ScreenCoarse<kPairs>{buf, hl.coarse[ti]};
  else
    return ScreenXyz<P>{buf, t, c};
}

// Generic neighbour-pass kernels over a pass policy.
// ---------------------------------------------------------------------------

// Light: one work-item per target; the workgroup size is a launch shape
// (64, 128 or 256), the column tables live in dynamic LDS.  A heavy target
// (more candidates than fixed_threshold, or when that is 0 than the
// threshold word the previous pass's combine kernel set) gets one chunk item per kChunk candidates and a
// record, appended with one atomic per workgroup each.  The counters of
// parity pass & 1 belong to this pass; the kernel clears the other parity's
// counters for the next pass (their previous users finished earlier on the
// stream).  If the chunk list is full the lane sums its target itself, still
// chunk by chunk, so the canonical order holds either way.
template <class P, class S, bool kC>
__global__ __launch_bounds__(kBlock, PBF_PASS_WAVES) void k_light(typename P::Args a, int n,
                                                                  StepConsts c, S sc,
                                                                  const uint32_t* __restrict__ cs,
                                                                  HeavyLists hl, int pass,
                                                                  uint32_t fixed_threshold) {
  extern __shared__ uint2 seq_dyn[];
  __shared__ uint32_t key_sh[kBlock];
  __shared__ uint32_t order_sh[kBlock];
  __shared__ uint32_t bucket_sh[kRankBuckets];
  __shared__ uint32_t alloc_sh[2][kBlock / 64];
  uint32_t* rec_cnt = hl.counters + rec_counter(pass & 1);
  uint32_t* item_cnt = hl.counters + item_counter(pass & 1);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    hl.counters[rec_counter((pass + 1) & 1)] = 0u;
    hl.counters[item_counter((pass + 1) & 1)] = 0u;
  }
  const uint32_t word = hl.counters[kThresholdWord];
  const uint32_t thr = fixed_threshold ? fixed_threshold : (word ? word : kLightMax);
  const int tid = threadIdx.x;
  const int nb = (int)blockDim.x;
  const int block_base = (P::kXcdRanges ? xcd_runs<kLightRun>((int)blockIdx.x, (int)gridDim.x)
                                        : (int)blockIdx.x) *
                         nb;
  const int i = block_base + tid;
  const bool active = i < n;
  const SeqTable st{&seq_dyn[tid], nb};
  const CellStarts starts = cell_starts(cs, c.cells, n);
  typename P::Target t{};
  uint32_t m = 0;
  if (active) {
    t = P::target(a, (uint32_t)i, c);
    const SceneGeo g = sc.at((uint32_t)i, c);
    m = build_seq(st, cell_of(t.x.x, t.x.y, t.x.z, g, c.h), starts, g);
  }
  {
    // this pass's statistics for the next pass's threshold: per level, how
    // many of the wavefront's targets have level < m <= kLightMax
    unsigned long long w[kLevelWords] = {};
#pragma unroll
    for (int k = 0; k < kLevels; ++k) {
      const uint64_t b = __ballot(m > heavy_level(k) && m <= kLightMax);
      w[k / 3] += (unsigned long long)__popcll(b) << (kLevelBits * (k % 3));
    }
    if ((threadIdx.x & 63) == 0) {
      const int wave = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
      unsigned long long* slot =
          reinterpret_cast<unsigned long long*>(hl.counters + stat_slot(wave % kStatSlots));
#pragma unroll
      for (int j = 0; j < kLevelWords; ++j)
        if (w[j]) atomicAdd(&slot[j], w[j]);
    }
  }
  const bool is_heavy = active && m > thr;
  const uint32_t nch = is_heavy ? (m + kChunk - 1) / kChunk : 0u;
  const int wave = tid >> 6;
  const uint64_t hm = __builtin_amdgcn_ballot_w64(is_heavy);
  uint32_t item_total = 0u, item_off = 0u;
  if (hm) item_off = wave_exclusive_sum(nch, &item_total);
  if ((tid & 63) == 0) {
    alloc_sh[0][wave] = item_total;
    alloc_sh[1][wave] = (uint32_t)__popcll(hm);
  }
  if (tid < kRankBuckets) bucket_sh[tid] = 0u;
  __syncthreads();
  uint32_t heavy = 0u;
#pragma unroll
  for (int k = 0; k < kBlock / 64; ++k) heavy += k < (nb >> 6) ? alloc_sh[1][k] : 0u;
  bool in_lane = false;  // chunk list full: this lane sums its chunks itself
  if (heavy) {
    // Allocation, one atomic a workgroup and counter: every workgroup's go to
    // the same two words, where they queue.  (Two a wavefront, one after the
    // other: 1M dense step 2413 -> 2316 us, 512K dam 1334 -> 1237 us, 64 scenes
    // 8921 -> 8825 us without them.)  Partials are target-major (lane
    // l owns [first, first + nch)); the work items are chunk-major over the
    // wave (chunk 0 of every heavy lane, then chunk 1, ...), so the lanes of
    // a chunk kernel wavefront work on the same chunk of neighbouring
    // targets, which in a crowded cell share their candidate sequence: the
    // candidate loads coalesce instead of being gathered lane by lane.
    __syncthreads();
    if (tid < 2) {
      uint32_t sum = 0u, w[kBlock / 64];
#pragma unroll
      for (int k = 0; k < kBlock / 64; ++k) {
        w[k] = sum;
        sum += k < (nb >> 6) ? alloc_sh[tid][k] : 0u;
      }
      const uint32_t base = atomicAdd(tid ? rec_cnt : item_cnt, sum);
#pragma unroll
      for (int k = 0; k < kBlock / 64; ++k) alloc_sh[tid][k] = base + w[k];
    }
    __syncthreads();
    const uint32_t item_base = alloc_sh[0][wave];
    const uint32_t first = item_base + item_off;
    const bool wave_fits = item_base + item_total <= hl.item_cap;
    uint32_t maxnch = nch;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const uint32_t o = __shfl_xor(maxnch, off);
      maxnch = o > maxnch ? o : maxnch;
    }
    const uint64_t lt = (1ull << (threadIdx.x & 63)) - 1ull;
    uint32_t pos = item_base;
    for (uint32_t ch = 0; ch < maxnch; ++ch) {
      const bool has = nch > ch;
      const uint64_t bm = __ballot(has);
      const uint32_t u = pos + (uint32_t)__popcll(bm & lt);
      if (has && u < hl.item_cap)
        hl.items[u] = wave_fits ? make_uint4((uint32_t)i, ch, first + ch, 0u)
                                : make_uint4(~0u, 0u, 0u, 0u);
      pos += (uint32_t)__popcll(bm);
    }
    if (is_heavy)  // a record without items is skipped by the combine kernel
      hl.recs[alloc_sh[1][wave] + (uint32_t)__popcll(hm & lt)] =
          make_uint4(wave_fits ? (uint32_t)i : ~0u, first, nch, 0u);
    in_lane = is_heavy && !wave_fits;
  }
  // Lanes take the block's remaining targets in order of candidate count, so
  // each wavefront gets targets of similar cost instead of waiting on its
  // longest lane: a counting sort over buckets of 8 candidates in LDS
  // (bucket 0: idle slots and targets handed to the chunk kernels).  The
  // targets stay in this block's particle range, whose neighbourhoods
  // overlap.  Each target's sum is unchanged: only the lane that computes it
  // moves, so the order within a bucket (set by LDS atomics) does not matter.
  const uint32_t key = active && (!is_heavy || in_lane) ? m + 1u : 0u;
  key_sh[tid] = key;
  const uint32_t bucket =
      key == 0u ? 0u : 1u + min((key - 1u) >> 3, (uint32_t)kRankBuckets - 2u);
  const uint32_t within = atomicAdd(&bucket_sh[bucket], 1u);
  __syncthreads();
  if (tid < kRankBuckets) {  // the first wavefront scans the bucket counts
    uint32_t total;
    const uint32_t cnt_b = bucket_sh[tid];
    bucket_sh[tid] = wave_exclusive_sum(cnt_b, &total);
  }
  __syncthreads();
  order_sh[bucket_sh[bucket] + within] = (uint32_t)tid;
  __syncthreads();
  const int src = (int)order_sh[tid];
  const uint32_t ks = key_sh[src];
  if (ks == 0u) return;  // idle slot, or a target handed to the chunk kernels
  const uint32_t ms = ks - 1u;
  const uint32_t ti = (uint32_t)(block_base + src);
  const SeqTable sts{&seq_dyn[src], nb};
  t = P::target(a, ti, c);
  // the sweep's blocks are the canonical chunks: each is summed from zero
  // and added to the total in order (also for a heavy target whose chunk
  // list was full)
  typename P::Acc s, part;
  const MaskIO<P> mio{hl, ti, ms};
  auto add = [&](uint32_t j, const auto& d) { P::add(part, t, j, d, c, a); };
  auto block_end = [&] {
    P::accumulate(s, part);
    part = typename P::Acc{};
  };
  auto get_mask = [&](uint32_t b, uint32_t& lo, uint32_t& hi) { return mio.get(b, lo, hi); };
  auto put_mask = [&](uint32_t b, uint32_t lo, uint32_t hi) { mio.put(b, lo, hi); };
  const Float4Buf sb = screen_buf<P, kC>(a, hl, (uint32_t)n);
  // a pass on stored hit masks screens nothing: its hits of up to four
  // blocks run through one loop (kLightMax candidates), which balances the
  // lanes best
  constexpr int kGroup = MaskMode<P>::value == kMaskLoad ? (int)(kLightMax / kChunk) : kLightGroup;
  sweep_seq<P::kHitBatch, kGroup>(
      sts, ms, 0u, ms, screen_of<P, kC, false>(sb, hl, ti, t, c),
      [&](uint32_t j) { return P::load_f(a, j); }, add, block_end, get_mask, put_mask);
  P::finish(a, t, s, c, sc.at(ti, c));
}

// One work-item per chunk item (i, chunk, partial slot): the partial sum of
// kChunk consecutive candidates of a heavy target.  Grid-stride over the
// items; the grid size is a launch shape.
template <class P, class S, bool kC>
__global__ __launch_bounds__(kBlock, PBF_PASS_WAVES) void k_chunks(typename P::Args a, int n,
                                                                   StepConsts c, S sc,
                                                   const uint32_t* __restrict__ cs, HeavyLists hl,
                                                   int pass) {
  __shared__ uint2 seq[10][kBlock];
  const uint32_t items = hl.counters[item_counter(pass & 1)];
  const uint32_t total = items < hl.item_cap ? items : hl.item_cap;
  // only as many workgroups as there are items to go round, spread over all
  // XCDs
  const uint32_t need = (total + kBlock - 1) / kBlock;
  const int active = need < gridDim.x ? (int)need : (int)gridDim.x;
  if ((int)blockIdx.x >= active) return;
  const int vb =
      P::kXcdRanges ? xcd_runs<kChunkRun>((int)blockIdx.x, active) : (int)blockIdx.x;
  const uint32_t stride = (uint32_t)active * kBlock;
  const SeqTable st{&seq[0][threadIdx.x], kBlock};
  const CellStarts starts = cell_starts(cs, c.cells, n);
  const Float4Buf sb = screen_buf<P, kC>(a, hl, (uint32_t)n);
  for (uint32_t u = (uint32_t)vb * kBlock + threadIdx.x; u < total; u += stride) {
    const uint4 it = hl.items[u];
    if (it.x == ~0u) continue;
    const typename P::Target t = P::target(a, it.x, c);
    const SceneGeo g = sc.at(it.x, c);
    const uint32_t m = build_seq(st, cell_of(t.x.x, t.x.y, t.x.z, g, c.h), starts, g);
    typename P::Acc part;
    const uint32_t s0 = it.y * kChunk;
    const uint32_t s1 = s0 + kChunk < m ? s0 + kChunk : m;
    const MaskIO<P> mio{hl, it.x, m};
    sweep_seq<P::kHitBatch, 1>(
        st, m, s0, s1, screen_of<P, kC, true>(sb, hl, it.x, t, c),
        [&](uint32_t j) { return P::load_f(a, j); },
        [&](uint32_t j, const auto& d) { P::add(part, t, j, d, c, a); }, [] {},
        [&](uint32_t b, uint32_t& lo, uint32_t& hi) { return mio.get(b, lo, hi); },
        [&](uint32_t b, uint32_t lo, uint32_t hi) { mio.put(b, lo, hi); });
    *reinterpret_cast<typename P::Acc*>(hl.partials + (size_t)it.z * partial_words<P>()) = part;
  }
}

// One work-item per heavy target: chunk partials added in chunk order.
template <class P, class S>
__global__ __launch_bounds__(kBlock) void k_combine(typename P::Args a, int n, StepConsts c, S sc,
                                                    HeavyLists hl, int pass) {
  const uint32_t nrec = hl.counters[rec_counter(pass & 1)];
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    // the next pass's heavy threshold from this pass's statistics, which are
    // cleared for the next pass
    unsigned long long* slot =
        reinterpret_cast<unsigned long long*>(hl.counters + stat_slot((int)threadIdx.x));
    unsigned long long cnt[kLevels];
#pragma unroll
    for (int j = 0; j < kLevelWords; ++j) {
      const unsigned long long w = slot[j];
      slot[j] = 0ull;
#pragma unroll
      for (int f = 0; f < 3 && 3 * j + f < kLevels; ++f)
        cnt[3 * j + f] = (w >> (kLevelBits * f)) & ((1ull << kLevelBits) - 1ull);
    }
#pragma unroll
    for (int k = 0; k < kLevels; ++k)
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) cnt[k] += __shfl_xor(cnt[k], off);
    if (threadIdx.x == 0) {
      uint32_t thr = kLightMax;
#pragma unroll
      for (int k = kLevels - 1; k >= 0; --k)
        if (cnt[k] * kLevelShare <= (unsigned long long)n ||
            (k < kFewLevels && cnt[k] <= kFewHeavy))
          thr = heavy_level(k);
      hl.counters[kThresholdWord] = thr;
    }
  }
  const uint32_t stride = gridDim.x * kBlock;
  for (uint32_t r = blockIdx.x * kBlock + threadIdx.x; r < nrec; r += stride) {
    const uint4 rec = hl.recs[r];
    if (rec.x == ~0u) continue;
    const typename P::Target t = P::target(a, rec.x, c);
    typename P::Acc s;
    using PAcc = typename P::Acc;
    const float* base = hl.partials + (size_t)rec.y * partial_words<P>();
    auto part = [&](uint32_t k) {
      return *reinterpret_cast<const PAcc*>(base + (size_t)k * partial_words<P>());
    };
    // eight loads in flight, then the adds in chunk order
    uint32_t k = 0;
    for (; k + 8u <= rec.z; k += 8u) {
      PAcc p8[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) p8[q] = part(k + q);
#pragma unroll
      for (int q = 0; q < 8; ++q) P::accumulate(s, p8[q]);
    }
    for (; k < rec.z; ++k) P::accumulate(s, part(k));
    P::finish(a, t, s, c, sc.at(rec.x, c));
  }
}

int grid_for_items(long long items, int max_blocks) {
  const long long b = (items + kBlock - 1) / kBlock;
  return (int)(b < 1 ? 1 : (b > max_blocks ? max_blocks : b));
}

// Lanes per target for n particles: 0 = the light, chunk and combine kernels.
// Steps under graph replay, microseconds, fresh lattice / collapsing dam (20
// frames) / spread dam (50 frames): 16K particles 195 / 164 / 162 with 16
// lanes, 184 / 195 / 187 with 8, 400 / 584 / 594 with the lane kernels; 32K
// 214 / 313 / 225 with 8 lanes, 386 / 598 / 631 with the lane kernels; 93K 383 /
// 429 / 474 against 335 / 587 / 642, 130K 498 / 559 / 636 against 344 / 608 / 699.
// Where every target has much the same number of candidates the lane kernels win
// from about 85K on (360 against 331), in dams teams win up to 130K and beyond, by
// less and less; nothing the host knows tells the two apart, and the line keeps a
// lattice's loss to about a tenth.
// Piles of one to seven thousand particles in one cell are the teams' worst case
// (a team's item is 64 candidates of one target, of which every lane folds every
// term): 80,000 particles, 1,000 / 2,000 / 4,000 / 6,000 of them in one cell 641 /
// 1060 / 2411 / 4391 us a step against 552 / 610 / 761 / 953 with the lane kernels;
// 8,000 overflow those kernels' lists, 6724 against 8388.
// A fixed heavy threshold asks for the chunk kernels, so it keeps the lane
// kernels at every size.  Every choice sums in the canonical order.
constexpr int kTeam16Max = 20480;
constexpr int kTeam8Max = 90112;
inline int team_lanes(int n, const Shapes& sh) {
  if (sh.heavy != 0 || n > kTeam8Max) return 0;
  return n <= kTeam16Max ? 16 : 8;
}
inline int team_blocks(int n, int lanes) {
  const int targets = kTeamBlock / lanes;
  return (n + targets - 1) / targets;
}

// Whether a pass of n particles screens on the screening coordinates (if its
// policy can).  From about a million particles on the L1's accesses bound the
// chunk kernels and every load the light kernels: 1M dense step 2264 -> 2150 us,
// 4M sweeping-wall frame 15.65 -> 14.48 ms, 64 scenes 8.69 -> 8.25 ms.  Smaller
// passes wait on latency, and the hits' reloads no longer find the lines that
// screening positions brought.  Fresh lattice / dam after 20 and 50 frames,
// positions -> coordinates: 128K 392 / 653 / 694 -> 399 / 666 / 708 us, 512K 794 /
// 1202 / 991 -> 809 / 1171 / 1001, 1M 1349 / 2370 / 1578 -> 1338 / 2248 / 1532.
constexpr int kCoarseMin = (1 << 19) + 1;
inline bool coarse_screen(int n, const Shapes& sh) {
  return n >= kCoarseMin && team_lanes(n, sh) == 0;
}

template <class P, class S, bool kC>
void launch_lanes(const typename P::Args& a, int n, const StepConsts& c, const S& sc,
                  const uint32_t* cs, const HeavyLists& hl, int pass, const Shapes& sh,
                  hipStream_t st) {
  const int lb = sh.light_block;
  k_light<P, S, kC><<<(n + lb - 1) / lb, lb, light_lds_bytes(lb), st>>>(
      a, n, c, sc, cs, hl, pass, (uint32_t)sh.heavy);
  k_chunks<P, S, kC><<<grid_for_items(hl.item_cap, sh.chunk_blocks), kBlock, 0, st>>>(
      a, n, c, sc, cs, hl, pass);
  k_combine<P, S><<<grid_for_items(n, 512), kBlock, 0, st>>>(a, n, c, sc, hl, pass);
}

template <class P, class S>
void launch_pass_s(const typename P::Args& a, int n, const StepConsts& c, const S& sc,
                   const uint32_t* cs, const HeavyLists& hl, int pass, const Shapes& sh,
                   hipStream_t st) {
  const int team = team_lanes(n, sh);
  if (team == 16) {
    k_team<P, S, 16><<<team_blocks(n, 16), kTeamBlock, 0, st>>>(a, n, c, sc, cs);
    return;
  }
  if (team == 8) {
    k_team<P, S, 8><<<team_blocks(n, 8), kTeamBlock, 0, st>>>(a, n, c, sc, cs);
    return;
  }
  if constexpr (CoarseMode<P>::value) {
    if (coarse_screen(n, sh)) {
      launch_lanes<P, S, true>(a, n, c, sc, cs, hl, pass, sh, st);
      return;
    }
  }
  launch_lanes<P, S, false>(a, n, c, sc, cs, hl, pass, sh, st);
}

template <class P>
void launch_pass(const typename P::Args& a, int n, const StepConsts& c, const Scenes& scn,
                 const uint32_t* cs, const HeavyLists& hl, int pass, const Shapes& sh,
                 hipStream_t st) {
  if (scn.geo)
    launch_pass_s<P>(a, n, c, SceneTable{scn.geo, scn.sid}, cs, hl, pass, sh, st);
  else
    launch_pass_s<P>(a, n, c, OneScene{}, cs, hl, pass, sh, st);
}

}  // namespace
}  // namespace pbf
