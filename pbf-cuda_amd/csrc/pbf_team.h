// pbf_team.h — the neighbour pass for particle counts that leave the chip
// idle with one work-item per target: a team of G lanes per target.
//
// With one lane per target a pass of a few ten thousand particles is a few
// hundred wavefronts on 1,024 SIMDs, and lasts as long as one lane's serial
// walk through its candidates (~200 of them: 27 round trips of 8 loads, then
// the hits), plus a chunk and a combine launch whether or not there is a
// crowded target.  A team walks them G at a time, in one launch.
#pragma once

#include "pbf_device.h"

namespace pbf {
namespace {

// What the team kernel needs of a pass policy besides the lane kernels'
// hooks (pbf_pass.h): Term, one candidate's contribution; term(), which
// forms it; fold(), which adds it to a running sum with the operations
// of add(), so that folding the terms in order gives add()'s bits (a zero
// Term leaves every sum as it is); kNbIsScreen: the pair term needs nothing
// of the candidate but the element of screen().  A policy without Term folds
// whole sums (the adjoint's passes, whose order of addition is their own).
template <class P, class = void>
struct TeamTerm {
  static constexpr bool kNbIsScreen = false;
  using Term = typename P::Acc;
  template <class D>
  static __device__ __forceinline__ Term term(const typename P::Target& t, uint32_t j, const D& d,
                                              const StepConsts& c, const typename P::Args& a) {
    Term s{};
    P::add(s, t, j, d, c, a);
    return s;
  }
  static __device__ __forceinline__ void fold(typename P::Acc& s, const Term& p) {
    P::accumulate(s, p);
  }
};
template <class P>
struct TeamTerm<P, std::void_t<typename P::Term>> {
  static constexpr bool kNbIsScreen = P::kNbIsScreen;
  using Term = typename P::Term;
  template <class D>
  static __device__ __forceinline__ Term term(const typename P::Target& t, uint32_t j, const D& d,
                                              const StepConsts& c, const typename P::Args& a) {
    return P::term(t, d, c, a);
  }
  static __device__ __forceinline__ void fold(typename P::Acc& s, const Term& p) {
    P::fold(s, p);
  }
};


constexpr int kTeamBlock = 256;

// LDS storage of an X (LDS objects cannot have initializers).
template <class X>
struct alignas(X) LdsOf {
  static_assert(sizeof(X) % 4 == 0, "words");
  uint32_t v[sizeof(X) / 4];
  __device__ __forceinline__ X get() const { return *reinterpret_cast<const X*>(v); }
  __device__ __forceinline__ void put(const X& x) { *reinterpret_cast<X*>(v) = x; }
};

// Reductions over a team (aligned groups of G lanes) by data-parallel
// moves: neighbours 1 and 2 apart, then the mirrored half rows and rows,
// whose lanes already hold equal values.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
}
template <int G>
__device__ __forceinline__ uint32_t team_or(uint32_t v) {
  v |= dpp<0xB1>(v);
  v |= dpp<0x4E>(v);
  if (G >= 8) v |= dpp<0x141>(v);
  if (G >= 16) v |= dpp<0x140>(v);
  return v;
}
template <int G>
__device__ __forceinline__ uint32_t team_sum(uint32_t v) {
  v += dpp<0xB1>(v);
  v += dpp<0x4E>(v);
  if (G >= 8) v += dpp<0x141>(v);
  if (G >= 16) v += dpp<0x140>(v);
  return v;
}

// G lanes per target, T = 64 / G targets per wavefront.  The canonical
// 64-candidate chunks of the wavefront's targets, target by target, are its
// work items; a round gives every team one item, whichever target it belongs
// to, so a crowded target's chunks spread over the whole wavefront.  In an
// item the lanes take the candidates G at a time (neighbouring slots: the
// loads coalesce), the candidates that pass hit() are queued in LDS in
// order, the lanes evaluate the queue G terms at a time and every lane folds
// the team's terms in that order; the chunk sums are then added to their
// targets' totals in chunk order.  That is the canonical order of
// pbf_device.h, so the results are those of the lane kernels.
//
// Bound: instruction issue from ~30,000 particles on (a round of 512
// candidates issues ~240 vector instructions to map and screen them and ~110
// per batch of terms and folds, 2.5 times what the lane kernels need per
// candidate, because every lane of a team folds every term), latency below:
// the lambda pass fills 72% of the issue peak at 32,768 particles, 13% at 2,048,
// with 80% of the lanes active in an issued instruction.
// Measured, lambda pass: 2,048 particles 45 us in three launches -> 11 us in
// one (G = 16); 32,768 in the collapsing double dam 89 -> 30 us (G = 8).
template <class P, class S, int G>
__global__ __launch_bounds__(kTeamBlock) void k_team(typename P::Args a, int n, StepConsts c, S sc,
                                                     const uint32_t* __restrict__ cs) {
  using TT = TeamTerm<P>;
  using Term = typename TT::Term;
  using Acc = typename P::Acc;
  using Target = typename P::Target;
  // queue the candidate itself where the term needs nothing else and the
  // queue is small (16 bytes an entry cost occupancy at G = 8: 64K particles
  // ran 3-5% slower than with byte offsets reloaded), else its byte offset
  constexpr bool kVecQ = TT::kNbIsScreen && G >= 16;
  using Queued = std::conditional_t<kVecQ, float4, uint32_t>;
  constexpr int T = 64 / G;
  constexpr int W = kTeamBlock / 64;
  constexpr int kCols = 9;
  constexpr int kSteps = (int)kChunk / G;
  constexpr int kBatch = kSteps < 8 ? kSteps : 8;
  // non-empty columns of each target: (16 x (first slot - first position),
  // first position); unused entries begin at ~0u
  __shared__ uint2 tab_sh[W][T][kCols];
  __shared__ LdsOf<Target> tgt_sh[W][T];
  __shared__ uint32_t cnt_sh[W][T];
  __shared__ Queued queue_sh[W][T][kChunk];
  __shared__ LdsOf<Term> term_sh[W][64];
  __shared__ LdsOf<Acc> part_sh[W][T];

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int g = lane & (G - 1), team = lane / G;
  // One contiguous range per XCD, whatever P::kXcdRanges asks of the lane kernels:
  // an XCD then fetches its range and one halo, where runs (or launch order) have
  // every XCD fetch everything.  Contiguous -> runs of 16 workgroups where true,
  // launch order where false: 32K double dam under graph replay 562 -> 576 us, a 16K
  // rollout with gradients 15.28 -> 15.56 ms, dams of 64K after 20 / 60 frames 246 /
  // 236 -> 260 / 248 us, fresh ones of 85K 327 -> 309.  A pile is the case for runs, as
  // its targets share an XCD here: 80,000 particles, 1,000 / 4,000 of them in one cell
  // 641 / 2403 -> 536 / 1624 us a step, 1.51 / 5.34 -> 1.39 / 4.48 ms a scatter-mode
  // backward frame.
  const int i = (xcd_block_index() * (int)blockDim.x + (int)threadIdx.x) / G;
  const bool active = i < n;
  const uint32_t ti = (uint32_t)(active ? i : n - 1);
  const Target own = P::target(a, ti, c);
  const SceneGeo geo = sc.at(ti, c);
  const Cell q = cell_of(own.x.x, own.x.y, own.x.z, geo, c.h);

  // the nine columns (pbf_device.h: load_cols), one or more per lane
  {
    const int z0 = q.z > 0 ? q.z - 1 : 0;
    const int z1 = q.z + 1 < geo.dz ? q.z + 1 : geo.dz - 1;
#pragma unroll
    for (int k0 = 0; k0 < kCols; k0 += G) {
      const int k = k0 + g;
      const int X = q.x + k / 3 - 1, Y = q.y + k % 3 - 1;
      const bool in = (k < kCols) & (X >= 0) & (X < geo.dx) & (Y >= 0) & (Y < geo.dy);
      const uint32_t col = geo.base + (in ? (uint32_t)((X * geo.dy + Y) * geo.dz) : 0u);
      const uint32_t lo = cs[col + z0], hi = cs[col + z1 + 1];
      if (k < kCols) tab_sh[w][team][k] = make_uint2(lo, (in & (hi > lo)) ? hi - lo : 0u);
    }
  }
  wave_lds_sync();
  uint32_t m = 0;
  {
    uint2 e[kCols];
#pragma unroll
    for (int k = 0; k < kCols; ++k) e[k] = tab_sh[w][team][k];
    wave_lds_sync();
#pragma unroll
    for (int k0 = 0; k0 < kCols; k0 += G)
      if (k0 + g < kCols) tab_sh[w][team][k0 + g] = make_uint2(0u, ~0u);
    wave_lds_sync();
    int nk = 0;
#pragma unroll
    for (int k = 0; k < kCols; ++k) {
      if (g == k % G && e[k].y) tab_sh[w][team][nk] = make_uint2((e[k].x - m) << 4, m);
      nk += e[k].y ? 1 : 0;
      m += e[k].y;
    }
  }
  if (!active) m = 0;
  if (g == 0) {
    tgt_sh[w][team].put(own);
    cnt_sh[w][team] = m;
  }
  // first item of each team's target, in scalar registers
  const uint32_t nch = (m + kChunk - 1) / kChunk;
  uint32_t first[T + 1];
  first[0] = 0u;
  uint32_t my_first = 0u;
#pragma unroll
  for (int k = 0; k < T; ++k) {
    my_first = k == team ? first[k] : my_first;
    first[k + 1] = first[k] + (uint32_t)__builtin_amdgcn_readlane((int)nch, k * G);
  }
  const uint32_t items = first[T], my_end = my_first + nch;
  const Float4Buf sb = float4_buf(P::screen(a), (uint32_t)n);
  const uint32_t below = (1u << g) - 1u;  // the team's lanes before this one
  wave_lds_sync();

  Acc tot{};
  for (uint32_t r0 = 0; r0 < items; r0 += T) {
    const uint32_t item = r0 + (uint32_t)team;
    const bool has = item < items;
    // the target the item belongs to
    int tq = 0;
    uint32_t f = 0u;
#pragma unroll
    for (int k = 1; k < T; ++k) {
      const bool past = item >= first[k];
      tq = past ? k : tq;
      f = past ? first[k] : f;
    }
    const Target t = tgt_sh[w][tq].get();
    const uint32_t u0 = (item - f) * kChunk;
    const uint32_t left = cnt_sh[w][tq] - u0;
    const uint32_t len = has ? (left < kChunk ? left : kChunk) : 0u;
    // the columns that begin inside the chunk as bits of its positions, and
    // the column its first position lies in
    uint32_t lo = 0u, hi = 0u, col = 0u;
#pragma unroll
    for (int k0 = 0; k0 < kCols; k0 += G) {
      const int k = k0 + g;
      const uint32_t s = k < kCols ? tab_sh[w][tq][k].y : ~0u;
      const uint32_t d = s - u0;  // wraps past kChunk for s < u0
      col += s <= u0 ? 1u : 0u;
      lo |= ((d != 0u) & (d < 32u)) ? 1u << (d & 31u) : 0u;
      hi |= ((d >= 32u) & (d < 64u)) ? 1u << (d & 31u) : 0u;
    }
    lo = team_or<G>(lo);
    hi = team_or<G>(hi);
    col = team_sum<G>(col);
    // a team without an item has len = 0: its mapping only has to stay in the table
    const uint2* tab = tab_sh[w][tq] + (col ? col - 1u : 0u);
    const uint32_t off0 = (u0 + (uint32_t)g) << 4;
    const int rem = (int)len - g;

    // screen: kSteps candidates per lane, kBatch loads in flight together
    using Seen = std::conditional_t<kVecQ, float4, float3>;
    uint32_t cnt = 0u;
    Queued* queue = queue_sh[w][team];
    const uint32_t col_hi = (uint32_t)__popc(lo);
#pragma unroll
    for (int s0 = 0; s0 < kSteps; s0 += kBatch) {
      // byte offsets: the column of position p is the number of columns begun
      // at or before it; positions past len read whatever lies there (the
      // buffer load stays in bounds) and are masked off below
      uint32_t off[kBatch];
      Seen x[kBatch];
#pragma unroll
      for (int s = 0; s < kBatch; ++s) {
        const int p0 = (s0 + s) * G;  // position of the team's first lane
        const uint32_t upto = (2u << ((uint32_t)(p0 & 31) + (uint32_t)g)) - 1u;
        const uint32_t k =
            p0 < 32 ? (uint32_t)__popc(lo & upto) : (uint32_t)__popc(hi & upto) + col_hi;
        off[s] = tab[k].x + off0 + (uint32_t)p0 * 16u;
      }
#pragma unroll
      for (int s = 0; s < kBatch; ++s) {
        if constexpr (kVecQ)
          x[s] = load_f4_at(sb, off[s]);
        else
          x[s] = load_xyz_at(sb, off[s]);
      }
#pragma unroll
      for (int s = 0; s < kBatch; ++s) {
        const uint64_t b =
            __builtin_amdgcn_ballot_w64(rem > (s0 + s) * G) &
            __builtin_amdgcn_ballot_w64(P::hit(t, make_float3(x[s].x, x[s].y, x[s].z), c));
        const uint32_t word = lane < 32 ? (uint32_t)b : (uint32_t)(b >> 32);
        const uint32_t mine = __builtin_amdgcn_ubfe(word, (uint32_t)(team * G) & 31u, G);
        uint32_t at = cnt + (uint32_t)__popc(mine & below);
        asm("" : "+v"(at));  // one count-and-add, not two shifted addends
        if (__builtin_amdgcn_inverse_ballot_w64(b)) {
          if constexpr (kVecQ)
            queue[at] = x[s];
          else
            queue[at] = off[s];
        }
        cnt += (uint32_t)__popc(mine);
      }
    }
    wave_lds_sync();

    // evaluate G queued candidates per team at a time, fold them in order
    Acc part{};
    for (uint32_t r = 0; __builtin_amdgcn_ballot_w64(r < cnt) != 0ull; r += G) {
      const uint32_t k = r + (uint32_t)g;
      Term tm{};
      if (k < cnt) {
        if constexpr (kVecQ) {
          tm = TT::term(t, 0u, queue[k], c, a);
        } else {
          const uint32_t j = queue[k] >> 4;
          tm = TT::term(t, j, P::load_f(a, j), c, a);
        }
      }
      term_sh[w][lane].put(tm);
      wave_lds_sync();
#pragma unroll
      for (int e = 0; e < G; ++e) TT::fold(part, term_sh[w][team * G + e].get());
      wave_lds_sync();
    }
    // chunk sums to their targets, in chunk order
    if (g == 0) part_sh[w][team].put(part);
    wave_lds_sync();
    {
      const uint32_t e0 = my_first > r0 ? my_first : r0;
      const uint32_t e1 = my_end < r0 + T ? my_end : r0 + T;
      for (uint32_t e = e0; e < e1; ++e) P::accumulate(tot, part_sh[w][e - r0].get());
    }
    wave_lds_sync();
  }
  if (active && g == 0) P::finish(a, own, tot, c, geo);
}

}  // namespace
}  // namespace pbf
