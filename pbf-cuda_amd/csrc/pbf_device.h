// pbf_device.h — shared device-side definitions of the gfx950 PBF step.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace pbf {

// Geometry of one scene's box and grid.  A batch of scenes shares one global
// cell-id space: scene s owns ids [base, base + dx*dy*dz), so one stable sort
// of all particles by cell id leaves every scene's particles in its own
// contiguous range, in the order sorting that scene alone would give.
struct alignas(16) SceneGeo {
  float llx, lly, llz;  // box lower corner (llim)
  float ulx, uly, ulz;  // box upper corner (ulim)
  float lox, loy, loz;  // box clamp lower: llim + LIM_EPS, rounded to FP32
  float hix, hiy, hiz;  // box clamp upper: ulim - LIM_EPS, rounded to FP32
  int dx, dy, dz;       // grid dims, (int)ceilf((ulim-llim)/h)
  uint32_t base;        // first global cell id of the scene
};

// Per-step constants, built on the host once per step and passed by value
// (kernarg segment).  Field meanings follow the reference's functors
// (fluids/Simulator.cu:22-161) and constants (fluids/helper.h:4-9).
struct StepConsts {
  SceneGeo g;              // the scene of a single-scene step
  int cells;               // cells of all scenes
  float h, h2;             // kernel radius, h*h
  float h2_outer;          // prefilter bound: r2 >= h2_outer => both kernels are 0
  float keps;              // KERNAL_EPS
  float keps2_lo;          // 0.99 keps^2: r2 < keps2_lo => sqrtf(r2) < keps (no gradient)
  float poly6;             // 315/(64 pi h^9)
  float spiky;             // -45/(pi h^6)
  float spiky_rho0;        // spiky / pho0 (the lambda gradient, Simulator_kernel.cuh:92)
  float pho0;
  float lambda_eps;
  float coef_corr;         // -k_corr / W(delta_q)^n_corr
  float n_corr;
  int n_corr_int;          // n_corr when it is an integer in [0,16], else -1
  float k_boundary;        // k_boundaryDensity
  float wall_c;            // 2 pi / 3 (DensityBoundary)
  float max_dp;            // MAX_DP
  float dt, inv_dt;        // dt, 1/dt (FP32, as h_updateVelocity)
  float gz;                // -g
  float c_xsph;
  double inv_screen;       // 1 / (16 h): periods of the screening coordinates per unit
};

// Scene sources: where a kernel finds the geometry of particle i's scene.
// OneScene: the single scene in the kernarg constants.  SceneTable: a batch;
// sid[i] is the scene of index i, valid in input and in sorted order alike
// (both keep scene s in its own index range).
struct OneScene {
  __device__ __forceinline__ SceneGeo at(uint32_t, const StepConsts& c) const { return c.g; }
};
struct SceneTable {
  const SceneGeo* __restrict__ geo;
  const uint16_t* __restrict__ sid;
  __device__ __forceinline__ SceneGeo at(uint32_t i, const StepConsts&) const {
    return geo[sid[i]];
  }
};

// Workgroup index remapped so that each of the 8 XCDs (which receive
// workgroups round-robin and each own an L2) processes one contiguous range
// of particles: neighbouring particles, which share neighbour data, then
// share an L2.
__device__ __forceinline__ int xcd_block_index() {
  const int G = (int)gridDim.x;
  const int p = (int)blockIdx.x;
  const int per = G >> 3, rem = G & 7, x = p & 7;
  return x * per + (x < rem ? x : rem) + (p >> 3);
}

// Workgroup p of a grid of `grid`, remapped so that each XCD takes runs of kRun
// consecutive workgroups in turn: neighbours share an L2 as above, and crowded
// and empty regions fall to all XCDs.  The last, partial round of runs is split
// evenly (a grid of up to 8 runs: one contiguous range per XCD).
template <int kRun>
__device__ __forceinline__ int xcd_runs(int p, int grid) {
  const int full = grid / (8 * kRun) * (8 * kRun);
  const int x = p & 7;
  if (p < full) {
    const int j = p >> 3;
    return ((j / kRun) * 8 + x) * kRun + j % kRun;
  }
  const int left = grid - full;
  const int per = left >> 3, rem = left & 7;
  return full + x * per + (x < rem ? x : rem) + ((p - full) >> 3);
}

// One axis of the cell coordinate, (int)((p - llim)/h) clamped to
// [0, dim-1] in FP32 (fluids/Simulator.cu:30-36).  Clamping the quotient
// before truncating gives the same integer for every finite quotient and
// maps NaN to 0.  The division is IEEE (built with
// -fhip-fp32-correctly-rounded-divide-sqrt) so keys match the host oracle.
__device__ __forceinline__ int cell_coord(float p, float ll, float h, int dim) {
  const float q = (p - ll) / h;
  return (int)fminf(fmaxf(q, 0.0f), (float)(dim - 1));
}

struct Cell {
  int x, y, z;
};

__device__ __forceinline__ Cell cell_of(float x, float y, float z, const SceneGeo& g, float h) {
  return Cell{cell_coord(x, g.llx, h, g.dx), cell_coord(y, g.lly, h, g.dy),
              cell_coord(z, g.llz, h, g.dz)};
}

// Cell id, x-major and z fastest (xyzToId, fluids/Simulator.cu:52), offset
// by the scene's base.
__device__ __forceinline__ uint32_t cell_id(const Cell& q, const SceneGeo& g) {
  return g.base + (uint32_t)((q.x * g.dy + q.y) * g.dz + q.z);
}

// Canonical summation order, shared with the host oracle's FP32 mirror: a
// target's candidate sequence is summed in consecutive chunks of kChunk
// candidates, each summed sequentially from zero, the chunk sums added in
// chunk order (one chunk: the plain sequential sum).  The order does not
// depend on who computes the sum, so the kernels may split the work freely:
// a light target's work-item walks all its chunks; a heavy target's chunks
// go to one work-item each (the chunk kernel) and are added up by the
// combine kernel.  Crowded cells (particles piled into a corner) then cost a
// few chunk lengths instead of one lane thousands of dependent gathers.
constexpr uint32_t kChunk = 64;
// A target is heavy when it has more than kLightMax candidates, or more than
// the threshold the previous neighbour pass chose: the smallest level L of
// heavy_level() such that at most n / kLevelShare targets had L < m <=
// kLightMax, or, among the lowest kFewLevels, at most kFewHeavy (else
// kLightMax).  A light wavefront lasts as long as its longest
// lane, so in sparse water the few long lanes set the light kernel's tail and
// are better spread over the chunk kernel (threshold 64); in dense water long
// lanes are common, balance each other within the wavefronts, and spreading
// them would only lengthen the chunk lists (threshold up to kLightMax).  While
// their chunks leave the chip idle even that costs less than waiting for them,
// if no light target is left with more than about one chunk (kFewLevels):
// collapsing dams after 20 / 50 frames, 92K particles 797 / 833 -> 632 / 669 us a
// step, 128K 823 / 861 -> 656 / 697, 256K 858 / 829 -> 777 / 761, fresh lattices
// and 1M unchanged.  kFewHeavy = 65536 put a fresh 92K lattice's targets
// on the lists (397 -> 570 us), 16384 left 256K at 841 / 785; with every level
// a dense dam of 130,000 takes 592 us instead of 587.
// Which targets are heavy changes no result (the canonical order above),
// only the timing.
constexpr uint32_t kLightMax = 256;
constexpr int kLevels = 7;
__host__ __device__ constexpr uint32_t heavy_level(int k) {  // 64, 80, .., 128, 160, 192
  return k < 4 ? 64u + 16u * (uint32_t)k : 128u + 32u * (uint32_t)(k - 4);
}
constexpr uint32_t kLevelShare = 25;
constexpr int kFewLevels = 3;  // up to 96 candidates
constexpr uint32_t kFewHeavy = 32768;
// The per-level counts travel packed, three 21-bit fields to a 64-bit word
// (exact while a statistics slot counts fewer than 2^21 targets per level,
// i.e. below 2^27 targets; beyond that a count may spill into the next field
// and misjudge the threshold, which costs time only).
constexpr int kLevelBits = 21;
constexpr int kLevelWords = (kLevels + 2) / 3;

// Hit masks shared by the two passes of one solver iteration.  lambda_k and
// delta-p_k read the same positions x_k and walk the same candidate sequence,
// and every pair delta-p adds (KERNAL_EPS <= r < h, j != i) passes lambda's
// screening test (r^2 < h^2 padded): a pass policy with kMask = kMaskStore
// (lambda) records the 64-bit hit mask of each 64-candidate block of targets
// with at most kMaskBlocks blocks (2048 candidates: all but the deepest corner
// piles), and one with kMask = kMaskLoad (delta-p)
// uses those masks instead of screening.  Its add() still tests every pair it
// is handed, so the extra bits (coincident pairs, i itself) add nothing and
// the sums are those of its own screening.
constexpr int kMaskNone = 0, kMaskStore = 1, kMaskLoad = 2;
constexpr uint32_t kMaskBlocks = 32;
template <class P, class = void>
struct MaskMode {
  static constexpr int value = kMaskNone;
};
template <class P>
struct MaskMode<P, std::void_t<decltype(P::kMask)>> {
  static constexpr int value = P::kMask;
};

// A float4 array as a raw buffer resource, addressed by byte offsets: a
// 32-bit offset per load instead of a 64-bit address, and loads past the
// array's n elements return 0 instead of touching other memory.  The loads
// go through the LLVM buffer-load intrinsic with an explicit 3 x float
// result (12 bytes, buffer_load_dwordx3).
typedef int pbf_i32x4 __attribute__((ext_vector_type(4)));
typedef float pbf_f32x3 __attribute__((ext_vector_type(3)));
__device__ pbf_f32x3 pbf_raw_buffer_load_f32x3(pbf_i32x4 rsrc, int voffset, int soffset,
                                               int aux) __asm("llvm.amdgcn.raw.buffer.load.v3f32");
typedef float pbf_f32x4 __attribute__((ext_vector_type(4)));
__device__ pbf_f32x4 pbf_raw_buffer_load_f32x4(pbf_i32x4 rsrc, int voffset, int soffset,
                                               int aux) __asm("llvm.amdgcn.raw.buffer.load.v4f32");
struct Float4Buf {
  pbf_i32x4 r;
};
__device__ __forceinline__ Float4Buf raw_buf(const void* p, uint64_t bytes) {
  const uint64_t a = (uint64_t)p;
  Float4Buf b;
  b.r.x = (int)(uint32_t)(a & 0xFFFFFFFFull);
  b.r.y = (int)(uint32_t)(a >> 32);  // stride 0
  b.r.z = (int)(bytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t)bytes);
  b.r.w = 0x00020000;  // the raw (untyped) buffer format of gfx9
  return b;
}
__device__ __forceinline__ Float4Buf float4_buf(const float4* p, uint32_t n) {
  return raw_buf(p, (uint64_t)n * 16u);
}
// x, y, z of the element at byte offset `off` (a 12-byte load).
__device__ __forceinline__ float3 load_xyz_at(const Float4Buf& b, uint32_t off) {
  const pbf_f32x3 v = pbf_raw_buffer_load_f32x3(b.r, (int)off, 0, 0);
  return make_float3(v.x, v.y, v.z);
}

// The element at byte offset `off`.
__device__ __forceinline__ float4 load_f4_at(const Float4Buf& b, uint32_t off) {
  const pbf_f32x4 v = pbf_raw_buffer_load_f32x4(b.r, (int)off, 0, 0);
  return make_float4(v.x, v.y, v.z, v.w);
}

typedef int pbf_i32x2 __attribute__((ext_vector_type(2)));
__device__ pbf_i32x2 pbf_raw_buffer_load_i32x2(pbf_i32x4 rsrc, int voffset, int soffset,
                                               int aux) __asm("llvm.amdgcn.raw.buffer.load.v2i32");
__device__ pbf_i32x4 pbf_raw_buffer_load_i32x4(pbf_i32x4 rsrc, int voffset, int soffset,
                                               int aux) __asm("llvm.amdgcn.raw.buffer.load.v4i32");

// Screening coordinates of a position: x | y << 16 and z, each in units of
// h / 4096 modulo 2^16 (a period of 16 h), formed in FP64 and rounded down.  A
// candidate then takes 8 bytes and four integer instructions to screen
// instead of 12 bytes (in a 16-byte element) and six: the differences wrap
// into [-8 h, 8 h), and a pair closer than h differs by less than 4096 + 1 units
// per axis from its true difference, so its squared length stays below
// kScreenNear.  Pairs that alias modulo 16 h or lie just beyond h pass the test
// too; add() decides those exactly.
__device__ __forceinline__ uint32_t screen_coord(float x, double inv) {
  const double t = (double)x * inv;
  return (uint32_t)((t - floor(t)) * 65536.0) & 0xFFFFu;
}
__device__ __forceinline__ uint2 screen_coords(float x, float y, float z, const StepConsts& c) {
  return make_uint2(screen_coord(x, c.inv_screen) | screen_coord(y, c.inv_screen) << 16,
                    screen_coord(z, c.inv_screen));
}
// (h (1 + 1e-4) in units + sqrt(3) for the rounding of both ends)^2, rounded up
constexpr int kScreenNear = 4099 * 4099;
// Squared screening distance minus kScreenNear: negative for every pair within
// h (whose squares do not overflow).
__device__ __forceinline__ int screen_near(const uint2& a, const uint2& b) {
  typedef short s16x2 __attribute__((ext_vector_type(2)));
  const s16x2 dxy = __builtin_bit_cast(s16x2, a.x) - __builtin_bit_cast(s16x2, b.x);
  const s16x2 dz = __builtin_bit_cast(s16x2, a.y) - __builtin_bit_cast(s16x2, b.y);
  return __builtin_amdgcn_sdot2(dz, dz, __builtin_amdgcn_sdot2(dxy, dxy, -kScreenNear, false),
                                false);
}

// Entries of a column table: nine columns and the closing entry.
constexpr int kSeqEntries = 10;

// A work-item's candidate sequence as a compact column table in LDS: entry
// k < nk is (first slot of the k-th non-empty column, sequence position of
// its first candidate); entry nk is (0, m).  `tab` points at entry 0 of this
// work-item and `stride` separates entries (LDS laid out [entry][lane] so
// lanes touch consecutive words).
struct SeqTable {
  uint2* tab;
  int stride;
  __device__ __forceinline__ uint2 at(int k) const { return tab[k * stride]; }
};

// The cell-start table of a grid as the neighbour passes read it: a column's
// entries by one 16-byte load, or (apart) its two ends by a load each.  One load
// is half the cache accesses (1M dense step 2197 -> 2155 us, spread 1075 -> 1056
// us), but where a pass waits on latency it is the slower one (130,000
// particles 597 -> 609 us), and it cannot reach 2^30 cells.
constexpr int kJoinedStartsMin = (1 << 19) + 1;  // particles
struct CellStarts {
  const uint32_t* __restrict__ cs;
  Float4Buf buf;
  bool apart;
};
__device__ __forceinline__ CellStarts cell_starts(const uint32_t* cs, int cells, int n) {
  return CellStarts{cs, raw_buf(cs, ((uint64_t)(uint32_t)cells + 1u) * 4u),
                    n < kJoinedStartsMin || (uint32_t)cells >= 1u << 30};
}

// Candidate neighbours of a particle whose query cell is q, in the
// reference's order (fluids/Simulator_kernel.cuh:78-88): dx, then dy, then
// dz, j ascending.  The three cells (x,y,z-1..z+1) of one column are
// consecutive cell ids, so their particles form one contiguous sorted range,
// read from the cell-start table cs (cells + 1 entries; cs[c] = first sorted
// slot whose cell id is >= c): [cs[first cell], cs[last cell + 1]).  Walking
// that range is the same j sequence as walking the three cells in turn.
// The nine candidate columns of query cell q (column k = 3*(dx+1) + (dy+1))
// as (first slot, length), length 0 for a column outside the grid or empty
// (outside: a valid dummy address is read); returns the candidate count m.
// The loads of all columns are issued together: one memory round trip.
struct Cols {
  uint32_t lo[9], len[9];
};
__device__ __forceinline__ uint32_t load_cols(Cols& cl, const Cell& q, const CellStarts& t,
                                              const SceneGeo& g) {
  uint32_t hi[9], col[9];
  bool in[9];
  const int z0 = q.z > 0 ? q.z - 1 : 0;
  const int z1 = q.z + 1 < g.dz ? q.z + 1 : g.dz - 1;
  const int nz = z1 - z0;  // 2, at the grid's ends 1 or 0
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const int X = q.x + k / 3 - 1;
    const int Y = q.y + k % 3 - 1;
    in[k] = (X >= 0) & (X < g.dx) & (Y >= 0) & (Y < g.dy);
    col[k] = g.base + (in[k] ? (uint32_t)((X * g.dy + Y) * g.dz) : 0u);
  }
  if (t.apart) {
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      cl.lo[k] = t.cs[col[k] + z0];
      hi[k] = t.cs[col[k] + z1 + 1];
    }
  } else {
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      // entries z0 .. z0 + 3 (past the table's end: zeros, not used)
      const pbf_i32x4 e =
          pbf_raw_buffer_load_i32x4(t.buf.r, (int)((col[k] + (uint32_t)z0) << 2), 0, 0);
      cl.lo[k] = (uint32_t)e.x;
      hi[k] = (uint32_t)(nz == 2 ? e.w : (nz == 1 ? e.z : e.y));
    }
  }
  uint32_t m = 0;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    cl.len[k] = (in[k] & (hi[k] > cl.lo[k])) ? hi[k] - cl.lo[k] : 0u;
    m += cl.len[k];
  }
  return m;
}

// Writes the column table of `cl`, column k's first slot mapped by
// slot_of(k, first slot), and returns the candidate count m.  Branch-free
// compaction: every column writes its entry at the next free index, which
// only advances past non-empty columns (an empty column's entry is
// overwritten by the next one or by the closing entry).
template <class SlotOf>
__device__ __forceinline__ uint32_t write_seq(const SeqTable& st, const Cols& cl,
                                              SlotOf&& slot_of) {
  uint32_t m = 0;
  int nk = 0;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    st.tab[nk * st.stride] = make_uint2(slot_of(k, cl.lo[k]), m);
    nk += cl.len[k] ? 1 : 0;
    m += cl.len[k];
  }
  st.tab[nk * st.stride] = make_uint2(0u, m);
  return m;
}

__device__ __forceinline__ uint32_t build_seq(const SeqTable& st, const Cell& q,
                                              const CellStarts& starts, const SceneGeo& g) {
  Cols cl;
  load_cols(cl, q, starts, g);
  return write_seq(st, cl, [](int, uint32_t lo) { return lo; });
}

// Maps increasing sequence positions to sorted slots (positions must be < m
// and must not decrease between calls).  The cursor holds the current column
// (first slot b0, positions [c0, n0)) and the next one (first slot b1,
// positions [n0, n1)); a column exists after the current one exactly when
// n0 < m, so the lookahead never reads past the table's closing entry.
struct SeqCursor {
  const uint2* e;  // the current column's entry
  int stride;      // entries apart in LDS
  uint32_t m, b0, c0, n0, b1, n1;
  // With no column after the current one, b1 = n0 makes offsets8 map the
  // positions past the sequence's end to slots p (< m + 8).
  __device__ __forceinline__ void load_next() {
    if (n0 < m) {
      b1 = e[stride].x;
      n1 = e[2 * stride].y;
    } else {
      b1 = n0;
      n1 = n0;
    }
  }
  __device__ __forceinline__ void init(const SeqTable& t, uint32_t u, uint32_t total) {
    e = t.tab;
    stride = t.stride;
    m = total;
    if (u != 0u) {
      // starting inside the sequence (a chunk item): the column holding u
      // from all entries' first positions, read together.  Entries 0..nk-1
      // are columns (first position < m), entry nk closes the table with m;
      // entries after it are stale, so only the run of entries below m
      // counts.
      uint32_t y[kSeqEntries];
#pragma unroll
      for (int k = 0; k < kSeqEntries; ++k) y[k] = e[k * stride].y;
      int col = 0;
      bool live = true;
#pragma unroll
      for (int k = 1; k < kSeqEntries; ++k) {
        live = live && y[k - 1] < total;
        col += (live && y[k] <= u) ? 1 : 0;
      }
      e += col * stride;
    }
    const uint2 e0 = e[0], e1 = e[stride];
    b0 = e0.x;
    c0 = e0.y;
    n0 = e1.y;
    load_next();
  }
  __device__ __forceinline__ void shift() {
    e += stride;
    b0 = b1;
    c0 = n0;
    n0 = n1;
    load_next();
  }
  __device__ __forceinline__ uint32_t slot(uint32_t u) {
    while (u >= n0) shift();
    return b0 + (u - c0);
  }
  // Byte offsets (elements of 2^kShift bytes) of positions p0 .. p0+7: off[t] -
  // (t << kShift) is the offset of the current column's element for t < n0 - p0 and of
  // the next column's beyond, so each position costs one select.
  // Positions past the batch's last valid one get offsets the caller's
  // valid-bit mask discards: at most 7 elements past the end of the last
  // column or of the sequence's slot range (see load_next).  A batch
  // spanning more than two columns takes the per-position slot walk.
  template <int kShift>
  __device__ __forceinline__ void offsets8(uint32_t p0, uint32_t last_valid, uint32_t off[8]) {
    const uint32_t last = p0 + 7u < last_valid ? p0 + 7u : last_valid;
    if (last < n1) {
      const uint32_t s = n0 - p0;  // positions of the current column in the batch
      const uint32_t oa = (b0 + (p0 - c0)) << kShift;
      const uint32_t ob = (b1 + p0 - n0) << kShift;  // wraps for t < s: not selected
#pragma unroll
      for (int t = 0; t < 8; ++t) off[t] = ((uint32_t)t < s ? oa : ob) + ((uint32_t)t << kShift);
      if (last >= n0) shift();
    } else {
#pragma unroll
      for (int t = 0; t < 8; ++t) off[t] = slot(p0 + t < last_valid ? p0 + t : last_valid) << kShift;
    }
  }
  // The same for 8-byte elements loaded in pairs: pair k (positions p0 + 2k and
  // the next) at byte offset pair[k], whose second element is the right one
  // unless a column begins there.  In a batch of at most two columns (true)
  // that can be one position, alone = p0 + split, at `odd[0]`, if split is odd
  // (8: none); in any other (false) the second elements are at odd[k].
  __device__ __forceinline__ bool pairs8(uint32_t p0, uint32_t last_valid, uint32_t pair[4],
                                         uint32_t odd[4], uint32_t& split) {
    const uint32_t last = p0 + 7u < last_valid ? p0 + 7u : last_valid;
    if (last < n1) {
      const uint32_t s = n0 - p0;  // positions of the current column in the batch
      const uint32_t oa = (b0 + (p0 - c0)) << 3;
      const uint32_t ob = (b1 + p0 - n0) << 3;  // wraps below position s: not used there
#pragma unroll
      for (int k = 0; k < 4; ++k) pair[k] = (2u * (uint32_t)k < s ? oa : ob) + 16u * (uint32_t)k;
      odd[0] = ob + 8u * s;
      split = s < 8u && (s & 1u) ? s : 8u;
      if (last >= n0) shift();
      return true;
    }
    uint32_t off[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) off[t] = slot(p0 + t < last_valid ? p0 + t : last_valid) << 3;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      pair[k] = off[2 * k];
      odd[k] = off[2 * k + 1];
    }
    split = 8u;
    return false;
  }
};

// The reload cursor: positions only (no lookahead), fewer registers; the
// slot of position u in the current column is u + delta.
struct SeqCursor1 {
  const uint2* e;
  int stride;
  uint32_t delta, next;
  __device__ __forceinline__ void from(const SeqCursor& c) {
    e = c.e;
    stride = c.stride;
    delta = c.b0 - c.c0;
    next = c.n0;
  }
  __device__ __forceinline__ uint32_t slot(uint32_t u) {
    while (u >= next) {
      e += stride;
      const uint2 e0 = e[0];
      delta = e0.x - e0.y;
      next = e[stride].y;
    }
    return u + delta;
  }
};

// The hit mask of the candidates [bb, be) (at most 64, one canonical block)
// of a target's sequence as two 32-bit words: sc.batch() screens eight at a
// time, their loads in flight together.  c1 walks forward only.
template <class Screen>
__device__ __forceinline__ void screen_block(SeqCursor& c1, uint32_t bb, uint32_t be,
                                             const Screen& sc, uint32_t& lo, uint32_t& hi) {
  lo = hi = 0u;
#pragma unroll 1
  for (uint32_t u = bb; u < be; u += 8) {
    const uint32_t valid = be - u >= 8u ? 0xFFu : (1u << (be - u)) - 1u;
    const uint32_t bits = sc.batch(c1, u, be - 1u) & valid;
    const uint32_t at = u - bb;  // the same for every lane
    if (at < 32u)
      lo |= bits << at;
    else
      hi |= bits << (at - 32u);
  }
}

// Visits sequence positions [u0, u1) of a candidate sequence of m positions
// in order, calling add() only for candidates passing the screen's test (see
// ScreenXyz, ScreenCoarse).  The positions are taken in groups of NB blocks of
// 64: each block of the group
// is screened eight loads at a time (across column boundaries, so a sparse
// neighbourhood costs a few memory round trips, not one or two per column)
// into a hit mask, then the hits of the whole group are reloaded G at a time
// (a pass policy's kHitBatch) and accumulated in ascending order, with
// block_end() called after the last hit of each block that has any, in order.
// Running the hits of several blocks through one loop keeps the lanes of a
// wavefront busy: they wait on the largest hit count of the group instead of
// that of every block.  Candidates failing the test contribute exactly
// nothing in add() (and a block without hits sums to zero), so the sums equal
// the plain in-order sum.
// The screening is branch-free after the loads (all eight tests are
// evaluated and masked), so the compiler keeps the eight loads in flight
// together instead of sinking some of them into conditional blocks that
// wait for each load in turn; the tests must be branch-free as well.
// The masks are walked as 32-bit words, the first of which holds the next hit:
// a hit costs one find-first, one clear and one select per word, where 64-bit
// masks took twice the instructions (a lane whose next word is empty sits one
// hit out).
// get_mask(b, lo, hi) may supply block b's hit mask (b = position / 64; u0
// must be a multiple of 64) instead of screening it; put_mask(b, lo, hi)
// receives each mask the sweep screened.
template <int G, int NB, class Screen, class LoadF, class Add, class BlockEnd, class GetMask,
          class PutMask>
__device__ __forceinline__ void sweep_seq(const SeqTable& st, uint32_t m, uint32_t u0,
                                          uint32_t u1, const Screen& sc, LoadF&& load_f,
                                          Add&& add, BlockEnd&& block_end, GetMask&& get_mask,
                                          PutMask&& put_mask) {
  if (u0 >= u1) return;
  constexpr int NW = 2 * NB;
  SeqCursor c1;
  c1.init(st, u0, m);
  SeqCursor1 c2;
  c2.from(c1);
#pragma unroll 1
  for (uint32_t gb = u0; gb < u1; gb += 64u * NB) {
    uint32_t w[NW];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const uint32_t bb = gb + 64u * (uint32_t)q;
      w[2 * q] = w[2 * q + 1] = 0u;
      if (bb < u1 && !get_mask(bb >> 6, w[2 * q], w[2 * q + 1])) {
        const uint32_t be = u1 - bb < 64u ? u1 : bb + 64u;
        screen_block(c1, bb, be, sc, w[2 * q], w[2 * q + 1]);
        put_mask(bb >> 6, w[2 * q], w[2 * q + 1]);
      }
    }
    // w[0] holds the remaining hits of positions [base, base + 32); block: the
    // one being summed
    uint32_t base = gb, last = gb, block = gb >> 6;
#pragma unroll 1
    while (true) {
      uint32_t any = w[0];
#pragma unroll
      for (int k = 1; k < NW; ++k) any |= w[k];
      if (!any) break;
      uint32_t j[G], blk[G];
      bool h[G];
#pragma unroll
      for (int t = 0; t < G; ++t) {
        const bool used = w[0] == 0u;
#pragma unroll
        for (int k = 0; k < NW; ++k) w[k] = used ? (k + 1 < NW ? w[k + 1] : 0u) : w[k];
        base += used ? 32u : 0u;
        h[t] = w[0] != 0u;
        // no hit: repeat the last (the cursor only moves forward)
        const uint32_t pos = h[t] ? base + (uint32_t)__builtin_ctz(w[0]) : last;
        last = pos;
        w[0] &= w[0] - 1u;
        j[t] = c2.slot(pos);
        blk[t] = base >> 6;
      }
      decltype(load_f(0u)) d[G];
#pragma unroll
      for (int t = 0; t < G; ++t) d[t] = load_f(j[t]);
#pragma unroll
      for (int t = 0; t < G; ++t)
        if (h[t]) {
          if (NB > 1 && blk[t] != block) {
            block_end();
            block = blk[t];
          }
          add(j[t], d[t]);
        }
    }
    block_end();
  }
}

// Orders the wavefront's LDS accesses (its lanes run in lockstep and the LDS
// serves them in issue order, so only the compiler must not move them).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exclusive prefix sum of v over the active lanes of the wavefront; *total
// receives the sum.  All active lanes must call it.
__device__ __forceinline__ uint32_t wave_exclusive_sum(uint32_t v, uint32_t* total) {
  const int lane = threadIdx.x & 63;
  uint32_t incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t t = __shfl_up(incl, off);
    if (lane >= off) incl += t;
  }
  *total = __shfl(incl, 63);
  return incl - v;
}

// Work lists of the heavy targets of one neighbour pass.
struct HeavyLists {
  // per pass parity: the record and chunk-item counters (rec_counter,
  // item_counter); counters[kThresholdWord]: the heavy threshold for the next
  // pass (0: kLightMax), set by each combine kernel from the kStatSlots
  // per-level target counts (stat_slot) the light kernel's wavefronts add
  // to.  Each word or slot has a 256-byte line of its own:
  // atomics on one line serialise, and every light wavefront reads the
  // threshold
  uint32_t* counters;
  uint4* recs;         // per heavy target: (i, first partial slot, chunks, 0)
  uint4* items;        // per chunk: (i, chunk index, partial slot, 0); i = ~0u: unused
  float* partials;     // per partial slot the pass's running sum, packed (at most
                       // kPartialWords floats)
  uint32_t item_cap;   // capacity of items / partials
  // screening coordinates of the positions the pass screens, for the policies
  // that use them (kCoarse), in the order of screen()
  uint2* coarse;
  // hit masks of the current iteration: block b of target i at
  // masks[b * mask_stride + i], b < kMaskBlocks (null: not kept)
  uint64_t* masks;
  uint32_t mask_stride;
};
constexpr int kPartialWords = 8;
constexpr int kCounterLine = 64;  // words
constexpr int kThresholdWord = 4 * kCounterLine;
constexpr int kStatSlots = 64;
constexpr int kCounterWords = (5 + kStatSlots) * kCounterLine;
// Statistics slot k: kLevelWords words of packed per-level target counts.
__host__ __device__ __forceinline__ int stat_slot(int k) { return (5 + k) * kCounterLine; }
__host__ __device__ __forceinline__ int rec_counter(int parity) {
  return 2 * parity * kCounterLine;
}
__host__ __device__ __forceinline__ int item_counter(int parity) {
  return (2 * parity + 1) * kCounterLine;
}
static_assert(3 * kCounterLine < kThresholdWord, "words below the threshold: the counters");

// x^n for the s_corr exponent: repeated multiplication for small integer n
// (the reference default n=4), powf otherwise.
__device__ __forceinline__ float pow_corr(float w, const StepConsts& c) {
  if (c.n_corr_int == 4) {
    // the reference default; exactly the product the loop below forms for
    // n = 4 (1 * ((w*w) * (w*w)))
    const float w2 = w * w;
    return w2 * w2;
  }
  if (c.n_corr_int >= 0) {
    float r = 1.0f, b = w;
    int e = c.n_corr_int;
    while (e) {
      if (e & 1) r = r * b;
      b = b * b;
      e >>= 1;
    }
    return r;
  }
  return powf(w, c.n_corr);
}

// Arithmetic contract: the kernels are built with -ffp-contract=off, so every
// expression below is evaluated as written (IEEE FP32 +,-,*,/,sqrt and the
// explicit fmaf calls).  The host oracle's FP32 mirror executes the same
// sequence, which makes a correct GPU result equal to it bit for bit.

// Squared distance of two positions: dx*dx, then + dy*dy and + dz*dz as
// fused multiply-adds.
__device__ __forceinline__ float dist2(const float4& a, const float4& b, float& dx, float& dy,
                                       float& dz) {
  dx = a.x - b.x;
  dy = a.y - b.y;
  dz = a.z - b.z;
  float r2 = dx * dx;
  r2 = fmaf(dy, dy, r2);
  r2 = fmaf(dz, dz, r2);
  return r2;
}

// The same with the second position as a float3 (screening loads of x, y, z
// only).
__device__ __forceinline__ float dist2(const float4& a, const float3& b, float& dx, float& dy,
                                       float& dz) {
  dx = a.x - b.x;
  dy = a.y - b.y;
  dz = a.z - b.z;
  float r2 = dx * dx;
  r2 = fmaf(dy, dy, r2);
  r2 = fmaf(dz, dz, r2);
  return r2;
}

// |a - b|^2 - bound with the bound as the first addend: negative below it, up to
// rounding (~1e-7 of the bound).
__device__ __forceinline__ float near2(const float4& a, const float3& b, float bound) {
  const float dx = a.x - b.x, dy = a.y - b.y, dz = a.z - b.z;
  return fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, -bound)));
}

// x, y, z of element j of a float4 array (a 12-byte load).
__device__ __forceinline__ float3 load_xyz(const float4* __restrict__ a, uint32_t j) {
  const float* p = reinterpret_cast<const float*>(a + j);
  return make_float3(p[0], p[1], p[2]);
}

// Correctly rounded square root and quotient for the operand ranges of the
// pair terms, where no operand or result is zero, subnormal, infinite or NaN
// and no exponent is extreme: there the compiler's IEEE sequences
// (-fhip-fp32-correctly-rounded-divide-sqrt) apply no scaling and no
// special-case fix-up, and what remains is exactly the sequence below, so
// the results are the IEEE results bit for bit (tests/test_gpu_arith.py and
// test_gpu_root.py, over all roots).  root_pair: s = x rsq(x), corrected by its
// residual times half the estimate (inputs r2 in [KERNAL_EPS^2 * 0.99,
// h^2 * 1.0001); a smaller input, down to 0, yields a value below KERNAL_EPS
// or a NaN, neither of which passes the callers' r >= KERNAL_EPS).  The
// estimate serves 1 / r as well: div_root makes its reciprocal from it by the
// Newton step with which div_pair makes one from v_rcp_f32, then both take the
// quotient with two residual corrections (numerators from 1e-18 to 1e6 over
// denominators from KERNAL_EPS to 1e4).  Transcendental instructions take four
// times as long as others: root and quotient need one and twelve others, where
// v_sqrt_f32, corrected by its neighbours' residuals, and v_rcp_f32 needed two
// and fifteen.  A step of 130,000 particles 604 -> 591 us, 1M dense
// 2150 -> 2110, 64 scenes 8.24 -> 8.03 ms.
struct Root {
  float r, inv;  // the root; an estimate of its reciprocal
};
__device__ __forceinline__ Root root_pair(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  const float s = x * y;
  return Root{fmaf(fmaf(-s, s, x), 0.5f * y, s), y};
}
// 1 / b from an estimate within a few ulp.
__device__ __forceinline__ float recip_step(float b, float y) {
  return fmaf(fmaf(-b, y, 1.0f), y, y);
}
// The estimate a root's reciprocal starts from: one unit up.  At mantissas of
// all ones the Newton step from v_rsq_f32's own value ends on the midpoint
// next to 1 / b and rounds to the wrong side of it.
__device__ __forceinline__ float root_inv(const Root& b) {
  return __int_as_float(__float_as_int(b.inv) + 1);
}
__device__ __forceinline__ float div_recip(float a, float b, float r) {
  float q = a * r;
  const float rem = fmaf(-b, q, a);
  q = fmaf(rem, r, q);
  const float rem2 = fmaf(-b, q, a);
  return fmaf(rem2, r, q);
}
__device__ __forceinline__ float div_root(float a, const Root& b) {
  return div_recip(a, b.r, recip_step(b.r, root_inv(b)));
}
__device__ __forceinline__ float div_pair(float a, float b) {
  return div_recip(a, b, recip_step(b, __builtin_amdgcn_rcpf(b)));
}

// poly6 numerator times its coefficient, for r2 < h2: poly6 * (h2-r2)^3.
__device__ __forceinline__ float poly6_of(float r2, const StepConsts& c) {
  const float t = c.h2 - r2;
  return ((c.poly6 * t) * t) * t;
}

// DensityBoundary (fluids/Simulator.cu:139-161): per face, 0 beyond h,
// 2pi/3 at or behind the wall, (2pi/3)(h-d)^2(h+d) in between; faces summed
// in the reference's order.
__device__ __forceinline__ float wall_density_at(float d, const StepConsts& c) {
  if (d > c.h) return 0.0f;
  if (d <= 0.0f) return c.wall_c;
  return ((c.wall_c * (c.h - d)) * (c.h - d)) * (c.h + d);
}

__device__ __forceinline__ float boundary_density(float x, float y, float z, const SceneGeo& g,
                                                  const StepConsts& c) {
  float s = wall_density_at(g.ulx - x, c);
  s = s + wall_density_at(x - g.llx, c);
  s = s + wall_density_at(g.uly - y, c);
  s = s + wall_density_at(y - g.lly, c);
  s = s + wall_density_at(g.ulz - z, c);
  s = s + wall_density_at(z - g.llz, c);
  return s;
}

// Caller vector arrays: LAYOUT 4 = float4 (16 B), LAYOUT 3 = packed float3.
template <int LAYOUT>
__device__ __forceinline__ float4 load_vec(const float* __restrict__ a, uint32_t i) {
  if constexpr (LAYOUT == 4) {
    return reinterpret_cast<const float4*>(a)[i];
  } else {
    const float* p = a + (size_t)i * 3;
    return make_float4(p[0], p[1], p[2], 0.0f);
  }
}

template <int LAYOUT>
__device__ __forceinline__ void store_vec(float* __restrict__ a, uint32_t i, float x, float y,
                                          float z) {
  if constexpr (LAYOUT == 4) {
    reinterpret_cast<float4*>(a)[i] = make_float4(x, y, z, 0.0f);
  } else {
    float* p = a + (size_t)i * 3;
    p[0] = x;
    p[1] = y;
    p[2] = z;
  }
}

// Counts particle of key k into cnt[k] (all lanes of the wavefront call it;
// valid lanes are a prefix) and returns its arrival number in that cell: one
// atomic per run of equal keys over consecutive lanes, which get consecutive
// numbers.
__device__ __forceinline__ uint32_t count_arrival(uint32_t k, bool valid,
                                                  uint32_t* __restrict__ cnt) {
  const int lane = threadIdx.x & 63;
  const uint32_t prev = __shfl_up(k, 1);
  const uint64_t vm = __builtin_amdgcn_ballot_w64(valid);
  const uint64_t hm = __builtin_amdgcn_ballot_w64(valid & ((lane == 0) | (prev != k)));
  const uint64_t upto = hm & (~0ull >> (63 - lane));
  const uint64_t later = lane == 63 ? 0ull : (hm >> (lane + 1)) << (lane + 1);
  const int head = upto ? 63 - __clzll((long long)upto) : lane;
  const int end = later ? __ffsll((unsigned long long)later) - 1 : __popcll(vm);
  uint32_t base = 0u;
  if (valid && lane == head) base = atomicAdd(&cnt[k], (uint32_t)(end - head));
  return __shfl(base, head) + (uint32_t)(lane - head);
}

// Rank of entry i among the cell's entries list[lo, hi).  A cell of up to
// kRankEntries is read by each of its lanes, eight loads in flight; a larger
// one (a pile: consecutive slots, so whole wavefronts rank the same cell) by
// the wavefront together, four loads of 64 entries in flight: entries that all
// lie below or above the indexes to rank are counted at once (particles arrive
// nearly in input order, so most do), the others passed to all lanes one by one.
// One load at a time and every entry passed, density error of 2M particles, of
// which 5,000 / 20,000 lie in one cell: 487 / 1145 -> 451 / 999 us, in random
// input order 625 / 1419 -> 584 / 1211 (with the radix sort 563 / 1081 and 592 /
// 1109); a step of 200,000 with 5,000 in one cell 984 -> 942 (sort: 963).
constexpr uint32_t kRankEntries = 64;
__device__ __forceinline__ uint32_t rank_in_cell(const uint2* __restrict__ list, uint32_t lo,
                                                 uint32_t hi, uint32_t i, bool valid) {
  const int lane = threadIdx.x & 63;
  uint32_t rank = 0u;
  const bool big = valid && hi - lo > kRankEntries;
  if (valid && !big) {
    for (uint32_t s = lo; s < hi; s += 8u) {
      uint32_t e[8];
#pragma unroll
      for (int t = 0; t < 8; ++t) e[t] = list[s + t < hi ? s + t : hi - 1u].x;
#pragma unroll
      for (int t = 0; t < 8; ++t) rank += ((s + t < hi) & (e[t] < i)) ? 1u : 0u;
    }
  }
  uint64_t todo = __builtin_amdgcn_ballot_w64(big);
  while (todo) {
    const int src = __builtin_ctzll(todo);
    const uint32_t l = (uint32_t)__builtin_amdgcn_readlane((int)lo, src);
    const uint32_t h = (uint32_t)__builtin_amdgcn_readlane((int)hi, src);
    const bool mine = big & (lo == l);
    // the range of the indexes to rank
    uint32_t least = mine ? i : ~0u, most = mine ? i : 0u;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t a = __shfl_xor(least, d), b = __shfl_xor(most, d);
      least = a < least ? a : least;
      most = b > most ? b : most;
    }
    uint32_t r = 0u;
    for (uint32_t s = l; s < h; s += 256u) {
      uint32_t e[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t at = s + 64u * (uint32_t)q + (uint32_t)lane;
        e[q] = at < h ? list[at].x : ~0u;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint64_t below = __builtin_amdgcn_ballot_w64(e[q] < least);
        const uint64_t above = __builtin_amdgcn_ballot_w64(e[q] > most);
        if ((below | above) == ~0ull) {
          r += (uint32_t)__popcll(below);
          continue;
        }
#pragma unroll
        for (int t = 0; t < 64; ++t)
          r += (uint32_t)__builtin_amdgcn_readlane((int)e[q], t) < i ? 1u : 0u;
      }
    }
    if (mine) rank = r;
    todo &= ~__builtin_amdgcn_ballot_w64(mine);
  }
  return rank;
}

// Particles per cell, counted from the sorted keys (the input of the
// cell-start scan).  Equal keys are contiguous after the sort, so a run that
// lies inside one wavefront is that cell's only run and its first lane
// stores the count; a run touching a wavefront boundary (at most two per
// wavefront) may continue in the neighbouring wavefront, and each of its
// parts is added atomically.  The counts must be zero beforehand (the scan
// re-zeroes them).
__device__ __forceinline__ void count_sorted(const uint32_t* __restrict__ skey, int s, int n,
                                             uint32_t* __restrict__ cnt) {
  const int lane = threadIdx.x & 63;
  const bool valid = s < n;
  const uint32_t k = valid ? skey[s] : 0u;
  const uint32_t prev = __shfl_up(k, 1);
  const uint64_t vm = __ballot(valid);
  const bool head = valid && (lane == 0 || prev != k);
  const uint64_t hm = __ballot(head);
  if (head) {
    // run = [lane, next head or end of the valid lanes)
    const uint64_t later = lane == 63 ? 0ull : (hm >> (lane + 1)) << (lane + 1);
    const int end = later ? __ffsll((unsigned long long)later) - 1 : 64 - __clzll(vm);
    const int len = end - lane;
    const int after = s + len;  // sorted index just past the run
    const bool open_left = lane == 0 && s > 0 && skey[s - 1] == k;
    const bool open_right = !later && after < n && skey[after] == k;
    if (open_left || open_right)
      atomicAdd(&cnt[k], (uint32_t)len);
    else
      cnt[k] = (uint32_t)len;
  }
}

}  // namespace pbf
