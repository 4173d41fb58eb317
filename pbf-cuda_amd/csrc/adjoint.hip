// adjoint.hip — reverse-mode derivative of one PBF frame on gfx950.
//
// The frame is differentiated with its discrete choices held fixed (sort
// order, stale grid, candidate lists, kernel cutoffs, active clamps), along
// the trajectory the forward kernels computed, which a tape records: per
// solver iteration k the positions and lambdas xl[k], the lambda pass's
// (sum of gradients S, denominator D) and densities, and the correction
// before its clamps.  Derivatives follow the reference's formulas
// (fluids/Simulator_kernel.cuh:52-239): lambda_i = -(rho_i/pho0 - 1)/D_i with
// D_i = sum_{j!=i} |g_ij|^2 + |S_i|^2 + eps, g_ij = spikyGrad(x_i-x_j)/pho0;
// dp_i = sum_{j!=i} (lambda_i + lambda_j + s_corr) spikyGrad / pho0, clamped;
// XSPH v'_i = v_i + c sum_j 2 (v_j - v_i) W_ij / (rho_i + rho_j).
//
// Every backward neighbour pass is a pass policy of pbf_pass.h.  A pair term
// of target i (j in its candidate list cand(i)) depends on x_i and x_j; its
// derivatives belong to both.  The stale grid makes candidate lists
// one-sided (j in cand(i) does not imply i in cand(j)), and two modes
// collect the terms (see the comment before member_word below):
//  * scatter: i sweeps cand(i) on the sorted grid, gathers its own terms
//    and, where i is in cand(j), j's term about i; where it is not, i adds
//    d(its term)/dx_j to j with float atomics into "extra" arrays that a
//    later kernel folds in (their order of addition depends on timing);
//  * gather: i sweeps a grid built on the pass's own positions, which holds
//    every particle within h, and gathers every term that concerns it; no
//    atomics, every sum in a fixed order.
#include "pbf_adjoint.h"
#include "pbf_pass.h"

namespace pbf {

namespace {

// Sorted (stale-grid) cell of a particle from its sorted key.
__device__ __forceinline__ Cell cell_of_key(uint32_t key, const SceneGeo& g) {
  const uint32_t local = key - g.base;
  const uint32_t yz = (uint32_t)(g.dy * g.dz);
  const uint32_t x = local / yz;
  const uint32_t r = local - x * yz;
  const uint32_t y = r / (uint32_t)g.dz;
  return Cell{(int)x, (int)y, (int)(r - y * (uint32_t)g.dz)};
}

// Query cells packed 10 bits per axis (x << 20 | y << 10 | z), valid when
// every grid dimension is at most 1024; a pointwise kernel computes them once
// per particle and position set, so the pair terms compare bit fields
// instead of dividing three coordinates per pair.
__device__ __forceinline__ bool packed_query_cells(const StepConsts& c) {
  return c.g.dx <= 1024 && c.g.dy <= 1024 && c.g.dz <= 1024;
}
__device__ __forceinline__ uint32_t pack_cell(const Cell& q) {
  return ((uint32_t)q.x << 20) | ((uint32_t)q.y << 10) | (uint32_t)q.z;
}

// Whether a particle whose sorted cell is ci is a candidate of the particle
// at position xj (ci in the 3x3x3 block around xj's query cell); qj is xj's
// packed query cell (read only when the packing is valid).
__device__ __forceinline__ bool is_candidate_of(const Cell& ci, const float4& xj, uint32_t qj,
                                                const StepConsts& c) {
  if (packed_query_cells(c)) {
    const int qx = (int)(qj >> 20), qy = (int)((qj >> 10) & 1023u), qz = (int)(qj & 1023u);
    return abs(ci.x - qx) <= 1 && abs(ci.y - qy) <= 1 && abs(ci.z - qz) <= 1;
  }
  const Cell q = cell_of(xj.x, xj.y, xj.z, c.g, c.h);
  return abs(ci.x - q.x) <= 1 && abs(ci.y - q.y) <= 1 && abs(ci.z - q.z) <= 1;
}

// dW/dx_i of poly6 at d = x_i - x_j is this times d: -6 poly6 (h2 - r2)^2,
// with t = h2 - r2 (0 beyond h).
__device__ __forceinline__ float poly6_slope(float t, const StepConsts& c) {
  return (-6.0f * c.poly6 * t) * t;
}

// 1/x to about one ulp (v_rcp_f32 and one Newton step).  The adjoint only
// has to agree with the FP64 adjoint to a relative 1e-4, so each pair
// divides once and multiplies by the reciprocal where the forward formulas
// divide.
__device__ __forceinline__ float recip(float x) {
  return recip_step(x, __builtin_amdgcn_rcpf(x));
}

// Hessian of k (h - r)^2 d / r (the spiky gradient with coefficient k):
// phi I + psi d d^T, phi = k u^2 / r, psi = -k u (h + r) / r^3, u = h - r.
struct SpikyHess {
  float phi, psi;
};
__device__ __forceinline__ SpikyHess spiky_hess(float k, float r, float inv_r,
                                                const StepConsts& c) {
  const float u = c.h - r;
  return SpikyHess{k * u * u * inv_r, -k * u * (c.h + r) * (inv_r * inv_r * inv_r)};
}
// d s_corr / d w for s_corr = coef_corr * w^n_corr.
__device__ __forceinline__ float dscorr_dw(float w, const StepConsts& c) {
  if (c.n_corr_int == 0 || c.n_corr == 0.0f) return 0.0f;
  if (c.n_corr_int == 4) return c.coef_corr * c.n_corr * ((w * w) * w);
  if (c.n_corr_int > 0) {
    float r = 1.0f;
    for (int e = 1; e < c.n_corr_int; ++e) r = r * w;
    return c.coef_corr * c.n_corr * r;
  }
  return w > 0.0f ? c.coef_corr * c.n_corr * powf(w, c.n_corr - 1.0f) : 0.0f;
}

__device__ __forceinline__ float dot3(const float3& a, const float3& b) {
  return fmaf(a.z, b.z, fmaf(a.y, b.y, a.x * b.x));
}
// a p + b q
__device__ __forceinline__ float3 comb(float a, const float3& p, float b, const float3& q) {
  return make_float3(fmaf(a, p.x, b * q.x), fmaf(a, p.y, b * q.y), fmaf(a, p.z, b * q.z));
}

// The scattered pair sums: kScatterCopies copies of n float4 entries, stored
// component-major ([component][copy][n] floats) so the four atomic adds of
// one scatter land on four cache lines.  A workgroup adds to copy
// blockIdx.x % kScatterCopies.
__device__ __forceinline__ size_t scatter_copy(uint32_t n) {
  return (size_t)(blockIdx.x % kScatterCopies) * n;
}
// Adds (x, y, z[, w]) at copy offset e (scatter_copy(n) + j).
__device__ __forceinline__ void scatter_add(float4* ex, uint32_t n, size_t e, float x, float y,
                                            float z, float w, bool with_w) {
  float* f = reinterpret_cast<float*>(ex);
  const size_t cs = (size_t)kScatterCopies * n;
  atomicAdd(&f[e], x);
  atomicAdd(&f[cs + e], y);
  atomicAdd(&f[2 * cs + e], z);
  if (with_w) atomicAdd(&f[3 * cs + e], w);
}
// Sum of the copies of entry i (in copy order), which are cleared.
__device__ __forceinline__ float4 take_scattered(float4* __restrict__ ex, int i, int n) {
  float* f = reinterpret_cast<float*>(ex);
  const size_t cs = (size_t)kScatterCopies * n;
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int k = 0; k < kScatterCopies; ++k) {
      const size_t idx = q * cs + (size_t)k * n + i;
      v[q] = v[q] + f[idx];
      f[idx] = 0.0f;
    }
  return make_float4(v[0], v[1], v[2], v[3]);
}

// Two modes share each backward pass policy:
//  * scatter (kGather = false): targets in the frame's sorted order sweep the
//    sorted (stale) grid around their query cell, so every candidate's own
//    term counts; j's term about i is gathered when i is a candidate of j
//    and otherwise i's term about j is scattered to j (float atomics);
//  * gather (kGather = true): targets and candidates in the order of a grid
//    built on the pass's own positions (sorted by query cell).  A target
//    sweeps that grid around its query cell, which holds every particle
//    within h of it, and tests both memberships per pair from each
//    slot's sorted and query cell (member_word): its own term counts when j is
//    its candidate, j's term about it when it is j's candidate.  Every term
//    is gathered by the particle it belongs to, in a fixed order: no atomics.
//    A pair within h whose query cells are two apart (possible only through
//    rounding when |x_i - x_j| is within ~1e-6 h of h, where every term and
//    derivative is ~0) is the only pair this sweep can miss.

// The memberships of a gather-mode pair from one word per particle.  A sweep's
// candidate j of target t has its query cell q_j within one of q_t on each
// axis, so with a particle's sorted cell s kept as q + clamp(s - q, +-3) both
// tests, |s_j - q_t| <= 1 and |s_t - q_j| <= 1, hold exactly when they hold
// modulo 8.  Six fields of 5 bits: that sorted cell's x, y, z, then q's, each
// modulo 8 plus 9; a difference of fields then ends in (difference + 1) modulo
// 8, which is at most 2 where the test holds.
// The word travels in the w of an element that the pass loads anyway (the lambda pass, which
// has none free, loads it apart).  Two packed cells of 8 bytes a particle, compared axis by
// axis -> this: delta-p pass of 270,000 particles 108 -> 100 us, lambda pass 57 -> 53, XSPH pass
// 97 -> 86, a stored rollout of them 3330 -> 3205, one 4M-particle sweeping-wall frame with
// gradients 56.7 -> 55.3 ms.
constexpr uint32_t kMemberOnes = 0x02108421u;  // 1 in each field
__device__ __forceinline__ uint32_t member_word(uint32_t sorted, uint32_t query) {
  uint32_t w = 0u;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const int s = (int)((sorted >> (10 * k)) & 1023u), q = (int)((query >> (10 * k)) & 1023u);
    const int d = s - q < -3 ? -3 : (s - q > 3 ? 3 : s - q);
    w |= ((uint32_t)(q + d) & 7u) << (5 * k) | ((uint32_t)q & 7u) << (15 + 5 * k);
  }
  return w + 9u * kMemberOnes;
}
// A target's word as member_fails() takes it: its query cell under the
// candidates' sorted cells and the other way about, without the 9s.
__device__ __forceinline__ uint32_t member_target(uint32_t w) {
  const uint32_t v = w - 9u * kMemberOnes;
  return v >> 15 | (v & 0x7fffu) << 15;
}
// Bits in the low 15: j is no candidate of t; above: t is none of j.
__device__ __forceinline__ uint32_t member_fails(uint32_t target, uint32_t word) {
  return (((word - target) & 7u * kMemberOnes) + 5u * kMemberOnes) & 8u * kMemberOnes;
}

// Memberships of a pair (target t, candidate j): own = j is a candidate of
// t (t's own term about j exists), other = t is a candidate of j.
struct Members {
  bool own, other;
};
template <bool kGather>
__device__ __forceinline__ Members members(const Cell& ct, uint32_t tc, const float4& xj,
                                           uint32_t jc, const StepConsts& c) {
  if constexpr (kGather) {
    const uint32_t v = member_fails(tc, jc);
    return Members{(v & 0x7fffu) == 0u, v < 0x8000u};
  } else {
    // the sweep ran over t's candidates; jc: j's packed query cell
    return Members{true, is_candidate_of(ct, xj, jc, c)};
  }
}

// The adjoint vectors of a pair: i's own where its own term counts, minus
// j's where j's term about i counts.  The two terms of a pair are the same
// linear function of the vector, j's with the opposite sign, so each pass
// evaluates it once for the difference.  The passes wait for the pair's loads
// as much as they compute.  Both terms evaluated apart -> once, in fused
// multiply-adds: delta-p pass of 270,000 particles 120 -> 108 us, a stored
// rollout of them 3470 -> 3338, one 4M-particle sweeping-wall frame with
// gradients 58.2 -> 56.9 ms.
__device__ __forceinline__ float3 pair_vector(const Members& mb, const float4& own,
                                              const float4& other) {
  return make_float3((mb.own ? own.x : 0.0f) - (mb.other ? other.x : 0.0f),
                     (mb.own ? own.y : 0.0f) - (mb.other ? other.y : 0.0f),
                     (mb.own ? own.z : 0.0f) - (mb.other ? other.z : 0.0f));
}

// ---- XSPH -----------------------------------------------------------------
template <bool kGather>
struct BwdXsphPass {
  // scatter mode: workgroups in launch order, round-robin over the XCDs, so a
  // crowded cell's targets scatter from all eight XCDs, each into its own
  // copy; gather mode: runs of workgroups (the team kernel: one contiguous
  // range per XCD in both, so there such a cell uses one copy)
  static constexpr bool kXcdRanges = kGather;
  static constexpr bool kCoarse = kGather;
  // hits reloaded per round of the sweep
  static constexpr int kHitBatch = 4;
  struct Args {
    const float4* __restrict__ x;    // final positions
    const float4* __restrict__ vr;   // (v before XSPH, rho of the last lambda pass)
    const float4* __restrict__ gv;   // adjoint of v after XSPH; gather: w = member_word()
    const uint32_t* __restrict__ key;  // scatter: sorted keys
    float4* __restrict__ out_x;      // gathered (dL/dx, dL/drho)
    float4* __restrict__ out_v;      // gathered dL/dv (pair terms)
    float4* __restrict__ ex_x;       // scatter: (dL/dx, dL/drho), kScatterCopies x ex_n
    float4* __restrict__ ex_v;       // scatter: dL/dv, kScatterCopies x ex_n
    uint32_t ex_n;
    const uint32_t* __restrict__ qc;  // scatter: packed query cells of x
  };
  struct Target {
    float4 x, vr, gv;
    Cell cell;
    uint32_t c;  // gather: member_target()
    uint32_t i;
  };
  struct Acc {
    float vx = 0.0f, vy = 0.0f, vz = 0.0f, xx = 0.0f, xy = 0.0f, xz = 0.0f, r = 0.0f;
  };
  struct Nb {
    float4 x, vr, gv;
    uint32_t c;  // gather: member_word(), scatter: packed query cell
  };
  static __device__ __forceinline__ Target target(const Args& a, uint32_t i, const StepConsts& c) {
    const float4 gv = a.gv[i];
    if constexpr (kGather)
      return Target{a.x[i], a.vr[i], gv, Cell{}, member_target(__float_as_uint(gv.w)), i};
    else
      return Target{a.x[i], a.vr[i], gv, cell_of_key(a.key[i], c.g), 0u, i};
  }
  static __device__ __forceinline__ const float4* screen(const Args& a) { return a.x; }
  static __device__ __forceinline__ Nb load_f(const Args& a, uint32_t j) {
    const float4 gv = a.gv[j];
    return Nb{a.x[j], a.vr[j], gv, kGather ? __float_as_uint(gv.w) : a.qc[j]};
  }
  static __device__ __forceinline__ bool hit(const Target& t, const float3& xj,
                                             const StepConsts& c) {
    float dx, dy, dz;
    return dist2(t.x, xj, dx, dy, dz) < c.h2;
  }
  static constexpr bool kNear = true;
  static __device__ __forceinline__ float near(const Target& t, const float3& xj,
                                               const StepConsts& c) {
    return near2(t.x, xj, c.h2_outer);
  }
  static __device__ __forceinline__ void add(Acc& s, const Target& t, uint32_t j, const Nb& nb,
                                             const StepConsts& c, const Args& a) {
    float dx, dy, dz;
    const float r2 = dist2(t.x, nb.x, dx, dy, dz);
    if (!(r2 < c.h2)) return;
    const Members mb = members<kGather>(t.cell, t.c, nb.x, nb.c, c);
    if (!(mb.own || mb.other)) return;  // no term: nothing of j may enter (0 * inf)
    const float3 d = make_float3(dx, dy, dz);
    const float W = poly6_of(r2, c);
    const float p = poly6_slope(c.h2 - r2, c);
    const float inv_den = recip(t.vr.w + nb.vr.w);  // 1 / (rho_i + rho_j)
    const float k2 = 2.0f * c.c_xsph * inv_den;
    const float f = k2 * W;
    const float3 dv = make_float3(nb.vr.x - t.vr.x, nb.vr.y - t.vr.y, nb.vr.z - t.vr.z);
    const float3 B = pair_vector(mb, t.gv, nb.gv);
    const float u = dot3(B, dv);
    const float fx = (k2 * u) * p;
    const float fr = (f * inv_den) * u;  // 2 c W / (rho_i + rho_j)^2 times u
    s.vx = fmaf(-f, B.x, s.vx);
    s.vy = fmaf(-f, B.y, s.vy);
    s.vz = fmaf(-f, B.z, s.vz);
    s.xx = fmaf(fx, d.x, s.xx);
    s.xy = fmaf(fx, d.y, s.xy);
    s.xz = fmaf(fx, d.z, s.xz);
    s.r -= fr;
    if constexpr (!kGather) {
      if (!mb.other && j != t.i) {
        // j never visits i: deliver the own term's derivatives about j
        const size_t e = scatter_copy(a.ex_n) + j;
        scatter_add(a.ex_v, a.ex_n, e, f * B.x, f * B.y, f * B.z, 0.0f, false);
        scatter_add(a.ex_x, a.ex_n, e, -fx * d.x, -fx * d.y, -fx * d.z, -fr, true);
      }
    }
  }
  static __device__ __forceinline__ void accumulate(Acc& tot, const Acc& p) {
    tot.vx += p.vx;
    tot.vy += p.vy;
    tot.vz += p.vz;
    tot.xx += p.xx;
    tot.xy += p.xy;
    tot.xz += p.xz;
    tot.r += p.r;
  }
  static __device__ __forceinline__ void finish(const Args& a, const Target& t, const Acc& s,
                                                const StepConsts&, const SceneGeo&) {
    a.out_x[t.i] = make_float4(s.xx, s.xy, s.xz, s.r);
    a.out_v[t.i] = make_float4(s.vx, s.vy, s.vz, 0.0f);
  }
};

// ---- delta-p ----------------------------------------------------------------
template <bool kGather>
struct BwdDeltaPass {
  // scatter mode: round-robin workgroups (see BwdXsphPass); gather mode: runs of
  // workgroups
  static constexpr bool kXcdRanges = kGather;
  // hit masks for the lambda pass of the same iteration, which sweeps the
  // same candidates of the same positions (its hit test below)
  static constexpr int kMask = kMaskStore;
  // hits reloaded per round of the sweep
  static constexpr int kHitBatch = 4;
  struct Args {
    const float4* __restrict__ xl;   // (x, lambda) of the iteration
    const float4* __restrict__ A;    // (adjoint of the correction sum (before / pho0), as
                                     //  float bits scatter: packed query cell of xl,
                                     //  gather: member_word())
    const uint32_t* __restrict__ key;  // scatter: sorted keys
    float4* __restrict__ out;        // gathered (dL/dx, dL/dlambda)
    float4* __restrict__ ex;         // scatter: (dL/dx, dL/dlambda), kScatterCopies x ex_n
    uint32_t ex_n;
  };
  struct Target {
    float4 x, A;
    Cell cell;
    uint32_t c;  // gather: member_target()
    uint32_t i;
  };
  struct Acc {
    float x = 0.0f, y = 0.0f, z = 0.0f, l = 0.0f;
  };
  struct Nb {
    float4 x, A;
    uint32_t c;  // gather: member_word(), scatter: packed query cell
  };
  static __device__ __forceinline__ Target target(const Args& a, uint32_t i, const StepConsts& c) {
    const float4 A = a.A[i];
    if constexpr (kGather)
      return Target{a.xl[i], A, Cell{}, member_target(__float_as_uint(A.w)), i};
    else
      return Target{a.xl[i], A, cell_of_key(a.key[i], c.g), 0u, i};
  }
  static __device__ __forceinline__ const float4* screen(const Args& a) { return a.xl; }
  static __device__ __forceinline__ Nb load_f(const Args& a, uint32_t j) {
    const float4 A = a.A[j];
    return Nb{a.xl[j], A, __float_as_uint(A.w)};
  }
  static __device__ __forceinline__ bool hit(const Target& t, const float3& xj,
                                             const StepConsts& c) {
    float dx, dy, dz;
    // i itself and coincident pairs (r2 = 0) add nothing; pairs closer than
    // KERNAL_EPS add nothing here either (add() drops them) but are hits of
    // the lambda pass, which uses these masks.  With coincident pairs let
    // through (near(), or the screening coordinates) the chunk items of piles
    // take 1437 us instead of 935 (4M particles under the sweeping wall).
    const float r2 = dist2(t.x, xj, dx, dy, dz);
    return (r2 < c.h2_outer) & (r2 > 0.0f);
  }
  static __device__ __forceinline__ void add(Acc& s, const Target& t, uint32_t j, const Nb& nb,
                                             const StepConsts& c, const Args& a) {
    if (j == t.i) return;
    float dx, dy, dz;
    const float r2 = dist2(t.x, nb.x, dx, dy, dz);
    if (!(r2 < c.h2_outer)) return;
    const Root root = root_pair(r2);
    const float r = root.r;
    if (!(r >= c.keps && r < c.h)) return;
    const Members mb = members<kGather>(t.cell, t.c, nb.x, nb.c, c);
    if (!(mb.own || mb.other)) return;  // no term: nothing of j may enter (0 * inf)
    const float3 d = make_float3(dx, dy, dz);
    const float tt = fmaxf(c.h2 - r2, 0.0f);
    const float w = ((c.poly6 * tt) * tt) * tt;
    const float q = (t.x.w + nb.x.w) + c.coef_corr * pow_corr(w, c);
    const float ds = dscorr_dw(w, c) * poly6_slope(tt, c);  // d s_corr / dx_i is this times d
    const SpikyHess H = spiky_hess(c.spiky, r, recip_step(r, root.inv), c);
    // own term A_i . (q G(d)), j's term about i -q A_j . G(d), G = phi d
    const float3 A = pair_vector(mb, t.A, nb.A);
    const float Ad = dot3(A, d);
    const float AG = H.phi * Ad;
    const float3 g = comb(q * H.phi, A, fmaf(q * H.psi, Ad, AG * ds), d);
    s.x += g.x;
    s.y += g.y;
    s.z += g.z;
    s.l += AG;
    if constexpr (!kGather) {
      if (!mb.other) {
        const size_t e = scatter_copy(a.ex_n) + j;
        scatter_add(a.ex, a.ex_n, e, -g.x, -g.y, -g.z, AG, true);
      }
    }
  }
  static __device__ __forceinline__ void accumulate(Acc& tot, const Acc& p) {
    tot.x += p.x;
    tot.y += p.y;
    tot.z += p.z;
    tot.l += p.l;
  }
  static __device__ __forceinline__ void finish(const Args& a, const Target& t, const Acc& s,
                                                const StepConsts&, const SceneGeo&) {
    a.out[t.i] = make_float4(s.x, s.y, s.z, s.l);
  }
};

// ---- lambda (density and gradient norms) ------------------------------------
template <bool kGather>
struct BwdLambdaPass {
  // scatter mode: round-robin workgroups (see BwdXsphPass); gather mode: runs of
  // workgroups
  static constexpr bool kXcdRanges = kGather;
  // the delta-p pass's hit masks (its hit test is this pass's)
  static constexpr int kMask = kMaskLoad;
  // hits reloaded per round of the sweep
  static constexpr int kHitBatch = 4;
  struct Args {
    const float4* __restrict__ xr;   // (x, dL/drho)
    const float4* __restrict__ sd;   // (S, dL/dD)
    const uint32_t* __restrict__ key;  // scatter: sorted keys
    const float4* gin;  // adjoint of x before the pass (sorted order)
    float4* gout;       // gin + gathered (sorted order; may alias gin)
    const float4* __restrict__ more;  // gather: what k_bwd_lambda_pre adds to gin (query order)
    float4* __restrict__ ex;         // scatter: dL/dx, kScatterCopies x ex_n
    uint32_t ex_n;
    const uint32_t* __restrict__ qc;   // scatter: packed query cells of x, gather: member_word()s
    const uint32_t* __restrict__ slot;  // gather: sorted slot of each query slot
  };
  struct Target {
    float4 x, sd;
    Cell cell;
    uint32_t c;  // gather: member_target()
    uint32_t i;
  };
  struct Acc {
    float x = 0.0f, y = 0.0f, z = 0.0f;
  };
  struct Nb {
    float4 x, sd;
    uint32_t c;  // gather: member_word(), scatter: packed query cell
  };
  static __device__ __forceinline__ Target target(const Args& a, uint32_t i, const StepConsts& c) {
    if constexpr (kGather)
      return Target{a.xr[i], a.sd[i], Cell{}, member_target(a.qc[i]), i};
    else
      return Target{a.xr[i], a.sd[i], cell_of_key(a.key[i], c.g), 0u, i};
  }
  static __device__ __forceinline__ const float4* screen(const Args& a) { return a.xr; }
  static __device__ __forceinline__ Nb load_f(const Args& a, uint32_t j) {
    return Nb{a.xr[j], a.sd[j], a.qc[j]};
  }
  static __device__ __forceinline__ bool hit(const Target& t, const float3& xj,
                                             const StepConsts& c) {
    float dx, dy, dz;
    // coincident pairs (and i itself) have d = 0: every term below vanishes
    // (the delta-p pass stores masks of this test)
    const float r2 = dist2(t.x, xj, dx, dy, dz);
    return (r2 < c.h2_outer) & (r2 > 0.0f);
  }
  static __device__ __forceinline__ void add(Acc& s, const Target& t, uint32_t j, const Nb& nb,
                                             const StepConsts& c, const Args& a) {
    float dx, dy, dz;
    const float r2 = dist2(t.x, nb.x, dx, dy, dz);
    if (!(r2 < c.h2_outer)) return;
    const float3 d = make_float3(dx, dy, dz);
    const Members mb = members<kGather>(t.cell, t.c, nb.x, nb.c, c);
    if (!(mb.own || mb.other)) return;  // no term: nothing of j may enter (0 * inf)
    // density: the coefficient of d in both terms (from h on there is no term,
    // whatever the adjoint: 0 * inf)
    float k = r2 < c.h2 ? ((mb.own ? t.x.w : 0.0f) + (mb.other ? nb.x.w : 0.0f)) *
                              poly6_slope(c.h2 - r2, c)
                        : 0.0f;
    float phi = 0.0f;
    float3 V = make_float3(0.0f, 0.0f, 0.0f);
    const Root root = root_pair(r2);
    const float r = root.r;
    if (r >= c.keps && r < c.h && j != t.i) {
      // gradient norms: 2 D_i H (g + S_i) + 2 D_j H (g - S_j), g = phi d
      const SpikyHess H = spiky_hess(c.spiky_rho0, r, recip_step(r, root.inv), c);
      const float4 si = mb.own ? t.sd : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      const float4 sj = mb.other ? nb.sd : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      const float ki = 2.0f * si.w;
      const float kj = 2.0f * sj.w;
      const float3 S = make_float3(fmaf(ki, si.x, -kj * sj.x), fmaf(ki, si.y, -kj * sj.y),
                                   fmaf(ki, si.z, -kj * sj.z));
      const float kg = (ki + kj) * H.phi;
      V = make_float3(fmaf(kg, d.x, S.x), fmaf(kg, d.y, S.y), fmaf(kg, d.z, S.z));
      phi = H.phi;
      k = fmaf(H.psi, dot3(V, d), k);
    }
    const float3 g = comb(phi, V, k, d);
    s.x += g.x;
    s.y += g.y;
    s.z += g.z;
    if constexpr (!kGather) {
      if (!mb.other && j != t.i)
        scatter_add(a.ex, a.ex_n, scatter_copy(a.ex_n) + j, -g.x, -g.y, -g.z, 0.0f, false);
    }
  }
  static __device__ __forceinline__ void accumulate(Acc& tot, const Acc& p) {
    tot.x += p.x;
    tot.y += p.y;
    tot.z += p.z;
  }
  static __device__ __forceinline__ void finish(const Args& a, const Target& t, const Acc& s,
                                                const StepConsts&, const SceneGeo&) {
    const uint32_t k = kGather ? a.slot[t.i] : t.i;
    float4 g = a.gin[k];
    if constexpr (kGather) {
      const float4 o = a.more[t.i];
      g = make_float4(g.x + o.x, g.y + o.y, g.z + o.z, 0.0f);
    }
    a.gout[k] = make_float4(g.x + s.x, g.y + s.y, g.z + s.z, 0.0f);
  }
};

// ---- pointwise kernels -------------------------------------------------------
// In gather mode the pass outputs are in query order: work-item u handles
// query slot u, whose sorted slot is perm[u]; sorted-order arrays are read
// and written at perm[u].  In scatter mode both orders are the sorted one.

// After the XSPH pass: dL/dx_final, dL/dx_start (from v = (x - x0)/dt) and
// dL/drho of the last lambda pass; scatter mode: adds and clears the extras.
template <bool kGather>
__global__ __launch_bounds__(kBlock) void k_bwd_velocity(
    int n, StepConsts c, const uint32_t* __restrict__ perm, const float4* __restrict__ gx_out,
    const float4* __restrict__ gv_out, const float4* __restrict__ out_x,
    const float4* __restrict__ out_v, float4* __restrict__ ex_x, float4* __restrict__ ex_v,
    float4* __restrict__ gx, float4* __restrict__ gx0, float* __restrict__ grho) {
  const int u = blockIdx.x * kBlock + threadIdx.x;
  if (u >= n) return;
  const int i = kGather ? (int)perm[u] : u;
  float4 ex = make_float4(0.0f, 0.0f, 0.0f, 0.0f), ev = ex;
  if constexpr (!kGather) {
    ex = take_scattered(ex_x, u, n);
    ev = take_scattered(ex_v, u, n);
  }
  const float4 ox = out_x[u], ov = out_v[u], go = gx_out[i], gvo = gv_out[i];
  const float vx = gvo.x + ov.x + ev.x, vy = gvo.y + ov.y + ev.y, vz = gvo.z + ov.z + ev.z;
  gx[i] = make_float4(go.x + ox.x + ex.x + vx * c.inv_dt, go.y + ox.y + ex.y + vy * c.inv_dt,
                      go.z + ox.z + ex.z + vz * c.inv_dt, 0.0f);
  gx0[i] = make_float4(-vx * c.inv_dt, -vy * c.inv_dt, -vz * c.inv_dt, 0.0f);
  grho[i] = ox.w + ex.w;
}

// Query cell of position x: written packed (qc, scatter mode) or as the key of
// the pass's grid (qkey, gather mode) with, in qval, its sorted slot (the radix
// sort) or its arrival number in that cell (cnt not null: the counted grid).
// All lanes of the wavefront call it; invalid ones write nothing.
__device__ __forceinline__ uint32_t note_query_cell(int i, bool valid, const float4& x,
                                                    const StepConsts& c,
                                                    uint32_t* __restrict__ qc,
                                                    uint32_t* __restrict__ qkey,
                                                    uint32_t* __restrict__ qval,
                                                    uint32_t* __restrict__ cnt) {
  const Cell q = cell_of(x.x, x.y, x.z, c.g, c.h);
  const uint32_t packed = pack_cell(q);
  if (qc && valid) qc[i] = packed;
  if (qkey) {
    const uint32_t k = cell_id(q, c.g);
    const uint32_t v = cnt ? count_arrival(k, valid, cnt) : (uint32_t)i;
    if (valid) {
      qkey[i] = k;
      qval[i] = v;
    }
  }
  return packed;
}

// Position update of iteration k (fluids/Simulator_kernel.cuh:184-192):
// x' = clamp_box(x + clamp(dp, +-MAX_DP)).  gx = dL/dx' -> gxn = identity
// part of dL/dx, A = dL/d(correction sum), r0 += dL/dpho0 through the / pho0;
// A.w holds the packed query cell of x, also noted for the passes (see
// note_query_cell); gather mode (pc: packed sorted cells): the membership word,
// made here, where pc is read in order, instead of after the gather: 4M gather
// 190 -> 173 us, a stored rollout of 270,000 particles 3112 -> 3062.
__global__ __launch_bounds__(kBlock) void k_bwd_clamp(
    int n, StepConsts c, const float4* __restrict__ gx, const float4* __restrict__ xl,
    const float4* __restrict__ dp, const uint32_t* __restrict__ pc, float4* __restrict__ gxn,
    float4* __restrict__ A,
    uint32_t* __restrict__ qc, uint32_t* __restrict__ qkey, uint32_t* __restrict__ qval,
    uint32_t* __restrict__ cnt, double* __restrict__ r0, const int* __restrict__ escale) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (blockIdx.x * kBlock >= n) return;  // whole workgroup past the end
  const int ii = i < n ? i : n - 1;
  const float4 x = xl[ii];
  const uint32_t q = note_query_cell(i, i < n, x, c, qc, qkey, qval, cnt);
  if (i >= n) return;
  const float4 g = gx[i], u = dp[i];
  const float gv[3] = {g.x, g.y, g.z}, xv[3] = {x.x, x.y, x.z}, uv[3] = {u.x, u.y, u.z};
  const float lo[3] = {c.g.lox, c.g.loy, c.g.loz}, hi[3] = {c.g.hix, c.g.hiy, c.g.hiz};
  float e[3], a[3];
  double rr = 0.0;
  for (int d = 0; d < 3; ++d) {
    const float y = xv[d] + fminf(fmaxf(uv[d], -c.max_dp), c.max_dp);
    e[d] = (y > lo[d] && y < hi[d]) ? gv[d] : 0.0f;
    const float db = (uv[d] > -c.max_dp && uv[d] < c.max_dp) ? e[d] : 0.0f;
    rr += (double)db * (-(double)uv[d] / (double)c.pho0);
    a[d] = db / c.pho0;
  }
  gxn[i] = make_float4(e[0], e[1], e[2], 0.0f);
  A[i] = make_float4(a[0], a[1], a[2], __uint_as_float(pc ? member_word(pc[i], q) : q));
  r0[i] += escale ? ldexp(rr, *escale) : rr;
}

// Query cells of the final positions (for the XSPH pass).
__global__ __launch_bounds__(kBlock) void k_bwd_qcell(int n, StepConsts c,
                                                      const float4* __restrict__ x,
                                                      uint32_t* __restrict__ qc,
                                                      uint32_t* __restrict__ qkey,
                                                      uint32_t* __restrict__ qval,
                                                      uint32_t* __restrict__ cnt) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (blockIdx.x * kBlock >= n) return;
  note_query_cell(i, i < n, x[i < n ? i : n - 1], c, qc, qkey, qval, cnt);
}

// Gather mode, once per frame: packed sorted (stale-grid) cell of each
// sorted slot.
__global__ __launch_bounds__(kBlock) void k_bwd_sorted_cells(int n, StepConsts c,
                                                             const uint32_t* __restrict__ key,
                                                             uint32_t* __restrict__ pc) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  pc[i] = pack_cell(cell_of_key(key[i], c.g));
}

// Gather mode: the query slot and sorted slot of work-item t.  From the radix
// sort (list null): slot t of the sorted query keys skey, whose sorted slot is
// perm[t]; counts the particles per cell into cnt (all zero beforehand).  From
// the counted grid: entry t of list, ranked within its cell; writes perm and
// clears cnt.  All lanes of the wavefront call it; s is in range for every
// lane, u only for valid ones.
struct QuerySlot {
  uint32_t u, s;
  bool valid;
};
__device__ __forceinline__ QuerySlot query_slot(int n, const uint32_t* __restrict__ skey,
                                                uint32_t* perm, const uint2* __restrict__ list,
                                                const uint32_t* __restrict__ cs,
                                                uint32_t* __restrict__ cnt) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  const bool valid = t < n;
  if (list) {
    const uint2 e = list[valid ? t : n - 1];
    const uint32_t lo = cs[e.y], hi = cs[e.y + 1];
    const uint32_t u = lo + rank_in_cell(list, lo, hi, e.x, valid);
    const bool ok = valid && u < (uint32_t)n;  // always, for consistent counts
    if (ok) {
      cnt[e.y] = 0u;
      perm[u] = e.x;
    }
    return QuerySlot{u, e.x < (uint32_t)n ? e.x : 0u, ok};
  }
  count_sorted(skey, t, n, cnt);
  const uint32_t s = valid ? perm[t] : 0u;
  return QuerySlot{(uint32_t)t, s < (uint32_t)n ? s : 0u, valid};
}

// Gather mode: the inputs of an iteration's delta-p pass in query order.
__global__ __launch_bounds__(kBlock) void k_bwd_gather_iter(
    int n, const uint32_t* __restrict__ skey, uint32_t* perm, const uint2* __restrict__ list,
    const uint32_t* __restrict__ cs, const float4* __restrict__ xl, const float4* __restrict__ A,
    float4* __restrict__ xq, float4* __restrict__ aq, uint32_t* __restrict__ mw,
    uint32_t* __restrict__ cnt) {
  if (blockIdx.x * kBlock >= n) return;  // whole workgroup past the end
  const QuerySlot q = query_slot(n, skey, perm, list, cs, cnt);
  if (!q.valid) return;
  const float4 a = A[q.s];
  xq[q.u] = xl[q.s];
  aq[q.u] = a;
  mw[q.u] = __float_as_uint(a.w);
}

// Gather mode: the inputs of the XSPH pass in query order.
__global__ __launch_bounds__(kBlock) void k_bwd_gather_xsph(
    int n, StepConsts c, const uint32_t* __restrict__ skey, uint32_t* perm,
    const uint2* __restrict__ list, const uint32_t* __restrict__ cs,
    const float4* __restrict__ x, const float4* __restrict__ vr, const float4* __restrict__ gv,
    const uint32_t* __restrict__ pc, float4* __restrict__ xq, float4* __restrict__ vrq,
    float4* __restrict__ gvq, uint2* __restrict__ coarse, uint32_t* __restrict__ cnt) {
  if (blockIdx.x * kBlock >= n) return;  // whole workgroup past the end
  const QuerySlot q = query_slot(n, skey, perm, list, cs, cnt);
  if (!q.valid) return;
  const float4 p = x[q.s];
  const Cell qc = cell_of(p.x, p.y, p.z, c.g, c.h);
  xq[q.u] = p;
  if (coarse) coarse[q.u] = screen_coords(p.x, p.y, p.z, c);
  vrq[q.u] = vr[q.s];
  const float4 b = gv[q.s];
  gvq[q.u] = make_float4(b.x, b.y, b.z, __uint_as_float(member_word(pc[q.s], pack_cell(qc))));
}

// DensityBoundary slope (fluids/Simulator.cu:139-161) at wall distance d.
__device__ __forceinline__ float wall_slope(float d, const StepConsts& c) {
  if (d > c.h || d <= 0.0f) return 0.0f;
  return -c.wall_c * (c.h - d) * (c.h + 3.0f * d);
}

// lambda = -(rho/pho0 - 1)/D: from dL/dlambda (gathered, plus in scatter
// mode the scattered extras, which it clears) to dL/drho, dL/dD; writes the
// lambda pass's per-particle inputs (xr, sdb: in the pass's order).  Scatter
// mode folds the delta-p pair terms into gxn.  Gather mode leaves them, with the wall
// terms, in out, for the lambda pass to add where it touches that slot of gx
// anyway, takes the positions in query order (xl) and keeps r0 (whose sum is
// all that counts) by query slot: of the accesses through perm, sd and
// rho remain.  4M particles under the sweeping wall, every array through perm ->
// this: 277 -> 113 us, their frame with gradients 54.7 -> 53.8 ms.
template <bool kGather>
__global__ __launch_bounds__(kBlock) void k_bwd_lambda_pre(
    int n, StepConsts c, int last, const uint32_t* __restrict__ perm, float4* __restrict__ out,
    float4* __restrict__ ex, const float4* __restrict__ xl, const float4* __restrict__ sd,
    const float* __restrict__ rho, const float* __restrict__ grho_x, float4* __restrict__ gxn,
    float4* __restrict__ xr, float4* __restrict__ sdb, double* __restrict__ r0,
    const int* __restrict__ escale) {
  const int u = blockIdx.x * kBlock + threadIdx.x;
  if (u >= n) return;
  const int i = kGather ? (int)perm[u] : u;
  float4 e = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if constexpr (!kGather) e = take_scattered(ex, u, n);
  const float4 o = out[u], x = xl[u], s = sd[i];
  const float gl = o.w + e.w;
  const float D = s.w, rh = rho[i];
  const float C = rh / c.pho0 - 1.0f;
  const float gC = -gl / D;
  const float gD = gl * C / (D * D);
  float gr = gC / c.pho0;
  if (last) gr += grho_x[i];
  const double dr0 = (double)gC * (-(double)rh / ((double)c.pho0 * (double)c.pho0)) +
                     (double)gD * (-2.0 * ((double)D - (double)c.lambda_eps) / (double)c.pho0);
  r0[u] += escale ? ldexp(dr0, *escale) : dr0;
  float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if constexpr (!kGather) g = gxn[u];
  g.x += o.x + e.x;
  g.y += o.y + e.y;
  g.z += o.z + e.z;
  if (c.k_boundary != 0.0f) {
    const float k = gr * c.k_boundary;
    g.x += k * (wall_slope(x.x - c.g.llx, c) - wall_slope(c.g.ulx - x.x, c));
    g.y += k * (wall_slope(x.y - c.g.lly, c) - wall_slope(c.g.uly - x.y, c));
    g.z += k * (wall_slope(x.z - c.g.llz, c) - wall_slope(c.g.ulz - x.z, c));
  }
  (kGather ? out : gxn)[u] = g;
  xr[u] = make_float4(x.x, x.y, x.z, gr);
  sdb[u] = make_float4(s.x, s.y, s.z, gD);
}

// Scatter mode: gx = gxn + scattered extras; clears the extras.
__global__ __launch_bounds__(kBlock) void k_bwd_fold(int n, const float4* __restrict__ gxn,
                                                     float4* __restrict__ ex,
                                                     float4* __restrict__ gx) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const float4 g = gxn[i], e = take_scattered(ex, i, n);
  gx[i] = make_float4(g.x + e.x, g.y + e.y, g.z + e.z, 0.0f);
}

// Per-frame rescaling of the adjoint state (tapes with PBF_TAPE_RESCALE):
// the largest finite |value| of two arrays of layout L (4: each fourth value is
// padding, which counts for nothing), as float bits (all values are
// non-negative, so the unsigned order of the bits is the float order) ...
template <int L>
__global__ __launch_bounds__(kBlock) void k_absmax(const float* __restrict__ a, int na,
                                                   const float* __restrict__ b, int nb,
                                                   uint32_t* __restrict__ out) {
  uint32_t m = 0u;
  const int stride = gridDim.x * kBlock;
  for (int k = blockIdx.x * kBlock + threadIdx.x; k < na + nb; k += stride) {
    if (L == 4 && (k & 3) == 3) continue;
    const float v = fabsf(k < na ? a[k] : b[k - na]);
    const uint32_t bits = __float_as_uint(v);
    m = (v <= 3.4028235e38f && bits > m) ? bits : m;  // NaN and inf are left out
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint32_t o = __shfl_xor(m, off);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63) == 0 && m) atomicMax(out, m);
}

// ... and both arrays multiplied by 2^e (exact) so that the largest becomes
// [1, 2); escale -= e (true values = stored x 2^escale).  Every workgroup
// derives e from the same maximum; workgroup 0 updates escale.
__global__ __launch_bounds__(kBlock) void k_rescale(float* __restrict__ a, int na,
                                                    float* __restrict__ b, int nb,
                                                    const uint32_t* __restrict__ maxbits,
                                                    int* __restrict__ escale) {
  const float mx = __uint_as_float(*maxbits);
  const int e = mx > 0.0f ? -ilogbf(mx) : 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) *escale -= e;
  if (e == 0) return;
  const int stride = gridDim.x * kBlock;
  for (int k = blockIdx.x * kBlock + threadIdx.x; k < na + nb; k += stride) {
    float* p = k < na ? a + k : b + (k - na);
    *p = ldexpf(*p, e);
  }
}

// Prediction x[0] = x + dt (v + dt g) (fluids/Simulator_kernel.cuh:14-15),
// back to the frame's input order through the sort permutation.
template <int L>
__global__ __launch_bounds__(kBlock) void k_bwd_predict(int n, StepConsts c,
                                                        const uint32_t* __restrict__ sval,
                                                        const float4* __restrict__ gx,
                                                        const float4* __restrict__ gx0,
                                                        float* __restrict__ gpos,
                                                        float* __restrict__ gvel) {
  const int s = blockIdx.x * kBlock + threadIdx.x;
  if (s >= n) return;
  const uint32_t src = sval[s] < (uint32_t)n ? sval[s] : 0u;
  const float4 g = gx[s], g0 = gx0[s];
  store_vec<L>(gpos, src, g0.x + g.x, g0.y + g.y, g0.z + g.z);
  store_vec<L>(gvel, src, c.dt * g.x, c.dt * g.y, c.dt * g.z);
}

__global__ void k_fill_u32_one(uint32_t* __restrict__ a) {
  if (threadIdx.x == 0) *a = 0u;
}

__global__ __launch_bounds__(kBlock) void k_fill_f4(float4* __restrict__ a, int n) {
  const int stride = gridDim.x * kBlock;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += stride)
    a[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

__global__ __launch_bounds__(kBlock) void k_fill_f64(double* __restrict__ a, int n) {
  const int stride = gridDim.x * kBlock;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) a[i] = 0.0;
}

// A caller's vector array of layout 3 as float4.
__global__ __launch_bounds__(kBlock) void k_to_f4(const float* __restrict__ a, int n,
                                                  float4* __restrict__ out) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  out[i] = load_vec<3>(a, (uint32_t)i);
}

// Sum of n doubles in a fixed order (independent of the hardware's
// scheduling): kSumParts contiguous segments, each summed by one workgroup
// (strided per work-item, then a fixed tree), then the segment sums by one
// workgroup.  part holds kSumParts doubles.
constexpr int kSumParts = 1024;

__device__ __forceinline__ double block_sum(double v) {
  __shared__ double sh[kBlock];
  sh[threadIdx.x] = v;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  return sh[0];
}

__global__ __launch_bounds__(kBlock) void k_sum_parts(const double* __restrict__ a, int n,
                                                      double* __restrict__ part) {
  const long long seg = ((long long)n + kSumParts - 1) / kSumParts;
  const long long lo = (long long)blockIdx.x * seg;
  const long long hi = lo + seg < n ? lo + seg : n;
  double v = 0.0;
  for (long long i = lo + threadIdx.x; i < hi; i += kBlock) v += a[i];
  const double t = block_sum(v);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

__global__ __launch_bounds__(kBlock) void k_sum_total(const double* __restrict__ part,
                                                      double* __restrict__ out) {
  double v = 0.0;
  for (int i = threadIdx.x; i < kSumParts; i += kBlock) v += part[i];
  const double t = block_sum(v);
  if (threadIdx.x == 0) out[0] = t;
}

int fill_blocks(int n) {
  const int b = (n + kBlock - 1) / kBlock;
  return b < 1 ? 1 : (b > 4096 ? 4096 : b);
}

}  // namespace

void launch_bwd_frame(const BwdFrame& f, int n, const StepConsts& c, hipStream_t st) {
  if (f.q) k_bwd_sorted_cells<<<blocks_for(n), kBlock, 0, st>>>(n, c, f.key, f.q->pc);
}

namespace {
// Gather mode: the query grid of a pass from the keys in q.k0 (with, in q.v0,
// the sorted slots or the arrival numbers, see note_query_cell), before and
// after the kernel that gathers the pass's inputs through query_slot.
struct QueryOrder {
  const uint32_t* skey = nullptr;
  uint32_t* perm = nullptr;
  const uint2* list = nullptr;
};
// One frame forward and backward on a stored tape, radix sort -> counted: 32K
// particles 1101 -> 919 us, 262K 2098 -> 1826, 1M 4971 -> 4662 (fresh lattice) and
// 7470 -> 7300 (collapsing dam); the 4M sweeping-wall frame 64.0 -> 64.3 ms, its
// ten grids' atomics costing more than the sort.
constexpr int kCountedQueryMax = 1 << 20;
bool counted_query(int n) { return n <= kCountedQueryMax; }
QueryOrder order_query(const BwdQuery& q, int n, const StepConsts& c, const HeavyLists& hl,
                       hipStream_t st) {
  QueryOrder o;
  if (counted_query(n)) {
    // the work lists' records are free between neighbour passes
    uint2* list = reinterpret_cast<uint2*>(hl.recs);
    launch_count_place(q.k0, q.v0, list, n, c.cells, q.tile_sum, q.cs, q.cnt, st);
    o.list = list;
    o.perm = q.v1;
    return o;
  }
  const int which =
      radix_sort_pairs(q.k0, q.v0, q.k1, q.v1, n, q.key_bits, q.hist, q.totals, st);
  o.skey = which ? q.k1 : q.k0;
  o.perm = which ? q.v1 : q.v0;
  return o;
}
void finish_query(const BwdQuery& q, int n, const StepConsts& c, hipStream_t st) {
  if (!counted_query(n)) launch_cell_starts(q.cnt, c.cells, q.tile_sum, q.cs, st);
}
}  // namespace

void launch_bwd_xsph(const BwdFrame& f, int n, const StepConsts& c, const uint32_t* cs,
                     const HeavyLists& hl, int pass, const Shapes& sh, hipStream_t st) {
  if (f.q) {
    const BwdQuery& q = *f.q;
    k_bwd_qcell<<<blocks_for(n), kBlock, 0, st>>>(n, c, f.x_final, nullptr, q.k0, q.v0,
                                                  counted_query(n) ? q.cnt : nullptr);
    const QueryOrder o = order_query(q, n, c, hl, st);
    k_bwd_gather_xsph<<<blocks_for(n), kBlock, 0, st>>>(n, c, o.skey, o.perm, o.list, q.cs,
                                                        f.x_final, f.vr, f.gv_out, q.pc, q.xq,
                                                        q.vrq, q.gvq,
                                                        coarse_of(hl, n, sh), q.cnt);
    finish_query(q, n, c, st);
    using P = BwdXsphPass<true>;
    launch_pass<P>(P::Args{q.xq, q.vrq, q.gvq, nullptr, f.out_x, f.out_v, nullptr, nullptr,
                           (uint32_t)n, nullptr},
                   n, c, Scenes{}, q.cs, hl, pass, sh, st);
    k_bwd_velocity<true><<<blocks_for(n), kBlock, 0, st>>>(n, c, o.perm, f.gx_out, f.gv_out,
                                                           f.out_x, f.out_v, nullptr, nullptr,
                                                           f.gx, f.gx0, f.grho_x);
    return;
  }
  k_bwd_qcell<<<blocks_for(n), kBlock, 0, st>>>(n, c, f.x_final, f.qc, nullptr, nullptr, nullptr);
  using P = BwdXsphPass<false>;
  launch_pass<P>(P::Args{f.x_final, f.vr, f.gv_out, f.key, f.out_x, f.out_v, f.ex_x, f.ex_v,
                         (uint32_t)n, f.qc},
                 n, c, Scenes{}, cs, hl, pass, sh, st);
  k_bwd_velocity<false><<<blocks_for(n), kBlock, 0, st>>>(n, c, nullptr, f.gx_out, f.gv_out,
                                                          f.out_x, f.out_v, f.ex_x, f.ex_v,
                                                          f.gx, f.gx0, f.grho_x);
}

void launch_bwd_iteration(const BwdFrame& f, const BwdIter& it, int last, int n,
                          const StepConsts& c, const uint32_t* cs, const HeavyLists& hl, int pass,
                          const Shapes& sh, hipStream_t st) {
  if (f.q) {
    const BwdQuery& q = *f.q;
    k_bwd_clamp<<<blocks_for(n), kBlock, 0, st>>>(n, c, f.gx, it.xl, it.dp, q.pc, f.gxn, f.A,
                                                  nullptr, q.k0, q.v0,
                                                  counted_query(n) ? q.cnt : nullptr, f.r0,
                                                  f.escale);
    const QueryOrder o = order_query(q, n, c, hl, st);
    k_bwd_gather_iter<<<blocks_for(n), kBlock, 0, st>>>(n, o.skey, o.perm, o.list, q.cs, it.xl,
                                                        f.A, q.xq, q.aq, q.mw, q.cnt);
    finish_query(q, n, c, st);
    using PD = BwdDeltaPass<true>;
    launch_pass<PD>(PD::Args{q.xq, q.aq, nullptr, f.out_x, nullptr, (uint32_t)n}, n, c,
                    Scenes{}, q.cs, hl, pass, sh, st);
    k_bwd_lambda_pre<true><<<blocks_for(n), kBlock, 0, st>>>(n, c, last, o.perm, f.out_x,
                                                             nullptr, q.xq, it.sd, it.rho,
                                                             f.grho_x, nullptr, q.xr, q.sdb,
                                                             f.r0, f.escale);
    using PL = BwdLambdaPass<true>;
    launch_pass<PL>(PL::Args{q.xr, q.sdb, nullptr, f.gxn, f.gx, f.out_x, nullptr, (uint32_t)n,
                             q.mw, o.perm},
                    n, c, Scenes{}, q.cs, hl, pass + 1, sh, st);
    return;
  }
  k_bwd_clamp<<<blocks_for(n), kBlock, 0, st>>>(n, c, f.gx, it.xl, it.dp, nullptr, f.gxn, f.A,
                                                f.qc, nullptr, nullptr, nullptr, f.r0, f.escale);
  using PD = BwdDeltaPass<false>;
  launch_pass<PD>(PD::Args{it.xl, f.A, f.key, f.out_x, f.ex_x, (uint32_t)n}, n, c,
                  Scenes{}, cs, hl, pass, sh, st);
  k_bwd_lambda_pre<false><<<blocks_for(n), kBlock, 0, st>>>(n, c, last, nullptr, f.out_x, f.ex_x,
                                                            it.xl, it.sd, it.rho, f.grho_x, f.gxn,
                                                            f.xr, f.sdb, f.r0, f.escale);
  using PL = BwdLambdaPass<false>;
  launch_pass<PL>(PL::Args{f.xr, f.sdb, f.key, f.gxn, f.gxn, nullptr, f.ex_x, (uint32_t)n, f.qc, nullptr},
                  n, c, Scenes{}, cs, hl, pass + 1, sh, st);
  k_bwd_fold<<<blocks_for(n), kBlock, 0, st>>>(n, f.gxn, f.ex_x, f.gx);
}

void launch_bwd_predict(int layout, const BwdFrame& f, const uint32_t* sval, int n,
                        const StepConsts& c, float* gpos, float* gvel, hipStream_t st) {
  if (layout == 3)
    k_bwd_predict<3><<<blocks_for(n), kBlock, 0, st>>>(n, c, sval, f.gx, f.gx0, gpos, gvel);
  else
    k_bwd_predict<4><<<blocks_for(n), kBlock, 0, st>>>(n, c, sval, f.gx, f.gx0, gpos, gvel);
}

void launch_rescale(int layout, float* a, float* b, int n, uint32_t* maxbits, int* escale,
                    hipStream_t st) {
  k_fill_u32_one<<<1, 64, 0, st>>>(maxbits);
  const int m = n * layout;
  const int blocks = fill_blocks(m + m);
  if (layout == 4)
    k_absmax<4><<<blocks, kBlock, 0, st>>>(a, m, b, m, maxbits);
  else
    k_absmax<3><<<blocks, kBlock, 0, st>>>(a, m, b, m, maxbits);
  k_rescale<<<blocks, kBlock, 0, st>>>(a, m, b, m, maxbits, escale);
}

void launch_fill_f4(float4* a, int n, hipStream_t st) {
  k_fill_f4<<<fill_blocks(n), kBlock, 0, st>>>(a, n);
}

void launch_fill_f64(double* a, int n, hipStream_t st) {
  k_fill_f64<<<fill_blocks(n), kBlock, 0, st>>>(a, n);
}

void launch_to_f4(const float* a, int n, float4* out, hipStream_t st) {
  k_to_f4<<<blocks_for(n), kBlock, 0, st>>>(a, n, out);
}

void launch_sum_f64(const double* a, int n, double* part, double* out, hipStream_t st) {
  k_sum_parts<<<kSumParts, kBlock, 0, st>>>(a, n, part);
  k_sum_total<<<1, kBlock, 0, st>>>(part, out);
}

}  // namespace pbf
