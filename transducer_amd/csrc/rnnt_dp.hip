// Lattice recursions of the RNN-T loss for gfx950: alpha, dalpha and the viterbi best path,
// plus the small data-movement kernels that feed them.
//
// One wavefront walks one utterance's (t,u) lattice along anti-diagonals.  Lane L owns C
// consecutive label positions u = L*C .. L*C+C-1 and, at step s, the cells (t = s-u, u).  A
// finished cell pushes two scores forward, with the reference's exact association
// (transducer/transducer_cpu.cpp:45-48, 61-69):
//     stay(t,u) = ((x + E[t,blank]) + P[u,blank]) - LN[t,u]   -> consumed by (t+1,u), same lane
//     emit(t,u) = ((x + E[t,l_u])   + P[u,l_u])   - LN[t,u]   -> consumed by (t,u+1)
// The hand-over to the next label position stays in registers inside a lane and crosses lanes
// with one DPP wave shift; there is no barrier and no memory access on the dependent chain.
// Operands are read from "skewed" planes, indexed by anti-diagonal t+u in groups of four
// (plane_at in rnnt_internal.h), so that four steps are one 16-byte load per lane and the lanes'
// loads are neighbours in memory; they are requested several groups ahead.  This file is compiled with -ffp-contract=off: the rounding
// sequence of every cell must equal the reference's.
//
// The file is compiled in parts side by side (-DRNNT_DP_PART=0..4: everything else, the alpha
// walk in its narrow and its wide forms, the dalpha walk, the best-path walk; all of it without
// the macro): a part holds the launchers that instantiate its kernels.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <type_traits>

#include "rnnt_internal.h"
#include "rnnt_blocks.h"
#include "rnnt_libm.h"
#include "rnnt_split.h"

#ifndef RNNT_DP_PART
#define RNNT_DP_PART -1
#endif
#define RNNT_IN_PART(n) (RNNT_DP_PART < 0 || RNNT_DP_PART == (n))

namespace rnnt {

namespace {

constexpr float kNegInf = -__builtin_huge_valf();
// Label-move score handed on by a cell outside the lattice in the alpha walk: far below any
// alpha, so a log-sum-exp returns the other operand untouched -- as -inf would -- but FINITE.
// The blank-move score of such a cell is -inf; an idle lane therefore forms
// lse(kOutside, -inf) = kOutside on the fast path, never inf - inf (which only the library path
// can sort out, and an idle lane would then send its whole wavefront there at every step).
// A cell INSIDE the lattice never sees this value: its left neighbour is inside too, and the
// first column is handed -inf (below), so -inf scores of the caller propagate exactly as in
// the reference (transducer/transducer_cpu.cpp:16-24,43-60).
constexpr float kOutside = -1.0e30f;
constexpr float kPosInf = __builtin_huge_valf();

// lane L receives the value of lane L-1; lane 0 receives `fill`.
__device__ inline float wave_shr1(float x, float fill) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(fill), __float_as_int(x),
                                                    0x138 /* wave_shr:1 */, 0xf, 0xf, false));
}
// lane L receives the value of lane L+1; lane 63 receives `fill`.
__device__ inline float wave_shl1(float x, float fill) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(fill), __float_as_int(x),
                                                    0x130 /* wave_shl:1 */, 0xf, 0xf, false));
}

// exp(x) for x <= 0 straight on the hardware transcendental unit
// (v_exp_f32 and v_log_f32 work in base 2 and are good to about one ulp).  In the one place they
// are used -- log1p(exp(-|a-b|)) below -- the rounding of x*log2(e) costs at most 2.4e-8
// absolute in the result (it is largest where exp(x) is small), i.e. less than half an ulp of
// the value log 2 that the result never exceeds.
__device__ inline float exp_neg(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }

// log1p(y) for y in [0,1]:  log(1+y) with the rounding error of the sum 1+y folded back in, divided
// by 1 + y to three digits (1 - y/2: the lost part is at most 2^-24, so a seventh of it is below a
// tenth of the result's last bit, and two instructions stand in for a reciprocal's four-cycle
// quarter-rate slot).  Within about one ulp of the correctly rounded value over the whole range.
__device__ inline float log1p_unit(float y) {
  const float w = 1.0f + y;
  const float lost = y - (w - 1.0f);
  return __builtin_fmaf(__builtin_amdgcn_logf(w), 0.693147180559945309f,
                        lost * __builtin_fmaf(y, -0.5f, 1.0f));
}

// log1p(exp(d)) for d <= 0 on the hardware transcendental units: within a few ulp of the C
// library's value at a seventh of its instructions.
__device__ inline float softplus_fast(float d) { return log1p_unit(exp_neg(d)); }

// Bound on |softplus_fast(d) - log1pf(expf(d))| (the library's floats) as a function of the fast
// value lf: lf * (kFastRelA + kFastRelB * |d|) + 2^-125.  The first term covers the rounding of both
// evaluations (a few ulp of lf), the second the rounding of d * log2(e) ahead of v_exp_f32,
// whose effect on the result grows with |d|.  The bound is not taken from data sheets: the
// fast value is compared with the exact one for EVERY float d <= 0 (rnnt_hip_lse_bound_check,
// run by the tests on the device itself).  Measured on gfx950, the largest distance as a share of
// the bound: 0.84 for |d| <= 1.5, 0.87 up to 4, 0.90 from there to 87, 0.50 beyond; the tests let it be
// 0.95.  The constants are what decides how often a wavefront of the alpha walk takes the library
// path (its chance per lane is twice the bound / the sum's spacing), so they are not rounder than
// that: with 5 and 1.25 the walk of B=32 T=2000 U=100 takes 255 us instead of 226.
constexpr float kFastRelA = 2.1f * 0x1p-23f;
constexpr float kFastRelB = 0.65f * 0x1p-23f;
// The bound for fast value lf at argument d.  The clamp to 1 (free: an output modifier of the
// multiply-add) keeps 0 * inf out of it at d = -inf; the added 2^-125 covers d below -87.3, where the
// library's value is a subnormal number and the hardware units return 0.
__device__ inline float fast_bound(float lf, float d) {
  const float rel = __builtin_fmaf(fabsf(d), kFastRelB, kFastRelA);
  return __builtin_fmaf(lf, fminf(rel, 1.0f), 0x1p-125f);
}

// transducer/transducer_cpu.cpp:16-24 with the C library's own expf and log1pf (rnnt_libm.h):
// the same bits as the reference's CPU backend for every pair of operands.
__device__ __forceinline__ float lse2_libm(float a, float b, const unsigned long long* tab) {
  // One operand -inf: |a - b| = inf, expf gives 0, log1pf(0) = 0 and the sum is the other
  // operand exactly, as the reference's early returns have it; only both -inf needs a guard.
  const float hi = a > b ? a : b;
  const float r = hi + log1pf_glibc(expf_glibc_nonpositive(-fabsf(a - b), tab));
  return (hi == kNegInf) ? kNegInf : r;
}

// The same bits, mostly without the library's ~100 instructions.  What the recursion keeps is
// r = fl(hi + l) with l = log1pf(expf(d)) at most log 2, and from a few hundred steps into a
// lattice |hi| is in the thousands: the sum's spacing is then thousands of times the
// uncertainty of a fast l, so nearly every fast sum is provably the library's sum.  The library's l
// lies in [lf - e, lf + e], e the bound above, and rounding is monotone: where fl(hi + lo) and
// fl(hi + up) are the same float, lo = fl(lf - e) and up = fl(lf + e), that float is the library's
// sum as well.  (l is a float, so lf - e <= l gives fl(lf - e) <= l: the rounding of the two ends
// costs nothing.)  No exponents are looked at, and the sum itself falls out of the proof: eight
// instructions, where forming the sum, its exact remainder and half the spacing of floats below
// it took twelve.  NaN operands and two operands of -inf (inf - inf) fail by themselves.  When a lane
// fails, its wavefront takes the library path (Ziv's strategy); either way the result is the
// library's, bit for bit.
struct FastLse {
  float lo, up;  // fl(hi + l) is the library's sum where the two are the same
};
// max without the two instructions that quiet its operands first (a NaN fails the proof anyway)
__device__ inline float max_raw(float a, float b) {
  float r;
  asm("v_max_f32_e32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline FastLse lse2_fast(float a, float b) {
  const float hi = max_raw(a, b);
  const float d = -fabsf(a - b);
  const float lf = softplus_fast(d);
  const float e = fast_bound(lf, d);
  FastLse r;
  r.lo = hi + (lf - e);
  r.up = hi + (lf + e);
  return r;
}

// Raises the device's trouble flag.  A store to GLOBAL memory by its address space: through a
// generic pointer it would be a flat instruction, which may go to LDS as well, and with one of
// those possibly in flight the compiler waits for every load in flight at the next use of any
// loaded value -- on the walk's fast path too, where the branch that raises the flag is never
// taken.
__device__ inline void raise_trouble(int* trouble) {
  typedef __attribute__((address_space(1))) int global_int;
  __hip_atomic_store((global_int*)trouble, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The wait of an upper wavefront for the progress counter of the one below it (LDS, same
// workgroup).  The lower wavefront never waits for an upper one, so the counter always gets
// there; the trip bound only turns a logic slip of a future edit into an error report instead
// of a hung device: when it runs out the wavefront raises the device's trouble flag, stops
// waiting for good (returns a count no later `need` exceeds) and finishes its walk on whatever
// the hand-over array holds.  The host reads the flag with rnnt_hip_check_kernels().
__device__ inline int bounded_wait(const int* counter, int have, int need, int spin_limit,
                                   int* __restrict__ trouble) {
  int spins = 0;
  while (have < need) {
    have = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    asm volatile("" ::: "memory");
    if (have < need) {
      if (spins++ >= spin_limit) {
        if ((threadIdx.x & 63) == 0) raise_trouble(trouble);
        return 0x7fffffff;
      }
      __builtin_amdgcn_s_sleep(1);
    }
  }
  return have;
}

__device__ inline float f4get(const float4& v, int j) {
  return j == 0 ? v.x : (j == 1 ? v.y : (j == 2 ? v.z : v.w));
}
__device__ inline void f4set(float4& v, int j, float x) {
  if (j == 0) v.x = x; else if (j == 1) v.y = x; else if (j == 2) v.z = x; else v.w = x;
}

// ------------------------------------------------------------------ skew / unskew
// row-major [B,T,U] <-> skewed planes.  A block takes 64 label positions x 64 anti-diagonals
// (16 groups of four: 1 KB of contiguous plane memory each) and their 127 frames t = dd - u, and
// transposes through LDS so that the plane side moves 16-byte pieces next to each other and the
// row-major side rows of consecutive label positions.  Only cells inside the utterance's
// (T_b, U_b) extent are touched.  Grid: (anti-diagonal blocks, label blocks, B).
__global__ __launch_bounds__(256) void skew_kernel(const float* __restrict__ src,
                                                   float* __restrict__ dstS,
                                                   const int* __restrict__ inLen,
                                                   const int* __restrict__ labLen, Dims d) {
  __shared__ float tile[64][65];  // [label position][anti-diagonal]
  const int b = blockIdx.z, dd0 = blockIdx.x * 64, u0 = blockIdx.y * 64;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  const int t_first = dd0 - u0 - 63;  // frames t_first .. t_first + 126 meet the tile
  if (u0 >= Ub || t_first >= Tb || t_first + 126 < 0) return;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const float* s = src + (size_t)b * d.T * d.U;
  // (all of a thread's 32 values are requested before the first goes to LDS: taken one by one,
  // each waited a memory round trip -- 0.45 ms for the 128 MB of B=8 T=10000 U=401)
  float v[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const int r = ty + 4 * i, t = t_first + r, u = u0 + tx, c = tx + r - 63;
    const bool wanted = c >= 0 && c < 64 && t >= 0 && t < Tb && u < Ub;
    v[i] = wanted ? s[(size_t)t * d.U + u] : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const int c = tx + ty + 4 * i - 63;
    if (c >= 0 && c < 64) tile[tx][c] = v[i];
  }
  __syncthreads();
  const size_t plane_b = (size_t)b * d.Ua * d.Dp;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int f = k * 256 + threadIdx.x, gl = f >> 6, ul = f & 63;
    const int u = u0 + ul, g = (dd0 >> 2) + gl, tq = 4 * g - u;  // frame of the group's first cell
    if (u >= Ub || tq + 3 < 0 || tq >= Tb) continue;
    float* dst = dstS + plane_b + ((size_t)g * d.Ua + u) * 4;
    if (tq >= 0 && tq + 3 < Tb) {
      *reinterpret_cast<float4*>(dst) = make_float4(tile[ul][4 * gl], tile[ul][4 * gl + 1],
                                                    tile[ul][4 * gl + 2], tile[ul][4 * gl + 3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (tq + j >= 0 && tq + j < Tb) dst[j] = tile[ul][4 * gl + j];
    }
  }
}

__global__ __launch_bounds__(256) void unskew_kernel(const float* __restrict__ srcS,
                                                     float* __restrict__ dst,
                                                     const int* __restrict__ inLen,
                                                     const int* __restrict__ labLen, Dims d) {
  __shared__ float tile[64][65];  // [label position][anti-diagonal]
  const int b = blockIdx.z, dd0 = blockIdx.x * 64, u0 = blockIdx.y * 64;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  const int t_first = dd0 - u0 - 63;
  if (u0 >= Ub || t_first >= Tb || t_first + 126 < 0) return;
  const size_t plane_b = (size_t)b * d.Ua * d.Dp;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int f = k * 256 + threadIdx.x, gl = f >> 6, ul = f & 63;
    const int u = u0 + ul, g = (dd0 >> 2) + gl, tq = 4 * g - u;
    float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    // (a group that holds a cell of the lattice lies inside the plane: 4g < T + U)
    if (u < Ub && tq + 3 >= 0 && tq < Tb)
      v = *reinterpret_cast<const float4*>(srcS + plane_b + ((size_t)g * d.Ua + u) * 4);
    tile[ul][4 * gl] = v.x;
    tile[ul][4 * gl + 1] = v.y;
    tile[ul][4 * gl + 2] = v.z;
    tile[ul][4 * gl + 3] = v.w;
  }
  __syncthreads();
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  float* o = dst + (size_t)b * d.T * d.U;
  for (int i = 0; i < 32; ++i) {
    const int r = ty + 4 * i, t = t_first + r, u = u0 + tx, c = tx + r - 63;
    if (c >= 0 && c < 64 && t >= 0 && t < Tb && u < Ub) o[(size_t)t * d.U + u] = tile[tx][c];
  }
}

// ------------------------------------------------------------------ gather
// elS(u, t+u) = E[t, label_u]; eb[t] = E[t, blank]; pb[u] = P[u, blank]; pl[u] = P[u, label_u].
// Tiles of 64 label positions x 64 anti-diagonals like skew_kernel (same grid), the source being
// E[t, label_u] instead of a row-major [T, U] array: a wavefront reads one frame's scores of 64
// labels (scattered over the frame's row either way), and the plane side is written as 16-byte
// pieces next to each other.  (One block per label position and 256 frames, every thread writing
// its own 4-byte cell: 0.38 ms against 0.13 at B=8 T=10000 U=401 V=32.)  The blocks of the first
// label tile also leave eb for their 64 anti-diagonals' frames, those of the first anti-diagonal
// block pb and pl for their 64 positions.
template <typename TIO>
__global__ __launch_bounds__(256) void gather_kernel(const TIO* __restrict__ E,
                                                     const TIO* __restrict__ P,
                                                     const int* __restrict__ labels,
                                                     const int* __restrict__ inLen,
                                                     const int* __restrict__ labLen, Planes p,
                                                     Dims d) {
  __shared__ float tile[64][65];  // [label position][anti-diagonal]
  const int b = blockIdx.z, dd0 = blockIdx.x * 64, u0 = blockIdx.y * 64;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (u0 >= Ub) return;
  const TIO* Eb = E + (size_t)b * d.T * d.V;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  if (blockIdx.y == 0 && threadIdx.x < 64) {  // frames dd0 .. dd0 + 63 (dd0 runs past T)
    const int t = dd0 + threadIdx.x;
    if (t < Tb) p.eb[(size_t)b * d.Tp + d.Eo + t] = ldf(Eb + (size_t)t * d.V + d.blank);
  }
  const int u_mine = u0 + tx;
  const bool has_label = labels != nullptr && u_mine + 1 < Ub;
  const int l = has_label ? label_at(labels, d, b, u_mine) : d.blank;
  if (blockIdx.x == 0 && ty == 0 && u_mine < Ub) {
    const TIO* Pu = P + ((size_t)b * d.U + u_mine) * d.V;
    p.pb[(size_t)b * d.Ua + u_mine] = ldf(Pu + d.blank);
    p.pl[(size_t)b * d.Ua + u_mine] = has_label ? ldf(Pu + l) : 0.0f;
  }
  const int t_first = dd0 - u0 - 63;  // frames t_first .. t_first + 126 meet the tile
  if (labels == nullptr || t_first >= Tb || t_first + 126 < 0) return;
  float v[32];
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const int r = ty + 4 * i, t = t_first + r, c = tx + r - 63;
    const bool wanted = c >= 0 && c < 64 && t >= 0 && t < Tb && has_label;
    v[i] = wanted ? ldf(Eb + (size_t)t * d.V + l) : 0.0f;
  }
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const int c = tx + ty + 4 * i - 63;
    if (c >= 0 && c < 64) tile[tx][c] = v[i];
  }
  __syncthreads();
  const size_t plane_b = (size_t)b * d.Ua * d.Dp;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int f = k * 256 + threadIdx.x, gl = f >> 6, ul = f & 63;
    const int u = u0 + ul, g = (dd0 >> 2) + gl, tq = 4 * g - u;  // frame of the group's first cell
    if (u + 1 >= Ub || tq + 3 < 0 || tq >= Tb) continue;         // (the last position has no label)
    float* dst = p.elS + plane_b + ((size_t)g * d.Ua + u) * 4;
    if (tq >= 0 && tq + 3 < Tb) {
      *reinterpret_cast<float4*>(dst) = make_float4(tile[ul][4 * gl], tile[ul][4 * gl + 1],
                                                    tile[ul][4 * gl + 2], tile[ul][4 * gl + 3]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (tq + j >= 0 && tq + j < Tb) dst[j] = tile[ul][4 * gl + j];
    }
  }
}

// The same per cell: grid (ceil(T/256), U, B), a block serves 256 frames of one label position
// and every thread writes its own cell.  For large vocabularies, where a frame's scores of 64
// labels are 64 cache lines whichever way they are read and this form keeps more requests in
// flight (B=32 T=2000 U=101 V=10000: 0.17 ms a launch against 0.185 by tiles).
template <typename TIO>
__global__ __launch_bounds__(256) void gather_cells_kernel(const TIO* __restrict__ E,
                                                           const TIO* __restrict__ P,
                                                           const int* __restrict__ labels,
                                                           const int* __restrict__ inLen,
                                                           const int* __restrict__ labLen,
                                                           Planes p, Dims d) {
  const int b = blockIdx.z, u = blockIdx.y;
  const int t = blockIdx.x * 256 + threadIdx.x;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (u >= Ub) return;
  const bool has_label = labels != nullptr && (u + 1 < Ub);
  const int l = has_label ? label_at(labels, d, b, u) : d.blank;
  const TIO* Eb = E + (size_t)b * d.T * d.V;
  if (t < Tb) {
    if (has_label) p.elS[plane_at(d, b, u, t + u)] = ldf(Eb + (size_t)t * d.V + l);
    if (u == 0) p.eb[(size_t)b * d.Tp + d.Eo + t] = ldf(Eb + (size_t)t * d.V + d.blank);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const TIO* Pu = P + ((size_t)b * d.U + u) * d.V;
    p.pb[(size_t)b * d.Ua + u] = ldf(Pu + d.blank);
    p.pl[(size_t)b * d.Ua + u] = has_label ? ldf(Pu + l) : 0.0f;
  }
}

// ------------------------------------------------------------------ alpha
// transducer/transducer_cpu.cpp:30-79 (one utterance per wavefront).
// A cell that has not started yet (t < 0) hands on "nothing" -- -inf upwards (blank move),
// kOutside to the right (label move) -- which makes the log-sum-exp of a first-row or
// first-column cell return its one real operand untouched: exactly the reference's special
// cases (:49-60), also when that operand is -inf (both operands are then -inf and the library
// path returns -inf).  Cells past the utterance (t >= T_b, u >= U_b) hand on the same and are
// never read by a valid cell.
// This kernel takes several label positions a lane: label axes past 256 positions that
// alpha_walk_kernel (one a lane, below) does not take side by side.
// W > 1: the label positions are dealt to W wavefronts of one workgroup (wavefront w owns
// positions [64 C w, 64 C (w+1))), because the walk is bound by how fast ONE wavefront issues
// the instructions of its cells.  The only value that crosses
// a wavefront boundary is the label-move score of the boundary cell, one float per step: the
// lower wavefront leaves it in an LDS array indexed by step and then publishes how far it has
// got; the upper one runs a few groups behind, so it finds its inputs there without waiting and
// re-reads the progress counter only once every few groups.  The lowest
// wavefront waits for nobody and every wavefront runs all groups, so the waits are bounded.
// A label axis longer than one workgroup's 64 C W positions is walked block by block, one launch
// per block of 64 C W positions (u_base = its first one), lowest block first.  The only values
// that cross a block boundary are the label-move scores of the block's last column, one per
// step: a launch leaves them in `ghout` ([B][hand_stride], entry s = score entering step s;
// null for the last block) and the next one reads them from `ghin` (null for the first block).
// kMulti: this launch is one of several blocks (the hand-over code is compiled in only then: in
// the single-block kernel even an unused hand-over load costs the walk its prefetch distance).
template <int C, int W, bool kMulti>
__global__ __launch_bounds__(64 * W) void alpha_kernel(Planes p, const int* __restrict__ inLen,
                                                       const int* __restrict__ labLen,
                                                       float* __restrict__ costs, Dims d,
                                                       int hand_stride, int spin_limit,
                                                       int* __restrict__ trouble, int u_base,
                                                       const float* __restrict__ ghin,
                                                       float* __restrict__ ghout) {
  extern __shared__ __attribute__((aligned(16))) float hand[];  // [W-1][hand_stride]: entry s =
                                                                // score handed to step s
  __shared__ int done[W];          // steps a wavefront has published
  __shared__ __attribute__((aligned(16))) float nothing[4];
  __shared__ unsigned long long etab[32];  // expf's table (rnnt_libm.h)
  const int b = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Tb == 0 || Ub == 0) {  // :39-41
    if (threadIdx.x == 0 && u_base == 0) costs[b] = kPosInf;
    return;
  }
  if (u_base >= Ub) return;  // a block past this utterance's labels: nobody reads what it would leave
  const int nsteps = Tb + Ub - 1;
  const int ngroups = (nsteps + 3) >> 2;
  const int u0 = u_base + (wave * 64 + lane) * C;
  const int gstride = plane_group_stride(d);
  const bool first_column = u_base == 0 && wave == 0;  // lane 0 owns the lattice's column u = 0
  const float* gin = (kMulti && ghin) ? ghin + (size_t)b * hand_stride : nullptr;
  float* gout = (kMulti && ghout) ? ghout + (size_t)b * hand_stride : nullptr;
  if (kMulti && gout && threadIdx.x == 0) gout[0] = kOutside;  // nothing enters step 0
  exp2_table_to_lds(etab);
  if (W > 1) {
    if (threadIdx.x < W) done[threadIdx.x] = 0;
    if (threadIdx.x < W - 1) hand[threadIdx.x * hand_stride] = kOutside;  // nothing enters step 0
    if (threadIdx.x < 4) nothing[threadIdx.x] = kNegInf;
  }
  __syncthreads();
  // a wavefront past this utterance's labels: nobody reads what it would hand on
  const int u_lo = u_base + wave * 64 * C;
  if (W > 1 && u_lo >= Ub) return;
  float* hand_out = hand + wave * hand_stride;                     // wave < W-1
  // wave > 0; wavefront 0 finds there that nothing comes in (-inf: see run_group)
  const float* hand_in = wave > 0 ? hand + (wave - 1) * hand_stride : nothing;
  // E[t,blank] for the cells of step s sits at ebp[s - u]; column c at step s = 4g+j reads
  // ebl[4g + j - c], so one run of C+3 values serves all columns of a group
  const float* ebl = p.eb + (size_t)b * d.Tp + d.Eo - min(u0, Ub - 1);

  float stay[C], emit[C], pbv[C], plv[C];
  unsigned tlim[C];  // frames of this column: T_b, or 0 for a label position past the utterance
  const float* lnp[C];
  const float* elp[C];
  float* ap[C];
  // Operands of a position past the utterance's last one are the last one's (its label score the
  // last label's), and its moves carry kOutside on top: whatever it meets is an ordinary number
  // far below any alpha, so that the interior groups below need no test for it.
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const bool real = u0 + c < Ub;
    tlim[c] = real ? (unsigned)Tb : 0u;
    lnp[c] = p.lnS + plane_group0(d, b, min(u0 + c, Ub - 1));
    elp[c] = p.elS + plane_group0(d, b, max(min(u0 + c, Ub - 2), 0));
    ap[c] = p.aS + plane_group0(d, b, u0 + c);  // u0 + c < Ua always
    pbv[c] = real ? p.pb[(size_t)b * d.Ua + u0 + c] : kOutside;
    plv[c] = real ? p.pl[(size_t)b * d.Ua + u0 + c] : kOutside;
    // :43 alpha[0,0] = 0: cell (0,0) finds 0 coming up from below and nothing from the left
    stay[c] = (u0 + c == 0) ? 0.0f : kNegInf;
    emit[c] = kOutside;
  }

  const int nwhole = nsteps >> 2;  // groups with all four steps
  // Interior groups [in_lo, in_hi): step 4g is past the first frame of the wavefront's last
  // position (rounded up to whole lanes), step 4g + 3 not past the last frame of its first one.
  // Their operands are addressed by 32-bit offsets from the utterance's own (uniform) plane
  // origins: one addition per load where 64-bit pointers took five instructions.
  const int top = min(u_lo + 64 * C, ((Ub + C - 1) / C) * C) - 1;
  const bool small_plane = 4ull * (unsigned long long)d.Ua * (unsigned)d.Dp < (1ull << 32);
  const int in_lo = (top + 3) >> 2;
  const int in_hi = (small_plane && Ub > 1) ? min((Tb + u_lo) >> 2, nwhole) : 0;
  const char* ln_b = reinterpret_cast<const char*>(p.lnS + plane_group0(d, b, 0));
  const char* el_b = reinterpret_cast<const char*>(p.elS + plane_group0(d, b, 0));
  char* a_b = reinterpret_cast<char*>(p.aS + plane_group0(d, b, 0));
  const char* eb_b = reinterpret_cast<const char*>(p.eb + (size_t)b * d.Tp);
  unsigned ln_o[C], el_o[C], a_o[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    ln_o[c] = 16u * (unsigned)min(u0 + c, Ub - 1);
    el_o[c] = 16u * (unsigned)max(min(u0 + c, Ub - 2), 0);
    a_o[c] = 16u * (unsigned)(u0 + c);
  }
  const unsigned eb_o = 4u * (unsigned)(d.Eo - min(u0, Ub - 1) - (C - 1));

  struct Group {
    float4 ln[C], el[C];
    float eb[C + 3];
    float4 gh;  // scores entering the block's first column from the block below
  };
  auto load_group = [&](int g) -> Group {
    Group r;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      r.ln[c] = *reinterpret_cast<const float4*>(lnp[c] + (size_t)g * gstride);
      r.el[c] = *reinterpret_cast<const float4*>(elp[c] + (size_t)g * gstride);
    }
#pragma unroll
    for (int k = 0; k < C + 3; ++k) r.eb[k] = ebl[4 * g + k - (C - 1)];
    if constexpr (kMulti) {
      r.gh = make_float4(kOutside, kOutside, kOutside, kOutside);
      if (gin) r.gh = *reinterpret_cast<const float4*>(gin + 4 * g);  // uniform
    }
    return r;
  };

  int avail = 0;  // steps the wavefront below is known to have published
  auto wait_for = [&](int need) {
    // LDS serves a wavefront's requests in order, so no hardware fence is needed on either
    // side (a release/acquire pair would also wait for the global prefetches in flight);
    // the empty asm statements only keep the compiler from moving LDS accesses across
    avail = bounded_wait(&done[wave - 1], avail, need, spin_limit, trouble);
  };
  // What enters a wavefront above the first during a group is asked for one group ahead (its
  // latency would otherwise stand at the head of every group), into two register sets in turn.
  // The first wavefront's interior groups ask as well, always for the same four entries that say
  // that nothing comes in, and never wait: no branch on the wavefront's place in the hot loop.
  if (wave == 0) avail = 0x7fffffff;
  auto fetch_hand = [&](int g, float4& h) {
    if (W == 1 || g >= ngroups) return;
    const int need = 4 * g + 3;  // the scores entering steps 4g .. 4g+3 left steps 4g-1 .. 4g+2
    if (__builtin_expect(avail < need, 0)) wait_for(need);
    h = *reinterpret_cast<const float4*>(hand_in + (wave > 0 ? 4 * g : 0));
  };
  // kWhole: all four steps of the group exist (every group but the last; no test per step)
  // kInterior: all four steps of every position of this wavefront (those past the utterance's
  // last one aside, see above) are inside the lattice, and no bounds are looked at; that is all
  // but the first and last 64 C steps or so.
  auto run_group = [&](int g, const Group& cur, const float4& hand_cur, float4& hand_next,
                       auto whole, auto interior) {
    constexpr bool kWhole = decltype(whole)::value;
    constexpr bool kInterior = decltype(interior)::value;
    float4 aout[C];
    // what enters the wavefront's first column from the left: for the lattice's own first
    // column (u = 0) nothing, which is -inf while its cells are inside the lattice (:49-52 adds
    // nothing there, so a -inf blank score must come out as -inf) and kOutside once they are
    // past the last frame (the idle lane's pair is then (kOutside, -inf) again)
    float4 hin;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      f4set(hin, j, (first_column && (kInterior || 4 * g + j < Tb)) ? kNegInf : kOutside);
    if constexpr (kMulti) {
      if (gin) hin = cur.gh;  // wavefront 0: from the block below
    }
    if constexpr (W > 1) {
      if (kInterior && !kMulti) hin = hand_cur;
      else if (wave > 0) hin = hand_cur;
      fetch_hand(g + 1, hand_next);
    }
    float gsend[4];  // what this lane's last column hands to the right after each step
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = 4 * g + j;
      gsend[j] = kOutside;
      if (kWhole || s < nsteps) {  // uniform; a step past the last must not touch the scores
        const float from_left = wave_shr1(emit[C - 1], f4get(hin, j));  // lane 0: hin
#pragma unroll
        for (int c = C - 1; c >= 0; --c) {
          const float left = (c == 0) ? from_left : emit[c - 1];
          const float ln = f4get(cur.ln[c], j);
          float a, sb, se;
          auto moves = [&](float x) {
            a = x;
            sb = a + cur.eb[j - c + (C - 1)];
            sb = sb + pbv[c];
            sb = sb - ln;
            se = a + f4get(cur.el[c], j);
            se = se + plv[c];
            se = se - ln;
          };
          // the moves go on from the fast sum while its proof is still on its way
          const FastLse fast = lse2_fast(left, stay[c]);
          moves(fast.lo);
          asm volatile("" : "+v"(sb), "+v"(se));
          if (__builtin_expect(
                  __builtin_amdgcn_ballot_w64(!(fast.lo == fast.up)) != 0ull, 0))
            moves(lse2_libm(left, stay[c], etab));
          // a cell of the lattice: 0 <= t = s - u < T_b (one unsigned comparison).  Cells before
          // the first frame or past the last one hand kOutside on, so whatever the planes hold
          // outside the utterance never enters a log-sum-exp (where it would cost the whole
          // wavefront the library path).
          const bool inside = kInterior || (unsigned)(s - (u0 + c)) < tlim[c];
          stay[c] = inside ? sb : kNegInf;
          emit[c] = inside ? se : kOutside;
          f4set(aout[c], j, a);
        }
        gsend[j] = emit[C - 1];
      }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if constexpr (kInterior)
        *reinterpret_cast<float4*>(a_b + (size_t)(a_o[c] + (unsigned)g * (4u * (unsigned)gstride))) = aout[c];
      else
        *reinterpret_cast<float4*>(ap[c] + (size_t)g * gstride) = aout[c];
    }
    if constexpr (kMulti) {
      if (gout && wave == W - 1 && lane == 63) {  // entries 4g+1 .. 4g+4 for the block above
#pragma unroll
        for (int j = 0; j < 4; ++j) gout[4 * g + 1 + j] = gsend[j];
      }
    }
    if (W > 1 && wave < W - 1 && lane == 63) {  // entries 4g+1 .. 4g+4, then the progress
#pragma unroll
      for (int j = 0; j < 4; ++j) hand_out[4 * g + 1 + j] = gsend[j];
      asm volatile("" ::: "memory");
      __hip_atomic_store(&done[wave], 4 * g + 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };
  // four register sets rotate (no copies): a group's loads are requested four groups (16
  // steps, more than a microsecond) ahead -- the planes of a long batch do not fit L2
  auto clamp_g = [&](int g) { return g < ngroups ? g : ngroups - 1; };
  Group q0 = load_group(0), q1 = load_group(clamp_g(1)), q2 = load_group(clamp_g(2)),
        q3 = load_group(clamp_g(3));
  if (W > 1 && wave > 0) wait_for(min(4 * ngroups, 4 * 8 * wave));  // fall a few groups behind
  const std::true_type whole, interior;
  const std::false_type partial, edge;
  auto load_inner = [&](int g) -> Group {
    Group r;
    const unsigned by = (unsigned)g * (4u * (unsigned)gstride);  // bytes
#pragma unroll
    for (int c = 0; c < C; ++c) {
      r.ln[c] = *reinterpret_cast<const float4*>(ln_b + (size_t)(ln_o[c] + by));
      r.el[c] = *reinterpret_cast<const float4*>(el_b + (size_t)(el_o[c] + by));
    }
    const unsigned eo = eb_o + 16u * (unsigned)g;
#pragma unroll
    for (int k = 0; k < C + 3; ++k)
      r.eb[k] = reinterpret_cast<const float*>(eb_b + (size_t)eo)[k];
    if constexpr (kMulti) {
      r.gh = make_float4(kOutside, kOutside, kOutside, kOutside);
      if (gin) r.gh = *reinterpret_cast<const float4*>(gin + 4 * g);  // uniform
    }
    return r;
  };
  float4 h0 = make_float4(kOutside, kOutside, kOutside, kOutside), h1 = h0;
  fetch_hand(0, h0);
  int g = 0;
  for (; g + 4 <= nwhole; g += 4) {
    // (with eight or sixteen positions a lane the registers are what is short)
    if constexpr (C <= 4) {
      for (; g >= in_lo && g + 4 <= in_hi && g + 8 <= ngroups; g += 4) {
        run_group(g, q0, h0, h1, whole, interior);
        q0 = load_inner(g + 4);
        run_group(g + 1, q1, h1, h0, whole, interior);
        q1 = load_inner(g + 5);
        run_group(g + 2, q2, h0, h1, whole, interior);
        q2 = load_inner(g + 6);
        run_group(g + 3, q3, h1, h0, whole, interior);
        q3 = load_inner(g + 7);
      }
      if (g + 4 > nwhole) break;
    }
    run_group(g, q0, h0, h1, whole, edge);
    q0 = load_group(clamp_g(g + 4));
    run_group(g + 1, q1, h1, h0, whole, edge);
    q1 = load_group(clamp_g(g + 5));
    run_group(g + 2, q2, h0, h1, whole, edge);
    q2 = load_group(clamp_g(g + 6));
    run_group(g + 3, q3, h1, h0, whole, edge);
    q3 = load_group(clamp_g(g + 7));
  }
  // the last one to four groups, the very last of which may be partial
  if (g < ngroups) run_group(g, q0, h0, h1, partial, edge);
  if (g + 1 < ngroups) run_group(g + 1, q1, h1, h0, partial, edge);
  if (g + 2 < ngroups) run_group(g + 2, q2, h0, h1, partial, edge);
  if (g + 3 < ngroups) run_group(g + 3, q3, h1, h0, partial, edge);
  // :73-78 the blank move out of the last cell, negated; that cell was the last one its
  // column processed
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (u0 + c == Ub - 1) costs[b] = -stay[c];
}

// ------------------------------------------------------------------ hand-over between wavefronts
// A lattice walk deals 64 neighbouring label positions to a wavefront, one a lane.  The one value
// a step that crosses from a wavefront to the next goes through a ring in LDS, four steps (a
// "quad") at a time: entry g of boundary w is what wavefront w takes in for group g.  prog[w + 1]
// counts the groups wavefront w has handed on; prog[w] is what it may take, and prog[w + 2] says
// how far the taker of its own quads has got, so a quad is overwritten only once it has been read.
// Wavefronts that have no neighbour on a side find kForever there.
// Every lane writes the quad, lane `from` into the ring and the others into a dump that nobody
// reads: a branch around the write would cost the walk 5.4 ns, whether taken or not, and switching
// lanes off and on again as much.  A group's quad is written during the next group, after the
// operands of that group's hand-over have arrived: LDS answers a wavefront in order, and a write
// right ahead of a wait for a read would be waited for as well.
constexpr int kRingGroups = 64;   // a power of two and a multiple of four
constexpr int kForever = 0x3fffffff;
// entries of 64 bits per utterance and boundary of blocks that run side by side: the value of a
// step and the step + 1 above it, so that a reader can tell a written entry by itself -- one store,
// no fence, no separate counter
__device__ inline unsigned long long live_entry(int s, float x) {
  return ((unsigned long long)(unsigned)(s + 1) << 32) | (unsigned long long)__float_as_uint(x);
}
__device__ inline int prog_load(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline void prog_store(int* p, int x) {
  __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Waits for the neighbours of a wavefront that is about to run group g of n, and returns the group up
// to which it need not look again.  `in`: groups handed on to it, `out`: how far the taker of its own has
// got (both as far as known in have_in, have_out).  Asked ahead of every second group: groups g and
// g + 1 take in the quads up to g + 2, each asking for the next group's, so g + 3 have to be there;
// two more are waited for, so that the next look finds what it needs.  They write the quads up to g,
// over those up to g - kRingGroups, and a taker that tells x has read every quad below x: up to
// x + kRingGroups nothing unread is lost, and four less is allowed.  A walk that had to wait goes on
// fourteen groups ahead of that line.
__device__ __forceinline__ int hand_over_until(const int* in, const int* out, int& have_in,
                                               int& have_out, int g, int n, int spin_limit,
                                               int* __restrict__ trouble) {
  have_in = bounded_wait(in, have_in, min(g + 5, n), spin_limit, trouble);
  have_out = bounded_wait(out, have_out, g + 18 - kRingGroups, spin_limit, trouble);
  return min(have_in >= n ? kForever : have_in - 3, min(have_out, kForever) + kRingGroups - 4);
}

// The wavefront beside the walking ones of a block that runs side by side with others: brings what
// the block before it has left in memory (`src`) into the ring of the first walking wavefront, and
// takes what the last one hands on out to `dst`, up to 64 quads in a turn.  It keeps the
// tagged entries, their waits and their addresses out of the walk.  at(g, i): the step of value
// i = 0..3 of group g (four steps in a row).  Groups are numbered in walking order; quads [in, n_in) are
// brought, [out, n_out) taken; group g's lies in slot g + kShift of a ring.  Bounded like every wait
// here: when nothing has moved for spin_limit turns it raises the trouble flag and lets everybody go
// on with whatever the rings hold.
template <int kShift, typename At>
__device__ inline void live_carrier(const unsigned long long* __restrict__ src,
                                    unsigned long long* __restrict__ dst, int in, int n_in, int out,
                                    int n_out, At at, float* ring_in, int* prog_in, const int* prog_first,
                                    const float* ring_out, const int* prog_last, int* prog_out,
                                    int spin_limit, int* __restrict__ trouble) {
  const int lane = threadIdx.x & 63, quad = lane >> 2, value = lane & 3;
  int idle = 0;
  in = src ? in : n_in;
  out = dst ? out : n_out;
  while (in < n_in || out < n_out) {
    bool moved = false;
    unsigned long long e[4];
    const int room = in < n_in ? min(prog_load(prog_first) + kRingGroups - 4, n_in) - in : 0;
    asm volatile("" ::: "memory");
    if (room > 0) {  // (asked for ahead of the other side's work: the answer takes a microsecond)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        e[k] = __hip_atomic_load(src + at(min(in + 16 * k + quad, n_in - 1), value), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
    }
    if (out < n_out) {
      const int m = min(min(prog_load(prog_last), n_out) - out, 64);
      asm volatile("" ::: "memory");
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int g = out + 16 * k + quad;
        if (16 * k + quad < m) {
          const float x = ring_out[4 * ((g + kShift) & (kRingGroups - 1)) + value];
          const int s = at(g, value);
          __hip_atomic_store(dst + s, live_entry(s, x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      if (m > 0) {
        out += m;
        asm volatile("" ::: "memory");
        if (lane == 0) prog_store(prog_out, out);
        moved = true;
      }
    }
    if (room > 0) {
      int ready = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int g = in + 16 * k + quad;
        const bool here = 16 * k + quad < room && (unsigned)(e[k] >> 32) == (unsigned)(at(g, value) + 1);
        const unsigned long long missing = __builtin_amdgcn_ballot_w64(!here);
        if (ready == 16 * k) ready += missing ? __builtin_ctzll(missing) >> 2 : 16;
        if (16 * k + quad < ready)
          ring_in[4 * ((g + kShift) & (kRingGroups - 1)) + value] = __uint_as_float((unsigned)e[k]);
      }
      if (ready > 0) {
        in += ready;
        asm volatile("" ::: "memory");  // (LDS serves a wavefront's requests in order)
        if (lane == 0) prog_store(prog_in, in < n_in ? in : kForever);
        moved = true;
      }
    }
    // (not more often than pays: its requests go the same way as the walk's operands)
    __builtin_amdgcn_s_sleep(16);
    if (moved) {
      idle = 0;
    } else if (idle++ >= spin_limit) {
      if (lane == 0) {
        raise_trouble(trouble);
        prog_store(prog_in, kForever);
        prog_store(prog_out, kForever);
      }
      return;
    }
  }
}

// ------------------------------------------------------------------ alpha, one position a lane
// One cell on the fast path of lse2_fast and the two moves out of it, in an order of its own: a
// lone wavefront issues an instruction every four cycles (1.67 ns), dependent or not, exp and log
// take two turns, and a branch on a mask that was compared just before it stalls for 6 ns.  So what
// counts is the number of instructions -- 25, fifteen for the sum, four for its proof, six for the
// moves -- and that the comparison stands ahead of the moves.  Between a transcendental and the use of its result,
// and between the last write of `emit` and the lane shift that follows this block, stand the
// independent instructions the hardware asks for.
struct AlphaCell {
  float a, stay, emit;
  unsigned long long fail;  // lanes whose sum is not proven to be the library's
};
__device__ inline AlphaCell alpha_cell(float left, float stay, float eb, float el, float pb,
                                       float pl, float ln) {
  AlphaCell r;
  float t, y, k, w, l, hi;
  asm volatile(
      "v_sub_f32_e32 %[t], %[left], %[stay]\n\t"
      "v_mul_f32_e64 %[y], |%[t]|, %[nl2e]\n\t"
      "v_exp_f32_e32 %[y], %[y]\n\t"
      "v_max_f32_e32 %[hi], %[left], %[stay]\n\t"
      "v_fma_f32 %[k], |%[t]|, %[relb], %[rela] clamp\n\t"
      "v_add_f32_e32 %[w], 1.0, %[y]\n\t"
      "v_log_f32_e32 %[l], %[w]\n\t"
      "v_add_f32_e32 %[w], -1.0, %[w]\n\t"
      "v_fma_f32 %[t], %[y], -0.5, 1.0\n\t"
      "v_sub_f32_e32 %[w], %[y], %[w]\n\t"
      "v_mul_f32_e32 %[t], %[w], %[t]\n\t"
      "v_fmac_f32_e32 %[t], 0x3f317218, %[l]\n\t"         // log1p(exp(-|left - stay|))
      "v_fmaak_f32 %[k], %[t], %[k], 0x01000000\n\t"      // its bound (fast_bound)
      "v_sub_f32_e32 %[w], %[t], %[k]\n\t"
      "v_add_f32_e32 %[t], %[t], %[k]\n\t"
      "v_add_f32_e32 %[a], %[hi], %[w]\n\t"
      "v_add_f32_e32 %[hi], %[hi], %[t]\n\t"
      "v_cmp_neq_f32_e64 %[fail], %[a], %[hi]\n\t"
      "v_add_f32_e32 %[em], %[el], %[a]\n\t"
      "v_add_f32_e32 %[st], %[eb], %[a]\n\t"
      "v_add_f32_e32 %[em], %[pl], %[em]\n\t"
      "v_sub_f32_e32 %[em], %[em], %[ln]\n\t"
      "v_add_f32_e32 %[st], %[pb], %[st]\n\t"
      "v_sub_f32_e32 %[st], %[st], %[ln]"
      : [a] "=&v"(r.a), [st] "=&v"(r.stay), [em] "=&v"(r.emit), [fail] "=&s"(r.fail), [t] "=&v"(t),
        [y] "=&v"(y), [k] "=&v"(k), [w] "=&v"(w), [l] "=&v"(l), [hi] "=&v"(hi)
      : [left] "v"(left), [stay] "v"(stay), [eb] "v"(eb), [el] "v"(el), [pb] "v"(pb), [pl] "v"(pl),
        [ln] "v"(ln), [nl2e] "s"(-1.44269504088896341f), [relb] "s"(kFastRelB),
        [rela] "v"(kFastRelA));
  return r;
}

typedef float quad_t __attribute__((ext_vector_type(4)));
typedef float quad4_t __attribute__((ext_vector_type(4), aligned(4)));
// A piece of memory addressed as a buffer: an access takes a lane's own constant offset and a scalar
// one that walks, and no address is formed in vector registers.
struct Buffer {
  __amdgpu_buffer_rsrc_t r;
  __device__ Buffer(const void* p, size_t bytes) {
    int n = (int)buffer_bytes(bytes), flags = 0x00020000;
    // (opaque: words that several descriptors have in common would be copied around at every use)
    asm volatile("" : "+s"(n), "+s"(flags));
    r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, n, flags);
  }
  __device__ quad_t load(unsigned lane_off, unsigned off) const {
    return __builtin_bit_cast(quad_t, __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0));
  }
  __device__ void store(unsigned lane_off, unsigned off, quad_t x) const {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, x), r, lane_off, off, 0);
  }
};

// The walk of one utterance with one label position a lane: W wavefronts of 64 positions; kLive:
// live_n such blocks of the label axis at the same time, as many workgroups on as many CUs of one
// XCD, with a wavefront more that carries the scores between them (live_carrier).  Workgroups are
// dispatched in launch order and a block has a smaller index than the block above it, so the block
// that is waited for is always running or done.
// A step is 25 instructions, the lane shift, a branch (5.4 ns, whether taken or not) and 40
// instructions per group of four for operands, hand-over and progress: 59 ns measured on one
// wavefront, 65 with a neighbour.  A step with a lane whose sum is not proven takes about 0.3 us
// more (the chance falls with the size of the alphas: nearly every step up to 100 or so, one in
// ten at 1000, one in a hundred at 10000).  Whole walks, B=8 T=2000: 85 ns a step at 51 positions, 92
// at 101 (93 and 111 with 29 instructions, the comparison right ahead of its branch, whole
// hand-over arrays in LDS whose writes the next group waited for); B=8 T=10000, 401
// positions 84 (128 with the entries between blocks asked for and checked inside the walk).
// A wavefront runs the groups from its first position's first cell to its last one's last.  While all of
// them ran all groups, most instructions of a lattice with more label positions than frames were for
// cells outside, and two workgroups on a CU, short of issue slots, were slower than the walk before
// this one: B=64 T=100, 1025 positions 317 us then, 371 with all groups, 239 so; B=4 238 and 206.
template <int W, bool kLive>
__global__ __launch_bounds__(64 * (W + (kLive ? 1 : 0))) void alpha_walk_kernel(
    Planes p, const int* __restrict__ inLen, const int* __restrict__ labLen,
    float* __restrict__ costs, Dims d, int spin_limit, int* __restrict__ trouble,
    unsigned long long* __restrict__ live, int live_n) {
  constexpr bool kHand = W > 1 || kLive;
  __shared__ __attribute__((aligned(16))) float ring[W + 1][kHand ? 4 * kRingGroups : 4];
  __shared__ __attribute__((aligned(16))) float nothing[16];
  __shared__ __attribute__((aligned(16))) float dump[kHand ? 4 * 64 + 16 : 4];
  __shared__ int prog[W + 2];
  __shared__ unsigned long long etab[32];  // expf's table (rnnt_libm.h)
  // live blocks: workgroups go round the 8 XCDs in launch order; ids i, i + 8, i + 16 .. share
  // one, and with it the L2 the boundary scores cross in.  Eight utterances take 8 live_n
  // consecutive ids, block by block, lowest block first.
  const int live_block = kLive ? (int)(blockIdx.x >> 3) % live_n : 0;
  const int b = kLive ? (int)(blockIdx.x / (8 * live_n)) * 8 + (blockIdx.x & 7) : blockIdx.x;
  if (kLive && b >= d.B) return;
  const int u_base = live_block * 64 * W;
  const int lane = threadIdx.x & 63;
  const int wave = (W > 1 || kLive) ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Tb == 0 || Ub == 0) {  // :39-41
    if (threadIdx.x == 0 && u_base == 0) costs[b] = kPosInf;
    return;
  }
  if (u_base >= Ub) return;  // a block past this utterance's labels: nobody reads what it would leave
  // groups a wavefront of positions u .. u + 63 runs
  auto begin_of = [](int u) { return u >> 2; };
  auto end_of = [&](int u) { return ((Tb - 1 + min(u + 63, Ub - 1)) >> 2) + 1; };
  // a block below and a block above this one (for this utterance)
  const bool live_in = kLive && live_block > 0;
  const bool live_out = kLive && live_block < live_n - 1 && u_base + 64 * W < Ub;
  exp2_table_to_lds(etab);
  if (threadIdx.x < 16) nothing[threadIdx.x] = kNegInf;
  if (threadIdx.x < W + 2) {
    // (counted from where each of them starts; a wavefront also needs the quad ahead of its first
    // group, whose last value enters its first step)
    const int w = (int)threadIdx.x - 1;  // the wavefront whose progress this is
    prog[threadIdx.x] = w < 0 ? (live_in ? begin_of(u_base) - 1 : kForever)
                        : w == W ? (live_out ? begin_of(u_base + 64 * W) - 1 : kForever)
                                 : (u_base + 64 * w < Ub ? begin_of(u_base + 64 * w) : kForever);
  }
  __syncthreads();
  if (kLive && wave == W) {
    const unsigned long long* src =
        live_in ? live + ((size_t)(live_block - 1) * d.B + b) * d.Dp : nullptr;
    unsigned long long* dst = live_out ? live + ((size_t)live_block * d.B + b) * d.Dp : nullptr;
    // what enters step s: value i of group g is what enters step 4g + 1 + i (nothing enters step 0)
    live_carrier<0>(src, dst, begin_of(u_base) - 1, end_of(u_base - 64), begin_of(u_base + 64 * W) - 1,
                    end_of(u_base + 64 * (W - 1)), [](int g, int i) { return 4 * g + 1 + i; }, ring[0],
                    &prog[0], &prog[1], ring[W], &prog[W], &prog[W + 1], spin_limit, trouble);
    return;
  }
  const int u_lo = u_base + wave * 64;
  if (u_lo >= Ub) return;  // a wavefront past this utterance's labels
  if (kLive) __builtin_amdgcn_s_setprio(3);  // ahead of the carrier on the same SIMD
  const int u = u_lo + lane;
  const bool real = u < Ub;
  const bool first_column = u_lo == 0;  // lane 0 owns the lattice's column u = 0
  // Operands of a position past the utterance's last one are the last one's (its label score the
  // last label's), and its moves carry kOutside on top: whatever it meets is an ordinary number
  // far below any alpha, so that the interior groups below need no test for it.
  // (loaded in every lane: a branch here would leave the uniform sizes behind it in vector registers)
  float pb = p.pb[(size_t)b * d.Ua + u], pl = p.pl[(size_t)b * d.Ua + u];  // u < Ua
  asm volatile("" : "+v"(pb), "+v"(pl));
  pb = real ? pb : kOutside;
  pl = real ? pl : kOutside;
  const unsigned tlim = real ? (unsigned)Tb : 0u;
  // :43 alpha[0,0] = 0: cell (0,0) finds 0 coming up from below and nothing from the left
  float stay = u == 0 ? 0.0f : kNegInf, emit = kOutside, final = 0.0f;

  // Interior groups [in_lo, in_hi): step 4g is past the first frame of the wavefront's last
  // position, step 4g + 3 not past the last frame of its first one.
  const unsigned gbytes = kLive ? 16u * (unsigned)d.Ua : 1024u * W;  // from a group to the next
  const int g_begin = begin_of(u_lo), g_end = end_of(u_lo);
  const int in_lo = (min(u_lo + 64, Ub) + 2) >> 2;
  const int in_hi = Ub > 1 ? min((Tb + u_lo) >> 2, g_end - 1) : 0;
  // The planes as buffers that begin at group `origin` of the utterance (moved on before an offset
  // would outgrow 32 bits).  E[t,blank] of step s, lane by lane, sits at eb[Eo + s - u].
  const size_t plane = (size_t)gbytes * (unsigned)(d.Dp / 4);
  const char* ln_b = reinterpret_cast<const char*>(p.lnS + plane_group0(d, b, 0));
  const char* el_b = reinterpret_cast<const char*>(p.elS + plane_group0(d, b, 0));
  char* a_b = reinterpret_cast<char*>(p.aS + plane_group0(d, b, 0));
  const Buffer eb_q(p.eb + (size_t)b * d.Tp, 4ull * d.Tp);
  Buffer ln_q(ln_b, plane), el_q(el_b, plane), a_q(a_b, plane);
  int origin = 0;
  const int span = (int)((1u << 30) / gbytes);
  auto move_on = [&](int g) {
    origin = g;
    const size_t by = (size_t)g * gbytes;
    ln_q = Buffer(ln_b + by, plane - by);
    el_q = Buffer(el_b + by, plane - by);
    a_q = Buffer(a_b + by, plane - by);
  };
  const unsigned ln_o = 16u * (unsigned)min(u, Ub - 1);
  const unsigned el_o = 16u * (unsigned)max(min(u, Ub - 2), 0);
  const unsigned a_o = 16u * (unsigned)u;
  const unsigned eb_o = 4u * (unsigned)(d.Eo - min(u, Ub - 1));
  struct Ops {
    quad_t ln, el, eb;
  };
  auto load = [&](int g) -> Ops {
    const unsigned by = (unsigned)(g - origin) * gbytes;
    Ops r;
    r.ln = ln_q.load(ln_o, by);
    r.el = el_q.load(el_o, by);
    r.eb = eb_q.load(eb_o, 16u * (unsigned)g);
    return r;
  };
  auto load_to_end = [&](int g) -> Ops { return load(min(g, g_end - 1)); };

  // ---- hand-over
  int ok = kHand ? -1 : kForever;  // groups up to here may run without looking at the neighbours
  int have_in = 0, have_out = 0;
  auto refresh = [&](int g) {
    ok = hand_over_until(&prog[wave], &prog[wave + 2], have_in, have_out, g, g_end, spin_limit, trouble);
  };
  const float* take = kHand ? (first_column ? nothing : ring[wave]) : nullptr;
  const int take_mask = first_column ? 0 : kRingGroups / 4 - 1;
  float* give = kHand ? (lane == 63 ? ring[wave + 1] : dump + 4 * lane) : nullptr;
  const int give_mask = lane == 63 ? kRingGroups / 4 - 1 : 0;
  int* give_prog = lane == 63 ? &prog[wave + 1] : reinterpret_cast<int*>(dump + 4 * lane);
  quad_t pend = {kOutside, kOutside, kOutside, kOutside};  // what the last group handed on
  quad_t hand = {kNegInf, kNegInf, kNegInf, kNegInf};      // what enters the running group
  float carry = first_column ? kNegInf : kOutside;         // ... and its first step

  // A group: hands on what the last one left, asks for what the next one takes in, four steps.
  // kInner: an interior group, which needs no bounds.  At the lattice's edges every cell is asked
  // whether it is inside, and the blank move out of a position's last cell stays in `final`.
  auto run_group = [&](int g, const Ops& q, const float* take_next, float* give_last, auto tell,
                       auto inner) {
    constexpr bool kTell = decltype(tell)::value, kInner = decltype(inner)::value;
    quad_t next = hand;
    if constexpr (kHand) {
      *reinterpret_cast<quad_t*>(give_last) = pend;
      asm volatile("" ::: "memory");  // (LDS serves a wavefront's requests in order)
      if constexpr (kTell) prog_store(give_prog, g);
      next = *reinterpret_cast<const quad_t*>(take_next);
    }
    float in[4] = {carry, hand[0], hand[1], hand[2]};
    unsigned long long inside[4];
    if constexpr (!kHand || !kInner) {
      if constexpr (!kHand) in[0] = in[1] = in[2] = in[3] = kNegInf;
      if constexpr (!kInner) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // a cell of the lattice: 0 <= t = s - u < T_b (one unsigned comparison)
          inside[j] = __builtin_amdgcn_ballot_w64((unsigned)(4 * g + j - u) < tlim);
          // what enters the lattice's own first column: nothing, which is -inf while its cells are
          // inside the lattice (:49-52 adds nothing there, so a -inf blank score must come out as
          // -inf) and, as in any first column, kOutside once they are past the last frame (see
          // kOutside; nobody hands anything on for those steps)
          if (4 * g + j >= Tb + u_lo) in[j] = kOutside;
        }
      }
      // (set well ahead of the lane shifts that fill lane 0 from them)
      asm volatile("" : "+v"(in[0]), "+v"(in[1]), "+v"(in[2]), "+v"(in[3]));
    }
    quad_t a;
    quad_t em;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float left = wave_shr1(emit, in[j]);
      const AlphaCell c = alpha_cell(left, stay, q.eb[j], q.el[j], pb, pl, q.ln[j]);
      float x = c.a, sb = c.stay, se = c.emit;
      if (__builtin_expect(c.fail != 0ull, 0)) {
        x = lse2_libm(left, stay, etab);
        sb = x + q.eb[j];
        sb = sb + pb;
        sb = sb - q.ln[j];
        se = x + q.el[j];
        se = se + pl;
        se = se - q.ln[j];
      }
      if constexpr (kInner) {
        stay = sb;
        emit = se;
      } else {
        const bool is = __builtin_amdgcn_inverse_ballot_w64(inside[j]);
        final = is ? sb : final;
        stay = is ? sb : kNegInf;
        emit = is ? se : kOutside;
      }
      a[j] = x;
      em[j] = emit;
    }
    a_q.store(a_o, (unsigned)(g - origin) * gbytes, a);
    pend = em;
    carry = hand[3];
    hand = next;
  };

  // four sets of operands rotate: a group's loads are requested four groups (16 steps, more than a
  // microsecond) ahead -- the planes of a long batch do not fit L2
  Ops q0 = load_to_end(g_begin), q1 = load_to_end(g_begin + 1), q2 = load_to_end(g_begin + 2),
      q3 = load_to_end(g_begin + 3);
  if constexpr (kHand) {
    if (!first_column) {  // (g_begin is a multiple of sixteen)
      refresh(g_begin);
      carry = take[16 * (((g_begin >> 2) - 1) & take_mask) + 15];
      hand = *reinterpret_cast<const quad_t*>(take + 16 * ((g_begin >> 2) & take_mask));
    }
  }
  const std::true_type yes;
  const std::false_type no;
  int g = g_begin;
  auto block = [&](auto inner) {
    constexpr bool kInner = decltype(inner)::value;
    const float *tk = nullptr, *tk_next = nullptr;
    float *gv = nullptr, *gv_last = nullptr;
    if constexpr (kHand) {
      tk = take + 16 * ((g >> 2) & take_mask);
      tk_next = take + 16 * (((g >> 2) + 1) & take_mask);
      gv = give + 16 * ((g >> 2) & give_mask);
      gv_last = give + 16 * (((g >> 2) - 1) & give_mask) + 12;
      if (__builtin_expect(g > ok, 0)) refresh(g);
    }
    auto ahead = [&](int k) -> Ops {
      if constexpr (kInner) return load(g + 4 + k);
      return load_to_end(g + 4 + k);
    };
    run_group(g, q0, tk + 4, gv_last, yes, inner);
    q0 = ahead(0);
    run_group(g + 1, q1, tk + 8, gv, no, inner);
    q1 = ahead(1);
    if constexpr (kHand) {
      if (__builtin_expect(g + 2 > ok, 0)) refresh(g + 2);
    }
    run_group(g + 2, q2, tk + 12, gv + 4, yes, inner);
    q2 = ahead(2);
    run_group(g + 3, q3, tk_next, gv + 8, no, inner);
    q3 = ahead(3);
    // everything LDS was asked for is there by now; said here, the head of the next block need not
    // wait for what it has itself just asked for
    if constexpr (kHand) __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    g += 4;
  };
  while (g + 4 < g_end) {
    if (g - origin >= span) move_on(g);
    if (g >= in_lo && g + 4 <= in_hi && g + 8 <= g_end) {
      const int end = min(min(in_hi, g_end - 4), origin + span);
      do block(yes);
      while (g + 4 <= end);
    } else {
      block(no);
    }
  }
  // the last one to four groups
  while (g < g_end) {
    const float* tk = nullptr;
    float* gv = nullptr;
    if constexpr (kHand) {
      tk = take + 16 * (((g + 1) >> 2) & take_mask) + 4 * ((g + 1) & 3);
      gv = give + 16 * (((g - 1) >> 2) & give_mask) + 4 * ((g - 1) & 3);
      if (__builtin_expect(g > ok, 0)) refresh(g);
    }
    run_group(g, q0, tk, gv, yes, no);
    q0 = q1;
    q1 = q2;
    q2 = q3;
    ++g;
  }
  if constexpr (kHand) {
    *reinterpret_cast<quad_t*>(give + 16 * (((g_end - 1) >> 2) & give_mask) + 4 * ((g_end - 1) & 3)) = pend;
    asm volatile("" ::: "memory");
    prog_store(give_prog, kForever);
  }
  // :73-78 the blank move out of the last cell, negated
  if (u == Ub - 1) costs[b] = -final;
}

// ------------------------------------------------------------------ transition weights
// Everything of the dalpha recursion that does not depend on dalpha itself
// (transducer/transducer_cpu.cpp:124-135).  A thread takes the four anti-diagonals of a group at one
// label position: its operands and results are whole 16-byte pieces of the planes, and eight
// exponentials are under way at once.  Bound by those (about 25 instructions each, eight of them in
// double) and by the planes it reads and writes, about evenly: B=8 T=10000 U=401 141 us (700 MB,
// 5 TB/s), 261 with one entry to a thread; B=32 T=2000 U=101 29, 41.
// Every entry of the two weight planes is written -- zero where there is no such move or no such
// cell -- so the recursion below needs no bounds of its own.
__global__ __launch_bounds__(256) void weights_kernel(Planes p, const int* __restrict__ inLen,
                                                      const int* __restrict__ labLen, Dims d) {
  __shared__ unsigned long long etab[32];  // expf's table (rnnt_libm.h)
  exp2_table_to_lds(etab);
  __syncthreads();
  // piece i of the utterance's plane: group i / Ua of label position i % Ua (Ua is a power of two)
  const int b = blockIdx.z;
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int ngroups = d.Dp >> 2;
  if (i >= d.Ua * ngroups) return;
  const int u = i & (d.Ua - 1), g = i >> (31 - __clz(d.Ua));
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  const int t0 = 4 * g - u;  // frame of the first of the four cells
  const size_t o = (size_t)b * d.Ua * d.Dp + 4 * (size_t)i;  // = plane_at(d, b, u, 4 g)
  float4 wb = make_float4(0.0f, 0.0f, 0.0f, 0.0f), we = wb;
  if (u < Ub && t0 > -4 && t0 < Tb) {
    auto piece = [](const float* q) { return *reinterpret_cast<const float4*>(q); };
    const bool emits = u + 1 < Ub;
    // one step on: the same position's and the next one's, the last of the four from the next group
    const size_t next = g + 1 < ngroups ? 4 * (size_t)d.Ua : 0, right = emits ? 4 : 0;
    const float4 a = piece(p.aS + o), ln = piece(p.lnS + o), ar = piece(p.aS + o + right);
    const float4 el = piece(p.elS + o);
    const float a4 = p.aS[o + next], ar4 = p.aS[o + next + right];
    const float* eb = p.eb + (size_t)b * d.Tp + d.Eo;
    const float pb = p.pb[(size_t)b * d.Ua + u], pl = p.pl[(size_t)b * d.Ua + u];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = t0 + j;
      float x = f4get(a, j) + eb[min(max(t, 0), Tb - 1)];
      x = x + pb;
      x = x - f4get(ln, j);
      x = x - (j < 3 ? f4get(a, j < 3 ? j + 1 : 0) : a4);
      const float stay = expf_glibc(x, etab);
      x = f4get(a, j) + f4get(el, j);
      x = x + pl;
      x = x - f4get(ln, j);
      x = x - (j < 3 ? f4get(ar, j < 3 ? j + 1 : 0) : ar4);
      const float emit = expf_glibc(x, etab);
      const bool cell = t >= 0 && t < Tb;
      f4set(wb, j, cell && t + 1 < Tb ? stay : 0.0f);
      f4set(we, j, cell && emits ? emit : 0.0f);
    }
  }
  *reinterpret_cast<float4*>(p.wB + o) = wb;
  *reinterpret_cast<float4*>(p.wE + o) = we;
}

// ------------------------------------------------------------------ dalpha
// transducer/transducer_cpu.cpp:81-143 with the exponentials already taken:
// dalpha[t,u] = dalpha[t+1,u]*wB[t,u] + dalpha[t,u+1]*wE[t,u], walked from the last diagonal
// back to the first; the last cell is seeded with 1 (:95) before the walk.  Each lane also
// keeps the running sums that the reference subtracts from pgrads[u,blank] and pgrads[u,l_u],
// in the reference's own order (t descending).  Operands are prefetched beta_depth(C) groups
// of four steps ahead through as many rotating register sets.
// A label axis longer than 64 C positions is walked block by block (u_base = first position of
// the block), HIGHEST block first: what crosses a boundary here is dalpha of the upper block's
// first column, one value per diagonal, left in `ghout` ([B][hand_stride], entry s = its dalpha
// on diagonal s; null for the lowest block) and read by the block below from `ghin` (null for
// the highest block).
// register sets of the dalpha walk's prefetch: eight where a set is small, three (the first
// version's) where a lane owns so many label positions that more sets would spill
constexpr int beta_depth(int C) { return C <= 2 ? 8 : C <= 4 ? 4 : 3; }
// W wavefronts (one launch covering the whole label axis only): wavefront w owns positions
// (64 w + lane) C .. + C-1, so the HIGHEST wavefront leads.  Each but the lowest leaves dalpha of
// its first column in LDS, one value per diagonal, and counts the groups it has finished; the
// wavefront below reads them one group later (the same hand-over as between blocks, with the
// bounded wait of alpha_kernel).  Every wavefront runs all groups, past the utterance's labels
// too (zeros), so nobody waits for a wavefront that has left.
template <int C, int W, bool kMulti>
__global__ __launch_bounds__(64 * W) void beta_kernel(Planes p, const int* __restrict__ labels,
                                                      const int* __restrict__ inLen,
                                                      const int* __restrict__ labLen, Dims d,
                                                      int hand_stride, int u_base,
                                                      const float* __restrict__ ghin,
                                                      float* __restrict__ ghout, int spin_limit,
                                                      int* __restrict__ trouble) {
  static_assert(W == 1 || !kMulti, "several wavefronts only when one launch covers the label axis");
  extern __shared__ __attribute__((aligned(16))) float hand[];  // [W-1][hand_stride]: entry s =
                                                                // dalpha on diagonal s
  __shared__ int done[W];  // groups a wavefront has published
  const int b = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Tb == 0 || Ub == 0) return;  // :92-94
  if (u_base >= Ub) return;        // a block past this utterance's labels
  if (W > 1) {
    if (threadIdx.x < W) done[threadIdx.x] = 0;
    __syncthreads();
  }
  const int nsteps = Tb + Ub - 1;
  const int last = nsteps - 1;  // diagonal of the last cell
  // A lane's C positions are 64 apart (u0 + 64 c), so that the 64 lanes of a load or store touch
  // neighbouring 16-byte pieces of the plane, whole cache lines together; the price is a
  // lane-to-scalar move per position and step (lane 63's right neighbour is lane 0's next position).
  constexpr int kApart = 64;
  const int u0 = u_base + wave * 64 * C + lane;
  const int gstride = plane_group_stride(d);
  float* hand_out = hand + (wave > 0 ? wave - 1 : 0) * hand_stride;  // wave > 0
  const float* hand_in = hand + wave * hand_stride;                  // wave < W-1
  const int g_first = last >> 2;  // the group that holds the seed: the first one run
  int avail = 0;                  // groups the wavefront above is known to have published
  auto wait_for = [&](int need) {
    avail = bounded_wait(&done[wave + 1], avail, need, spin_limit, trouble);
  };
  // the block above exists for this utterance only if its first column does
  const float* gin =
      (kMulti && ghin && u_base + 64 * C < Ub) ? ghin + (size_t)b * hand_stride : nullptr;
  float* gout = (kMulti && ghout) ? ghout + (size_t)b * hand_stride : nullptr;
  float dcol[C], accB[C], accL[C];
  bool fold[C];  // label of this position equals blank: both sums share one accumulator
  const float* wbp[C];
  const float* wep[C];
  float* dp[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int u = u0 + kApart * c;
    const size_t row = plane_group0(d, b, u);
    wbp[c] = p.wB + row;
    wep[c] = p.wE + row;
    dp[c] = p.dS + row;
    dcol[c] = (u == Ub - 1) ? 1.0f : 0.0f;   // :95
    accB[c] = (u == Ub - 1) ? -1.0f : 0.0f;  // :97
    accL[c] = 0.0f;
    fold[c] = (u + 1 < Ub) && label_at(labels, d, b, u) == d.blank;
  }

  struct Group {
    float4 wb[C], we[C];
    float gh[4];  // dalpha of the block above's first column on diagonals 4g+1 .. 4g+4
  };
  auto load_group = [&](int g) -> Group {
    Group r;
    const int gc = g > 0 ? g : 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      r.wb[c] = *reinterpret_cast<const float4*>(wbp[c] + (size_t)gc * gstride);
      r.we[c] = *reinterpret_cast<const float4*>(wep[c] + (size_t)gc * gstride);
    }
    if constexpr (kMulti) {
#pragma unroll
      for (int j = 0; j < 4; ++j) r.gh[j] = gin ? gin[4 * gc + 1 + j] : 0.0f;  // uniform
    }
    return r;
  };
  // steps last-1 .. 0 are computed; the slot of step `last` receives the seed and the slots
  // after it (same group of four) zeros
  // with_fold: some position of this wavefront has the blank as its label, whose two sums then
  // share one accumulator.  Real transcripts have none, and the walk without the two selects per
  // cell is a fifth shorter (x - 0 is x, so the sums come out the same bits either way).
  // seeded: the group that holds the last diagonal (the first one run).  Every other group has
  // all four of its steps below `last`, and is compiled without the test per step (a scalar
  // compare, two mask moves and two branches: eight of the walk's sixteen instructions a step).
  auto run_group = [&](int g, const Group& w, auto with_fold, auto seeded) {
    constexpr bool kFold = decltype(with_fold)::value;
    constexpr bool kSeeded = decltype(seeded)::value;
    float4 dout[C];
    float gsend[4];  // dalpha of this lane's first column after each step
    float hh[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // dalpha of the wavefront above's first column on
                                             // diagonals 4g+1 .. 4g+4
    if (W > 1 && wave < W - 1) {
      wait_for(g_first - g + 1);  // diagonals 4g+1 .. 4g+3 are of its group g
#pragma unroll
      for (int j = 0; j < 4; ++j) hh[j] = hand_in[4 * g + 1 + j];  // uniform
    }
#pragma unroll
    for (int j = 3; j >= 0; --j) {
      const int s = 4 * g + j;
      if (kSeeded && s >= last) {  // uniform
#pragma unroll
        for (int c = 0; c < C; ++c) f4set(dout[c], j, s == last ? dcol[c] : 0.0f);
        if constexpr (kMulti || W > 1) gsend[j] = s == last ? dcol[0] : 0.0f;
      } else {
        // dalpha of the position to the right on the diagonal just done, s + 1: the next lane's,
        // and for lane 63 lane 0's next position -- or, right of the wavefront's last position,
        // what the block or the wavefront above handed over (nothing above: 0)
        float right[C];
        float above = 0.0f;  // right of the wavefront's last position
        if constexpr (kMulti) above = gin ? w.gh[j] : 0.0f;
        if (W > 1) above = wave < W - 1 ? hh[j] : 0.0f;
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const float past =  // what lane 63 receives
              c < C - 1 ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dcol[c + 1]), 0))
                        : above;
          right[c] = wave_shl1(dcol[c], past);
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const float ne = dcol[c] * f4get(w.wb[c], j);
          const float em = right[c] * f4get(w.we[c], j);
          const float dn = ne + em;
          if constexpr (kFold) {
            const float em_b = fold[c] ? em : 0.0f, em_l = fold[c] ? 0.0f : em;
            accB[c] = (accB[c] - ne) - em_b;
            accL[c] = accL[c] - em_l;
          } else {
            accB[c] = accB[c] - ne;
            accL[c] = accL[c] - em;
          }
          dcol[c] = dn;
          f4set(dout[c], j, dn);
        }
        if constexpr (kMulti || W > 1) gsend[j] = dcol[0];
      }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) *reinterpret_cast<float4*>(dp[c] + (size_t)g * gstride) = dout[c];
    if constexpr (kMulti) {
      if (gout && lane == 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) gout[4 * g + j] = gsend[j];
      }
    }
    if (W > 1 && wave > 0 && lane == 0) {  // entries 4g .. 4g+3, then the progress
#pragma unroll
      for (int j = 0; j < 4; ++j) hand_out[4 * g + j] = gsend[j];
      asm volatile("" ::: "memory");  // (LDS serves a wavefront's requests in order)
      __hip_atomic_store(&done[wave], g_first - g + 1, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };

  // beta_depth(C) register sets rotate (no copies): a group's weights are requested that many
  // groups ahead.  A step of this walk is a dozen instructions, so eight groups are 32 steps or
  // about a microsecond -- what a load that misses L2 takes; with two groups ahead (the first
  // version) the walk waited for its weights at nearly every group: 78 ns a step at U = 101.
  auto walk = [&](auto with_fold) __attribute__((always_inline)) {
    constexpr int kBetaDepth = beta_depth(C);
    int g = g_first;
    Group q[kBetaDepth];
#pragma unroll
    for (int i = 0; i < kBetaDepth; ++i) q[i] = load_group(g - i);
    // fall a few groups behind the wavefront above, so that the wait per group finds its
    // counter there already
    if (W > 1 && wave < W - 1) wait_for(min(g_first + 1, 8 * (W - 1 - wave)));
    // the first round, whose first group holds the seed (a short lattice may end inside it)
    const std::true_type seeded;
    const std::false_type plain;
    run_group(g, q[0], with_fold, seeded);
    q[0] = load_group(g - kBetaDepth);
#pragma unroll
    for (int i = 1; i < kBetaDepth; ++i) {
      if (g - i >= 0) run_group(g - i, q[i], with_fold, plain);
      q[i] = load_group(g - i - kBetaDepth);
    }
    g -= kBetaDepth;
    for (; g >= kBetaDepth - 1; g -= kBetaDepth) {
#pragma unroll
      for (int i = 0; i < kBetaDepth; ++i) {
        run_group(g - i, q[i], with_fold, plain);
        q[i] = load_group(g - i - kBetaDepth);
      }
    }
#pragma unroll
    for (int i = 0; i < kBetaDepth - 1; ++i)
      if (g - i >= 0) run_group(g - i, q[i], with_fold, plain);
  };
  bool any_fold = false;
#pragma unroll
  for (int c = 0; c < C; ++c) any_fold = any_fold || fold[c];
  if (__ballot(any_fold) != 0) walk(std::true_type{});
  else walk(std::false_type{});

#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int u = u0 + kApart * c;
    if (u < Ub) {
      p.gB[(size_t)b * d.Ua + u] = accB[c];
      p.gL[(size_t)b * d.Ua + u] = accL[c];
    }
  }
}

// ------------------------------------------------------------------ dalpha, one position a lane
// The same recursion with one label position a lane, dealt to wavefronts and to blocks side by side
// like alpha_walk_kernel's with the directions turned round: the HIGHEST wavefront leads (and the
// highest block has the smallest workgroup index); what crosses is dalpha of a wavefront's first
// column, quads of four diagonals through the rings.  Groups are counted in walking order, i = 0 the
// one that holds the seed; group i's quad lies in slot i + 3 of the ring, so that the groups after
// the seed's come in aligned blocks of four slots.
// A step is six instructions, a group of four about twenty more, and the hand-over as many again: 19 ns
// a step on one wavefront, 33 with a neighbour (20 and 36 when two positions a lane shared one
// wavefront, every load formed an address and was asked for eight groups ahead).  Beyond, the walk
// waits for memory, 12 bytes a cell: kDepth register sets rotate, a group's weights being requested
// that many groups ahead (a microsecond is about twelve groups).  B=8, 201 positions T=2000: 124 ->
// 80 us (the weights of a group used to be waited for together with what had just been handed
// over); 401 positions T=2000 193 -> 100, T=10000 766 -> 372.  The weight planes hold zeros
// wherever there is no move, so nothing asks for bounds.
template <int W, bool kLive>
__global__ __launch_bounds__(64 * (W + (kLive ? 1 : 0))) void beta_walk_kernel(
    Planes p, const int* __restrict__ labels, const int* __restrict__ inLen,
    const int* __restrict__ labLen, Dims d, int spin_limit, int* __restrict__ trouble,
    unsigned long long* __restrict__ live, int live_n) {
  constexpr bool kHand = W > 1 || kLive;
  constexpr int kDepth = W == 1 ? 16 : 12;
  __shared__ __attribute__((aligned(16))) float ring[W + 1][kHand ? 4 * kRingGroups : 4];
  __shared__ __attribute__((aligned(16))) float nothing[16];
  __shared__ __attribute__((aligned(16))) float dump[kHand ? 4 * 64 + 16 : 4];
  __shared__ int prog[W + 2];
  const int live_block = kLive ? live_n - 1 - (int)(blockIdx.x >> 3) % live_n : 0;
  const int b = kLive ? (int)(blockIdx.x / (8 * live_n)) * 8 + (blockIdx.x & 7) : blockIdx.x;
  if (kLive && b >= d.B) return;
  const int u_base = live_block * 64 * W;
  const int lane = threadIdx.x & 63;
  const int wave = kHand ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Tb == 0 || Ub == 0) return;  // :92-94
  if (u_base >= Ub) return;        // a block past this utterance's labels
  const int last = Tb + Ub - 2;    // diagonal of the last cell
  const int g_first = last >> 2;   // the group that holds the seed
  const int n = g_first + 1;
  const bool live_in = kLive && live_block < live_n - 1 && u_base + 64 * W < Ub;
  const bool live_out = kLive && live_block > 0;
  if constexpr (kHand) {
    if (threadIdx.x < 16) nothing[threadIdx.x] = 0.0f;
    if (threadIdx.x < W + 2) {
      const int r = (int)threadIdx.x - 1;  // the wavefront, in walking order, whose progress this is
      prog[threadIdx.x] = r < 0 ? (live_in ? 0 : kForever)
                          : r == W ? (live_out ? 0 : kForever)
                                   : (u_base + 64 * (W - 1 - r) < Ub ? 0 : kForever);
    }
    __syncthreads();
  }
  if (kLive && wave == W) {
    const unsigned long long* src =
        live_in ? live + ((size_t)live_block * d.B + b) * d.Dp : nullptr;
    unsigned long long* dst =
        live_out ? live + ((size_t)(live_block - 1) * d.B + b) * d.Dp : nullptr;
    live_carrier<3>(src, dst, 0, n, 0, n, [&](int i, int k) { return 4 * (g_first - i) + k; }, ring[0],
                    &prog[0], &prog[1], ring[W], &prog[W], &prog[W + 1], spin_limit, trouble);
    return;
  }
  const int u_lo = u_base + wave * 64;
  if (u_lo >= Ub) return;  // a wavefront past this utterance's labels
  if (kLive) __builtin_amdgcn_s_setprio(3);  // ahead of the carrier on the same SIMD
  const int order = W - 1 - wave;
  const bool leads = !live_in && u_lo + 64 >= Ub;  // nothing comes in from above
  const int u = u_lo + lane;
  float dcol = u == Ub - 1 ? 1.0f : 0.0f;   // :95
  float accB = u == Ub - 1 ? -1.0f : 0.0f;  // :97
  float accL = 0.0f;
  // label of this position equals blank: both sums share one accumulator
  bool fold = false;
  if (d.U > 1) {  // (read in every lane: no divergent branch, see alpha_walk_kernel)
    const int label = label_at(labels, d, b, min(u, d.U - 2));
    fold = (u + 1 < Ub) & (label == d.blank);
  }

  const unsigned gbytes = kLive ? 16u * (unsigned)d.Ua : 1024u * W;  // from a group to the next
  const unsigned lane_o = 16u * (unsigned)u;
  // the planes as buffers that begin at group `origin` (moved down as the walk goes on, so that no
  // offset outgrows 32 bits)
  const int span = (int)((1u << 30) / gbytes);
  int origin = max(0, g_first - span);
  const char* wb_b = reinterpret_cast<const char*>(p.wB + plane_group0(d, b, 0));
  const char* we_b = reinterpret_cast<const char*>(p.wE + plane_group0(d, b, 0));
  char* d_b = reinterpret_cast<char*>(p.dS + plane_group0(d, b, 0));
  const size_t plane = (size_t)gbytes * (unsigned)(d.Dp / 4);
  const size_t by0 = (size_t)origin * gbytes;
  Buffer wb_q(wb_b + by0, plane - by0), we_q(we_b + by0, plane - by0), d_q(d_b + by0, plane - by0);
  auto move_to = [&](int g) {
    origin = g;
    const size_t by = (size_t)g * gbytes;
    wb_q = Buffer(wb_b + by, plane - by);
    we_q = Buffer(we_b + by, plane - by);
    d_q = Buffer(d_b + by, plane - by);
  };
  struct Ops {
    quad_t wb, we;
  };
  auto load = [&](int i) -> Ops {  // (what is asked for past the last group is never used)
    const unsigned by = (unsigned)(max(g_first - i, 0) - origin) * gbytes;
    Ops r;
    r.wb = wb_q.load(lane_o, by);
    r.we = we_q.load(lane_o, by);
    return r;
  };

  // ---- hand-over (see alpha_walk_kernel)
  int ok = kHand ? -1 : kForever;
  int have_in = 0, have_out = 0;
  auto refresh = [&](int i) {  // hand_over_until written out: called, the walk is scheduled 1.5 % worse
    have_in = bounded_wait(&prog[order], have_in, min(i + 5, n), spin_limit, trouble);
    have_out = bounded_wait(&prog[order + 2], have_out, i + 18 - kRingGroups, spin_limit, trouble);
    ok = min(have_in >= n ? kForever : have_in - 3, min(have_out, kForever) + kRingGroups - 4);
  };
  const float* take = kHand ? (leads ? nothing : ring[order]) : nullptr;
  const int take_mask = leads ? 0 : kRingGroups / 4 - 1;
  float* give = kHand ? (lane == 0 ? ring[order + 1] : dump + 4 * lane) : nullptr;
  const int give_mask = lane == 0 ? kRingGroups / 4 - 1 : 0;
  int* give_prog = lane == 0 ? &prog[order + 1] : reinterpret_cast<int*>(dump + 4 * lane);
  quad_t pend = {0.0f, 0.0f, 0.0f, 0.0f}, hand = pend;
  float carry = 0.0f;
  // dalpha of the position to the right on the diagonal just done: the next lane's, and for lane 63
  // what was handed over
  auto from_right = [&](float x, float in) {
    if constexpr (!kHand)
      return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130 /* wave_shl:1 */,
                                                        0xf, 0xf, true));
    return wave_shl1(x, in);
  };
  auto cell = [&](float wb, float we, float in, auto with_fold) {
    const float right = from_right(dcol, in);
    const float ne = dcol * wb;
    const float em = right * we;
    dcol = ne + em;
    if constexpr (decltype(with_fold)::value) {
      const float em_b = fold ? em : 0.0f, em_l = fold ? 0.0f : em;
      accB = (accB - ne) - em_b;
      accL = accL - em_l;
    } else {
      accB = accB - ne;
      accL = accL - em;
    }
  };
  // with_fold: some position of this wavefront has the blank as its label.  Real transcripts have
  // none, and the walk without the two selects per cell is shorter (x - 0 is x, so the sums come
  // out the same bits either way).
  auto walk = [&](auto with_fold) __attribute__((always_inline)) {
    // the group that holds the seed: the slot of diagonal `last` receives it, those after it zeros
    Ops first = load(0);
    Ops q[kDepth];
#pragma unroll
    for (int k = 0; k < kDepth; ++k) q[k] = load(1 + k);
    if constexpr (kHand) {
      if (!leads) {
        refresh(0);
        hand = *reinterpret_cast<const quad_t*>(take + 12);
      }
    }
    {
      quad_t out, next = hand;
      if constexpr (kHand) next = *reinterpret_cast<const quad_t*>(take + 16 * (1 & take_mask));
      const float in[4] = {hand[1], hand[2], hand[3], carry};
#pragma unroll
      for (int j = 3; j >= 0; --j) {
        const int s = 4 * g_first + j;
        if (s < last) cell(first.wb[j], first.we[j], in[j], with_fold);  // uniform
        out[j] = s <= last ? dcol : 0.0f;
      }
      d_q.store(lane_o, (unsigned)(g_first - origin) * gbytes, out);
      pend = out;
      carry = hand[0];
      hand = next;
    }
    auto run_group = [&](int i, const Ops& w, const float* take_next, float* give_last, auto tell) {
      quad_t next = hand;
      if constexpr (kHand) {
        *reinterpret_cast<quad_t*>(give_last) = pend;
        asm volatile("" ::: "memory");  // (LDS serves a wavefront's requests in order)
        if constexpr (decltype(tell)::value) prog_store(give_prog, i);
        next = *reinterpret_cast<const quad_t*>(take_next);
        __builtin_amdgcn_sched_barrier(0);  // (asked for ahead of the steps, not among them)
      }
      const float in[4] = {hand[1], hand[2], hand[3], carry};
      quad_t out;
#pragma unroll
      for (int j = 3; j >= 0; --j) {
        cell(w.wb[j], w.we[j], in[j], with_fold);
        out[j] = dcol;
      }
      d_q.store(lane_o, (unsigned)(g_first - i - origin) * gbytes, out);
      pend = out;
      carry = hand[0];
      hand = next;
    };
    // groups i .. i + 3, an aligned block of slots; kWhole: all of them exist, and sixteen more are asked for
    auto four = [&](int i, Ops* w, auto whole) {
      constexpr bool kWhole = decltype(whole)::value;
      const float *tk = nullptr, *tk_next = nullptr;
      float *gv = nullptr, *gv_last = nullptr;
      const int slot = (i + 3) >> 2;
      if constexpr (kHand) {
        tk = take + 16 * (slot & take_mask);
        tk_next = take + 16 * ((slot + 1) & take_mask);
        gv = give + 16 * (slot & give_mask);
        gv_last = give + 16 * ((slot - 1) & give_mask) + 12;
        if (__builtin_expect(i > ok, 0)) refresh(i);
      }
      run_group(i, w[0], tk + 4, gv_last, std::true_type{});
      if (kWhole) w[0] = load(i + kDepth);
      if (kWhole || i + 1 < n) run_group(i + 1, w[1], tk + 8, gv, std::false_type{});
      if (kWhole) w[1] = load(i + 1 + kDepth);
      if (kWhole || i + 2 < n) {
        if constexpr (kHand) {
          if (__builtin_expect(i + 2 > ok, 0)) refresh(i + 2);
        }
        run_group(i + 2, w[2], tk + 12, gv + 4, std::true_type{});
      }
      if (kWhole) w[2] = load(i + 2 + kDepth);
      if (kWhole || i + 3 < n) run_group(i + 3, w[3], tk_next, gv + 8, std::false_type{});
      if (kWhole) w[3] = load(i + 3 + kDepth);
      if constexpr (kHand && kWhole) __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): see alpha
    };
    int i = 1;
    for (; i + kDepth <= n; i += kDepth) {
      const int lowest = max(0, g_first - i - 2 * kDepth);
      if (lowest < origin) move_to(max(0, lowest - span));
#pragma unroll
      for (int k = 0; k < kDepth; k += 4) four(i + k, &q[k], std::true_type{});
    }
#pragma unroll
    for (int k = 0; k < kDepth; k += 4)
      if (i + k < n) four(i + k, &q[k], std::false_type{});
    if constexpr (kHand) {
      *reinterpret_cast<quad_t*>(give + 16 * (((n + 2) >> 2) & give_mask) + 4 * ((n + 2) & 3)) = pend;
      asm volatile("" ::: "memory");
      prog_store(give_prog, n);
    }
  };
  if (__ballot(fold) != 0) walk(std::true_type{});
  else walk(std::false_type{});
  if (u < Ub) {
    p.gB[(size_t)b * d.Ua + u] = accB;
    p.gL[(size_t)b * d.Ua + u] = accL;
  }
}

// ------------------------------------------------------------------ sparse gradient terms
// The blank/label terms of transducer/transducer_cpu.cpp:95-141, scattered into egrads from what
// frame_terms_block (below) leaves: bsum[b][t], the finished value of column `blank` of frame t,
// and emT[b][u][t], the label move's term of every cell.  One thread per frame walks the label
// positions from last to first, which is the order in which the reference subtracts into a row
// of egrads, so repeated labels round the same way; a label position's terms of 256 consecutive
// frames are 1 KB in a row.  pgrads comes from the sums the dalpha kernel kept.  add == 0: the
// terms are stored (the arrays were zero-filled); add != 0: scale[b] (1 when scale is null)
// times the term is added to what the arrays hold.
__global__ __launch_bounds__(256) void sparse_e_kernel(const float* __restrict__ bsum,
                                                       const float* __restrict__ emT,
                                                       float* __restrict__ egrads,
                                                       const int* __restrict__ labels,
                                                       const int* __restrict__ inLen,
                                                       const int* __restrict__ labLen,
                                                       const float* __restrict__ scale, int add,
                                                       Dims d) {
  const int b = blockIdx.y;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Ub == 0 || t >= Tb) return;
  float* __restrict__ row = egrads + ((size_t)b * d.T + t) * d.V;
  const int* __restrict__ lab = labels + (size_t)b * (d.U - 1);
  const float* __restrict__ em = emT + (size_t)b * d.U * d.T + t;
  const float sc = scale ? scale[b] : 1.0f;
  const float blank_total = bsum[(size_t)b * d.T + t];
  // Positions are taken eight at a time, last to first; the terms of the next eight are
  // requested before the current eight are folded in, so the loop runs at the rate of the
  // memory pipe rather than one round trip per label position.
  constexpr int kChunk = 8;
  struct Chunk { float em[kChunk]; };
  auto load_chunk = [&](int uhi) -> Chunk {  // positions uhi, uhi-1, ..., uhi-7 (those >= 0)
    Chunk c;
#pragma unroll
    for (int k = 0; k < kChunk; ++k) c.em[k] = em[(size_t)max(uhi - k, 0) * d.T];
    return c;
  };
  Chunk cur = load_chunk(Ub - 2);  // the last position has no label move
  for (int uhi = Ub - 2; uhi >= 0; uhi -= kChunk) {
    const Chunk nxt = load_chunk(uhi - kChunk);
#pragma unroll
    for (int k = 0; k < kChunk; ++k) {
      const int u = uhi - k;
      if (u >= 0) {
        const int l = clampi(lab[u], 0, d.V - 1);
        // Label columns are updated with no-return hardware adds: nothing waits on them,
        // and since this thread alone touches row t and its requests to one address stay
        // in order, repeated labels still accumulate in the reference's order.  (A label move
        // whose label is the blank is already part of the blank total.)
        if (l != d.blank) unsafeAtomicAdd(&row[l], add ? sc * (-cur.em[k]) : -cur.em[k]);
      }
    }
    cur = nxt;
  }
  if (add) row[d.blank] += sc * blank_total;
  else row[d.blank] = blank_total;
}

// The same terms for a small vocabulary, added (times scale[b]) onto an egrads that holds the
// dense part.  With few columns the hardware adds of sparse_e_kernel all land in a few cache
// lines per row and queue up at L2 (B=8, T=2000, U=100, V=100: 0.08 ms for 1.6 M adds), so
// here a workgroup keeps its frames' rows in LDS (64 x V floats, odd pitch: lane t owns row t, all
// lanes hit column l together, no conflicts).  Each of the four wavefronts takes the columns of one
// remainder by four: it picks their positions out of 64 labels at a time with a ballot and subtracts
// their terms in the reference's order, the next eight requested ahead (a subtraction in LDS waits
// for the one before it, 0.1 us; LDS adds that nothing waits for are no faster: B=8 T=10000 U=401
// V=32 the whole step 2073 us with one wavefront subtracting, 2165 with one adding).  Then all four add
// the rows to egrads, one contiguous piece of memory (B=8 T=2000 U=101 V=100: 20 us with one
// wavefront subtracting, 15 with four; T=10000 U=401 V=32 53 and 45).
// `frames` (at most 64) rows a workgroup; 32 where the LDS of 64 would pass 64 KB (B=16 T=2000 U=101
// V=500: 162 us with hardware adds, 58 so).  Dynamic LDS: frames * (V | 1) floats.
__global__ __launch_bounds__(256) void sparse_e_rows_kernel(const float* __restrict__ bsum,
                                                            const float* __restrict__ emT,
                                                            float* __restrict__ egrads,
                                                            const int* __restrict__ labels,
                                                            const int* __restrict__ inLen,
                                                            const int* __restrict__ labLen,
                                                            const float* __restrict__ scale,
                                                            Dims d, int frames) {
  extern __shared__ float rows[];
  const int b = blockIdx.y, t0 = blockIdx.x * frames, tid = threadIdx.x;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Ub == 0 || t0 >= Tb) return;
  const int pitch = d.V | 1;
  for (int i = tid; i < frames * pitch; i += 256) rows[i] = 0.0f;
  __syncthreads();
  {
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t = min(t0 + lane, Tb - 1);  // lanes past the utterance walk its last frame, unused
    const bool own = lane < frames;
    float* mine = rows + min(lane, frames - 1) * pitch;
    const int* __restrict__ lab = labels + (size_t)b * (d.U - 1);
    const float* __restrict__ em = emT + (size_t)b * d.U * d.T + t;
    if (wave == 0 && own) mine[d.blank] += bsum[(size_t)b * d.T + t];
    constexpr int kBatch = 8;
    struct Batch { float e[kBatch]; int l[kBatch]; };
    // lane k of a look holds the label of position c0 + k (the blank's where there is none)
    auto look = [&](int c0) -> int {
      const int u = c0 + lane, l = clampi(lab[clampi(u, 0, Ub - 2)], 0, d.V - 1);
      return u < Ub - 1 ? l : d.blank;
    };
    const int last = Ub >= 2 ? (Ub - 2) & ~63 : -1;
    int next = last >= 0 ? look(last) : 0;
    for (int c0 = last; c0 >= 0; c0 -= 64) {
      const int here = next;
      next = look(max(c0 - 64, 0));
      unsigned long long m = __ballot(here != d.blank && (here & 3) == wave);
      auto request = [&]() -> Batch {  // the next moves, highest position first; l = -1: no more
        Batch x;
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          const int at = m ? 63 - __builtin_clzll(m) : 0;
          x.l[k] = m ? __builtin_amdgcn_readlane(here, at) : -1;
          x.e[k] = em[(size_t)(c0 + at) * d.T];
          m &= ~(1ull << at);
        }
        return x;
      };
      Batch cur = request();
      while (cur.l[0] >= 0) {
        const Batch nxt = request();
#pragma unroll
        for (int k = 0; k < kBatch; ++k)
          if (cur.l[k] >= 0 && own) mine[cur.l[k]] -= cur.e[k];
        cur = nxt;
      }
    }
  }
  __syncthreads();
  const float sc = scale ? scale[b] : 1.0f;
  const int n = min(frames, Tb - t0) * d.V;
  float* base = egrads + ((size_t)b * d.T + t0) * d.V;
  for (int i0 = tid; i0 < n; i0 += 8 * 256) {
    float have[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) have[k] = base[min(i0 + 256 * k, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int i = i0 + 256 * k;
      if (i < n) {
        const float x = rows[i / d.V * pitch + i % d.V];
        if (x != 0.0f) base[i] = have[k] + sc * x;
      }
    }
  }
}

// What the reference subtracts from egrads besides the dense part, per lattice cell
// (transducer/transducer_cpu.cpp:96,106,138), in the form the dense egrads kernel folds into its
// write-out:
//   bsum[b][t]    the total that lands in column `blank` of frame t: -1 for the last frame (:96),
//                 every blank move's dalpha[t+1,u] wB[t,u], and the label moves whose label is the
//                 blank -- the value sparse_e_kernel would leave in that column;
//   emT[b][u][t]  the label move's dalpha[t,u+1] wE[t,u] of every cell ([B][U][T]: the kernel that
//                 folds them in reads one label position's frames in a row).
// One lane per frame subtracts its frame's terms in the reference's order, label positions last
// to first.  The operands come through LDS: for eight label positions at a time a wavefront copies the
// groups of anti-diagonals its 64 frames meet there -- 128 contiguous bytes a group and plane --
// with 16-byte loads, requested one round ahead, and each lane then picks its own cells (read
// straight from the planes, the 64 frames would touch 17 cache lines per load).
// kShared: a workgroup takes 64 frames and 32 label positions a round, eight to a wavefront; the
// wavefronts form the products side by side and leave those of the blank moves in LDS, where the
// first one subtracts them in order.  Without: a wavefront takes 64 frames and all their positions by
// itself, without barriers.  The latter moves more bytes at a time where there are workgroups enough
// (us for post_beta_kernel at B=32 T=2000 U=101 47 against 65, B=8 T=10000 U=401 249 against 290), and
// is thirteen round trips one after the other where there are not (B=8 T=2000 U=101 30 against
// 21, B=32 T=400 U=102 31 against 23; B=16 T=2000 U=101, 128
// workgroups of the other kind, 34 against 37): shared up to 96 of them.
constexpr int kBsFrames = 64, kBsPos = 8;
constexpr int kBsGroups = (kBsFrames + kBsPos + 3) / 4 + 1;  // groups of four anti-diagonals a chunk meets
// floats per staged group; the pitches put the 16-byte pieces of consecutive groups on different banks
constexpr int kBsPitch = 4 * kBsPos + 4;         // wB, wE: eight positions
constexpr int kBsPitchD = 4 * (kBsPos + 1) + 8;  // dalpha: nine (a cell's label move enters position u+1)
constexpr int kBsPieces = (kBsGroups * kBsPos + 63) / 64;         // 16-byte pieces a lane copies per plane
constexpr int kBsPiecesD = (kBsGroups * (kBsPos + 1) + 63) / 64;
constexpr int kBsWave = kBsGroups * (2 * kBsPitch + kBsPitchD);   // floats of LDS a wavefront stages in
constexpr int kBsSums = 2 * 4 * kBsPos * kBsFrames;  // floats: the products of a round, stay and label moves
constexpr int kBsAll = 4 * kBsWave + kBsSums;
constexpr int post_beta_lds(bool shared) {  // floats: either kind of block
  return std::max(shared ? kBsAll : 4 * kBsWave, 64 * 65);
}
template <bool kShared>
__device__ __forceinline__ void frame_terms_block(const Planes& p, float* __restrict__ bsum,
                                                  float* __restrict__ emT,
                                                  const int* __restrict__ labels,
                                                  const int* __restrict__ inLen,
                                                  const int* __restrict__ labLen, const Dims& d,
                                                  int bx, int b, float* __restrict__ lds) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int t0 = (kShared ? bx : 4 * bx + wave) * kBsFrames, t = t0 + lane;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Ub == 0 || t0 >= Tb) return;  // the whole workgroup (wavefront)
  const bool active = t < Tb;
  const int* __restrict__ lab = labels + (size_t)b * (d.U - 1);
  const float* __restrict__ dS = p.dS;
  const float* __restrict__ wB = p.wB;
  const float* __restrict__ wE = p.wE;
  float* stW = lds + wave * kBsWave;        // wB of anti-diagonal groups gbase ..
  float* stE = stW + kBsGroups * kBsPitch;  // wE
  float* stD = stE + kBsGroups * kBsPitch;  // dalpha
  float* stays = lds + 4 * kBsWave;                 // [position of the round][frame]
  float* emits = stays + 4 * kBsPos * kBsFrames;    // where the label is the blank
  const size_t plane_b = (size_t)b * d.Ua * d.Dp;
  const int ngroups_plane = d.Dp >> 2;
  const bool has_stay = t + 1 < Tb;
  float acc = (t == Tb - 1) ? -1.0f : 0.0f;
  // cell (t,u) reads the weights on anti-diagonal t+u and dalpha on t+u+1: positions ua .. ua+7
  // of the wavefront's frames meet groups (t0 + ua) / 4 .. (t0 + ua + 64 + 7) / 4
  struct Pieces { float4 w[kBsPieces], e[kBsPieces], d[kBsPiecesD]; };
  const float4 zero4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  auto request = [&](int ua) -> Pieces {
    Pieces r;
    const int gbase = (t0 + max(ua, 0)) >> 2;
#pragma unroll
    for (int i = 0; i < kBsPieces; ++i) {
      const int f = 64 * i + lane, g = gbase + f / kBsPos, ul = f % kBsPos;
      r.w[i] = zero4;
      r.e[i] = zero4;
      if (ua >= 0 && f < kBsGroups * kBsPos && g < ngroups_plane) {  // (ua + ul < Ua: a multiple of 64)
        const size_t o = plane_b + ((size_t)g * d.Ua + ua + ul) * 4;
        r.w[i] = *reinterpret_cast<const float4*>(wB + o);
        r.e[i] = *reinterpret_cast<const float4*>(wE + o);
      }
    }
#pragma unroll
    for (int i = 0; i < kBsPiecesD; ++i) {
      const int f = 64 * i + lane, g = gbase + f / (kBsPos + 1), ul = f % (kBsPos + 1);
      r.d[i] = zero4;
      // (position ua + 8 may be Ua itself: the address is then position 0 of the next group,
      // inside the plane since g + 1 groups exist, and no cell uses the value)
      if (ua >= 0 && f < kBsGroups * (kBsPos + 1) && g + 1 < ngroups_plane)
        r.d[i] = *reinterpret_cast<const float4*>(dS + plane_b + ((size_t)g * d.Ua + ua + ul) * 4);
    }
    return r;
  };
  // round by round from the last positions down; this wavefront's eight may lie past the
  // utterance's last one (their cells hold zeros or nothing and are not looked at)
  constexpr int kRound = (kShared ? 4 : 1) * kBsPos;
  const int u_off = kShared ? kBsPos * wave : 0;
  const int first = (Ub - 1) & ~(kRound - 1);
  Pieces cur = request(first + u_off);
  for (int u_round = first; u_round >= 0; u_round -= kRound) {
    const int ua = u_round + u_off, gbase = (t0 + ua) >> 2;
    // (LDS serves a wavefront's accesses in order; the fences only hold the compiler to it)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < kBsPieces; ++i) {
      const int f = 64 * i + lane;
      if (f < kBsGroups * kBsPos) {
        *reinterpret_cast<float4*>(stW + (f / kBsPos) * kBsPitch + 4 * (f % kBsPos)) = cur.w[i];
        *reinterpret_cast<float4*>(stE + (f / kBsPos) * kBsPitch + 4 * (f % kBsPos)) = cur.e[i];
      }
    }
#pragma unroll
    for (int i = 0; i < kBsPiecesD; ++i) {
      const int f = 64 * i + lane;
      if (f < kBsGroups * (kBsPos + 1))
        *reinterpret_cast<float4*>(stD + (f / (kBsPos + 1)) * kBsPitchD + 4 * (f % (kBsPos + 1))) =
            cur.d[i];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    cur = request(ua - kRound);
    if (active) {
#pragma unroll
      for (int k = kBsPos - 1; k >= 0; --k) {
        const int u = ua + k;
        if (u < Ub) {  // uniform
          const int dd = t + u;
          const int here = ((dd >> 2) - gbase) * kBsPitch + 4 * k + (dd & 3);
          const int next = (((dd + 1) >> 2) - gbase) * kBsPitchD + 4 * k + ((dd + 1) & 3);
          const float ne = stD[next] * stW[here];      // dalpha[t+1,u] wB[t,u]
          const float em = stD[next + 4] * stE[here];  // dalpha[t,u+1] wE[t,u]
          const bool has_label = u + 1 < Ub;
          if constexpr (kShared) {
            stays[(u_off + k) * kBsFrames + lane] = has_stay ? ne : 0.0f;
            emits[(u_off + k) * kBsFrames + lane] = em;
          } else {
            acc -= has_stay ? ne : 0.0f;
            if (has_label && clampi(lab[u], 0, d.V - 1) == d.blank) acc -= em;
          }
          emT[((size_t)b * d.U + u) * d.T + t] = has_label ? em : 0.0f;
        }
      }
    }
    if constexpr (kShared) {
      __syncthreads();
      if (wave == 0) {
#pragma unroll 8
        for (int k = min(kRound, Ub - u_round) - 1; k >= 0; --k) {
          acc -= stays[k * kBsFrames + lane];
          const int u = u_round + k;
          if (u + 1 < Ub && clampi(lab[u], 0, d.V - 1) == d.blank)
            acc -= emits[k * kBsFrames + lane];
        }
      }
      __syncthreads();
    }
  }
  if (active && (!kShared || wave == 0)) bsum[(size_t)b * d.T + t] = acc;
}

// W from the skewed planes the lattice kernels leave behind (dalpha and LN): no un-skewed copy of
// dalpha is needed first.  A block takes 64 label positions x 64 anti-diagonals (16 groups of
// four: 1 KB of contiguous memory a group and plane, read with 16-byte loads), forms W of those
// cells, and writes them to both orientations through an LDS tile.  Its frames are the 127
// t = dd - u; the blocks (64 by, 64 bx) over all anti-diagonals below Tw + Up tile the planes.
// Same arithmetic per cell as wplanes_kernel, same bits.
__device__ __forceinline__ void wplanes_skewed_block(
    const float* __restrict__ dS, const float* __restrict__ lnS, const float* __restrict__ mE,
    const float* __restrict__ mP, float* __restrict__ Wn, float* __restrict__ Wt,
    const int* __restrict__ inLen, const int* __restrict__ labLen, const Dims& d, int Up, int Tw,
    float (*tile)[65], int bx, int by, int b) {
  const int dd0 = bx * 64, u0 = by * 64;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  const size_t plane_b = (size_t)b * d.Ua * d.Dp;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int f = k * 256 + threadIdx.x, gl = f >> 6, ul = f & 63;
    const int u = u0 + ul, g = (dd0 >> 2) + gl;
    const int tq = 4 * g - u;  // frame of the group's first anti-diagonal
    float w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (u < Ub && tq + 3 >= 0 && tq < Tb) {  // (so 4g < T + U: the group lies inside the plane)
      const size_t o = plane_b + ((size_t)g * d.Ua + u) * 4;
      const float4 d4 = *reinterpret_cast<const float4*>(dS + o);
      const float4 l4 = *reinterpret_cast<const float4*>(lnS + o);
      const float mp = mP[(size_t)b * d.U + u];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = tq + j;
        if (t >= 0 && t < Tb) {
          const float me = mE[(size_t)b * d.T + t];
          w[j] = f4get(d4, j) * expf((me + mp) - f4get(l4, j)) * frame_exp_correction(me);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) tile[ul][4 * gl + j] = w[j];  // [label position][anti-diagonal]
  }
  __syncthreads();
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 16; ++i) {  // rows of Wt: one label position, 64 consecutive frames
    const int ul = ty + 4 * i, u = u0 + ul, t = dd0 + tx - u;
    if (t >= 0 && t < Tw && u < Up) Wt[((size_t)b * Up + u) * Tw + t] = tile[ul][tx];
  }
  for (int i = 0; i < 32; ++i) {  // rows of Wn: one frame, the label positions it has in the tile
    const int r = ty + 4 * i;     // frame dd0 - u0 - 63 + r meets position u0 + tx on dd0 + tx + r - 63
    const int t = dd0 - u0 - 63 + r, u = u0 + tx, c = tx + r - 63;
    if (c >= 0 && c < 64 && t >= 0 && t < Tw && u < Up)
      Wn[((size_t)b * Tw + t) * Up + u] = tile[tx][c];
  }
}

// W of 64 frames x 64 label positions as bf16 pieces, in the two slab images the fused gradient
// kernel copies into LDS as they are (WImages).  Same arithmetic per cell as above.
__device__ __forceinline__ void wimages_block(
    const float* __restrict__ dS, const float* __restrict__ lnS, const float* __restrict__ mE,
    const float* __restrict__ mP, const int* __restrict__ inLen, const int* __restrict__ labLen,
    const Dims& d, int Tw, float (*tile)[65], int bx, int by, int b, const WImages& img) {
  const int t0 = bx * 64, u0 = by * 64;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int u = u0 + ty + 4 * i, t = t0 + tx;
    float w = 0.0f;
    if (t < Tb && u < Ub) {
      const size_t o = plane_at(d, b, u, t + u);
      const float me = mE[(size_t)b * d.T + t];
      w = dS[o] * expf((me + mP[(size_t)b * d.U + u]) - lnS[o]) * frame_exp_correction(me);
    }
    tile[ty + 4 * i][tx] = w;  // [label position][frame]
  }
  __syncthreads();
  const int ntile = Tw >> 5;
  // frames x label positions (the egrads operand): pairs of neighbouring label positions
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int id = k * 256 + threadIdx.x, tl = id >> 5, j = id & 31;
    const int u = u0 + 2 * j;
    if (u < WImages::kCols) {
      unsigned ph, pm, pl;
      split_pair(tile[2 * j][tl], tile[2 * j + 1][tl], ph, pm, pl);
      unsigned* dst = img.e + ((size_t)b * ntile + ((t0 + tl) >> 5)) * (3 * WImages::kEPlane) +
                      ((t0 + tl) & 31) * (WImages::kCols / 2) + (u >> 1);
      dst[0] = ph;
      dst[WImages::kEPlane] = pm;
      dst[2 * WImages::kEPlane] = pl;
    }
  }
  // label positions x frames (the pgrads operand), the frames of a slab in the order the fused
  // kernel feeds them to the matrix instruction: slot = frame with bits 2 and 3 swapped (its own
  // inverse; pairs of neighbouring frames stay pairs)
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int id = k * 256 + threadIdx.x, ul = id >> 5, q = id & 31;
    const int sel = q >> 4, slot = 2 * (q & 15);
    const int f = (slot & 16) | ((slot & 4) << 1) | ((slot & 8) >> 1) | (slot & 2);
    unsigned ph, pm, pl;
    split_pair(tile[ul][32 * sel + f], tile[ul][32 * sel + f + 1], ph, pm, pl);
    unsigned* dst = img.p + ((size_t)b * ntile + (t0 >> 5) + sel) * (3 * WImages::kPPlane) +
                    (u0 + ul) * 16 + (slot >> 1);
    dst[0] = ph;
    dst[WImages::kPPlane] = pm;
    dst[2 * WImages::kPPlane] = pl;
  }
}


// W planes and per-frame blank totals in one launch: both only need the finished dalpha plane and
// neither needs the other, so the blocks of the second fill the device beside the first's
// instead of waiting behind a kernel boundary.  The last nw blocks form W (tile bx, by of
// utterance b; with `img` the tiles are 64 frames x 64 label positions and go to the slab images
// instead), the blocks before them the per-frame terms bsum and emT (bsum == nullptr: none).
template <bool kShared>
__global__ __launch_bounds__(256) void post_beta_kernel(Planes p, const float* __restrict__ mE,
                                                        const float* __restrict__ mP,
                                                        float* __restrict__ Wn,
                                                        float* __restrict__ Wt,
                                                        float* __restrict__ bsum,
                                                        float* __restrict__ emT,
                                                        const int* __restrict__ labels,
                                                        const int* __restrict__ inLen,
                                                        const int* __restrict__ labLen, Dims d,
                                                        int Up, int Tw, int wx, int wy, int nw,
                                                        int sx, WImages img) {
  __shared__ __attribute__((aligned(16))) float lds[post_beta_lds(kShared)];
  float (*tile)[65] = reinterpret_cast<float (*)[65]>(lds);
  // the per-frame blocks come first in the grid: each runs longer than a W tile, and started
  // last they would be the kernel's tail
  const int ns = gridDim.x - nw;
  if ((int)blockIdx.x >= ns) {
    const int n = blockIdx.x - ns;
    const int b = n / (wx * wy), r = n - b * (wx * wy);
    if (img.e)
      wimages_block(p.dS, p.lnS, mE, mP, inLen, labLen, d, Tw, tile, r % wx, r / wx, b, img);
    else
      wplanes_skewed_block(p.dS, p.lnS, mE, mP, Wn, Wt, inLen, labLen, d, Up, Tw, tile, r % wx,
                           r / wx, b);
  } else {
    const int m = blockIdx.x;
    frame_terms_block<kShared>(p, bsum, emT, labels, inLen, labLen, d, m % sx, m / sx, lds);
  }
}

__global__ __launch_bounds__(256) void sparse_p_kernel(Planes p, float* __restrict__ pgrads,
                                                       const int* __restrict__ labels,
                                                       const int* __restrict__ inLen,
                                                       const int* __restrict__ labLen,
                                                       const float* __restrict__ scale, int add,
                                                       Dims d) {
  const int b = blockIdx.y;
  const int u = blockIdx.x * 256 + threadIdx.x;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Tb == 0 || u >= Ub) return;
  float* row = pgrads + ((size_t)b * d.U + u) * d.V;
  const float gb = p.gB[(size_t)b * d.Ua + u], gl = p.gL[(size_t)b * d.Ua + u];
  const bool has_label = u + 1 < Ub;
  const int l = has_label ? label_at(labels, d, b, u) : d.blank;
  if (add) {
    const float sc = scale ? scale[b] : 1.0f;
    row[d.blank] += sc * gb;
    if (has_label && l != d.blank) row[l] += sc * gl;
  } else {
    row[d.blank] = gb;
    if (has_label && l != d.blank) row[l] = gl;
  }
}

// ------------------------------------------------------------------ max-plus table
// best[t,u] = max over v != blank of E[t,v]+P[u,v], arg = lowest such v
// (transducer/transducer_cpu.cpp:158-171).  Pure vector-ALU work (max-plus has no matrix form),
// so the kernel is laid out to spend its instructions on the add and the max:
//   * a workgroup of 8 wavefronts owns 128 frames x 64 label positions; a wavefront owns 8 label
//     positions, a lane two frames (lane, lane+64): 16 cells per lane (two workgroups share a
//     CU; with 16 wavefronts and 128 label positions per workgroup only one fits, and the
//     wavefronts idling past a short utterance's last label cost a whole slot);
//   * E and P stream through LDS in chunks of 32 columns (double-buffered, one barrier per
//     chunk); E is staged with the blank column, columns past V and frames past the utterance at
//     -inf; a lane reads its two rows of E 16 bytes at a time (row pitch 36 floats:
//     conflict-free), and the P values of the wavefront's 8 rows, which are the same for all its
//     lanes, with broadcast reads (one address per wavefront).  Scalar loads would bring them in
//     as scalar operands, but they return out of order, so only one row could be in flight and
//     the L2 latency of every row showed: measured 5.5 ms against 6.8 ms for a 4x4-cells
//     LDS-tiled first version;
//   * the running maximum is exact and order-free; per chunk a cell only notes whether the
//     chunk raised it, and the index is recovered afterwards by rescanning the first chunk that
//     reached the maximum.
// Wavefronts whose label positions lie past the utterance only help staging.
constexpr int kMpT = 128, kMpK = 32, kMpPitch = 36, kMpRows = 8;
constexpr int kMpWaves = 8, kMpU = kMpWaves * kMpRows, kMpThreads = 64 * kMpWaves;
// As many ranges of columns as bring the grid to kMpWanted workgroups (two fit a CU at a time, and
// the padded tiles of short utterances end at once), each range at least kMpMinChunks chunks long.
// The table of B=16 T=1500 U=81 V=2001 (384 tiles): 495 us before ranges, 344 with two, 359 with five;
// B=8 T=2000 U=101 V=1000 (256): 191, 146 with four, 158 with eight; B=32 of the same (1024): 641,
// 546 with one, 539 with two.
constexpr long kMpWanted = 1024, kMpMinChunks = 2, kMpMaxParts = 16;
constexpr int kMpEPasses = kMpT * (kMpK / 4) / kMpThreads;  // 16-byte pieces of the E chunk per thread

// The lowest column of a chunk at which a cell reaches its maximum `want`: the chunk's 32 columns
// of the cell's two rows come in as sixteen 16-byte loads, all requested before the first is
// looked at, and the sums are compared in registers.  (Looked up column by column, the way the
// reference scans, this was two dependent loads and a wait per column and cell: five hundred
// memory round trips in a row at the end of every wavefront.)
template <bool kVec, typename TIO>
__device__ inline int chunk_argmax(const TIO* __restrict__ e, const TIO* __restrict__ q, int chunk,
                                   float want, const Dims& d) {
  const int v0 = max(chunk, 0) * kMpK;
  float4 ev[kMpK / 4], pv[kMpK / 4];
#pragma unroll
  for (int g = 0; g < kMpK / 4; ++g) {
    const int v = v0 + 4 * g;
    // (kVec: a group of four is inside the row or past it as a whole, and one past it is
    // never looked at, so the clamped start only keeps the load inside the array)
    ev[g] = kVec ? load4(e + min(v, d.V - 4)) : load4_any(e, min(v, d.V - 1), d.V);
    pv[g] = kVec ? load4(q + min(v, d.V - 4)) : load4_any(q, min(v, d.V - 1), d.V);
  }
  int at = 0;  // :160 the scan starts from index 0 and keeps it if nothing beats -inf
  if (chunk >= 0) {
    // from the last column down, so that the lowest match is what remains
#pragma unroll
    for (int g = kMpK / 4 - 1; g >= 0; --g) {
      const float sum[4] = {ev[g].x + pv[g].x, ev[g].y + pv[g].y, ev[g].z + pv[g].z,
                            ev[g].w + pv[g].w};
#pragma unroll
      for (int j = 3; j >= 0; --j) {
        const int v = v0 + 4 * g + j;
        if (v < d.V && v != d.blank && sum[j] == want) at = v;
      }
    }
  }
  return at;
}

// kParts: a workgroup takes one of parts.n ranges of columns and leaves its cells' maxima and
// chunks in `parts` (maxplus_index_kernel goes on from there); without, it takes all columns and
// finishes its cells: that form redoes single tiles after the list pass.  Each workgroup walks its
// columns alone, so with one range few tiles are a long walk on a few CUs: the table of B=1 T=500
// U=41 V=1000 (four tiles) 124 -> 31 us with sixteen ranges.
// kVec: V is a multiple of 4, so four consecutive elements never straddle a row's end and every
// group of four is naturally aligned (16 bytes in fp32, 8 in bf16).
template <bool kVec, bool kParts, typename TIO>
__global__ __launch_bounds__(kMpThreads) void maxplus_kernel(const TIO* __restrict__ E,
                                                       const TIO* __restrict__ P,
                                                       const int* __restrict__ inLen,
                                                       const int* __restrict__ labLen,
                                                       float* __restrict__ best,
                                                       int* __restrict__ arg, Dims d,
                                                       const int* __restrict__ tile_fail,
                                                       const int* __restrict__ lists_on,
                                                       int fail_limit, MaxplusParts parts) {
  __shared__ __attribute__((aligned(16))) float Es[2][kMpT * kMpPitch];
  __shared__ __attribute__((aligned(16))) float Ps[2][kMpU * kMpK];
  const int part = kParts ? (int)(blockIdx.z % (unsigned)parts.n) : 0;
  const int b = kParts ? (int)(blockIdx.z / (unsigned)parts.n) : (int)blockIdx.z;
  const int t0 = blockIdx.x * kMpT, u0 = blockIdx.y * kMpU;
  // after the list pass (if it went past its sample): only the tiles in which too many cells
  // failed its test are redone
  if (tile_fail && lists_on[0] != 0 &&
      tile_fail[((size_t)b * gridDim.x + blockIdx.x) * gridDim.y + blockIdx.y] <= fail_limit)
    return;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (t0 >= Tb || u0 >= Ub) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const TIO* Eb = E + (size_t)b * d.T * d.V;
  const TIO* Pb = P + (size_t)b * d.U * d.V;
  const int ur0 = u0 + wave * kMpRows;  // first label position of this wavefront
  const bool active = ur0 < Ub;

  // staging role: thread -> row srow of the P tile and rows srow + (kMpThreads/8) * i of the E
  // tile, four columns from sc4
  const int srow = tid >> 3, sc4 = (tid & 7) * 4;
  const TIO* esrc[kMpEPasses];
  bool erow_ok[kMpEPasses];
#pragma unroll
  for (int i = 0; i < kMpEPasses; ++i) {
    const int t = t0 + srow + (kMpThreads / 8) * i;
    erow_ok[i] = t < Tb;
    esrc[i] = Eb + (size_t)min(t, Tb - 1) * d.V;
  }
  const TIO* psrc = Pb + (size_t)min(u0 + srow, Ub - 1) * d.V;  // rows past the utterance are
                                                                  // computed and dropped
  // the raw values are requested before a chunk's arithmetic and stored after it, so the wait
  // for them falls behind the arithmetic
  auto fetch = [&](const TIO* src, int k) -> float4 {
    const int v = k * kMpK + sc4;
    float4 x;
    if (kVec) {  // columns past V are re-read from the row's last four (E: masked below; P: any
                 // finite value will do there, E is -inf)
      x = load4(src + min(v, d.V - 4));
    } else {  // one wide load at the element's own alignment, one by one at the row's end
      x = load4_any(src, min(v, d.V - 1), d.V);
    }
    return x;
  };
  struct Staged {
    float4 e[kMpEPasses], p;
  };
  auto fetch_all = [&](int k) -> Staged {
    Staged r;
#pragma unroll
    for (int i = 0; i < kMpEPasses; ++i) r.e[i] = fetch(esrc[i], k);
    r.p = fetch(psrc, k);
    return r;
  };
  auto stash = [&](int buf, int k, const Staged& r) {
    const int v = k * kMpK + sc4;
#pragma unroll
    for (int i = 0; i < kMpEPasses; ++i) {
      float4 x = r.e[i];
      x.x = (erow_ok[i] && v < d.V && v != d.blank) ? x.x : kNegInf;
      x.y = (erow_ok[i] && v + 1 < d.V && v + 1 != d.blank) ? x.y : kNegInf;
      x.z = (erow_ok[i] && v + 2 < d.V && v + 2 != d.blank) ? x.z : kNegInf;
      x.w = (erow_ok[i] && v + 3 < d.V && v + 3 != d.blank) ? x.w : kNegInf;
      *reinterpret_cast<float4*>(&Es[buf][(srow + (kMpThreads / 8) * i) * kMpPitch + sc4]) = x;
    }
    *reinterpret_cast<float4*>(&Ps[buf][srow * kMpK + sc4]) = r.p;
  };

  float top[2][kMpRows];
  int chunk[2][kMpRows];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < kMpRows; ++r) { top[i][r] = kNegInf; chunk[i][r] = -1; }

  const int all = (d.V + kMpK - 1) / kMpK;
  const int first = kParts ? (int)((long)all * part / parts.n) : 0;
  const int nchunks = kParts ? (int)((long)all * (part + 1) / parts.n) : all;
  int cur = 0;
  stash(0, first, fetch_all(first));
  __syncthreads();
  for (int k = first; k < nchunks; ++k) {
    const int kn = min(k + 1, nchunks - 1);  // the last chunk re-reads its own
    const Staged nxt = fetch_all(kn);
    if (active) {
      float cm[2][kMpRows];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < kMpRows; ++r) cm[i][r] = kNegInf;
#pragma unroll
      for (int sub = 0; sub < kMpK / 8; ++sub) {
        float e[2][8];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float4 lo =
              *reinterpret_cast<const float4*>(&Es[cur][(lane + 64 * i) * kMpPitch + sub * 8]);
          const float4 hi =
              *reinterpret_cast<const float4*>(&Es[cur][(lane + 64 * i) * kMpPitch + sub * 8 + 4]);
          e[i][0] = lo.x; e[i][1] = lo.y; e[i][2] = lo.z; e[i][3] = lo.w;
          e[i][4] = hi.x; e[i][5] = hi.y; e[i][6] = hi.z; e[i][7] = hi.w;
        }
        const float* pw = &Ps[cur][wave * kMpRows * kMpK + sub * 8];
#pragma unroll
        for (int r = 0; r < kMpRows; ++r) {
          const float4 plo = *reinterpret_cast<const float4*>(pw + r * kMpK);
          const float4 phi = *reinterpret_cast<const float4*>(pw + r * kMpK + 4);
          const float pv[8] = {plo.x, plo.y, plo.z, plo.w, phi.x, phi.y, phi.z, phi.w};
#pragma unroll
          for (int c = 0; c < 8; c += 2) {
            cm[0][r] = fmaxf(fmaxf(cm[0][r], e[0][c] + pv[c]), e[0][c + 1] + pv[c + 1]);
            cm[1][r] = fmaxf(fmaxf(cm[1][r], e[1][c] + pv[c]), e[1][c + 1] + pv[c + 1]);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < kMpRows; ++r)
          if (cm[i][r] > top[i][r]) { top[i][r] = cm[i][r]; chunk[i][r] = k; }
    }
    stash(cur ^ 1, kn, nxt);
    __syncthreads();
    cur ^= 1;
  }
  if (!active) return;
  if constexpr (kParts) {  // maxplus_index_kernel compares the parts and looks the column up
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < kMpRows; ++r) {
        const int t = t0 + lane + 64 * i, u = ur0 + r;
        if (t < Tb && u < Ub) {
          const size_t o = parts.n > 1 ? (((size_t)part * d.B + b) * d.U + u) * d.T + t
                                       : plane_at(d, b, u, t + u);
          parts.top[o] = top[i][r];
          parts.chunk[o] = chunk[i][r];
        }
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < kMpRows; ++r) {
      const int t = t0 + lane + 64 * i, u = ur0 + r;
      // every lane goes through the loads with clamped rows; only cells of the utterance are written
      const int at = chunk_argmax<kVec>(Eb + (size_t)min(t, Tb - 1) * d.V,
                                        Pb + (size_t)min(u, Ub - 1) * d.V, chunk[i][r], top[i][r], d);
      if (t < Tb && u < Ub) {
        // straight into the skewed planes the lattice walk reads
        const size_t o = plane_at(d, b, u, t + u);
        best[o] = top[i][r];
        arg[o] = at;
      }
    }
}

// The table from what maxplus_kernel<.., true> left: the first range of columns that holds the
// largest maximum, then the lowest column of its chunk that reaches it.  A wavefront takes 64 frames
// of one label position.  Eight lanes look at a cell, four columns each, so that a load brings in
// eight cells' 128 contiguous bytes: with one lane to a cell every load touched 64 cache lines,
// and the look-up took as long as the maxima (365 of 668 us at B=32 T=2000 U=101 V=1000, as it
// did at the end of maxplus_kernel itself).
template <bool kVec, typename TIO>
__global__ __launch_bounds__(256) void maxplus_index_kernel(const TIO* __restrict__ E,
                                                            const TIO* __restrict__ P,
                                                            const int* __restrict__ inLen,
                                                            const int* __restrict__ labLen,
                                                            float* best, int* arg, Dims d,
                                                            MaxplusParts parts) {
  const int b = blockIdx.z, lane = threadIdx.x & 63, t0 = blockIdx.x * 64;
  const int u = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (t0 >= Tb || u >= Ub) return;  // uniform
  const int t = t0 + lane, tc = min(t, Tb - 1);
  const size_t w = plane_at(d, b, u, tc + u);
  float top;
  int chunk;
  if (parts.n > 1) {
    const size_t stride = (size_t)d.B * d.U * d.T;
    const size_t o = ((size_t)b * d.U + u) * d.T + tc;
    top = parts.top[o];
    chunk = parts.chunk[o];
    for (int s = 1; s < parts.n; ++s) {
      const float x = parts.top[s * stride + o];
      const int c = parts.chunk[s * stride + o];
      if (x > top) { top = x; chunk = c; }
    }
  } else {
    top = parts.top[w];
    chunk = parts.chunk[w];
  }
  const TIO* Eb = E + (size_t)b * d.T * d.V;
  const TIO* q = P + ((size_t)b * d.U + u) * d.V;
  float4 ev[8], pv[8];
  int v0[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {  // cells 8 i .. 8 i + 7
    const int cell = 8 * i + (lane >> 3);
    v0[i] = max(__shfl(chunk, cell), 0) * kMpK + 4 * (lane & 7);
    const TIO* e = Eb + (size_t)min(t0 + cell, Tb - 1) * d.V;
    // columns past V: see chunk_argmax
    ev[i] = kVec ? load4(e + min(v0[i], d.V - 4)) : load4_any(e, min(v0[i], d.V - 1), d.V);
    pv[i] = kVec ? load4(q + min(v0[i], d.V - 4)) : load4_any(q, min(v0[i], d.V - 1), d.V);
  }
  int at = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float want = __shfl(top, 8 * i + (lane >> 3));
    const float sum[4] = {ev[i].x + pv[i].x, ev[i].y + pv[i].y, ev[i].z + pv[i].z,
                          ev[i].w + pv[i].w};
    int found = 0x7fffffff;
#pragma unroll
    for (int j = 3; j >= 0; --j) {
      const int v = v0[i] + j;
      if (v < d.V && v != d.blank && sum[j] == want) found = v;
    }
    found = min(found, __shfl_xor(found, 1));
    found = min(found, __shfl_xor(found, 2));
    found = min(found, __shfl_xor(found, 4));
    const int got = __shfl(found, 8 * (lane & 7));
    at = (lane >> 3) == i ? got : at;
  }
  if (t >= Tb) return;
  best[w] = top;
  arg[w] = chunk < 0 ? 0 : at;  // :160 the scan starts from index 0 and keeps it
}

// ------------------------------------------------------------------ viterbi
// transducer/transducer_cpu.cpp:145-222.  Scores walk the lattice like alpha with
// max in place of log-sum-exp: no transcendental anywhere, so given the same LN the path is
// bit-exact.  Association: blank move ((s + e) + p) - LN (:192-195), label move
// (s + best) - LN (:197-199); "emit > stay" takes the label, ties go to blank (:200-206).
// The decision of every cell is one bit; each step's 64-lane ballot goes to `bits`
// (LDS when it fits, else global), and lane 0 walks them backwards at the end (:208-219).
// C cells per lane, W wavefronts (the label positions dealt to them as in alpha_kernel, with
// the same hand-over of the boundary score).
// The decision of a cell is one bit.  A lane keeps the bits of its own cells, 32 steps to a
// word, and stores a word when it is full: column u of the table `cols` holds the decisions of
// label position u over all steps.  The backtrace then does not walk the ~T+U moves one by one:
// at position u, reached at step s, the move that entered u is the highest set bit at or below
// s in column u (everything above it is blank moves), found with one or two word reads and a
// count-leading-zeros; U-1 such searches, by one lane, and the labels are fetched by all lanes
// afterwards.
// Dynamic LDS: one int per label position (steps at which labels were taken), the hand-over
// array (W > 1), the columns (kLdsBits; else they live in global memory).
template <int C, int W, bool kLdsBits, bool kMulti>
__global__ __launch_bounds__(64 * W) void viterbi_kernel(Planes p, const float* __restrict__ bestS,
                                                         const float* __restrict__ argS,
                                                         const int* __restrict__ inLen,
                                                         const int* __restrict__ labLen,
                                                         unsigned* __restrict__ gcols,
                                                         int* __restrict__ labels_out, Dims d,
                                                         int hand_stride, int nw, int spin_limit,
                                                         int* __restrict__ trouble, int u_base,
                                                         const float* __restrict__ ghin,
                                                         float* __restrict__ ghout,
                                                         int traces) {
  extern __shared__ __attribute__((aligned(16))) int dyn[];
  __shared__ int done[W];  // steps a wavefront has published
  __shared__ __attribute__((aligned(16))) float nothing[4];
  const int b = blockIdx.x;
  const int lane = threadIdx.x & 63, tidx = threadIdx.x;
  const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Tb == 0 || Ub == 0) return;  // :152-154
  // A label axis longer than 64 C W positions is walked block by block, lowest first, as in
  // alpha_kernel (u_base, ghin, ghout); the decision columns then live in global memory and the
  // launch of the highest block (traces != 0) follows the path back through all of them.
  const bool walks = u_base < Ub;
  if (!walks && !traces) return;
  const int nsteps = Tb + Ub - 1;
  const int ngroups = (nsteps + 3) >> 2;
  int* taken = dyn;                             // [U rounded up to 4]
  float* hand = reinterpret_cast<float*>(dyn + ((d.U + 3) & ~3));  // [W-1][hand_stride]
  unsigned* cols = kLdsBits
      ? reinterpret_cast<unsigned*>(hand + (W - 1) * hand_stride)     // [64 C W][nw]
      : gcols + (size_t)b * d.Ua * nw;                                // [Ua][nw]
  const float* gin = (kMulti && ghin) ? ghin + (size_t)b * hand_stride : nullptr;
  float* gout = (kMulti && ghout && walks) ? ghout + (size_t)b * hand_stride : nullptr;
  if (kMulti && gout && tidx == 0) gout[0] = kNegInf;  // nothing enters step 0
  if (W > 1) {
    if (tidx < W) done[tidx] = 0;
    if (tidx < W - 1) hand[tidx * hand_stride] = kNegInf;  // nothing enters step 0
    if (tidx < 4) nothing[tidx] = kNegInf;
  }
  for (int u = tidx; u < Ub; u += 64 * W) taken[u] = -1;
  __syncthreads();
  float* hand_out = hand + wave * hand_stride;                            // wave < W-1
  // wave > 0; wavefront 0 finds there that nothing comes in
  const float* hand_in = wave > 0 ? hand + (wave - 1) * hand_stride : nothing;
  // (a launch that only traces asks for its first groups' operands like any other, and never
  // uses them: it asks where the lowest block would, inside the arrays)
  const int u0 = (walks ? u_base : 0) + (wave * 64 + lane) * C;
  // E[t,blank] for the cells of step s sits at ebl[s - u]; column c at step 4g+j reads
  // ebl[4g + j - c], so one run of C+3 values serves all columns of a group
  const float* ebl = p.eb + (size_t)b * d.Tp + d.Eo - u0;
  const int gstride = plane_group_stride(d);

  float stay[C], emit[C], pbv[C];
  unsigned wbits[C];
  const float* lnp[C];
  const float* bsp[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int u = u0 + c, uc = u < d.U ? u : d.U - 1;
    const size_t row = plane_group0(d, b, uc);
    lnp[c] = p.lnS + row;
    bsp[c] = bestS + row;
    pbv[c] = p.pb[(size_t)b * d.Ua + uc];
    stay[c] = kNegInf;
    emit[c] = kNegInf;
    wbits[c] = 0u;
  }
  // Groups from in_lo on need not ask whether a cell has started: step 4g is past the first frame of
  // the wavefront's last position (positions past the utterance are never consulted, whatever
  // they run on).  Their operands are addressed by 32-bit offsets from the utterance's own (uniform) plane
  // origins.
  const int u_lo = (walks ? u_base : 0) + wave * 64 * C;
  const bool small_plane = 4ull * (unsigned long long)d.Ua * (unsigned)d.Dp < (1ull << 32);
  const int in_lo = small_plane ? (max(min(u_lo + 64 * C, Ub) - 1, 1) + 3) >> 2 : 0x7fffffff;
  const char* ln_b = reinterpret_cast<const char*>(p.lnS + plane_group0(d, b, 0));
  const char* bs_b = reinterpret_cast<const char*>(bestS + plane_group0(d, b, 0));
  const char* eb_b = reinterpret_cast<const char*>(p.eb + (size_t)b * d.Tp);
  unsigned row_o[C];
#pragma unroll
  for (int c = 0; c < C; ++c) row_o[c] = 16u * (unsigned)min(u0 + c, d.U - 1);
  const unsigned eb_o = 4u * (unsigned)(d.Eo - u0 - (C - 1));
  struct Group {
    float4 ln[C], bs[C];
    float eb[C + 3];
    float4 gh;  // scores entering the block's first column from the block below
  };
  auto load_group = [&](int g) -> Group {
    Group r;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      r.ln[c] = *reinterpret_cast<const float4*>(lnp[c] + (size_t)g * gstride);
      r.bs[c] = *reinterpret_cast<const float4*>(bsp[c] + (size_t)g * gstride);
    }
#pragma unroll
    for (int k = 0; k < C + 3; ++k) r.eb[k] = ebl[4 * g + k - (C - 1)];
    if constexpr (kMulti) {
      r.gh = make_float4(kNegInf, kNegInf, kNegInf, kNegInf);
      if (gin) r.gh = *reinterpret_cast<const float4*>(gin + 4 * g);  // uniform
    }
    return r;
  };
  auto load_inner = [&](int g) -> Group {
    Group r;
    const unsigned by = (unsigned)g * (4u * (unsigned)gstride);  // bytes
#pragma unroll
    for (int c = 0; c < C; ++c) {
      r.ln[c] = *reinterpret_cast<const float4*>(ln_b + (size_t)(row_o[c] + by));
      r.bs[c] = *reinterpret_cast<const float4*>(bs_b + (size_t)(row_o[c] + by));
    }
    const unsigned eo = eb_o + 16u * (unsigned)g;
#pragma unroll
    for (int k = 0; k < C + 3; ++k)
      r.eb[k] = reinterpret_cast<const float*>(eb_b + (size_t)eo)[k];
    if constexpr (kMulti) {
      r.gh = make_float4(kNegInf, kNegInf, kNegInf, kNegInf);
      if (gin) r.gh = *reinterpret_cast<const float4*>(gin + 4 * g);  // uniform
    }
    return r;
  };
  int avail = 0;  // steps the wavefront below is known to have published (see alpha_kernel)
  auto wait_for = [&](int need) {
    avail = bounded_wait(&done[wave - 1], avail, need, spin_limit, trouble);
  };
  // what enters a wavefront above the first is asked for a group ahead, as in alpha_kernel (the
  // first one asks for the four entries that say that nothing comes in)
  if (wave == 0) avail = 0x7fffffff;
  auto fetch_hand = [&](int g, float4& h) {
    if (W == 1 || g >= ngroups) return;
    const int need = 4 * g + 3;
    if (__builtin_expect(avail < need, 0)) wait_for(need);
    h = *reinterpret_cast<const float4*>(hand_in + (wave > 0 ? 4 * g : 0));
  };
  // A cell that has not started (t < 0) keeps -inf scores and never takes a label; cells past
  // the utterance run on whatever the planes hold and are never consulted by the backtrace.
  // The decision bits of 32 steps are shifted in from the right, one addition with carry a cell.
  auto run_group = [&](int g, const Group& cur, const float4& hand_cur, float4& hand_next,
                       auto interior) {
    constexpr bool kInterior = decltype(interior)::value;
    float4 hin = {kNegInf, kNegInf, kNegInf, kNegInf};
    if constexpr (kMulti) hin = cur.gh;  // wavefront 0: from the block below (or nothing)
    if constexpr (W > 1) {
      if (!kMulti) hin = hand_cur;
      else if (wave > 0) hin = hand_cur;
      fetch_hand(g + 1, hand_next);
    }
    float gsend[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = 4 * g + j;
      const float from_left = wave_shr1(emit[C - 1], f4get(hin, j));  // lane 0: hin
#pragma unroll
      for (int c = C - 1; c >= 0; --c) {
        const float left = (c == 0) ? from_left : emit[c - 1];
        const bool take = left > stay[c];  // :200-206 ties go to blank
        float x = take ? left : stay[c];
        if (!kInterior && j == 0 && g == 0) x = (u0 + c == 0) ? 0.0f : x;
        wbits[c] = wbits[c] + wbits[c] + (take ? 1u : 0u);
        const float ln = f4get(cur.ln[c], j);
        float sb = x + cur.eb[j - c + (C - 1)];
        sb = sb + pbv[c];
        sb = sb - ln;
        float se = x + f4get(cur.bs[c], j);
        se = se - ln;
        const bool started = kInterior || s >= u0 + c;
        stay[c] = started ? sb : kNegInf;
        emit[c] = started ? se : kNegInf;
      }
      gsend[j] = emit[C - 1];
    }
    if constexpr (kMulti) {
      if (gout && wave == W - 1 && lane == 63) {  // entries 4g+1 .. 4g+4 for the block above
#pragma unroll
        for (int j = 0; j < 4; ++j) gout[4 * g + 1 + j] = gsend[j];
      }
    }
    if ((g & 7) == 7 || g == ngroups - 1) {  // uniform: a word of 32 steps is complete
#pragma unroll
      for (int c = 0; c < C; ++c) {
        // (the last word may hold fewer steps: the first of them goes to bit 0 all the same)
        cols[(size_t)(u0 + c) * nw + (g >> 3)] = __brev(wbits[c] << (28 - 4 * (g & 7)));
        wbits[c] = 0u;
      }
    }
    if (W > 1 && wave < W - 1 && lane == 63) {  // entries 4g+1 .. 4g+4, then the progress
#pragma unroll
      for (int j = 0; j < 4; ++j) hand_out[4 * g + 1 + j] = gsend[j];
      asm volatile("" ::: "memory");
      __hip_atomic_store(&done[wave], 4 * g + 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };
  // four register sets rotate (no copies): a group's loads are requested four groups ahead
  auto clamp_g = [&](int g) { return g < ngroups ? g : ngroups - 1; };
  Group q0 = load_group(0), q1 = load_group(clamp_g(1)), q2 = load_group(clamp_g(2)),
        q3 = load_group(clamp_g(3));
  const int nwalk = walks ? ngroups : 0;  // a block past the utterance's labels only traces
  if (W > 1 && wave > 0 && walks)
    wait_for(min(4 * ngroups, 4 * 8 * wave));  // fall a few groups behind
  const std::true_type inner;
  const std::false_type edge;
  float4 h0 = make_float4(kNegInf, kNegInf, kNegInf, kNegInf), h1 = h0;
  if (walks) fetch_hand(0, h0);
  for (int g = 0; g < nwalk; g += 4) {
    if constexpr (C <= 4) {  // (beyond, the registers are what is short)
      for (; g >= in_lo && g + 8 <= ngroups; g += 4) {
        run_group(g, q0, h0, h1, inner);
        q0 = load_inner(g + 4);
        run_group(g + 1, q1, h1, h0, inner);
        q1 = load_inner(g + 5);
        run_group(g + 2, q2, h0, h1, inner);
        q2 = load_inner(g + 6);
        run_group(g + 3, q3, h1, h0, inner);
        q3 = load_inner(g + 7);
      }
    }
    run_group(g, q0, h0, h1, edge);
    q0 = load_group(clamp_g(g + 4));
    if (g + 1 < ngroups) run_group(g + 1, q1, h1, h0, edge);
    q1 = load_group(clamp_g(g + 5));
    if (g + 2 < ngroups) run_group(g + 2, q2, h0, h1, edge);
    q2 = load_group(clamp_g(g + 6));
    if (g + 3 < ngroups) run_group(g + 3, q3, h1, h0, edge);
    q3 = load_group(clamp_g(g + 7));
  }
  if (!kLdsBits) __threadfence();  // the columns in global memory, before another lane reads them
  __syncthreads();
  if (!traces) return;
  // Backtrace (:208-219): from (T_b - 1, U_b - 1); a set bit at (step, u) means "entered from
  // u - 1 with a label", a clear one "entered from t - 1 with a blank".
  if (tidx == 0) {
    int u = Ub - 1, s = nsteps - 1;
    while (u > 0) {
      int wi = s >> 5;
      unsigned m = cols[(size_t)u * nw + wi] & (0xFFFFFFFFu >> (31 - (s & 31)));
      while (m == 0u && wi > 0) {
        --wi;
        m = cols[(size_t)u * nw + wi];
      }
      if (m == 0u) break;  // ran out of frames: cannot happen on a lattice that was walked
      const int st = 32 * wi + 31 - __clz(m);
      taken[u - 1] = st;
      u -= 1;
      s = st - 1;
    }
  }
  __syncthreads();
  int* out = labels_out + (size_t)b * (d.U - 1);
  const int* argI = reinterpret_cast<const int*>(argS);
  for (int u1 = tidx; u1 < Ub - 1; u1 += 64 * W) {
    const int st = taken[u1];
    // (a label is never taken at step 0 on a lattice that was walked; the clamp keeps the read
    // inside the plane whatever the decision bits hold)
    if (st >= 0) out[u1] = argI[plane_at(d, b, u1, max(st - 1, 0))];
  }
}

// ------------------------------------------------------------------ backtrace
// transducer/transducer_cpu.cpp:208-219, from (T_b - 1, U_b - 1): a set bit at (step, u) means
// "entered from u - 1 with a label", a clear one "entered from t - 1 with a blank", so the step at
// which position v was entered is the highest set bit at or below the running step in column v.
// A wavefront finds it with one comparison over 64 words (lane k holds the k-th word down from the
// path's) and reads kBatch columns at a time; one lane that read a word, tested it and read the next
// took 100 ns a position from LDS (45 so) and most of a microsecond from memory.
// taken[v - 1]: the step at which position v was entered; it stays as it is where there is none.
template <int kBatch, typename Word>
__device__ inline void trace_path(int v, int s, int* taken, Word word) {
  const int lane = threadIdx.x & 63;
  while (v > 0 && s >= 0) {
    const int w0 = s >> 5;
    unsigned m[kBatch];
#pragma unroll
    for (int c = 0; c < kBatch; ++c)
      m[c] = word(max(v - c, 0), max(w0 - lane, 0));
    int step = -1, done = 0;
    bool more = true;
#pragma unroll
    for (int c = 0; c < kBatch; ++c) {
      if (more && v - c > 0 && s >= 0) {  // uniform
        const int k0 = w0 - (s >> 5);  // the lane whose word holds step s
        const unsigned upto = 0xFFFFFFFFu >> (31 - (s & 31));
        unsigned x = lane == k0 ? m[c] & upto : m[c];
        x = lane < k0 || lane > w0 ? 0u : x;
        const unsigned long long any = __builtin_amdgcn_ballot_w64(x != 0u);
        if (any == 0ull) {  // not in these 2048 steps
          s = min(s, 32 * (w0 - 63) - 1);
          more = false;
        } else {
          const int f = __builtin_ctzll(any);
          const unsigned y = __builtin_amdgcn_readlane(x, f);
          const int st = 32 * (w0 - f) + 31 - __builtin_clz(y);
          step = lane == c ? st : step;
          s = st - 1;
          done = c + 1;
        }
      }
    }
    if (lane < done) taken[v - 1 - lane] = step;
    v -= done;
  }
}
// The labels of the path.  (A label is never taken at step 0 on a lattice that was walked; the clamp
// keeps the read inside the plane whatever the decision bits hold.)
__device__ inline void put_labels(const int* taken, const float* __restrict__ argS,
                                  int* __restrict__ labels_out, const Dims& d, int b, int Ub,
                                  int threads) {
  int* out = labels_out + (size_t)b * (d.U - 1);
  const int* argI = reinterpret_cast<const int*>(argS);
  for (int v = threadIdx.x; v < Ub - 1; v += threads) {
    const int st = taken[v];
    if (st >= 0) out[v] = argI[plane_at(d, b, v, max(st - 1, 0))];
  }
}

// ------------------------------------------------------------------ best path, one position a lane
// The same walk with one label position a lane, its wavefronts, blocks and hand-over those of
// alpha_walk_kernel.  A step is nine instructions: the lane shift, one comparison, two that use it
// (the larger score; the decision shifted into the lane's word by an addition with carry), the five
// of the two moves.  Operands are asked for eight groups ahead.  32 ns a step on one wavefront, 43
// with a neighbour; B=8 T=2000, walk and backtrace: 101 positions 142 -> 107 us, 201 226 -> 129,
// 401 392 -> 181 (half of that was the backtrace, a word at a time from memory).
// kLdsBits: the decision columns fit into LDS, and the workgroup traces the path at the end.
// Otherwise they go to global memory and viterbi_trace_kernel follows.
template <int W, bool kLive, bool kLdsBits>
__global__ __launch_bounds__(64 * (W + (kLive ? 1 : 0))) void viterbi_walk_kernel(
    Planes p, const float* __restrict__ bestS, const float* __restrict__ argS,
    const int* __restrict__ inLen, const int* __restrict__ labLen, unsigned* __restrict__ gcols,
    int* __restrict__ labels_out, Dims d, int nw, int spin_limit, int* __restrict__ trouble,
    unsigned long long* __restrict__ live, int live_n) {
  static_assert(!kLive || !kLdsBits, "blocks side by side keep their columns in global memory");
  constexpr bool kHand = W > 1 || kLive;
  constexpr int kDepth = 8;
  extern __shared__ __attribute__((aligned(16))) int dyn[];  // kLdsBits: [U up to 4] steps at which
                                                             // labels were taken, then the columns
  __shared__ __attribute__((aligned(16))) float ring[W + 1][kHand ? 4 * kRingGroups : 4];
  __shared__ __attribute__((aligned(16))) float nothing[16];
  __shared__ __attribute__((aligned(16))) float dump[kHand ? 4 * 64 + 16 : 4];
  __shared__ int prog[W + 2];
  const int live_block = kLive ? (int)(blockIdx.x >> 3) % live_n : 0;
  const int b = kLive ? (int)(blockIdx.x / (8 * live_n)) * 8 + (blockIdx.x & 7) : blockIdx.x;
  if (kLive && b >= d.B) return;
  const int u_base = live_block * 64 * W;
  const int lane = threadIdx.x & 63;
  const int wave = kHand ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Tb == 0 || Ub == 0) return;  // :152-154
  if (u_base >= Ub) return;
  const int nsteps = Tb + Ub - 1;
  const int ngroups = (nsteps + 3) >> 2;
  const bool live_in = kLive && live_block > 0;
  const bool live_out = kLive && live_block < live_n - 1 && u_base + 64 * W < Ub;
  int* taken = dyn;
  unsigned* cols = kLdsBits ? reinterpret_cast<unsigned*>(dyn + ((d.U + 3) & ~3))  // [64 W][nw]
                            : gcols + (size_t)b * d.Ua * nw;                       // [Ua][nw]
  if (threadIdx.x < 16) nothing[threadIdx.x] = kNegInf;
  if (threadIdx.x < W + 2) {
    const int w = (int)threadIdx.x - 1;  // the wavefront whose progress this is
    prog[threadIdx.x] = w < 0 ? (live_in ? 0 : kForever)
                        : w == W ? (live_out ? 0 : kForever)
                                 : (u_base + 64 * w < Ub ? 0 : kForever);
  }
  if constexpr (kLdsBits)
    for (int u = threadIdx.x; u < Ub; u += 64 * W) taken[u] = -1;
  __syncthreads();
  if (kLive && wave == W) {
    const unsigned long long* src =
        live_in ? live + ((size_t)(live_block - 1) * d.B + b) * d.Dp : nullptr;
    unsigned long long* dst = live_out ? live + ((size_t)live_block * d.B + b) * d.Dp : nullptr;
    live_carrier<0>(src, dst, 0, ngroups, 0, ngroups, [](int g, int i) { return 4 * g + 1 + i; },
                    ring[0], &prog[0], &prog[1], ring[W], &prog[W], &prog[W + 1], spin_limit, trouble);
    return;
  }
  const int u_lo = u_base + wave * 64;
  const int u = u_lo + lane;
  if (u_lo < Ub) {  // uniform: else a wavefront past this utterance's labels
    if (kLive) __builtin_amdgcn_s_setprio(3);  // ahead of the carrier on the same SIMD
    const bool first_column = u_lo == 0;
    const float pb = p.pb[(size_t)b * d.Ua + min(u, d.U - 1)];
    // cell (0,0) finds 0 coming up from below (:157) and nothing from the left
    float stay = u == 0 ? 0.0f : kNegInf, emit = kNegInf;
    unsigned bits = 0;
    // Groups from in_lo on need not ask whether a cell has started; cells past the utterance run on
    // whatever the planes hold and are never consulted.
    const int in_lo = (min(u_lo + 64, Ub) + 2) >> 2;
    const unsigned gbytes = kLive ? 16u * (unsigned)d.Ua : 1024u * W;  // from a group to the next
    const size_t plane = (size_t)gbytes * (unsigned)(d.Dp / 4);
    const char* ln_b = reinterpret_cast<const char*>(p.lnS + plane_group0(d, b, 0));
    const char* bs_b = reinterpret_cast<const char*>(bestS + plane_group0(d, b, 0));
    // (buffers that begin at group `origin`, moved on before an offset would outgrow 32 bits)
    Buffer ln_q(ln_b, plane), bs_q(bs_b, plane);
    const Buffer eb_q(p.eb + (size_t)b * d.Tp, 4ull * d.Tp);
    int origin = 0;
    const int span = (int)((1u << 30) / gbytes);
    const unsigned lane_o = 16u * (unsigned)min(u, d.U - 1);
    const unsigned eb_o = 4u * (unsigned)(d.Eo - u);
    struct Ops {
      quad_t ln, bs, eb;
    };
    auto load = [&](int g) -> Ops {
      g = min(g, ngroups - 1);
      const unsigned by = (unsigned)(g - origin) * gbytes;
      Ops r;
      r.ln = ln_q.load(lane_o, by);
      r.bs = bs_q.load(lane_o, by);
      r.eb = eb_q.load(eb_o, 16u * (unsigned)g);
      return r;
    };
    // ---- hand-over (see alpha_walk_kernel)
    int ok = kHand ? -1 : kForever;
    int have_in = 0, have_out = 0;
    auto refresh = [&](int g) {
      ok = hand_over_until(&prog[wave], &prog[wave + 2], have_in, have_out, g, ngroups, spin_limit,
                           trouble);
    };
    const float* take = kHand ? (first_column ? nothing : ring[wave]) : nullptr;
    const int take_mask = first_column ? 0 : kRingGroups / 4 - 1;
    float* give = kHand ? (lane == 63 ? ring[wave + 1] : dump + 4 * lane) : nullptr;
    const int give_mask = lane == 63 ? kRingGroups / 4 - 1 : 0;
    int* give_prog = lane == 63 ? &prog[wave + 1] : reinterpret_cast<int*>(dump + 4 * lane);
    quad_t pend = {kNegInf, kNegInf, kNegInf, kNegInf}, hand = pend;
    float carry = kNegInf;
    auto run_group = [&](int g, const Ops& q, const float* take_next, float* give_last, auto tell,
                         auto inner) {
      constexpr bool kInner = decltype(inner)::value;
      quad_t next = hand;
      if constexpr (kHand) {
        *reinterpret_cast<quad_t*>(give_last) = pend;
        asm volatile("" ::: "memory");  // (LDS serves a wavefront's requests in order)
        if constexpr (decltype(tell)::value) prog_store(give_prog, g);
        next = *reinterpret_cast<const quad_t*>(take_next);
      }
      float in[4] = {carry, hand[0], hand[1], hand[2]};
      if constexpr (!kHand) {  // (set well ahead of the lane shifts that fill lane 0 from them)
        in[0] = in[1] = in[2] = in[3] = kNegInf;
        asm volatile("" : "+v"(in[0]), "+v"(in[1]), "+v"(in[2]), "+v"(in[3]));
      }
      quad_t em;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float left = wave_shr1(emit, in[j]);
        const bool takes = left > stay;  // :200-206 ties go to blank
        const float x = takes ? left : stay;
        bits = bits + bits + (takes ? 1u : 0u);
        float se = x + q.bs[j];
        float sb = x + q.eb[j];
        se = se - q.ln[j];
        sb = sb + pb;
        sb = sb - q.ln[j];
        if constexpr (kInner) {
          stay = sb;
          emit = se;
        } else {
          const bool started = 4 * g + j >= u;
          stay = started ? sb : kNegInf;
          emit = started ? se : kNegInf;
        }
        em[j] = emit;
      }
      pend = em;
      carry = hand[3];
      hand = next;
    };
    // a word of 32 steps, the first of them in bit 0 (the last word may hold fewer)
    auto put_word = [&](int g) {
      cols[(size_t)u * nw + (g >> 3)] = __brev(bits << (28 - 4 * (g & 7)));
      bits = 0u;
    };
    const std::true_type yes;
    const std::false_type no;
    Ops q[kDepth];
#pragma unroll
    for (int k = 0; k < kDepth; ++k) q[k] = load(k);
    if constexpr (kHand) {
      if (!first_column) {
        refresh(0);
        hand = *reinterpret_cast<const quad_t*>(take);
      }
    }
    // groups g .. g + 3, an aligned block of slots; kWhole: all of them exist
    auto four = [&](int g, Ops* w, auto whole, auto inner) {
      constexpr bool kWhole = decltype(whole)::value;
      const float *tk = nullptr, *tk_next = nullptr;
      float *gv = nullptr, *gv_last = nullptr;
      if constexpr (kHand) {
        tk = take + 16 * ((g >> 2) & take_mask);
        tk_next = take + 16 * (((g >> 2) + 1) & take_mask);
        gv = give + 16 * ((g >> 2) & give_mask);
        gv_last = give + 16 * (((g >> 2) - 1) & give_mask) + 12;
        if (__builtin_expect(g > ok, 0)) refresh(g);
      }
      run_group(g, w[0], tk + 4, gv_last, yes, inner);
      if (kWhole) w[0] = load(g + kDepth);
      if (kWhole || g + 1 < ngroups) run_group(g + 1, w[1], tk + 8, gv, no, inner);
      if (kWhole) w[1] = load(g + 1 + kDepth);
      if (kWhole || g + 2 < ngroups) {
        if constexpr (kHand) {
          if (__builtin_expect(g + 2 > ok, 0)) refresh(g + 2);
        }
        run_group(g + 2, w[2], tk + 12, gv + 4, yes, inner);
      }
      if (kWhole) w[2] = load(g + 2 + kDepth);
      if (kWhole || g + 3 < ngroups) run_group(g + 3, w[3], tk_next, gv + 8, no, inner);
      if (kWhole) w[3] = load(g + 3 + kDepth);
      if constexpr (kHand && kWhole) __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): see alpha
    };
    int g = 0;
    for (; g + 8 <= ngroups && g < in_lo; g += 8) {
      four(g, q, yes, no);
      four(g + 4, q + 4, yes, no);
      put_word(g + 7);
    }
    for (; g + 8 <= ngroups; g += 8) {
      if (g - origin >= span) {
        origin = g;
        const size_t by = (size_t)g * gbytes;
        ln_q = Buffer(ln_b + by, plane - by);
        bs_q = Buffer(bs_b + by, plane - by);
      }
      four(g, q, yes, yes);
      four(g + 4, q + 4, yes, yes);
      put_word(g + 7);
    }
    if (g < ngroups) {
      four(g, q, no, no);
      if (g + 4 < ngroups) four(g + 4, q + 4, no, no);
      put_word(ngroups - 1);
    }
    if constexpr (kHand) {
      *reinterpret_cast<quad_t*>(give + 16 * (((ngroups - 1) >> 2) & give_mask) +
                                 4 * ((ngroups - 1) & 3)) = pend;
      asm volatile("" ::: "memory");
      prog_store(give_prog, ngroups);
    }
  }
  if constexpr (kLdsBits) {
    __syncthreads();
    if (wave == 0)
      trace_path<8>(Ub - 1, nsteps - 1, taken, [&](int v, int w) { return cols[v * nw + w]; });
    __syncthreads();
    put_labels(taken, argS, labels_out, d, b, Ub, 64 * W);
  }
}

// The backtrace from decision columns in global memory, one wavefront an utterance.
// Dynamic LDS: one int per label position.
__global__ __launch_bounds__(64) void viterbi_trace_kernel(const float* __restrict__ argS,
                                                           const int* __restrict__ inLen,
                                                           const int* __restrict__ labLen,
                                                           const unsigned* __restrict__ gcols,
                                                           int* __restrict__ labels_out, Dims d,
                                                           int nw) {
  extern __shared__ __attribute__((aligned(16))) int taken[];
  const int b = blockIdx.x;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  if (Tb == 0 || Ub <= 1) return;
  for (int u = threadIdx.x; u < Ub; u += 64) taken[u] = -1;
  __syncthreads();
  const unsigned* cols = gcols + (size_t)b * d.Ua * nw;
  trace_path<24>(Ub - 1, Tb + Ub - 2, taken,
                 [&](int v, int w) { return cols[(size_t)v * nw + w]; });
  __syncthreads();
  put_labels(taken, argS, labels_out, d, b, Ub, 64);
}

// ------------------------------------------------------------------ chain-latency floor
// What ONE step of a lattice walk costs when nothing but its dependent chain is left: operands
// in registers, no loads, no stores, no bookkeeping, one wavefront alone on its SIMD.
//   kind 0: a cell of alpha_walk_kernel -- DPP hand-over, log-sum-exp on the hardware units with
//           the check that its sum is the C library's (alpha_cell; the operands are large, so no lane
//           falls back), the additions of its two moves;
//   kind 1: a cell of the dalpha walk -- DPP hand-over, two multiplies and an add;
//   kind 2: kind 0 with every lane on the library path (rnnt_libm.h: ~100 instructions, two of
//           them divisions): what a step costs while any lane of the wavefront falls back.
// The walks cannot run faster than steps x this; the ratio is what the prefetch, the stores and
// the second wavefront's hand-over cost on top.
template <int kKind>
__global__ __launch_bounds__(64) void chain_floor_kernel(float* __restrict__ sink, int steps,
                                                         float e, float p, float ln, float w) {
  __shared__ unsigned long long etab[32];
  exp2_table_to_lds(etab);
  __syncthreads();
  const int lane = threadIdx.x;
  float stay = -5000.0f - 0.37f * lane, emit = -5000.0f - 0.61f * lane, dcol = 1.0f / (1 + lane);
  auto step = [&]() {
    if (kKind != 1) {
      const float left = wave_shr1(emit, kOutside);
      AlphaCell c = alpha_cell(left, stay, e, p, p, e, ln);
      if (kKind == 2 || __builtin_expect(c.fail != 0ull, 0)) {
        const float a = lse2_libm(left, stay, etab);
        c.stay = a + e;
        c.stay = c.stay + p;
        c.stay = c.stay - ln;
        c.emit = a + p;
        c.emit = c.emit + e;
        c.emit = c.emit - ln;
      }
      stay = c.stay;
      emit = c.emit;
    } else {
      const float right = wave_shl1(dcol, 0.0f);
      const float ne = dcol * w;
      const float em = right * w;
      dcol = ne + em;
    }
  };
  // four at a time by hand: the compiler leaves a loop around the hand-written cell as it is
  int s = 0;
  for (; s + 4 <= steps; s += 4) {
    step();
    step();
    step();
    step();
  }
  for (; s < steps; ++s) step();
  sink[lane] = kKind != 1 ? stay + emit : dcol;
}

}  // namespace

namespace {
// The two library functions applied elementwise, for the tests that hold them to the host's C
// library bit for bit.
__global__ __launch_bounds__(256) void libm_probe_kernel(const float* __restrict__ x,
                                                         float* __restrict__ e,
                                                         float* __restrict__ l, long n) {
  __shared__ unsigned long long etab[32];
  exp2_table_to_lds(etab);
  __syncthreads();
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  e[i] = expf_glibc(x[i], etab);
  l[i] = log1pf_glibc(x[i]);
}
}  // namespace

namespace {
// For every float d with bit pattern in [lo, hi] (d <= 0): does the bound of lse2_fast cover
// the distance between the fast and the library value of log1p(exp(d))?  out[0] counts the
// patterns where it does not, out[1] keeps the largest ratio distance / bound (as float bits;
// ratios are non-negative, so their bit patterns order like integers).
__global__ __launch_bounds__(256) void lse_bound_kernel(unsigned lo, unsigned hi,
                                                        unsigned* __restrict__ out) {
  __shared__ unsigned long long etab[32];
  exp2_table_to_lds(etab);
  __syncthreads();
  unsigned bad = 0;
  float worst = 0.0f;
  const unsigned long long n = (unsigned long long)hi - lo + 1;
  for (unsigned long long i = (unsigned long long)blockIdx.x * 256 + threadIdx.x; i < n;
       i += (unsigned long long)gridDim.x * 256) {
    const float d = __uint_as_float(lo + (unsigned)i);
    const float exact = log1pf_glibc(expf_glibc_nonpositive(d, etab));
    const float lf = softplus_fast(d);
    const float bound = fast_bound(lf, d);
    const float dist = fabsf(lf - exact);
    if (!(dist <= bound)) {
      ++bad;
    } else if (bound > 0.0f) {
      worst = fmaxf(worst, dist / bound);
    }
  }
  if (bad) atomicAdd(&out[0], bad);
  atomicMax(&out[1], __float_as_uint(worst));
}
}  // namespace

#if RNNT_IN_PART(0)
int launch_lse_bound_check(unsigned lo, unsigned hi, unsigned* out, hipStream_t s) {
  hipLaunchKernelGGL(lse_bound_kernel, dim3(4096), dim3(256), 0, s, lo, hi, out);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return check_hip(err, "launch lse_bound_kernel", __FILE__, __LINE__);
  return kOk;
}

int launch_libm_probe(const float* x, float* e, float* l, long n, hipStream_t s) {
  if (n == 0) return kOk;
  const long blocks = (n + 255) / 256;
  if (blocks > 0x7fffffffl) return fail(kInvalid, "libm_probe: too many elements");
  hipLaunchKernelGGL(libm_probe_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, e, l, n);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return check_hip(err, "launch libm_probe_kernel", __FILE__, __LINE__);
  return kOk;
}

int launch_chain_floor(int kind, int steps, hipStream_t s) {
  int* words = nullptr;
  RNNT_TRY(trouble_flag(&words));
  float* sink = reinterpret_cast<float*>(words + 64);
  // scores that keep the recursion near zero: a step adds log 2 and takes it off again
  if (kind == 0)
    hipLaunchKernelGGL(chain_floor_kernel<0>, dim3(1), dim3(64), 0, s, sink, steps, 0.3f, 0.2f,
                       0.5f + 0.693147f, 0.5f);
  else if (kind == 2)
    hipLaunchKernelGGL(chain_floor_kernel<2>, dim3(1), dim3(64), 0, s, sink, steps, 0.3f, 0.2f,
                       0.5f + 0.693147f, 0.5f);
  else
    hipLaunchKernelGGL(chain_floor_kernel<1>, dim3(1), dim3(64), 0, s, sink, steps, 0.3f, 0.2f,
                       0.5f, 0.5f);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return check_hip(e, "launch chain_floor_kernel", __FILE__, __LINE__);
  return kOk;
}

// ------------------------------------------------------------------ trouble flag
// One int per device, raised by a lattice kernel whose bounded wait ran out (bounded_wait).  The
// array's name is a host-side handle, not a device address: the address is looked up once per
// device, with that device current, and kernels are given that pointer.
static __device__ int g_trouble_word[128];  // [0]: the flag; [64..127]: sink of the floor probe
constexpr int kMaxDevices = 64;
static int* g_trouble_ptr[kMaxDevices];
static std::mutex g_trouble_mutex;
int g_spin_limit = kDefaultSpinLimit;

int trouble_flag(int** out) {
  int dev = 0;
  RNNT_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail(kInvalid, "device index %d not supported", dev);
  std::lock_guard<std::mutex> lock(g_trouble_mutex);
  if (g_trouble_ptr[dev] == nullptr) {
    void* p = nullptr;
    RNNT_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(g_trouble_word)));
    g_trouble_ptr[dev] = static_cast<int*>(p);
  }
  *out = g_trouble_ptr[dev];
  return kOk;
}

// ------------------------------------------------------------------ workspace layout
static size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

// The two hand-over vectors of the planes hold the walks' tagged 64-bit entries as well: one
// array of [B][Dp] entries per boundary between blocks side by side.  In units of [B][Dp] floats
// each.
static int hand_arrays(const Dims& d, bool decode_only) {
  int w;
  return std::max(1, (decode_only ? viterbi_blocks(d)
                                  : std::max(alpha_blocks(d), beta_blocks(d, &w))) - 1);
}

size_t planes_bytes(const Dims& d, bool decode_only) {
  const size_t plane = align_up(sizeof(float) * (size_t)d.B * d.Ua * d.Dp + 64);
  return (decode_only ? 1 : 6) * plane + align_up(sizeof(float) * (size_t)d.B * d.Tp) +
         4 * align_up(sizeof(float) * (size_t)d.B * d.Ua) +
         2 * align_up(sizeof(float) * (size_t)d.B * d.Dp * hand_arrays(d, decode_only));
}

void carve_planes(void* base, const Dims& d, Planes* p, bool decode_only) {
  char* c = static_cast<char*>(base);
  const size_t plane = align_up(sizeof(float) * (size_t)d.B * d.Ua * d.Dp + 64);
  auto take = [&](size_t n) { float* r = reinterpret_cast<float*>(c); c += n; return r; };
  p->lnS = take(plane);
  p->elS = p->aS = p->wB = p->wE = p->dS = nullptr;
  if (!decode_only) {
    p->elS = take(plane); p->aS = take(plane);
    p->wB = take(plane); p->wE = take(plane); p->dS = take(plane);
  }
  p->eb = take(align_up(sizeof(float) * (size_t)d.B * d.Tp));
  const size_t bu = align_up(sizeof(float) * (size_t)d.B * d.Ua);
  p->pb = take(bu); p->pl = take(bu); p->gB = take(bu); p->gL = take(bu);
  const size_t bh = align_up(sizeof(float) * (size_t)d.B * d.Dp * hand_arrays(d, decode_only));
  p->hand[0] = take(bh); p->hand[1] = take(bh);
}

#endif

// ------------------------------------------------------------------ launchers
// tiles of 64 anti-diagonals x 64 label positions over all anti-diagonals t + u < T + U
static dim3 tile_grid(const Dims& d) {
  return dim3((d.T + d.U + 62) / 64, (d.U + 63) / 64, d.B);
}

#if RNNT_IN_PART(0)
int launch_skew(const float* src, float* dstS, const int* inLen, const int* labLen, const Dims& d,
                hipStream_t s) {
  if (d.B == 0 || d.T == 0 || d.U == 0) return kOk;
  hipLaunchKernelGGL(skew_kernel, tile_grid(d), dim3(256), 0, s, src, dstS, inLen, labLen, d);
  RNNT_LAUNCH_CHECK("skew_kernel");
  return kOk;
}

int launch_unskew(const float* srcS, float* dst, const int* inLen, const int* labLen,
                  const Dims& d, hipStream_t s) {
  if (d.B == 0 || d.T == 0 || d.U == 0) return kOk;
  hipLaunchKernelGGL(unskew_kernel, tile_grid(d), dim3(256), 0, s, srcS, dst, inLen, labLen, d);
  RNNT_LAUNCH_CHECK("unskew_kernel");
  return kOk;
}

template <typename TIO>
static int gather_any(const TIO* E, const TIO* P, const int* labels, const int* inLen,
                      const int* labLen, const Planes& p, const Dims& d, hipStream_t s) {
  if (d.B == 0 || d.T == 0 || d.U == 0) return kOk;
  if (d.V <= 1024)
    hipLaunchKernelGGL(gather_kernel<TIO>, tile_grid(d), dim3(256), 0, s, E, P, labels, inLen,
                       labLen, p, d);
  else
    hipLaunchKernelGGL(gather_cells_kernel<TIO>, dim3((d.T + 255) / 256, d.U, d.B), dim3(256), 0,
                       s, E, P, labels, inLen, labLen, p, d);
  RNNT_LAUNCH_CHECK("gather_kernel");
  return kOk;
}
int launch_gather(const float* E, const float* P, const int* labels, const int* inLen,
                  const int* labLen, const Planes& p, const Dims& d, hipStream_t s) {
  return gather_any(E, P, labels, inLen, labLen, p, d, s);
}
int launch_gather(const bf16_t* E, const bf16_t* P, const int* labels, const int* inLen,
                  const int* labLen, const Planes& p, const Dims& d, hipStream_t s) {
  return gather_any(E, P, labels, inLen, labLen, p, d, s);
}
int launch_gather(const f16_t* E, const f16_t* P, const int* labels, const int* inLen,
                  const int* labLen, const Planes& p, const Dims& d, hipStream_t s) {
  return gather_any(E, P, labels, inLen, labLen, p, d, s);
}

#endif

static __global__ void clear_words_kernel(int* x, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] = 0;
}

// Clears the tagged entries of n blocks side by side.
static int clear_live(unsigned long long* live, const Dims& d, int n, hipStream_t s) {
  const int words = 2 * d.B * d.Dp * (n - 1);
  hipLaunchKernelGGL(clear_words_kernel, dim3((words + 255) / 256), dim3(256), 0, s,
                     reinterpret_cast<int*>(live), words);
  RNNT_LAUNCH_CHECK("clear_words_kernel");
  return kOk;
}

int launch_alpha_wide(const Planes& p, const int* inLen, const int* labLen, float* costs,
                      const Dims& d, hipStream_t s, int C, int W, bool multi, size_t lds,
                      int* trouble, int u_base, const float* ghin, float* ghout);
#define CASE(C, W, M)                                                                        \
  case (M ? 10000 : 0) + C * 100 + W:                                                        \
    if (lds > 64 * 1024)                                                                     \
      RNNT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(alpha_kernel<C, W, M>),     \
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));   \
    hipLaunchKernelGGL((alpha_kernel<C, W, M>), dim3(d.B), dim3(64 * W), lds, s, p, inLen,  \
                       labLen, costs, d, stride, g_spin_limit, trouble, u_base, ghin,        \
                       ghout);                                                               \
    break;

#if RNNT_IN_PART(1)
static int launch_alpha_walk(const Planes& p, const int* inLen, const int* labLen, float* costs,
                             const Dims& d, hipStream_t s, int* trouble) {
  unsigned long long* live = reinterpret_cast<unsigned long long*>(p.hand[0]);
  const int n = alpha_blocks(d);
  if (n > 1) {
    RNNT_TRY(clear_live(live, d, n, s));
    hipLaunchKernelGGL((alpha_walk_kernel<4, true>), dim3(8 * n * ((d.B + 7) / 8)), dim3(320), 0, s,
                       p, inLen, labLen, costs, d, g_spin_limit, trouble, live, n);
  } else if (d.U <= 64) {
    hipLaunchKernelGGL((alpha_walk_kernel<1, false>), dim3(d.B), dim3(64), 0, s, p, inLen, labLen,
                       costs, d, g_spin_limit, trouble, live, 1);
  } else if (d.U <= 128) {
    hipLaunchKernelGGL((alpha_walk_kernel<2, false>), dim3(d.B), dim3(128), 0, s, p, inLen, labLen,
                       costs, d, g_spin_limit, trouble, live, 1);
  } else {
    hipLaunchKernelGGL((alpha_walk_kernel<4, false>), dim3(d.B), dim3(256), 0, s, p, inLen, labLen,
                       costs, d, g_spin_limit, trouble, live, 1);
  }
  RNNT_LAUNCH_CHECK("alpha_walk_kernel");
  return kOk;
}

int launch_alpha(const Planes& p, const int* inLen, const int* labLen, float* costs,
                 const Dims& d, hipStream_t s) {
  if (d.B == 0) return kOk;
  // cells per lane of a single wavefront; split over two wavefronts when the hand-over
  // array (one float per step and boundary) fits LDS
  const int cpl = block_cells_per_lane(d), nblocks = label_blocks(d);
  const int stride = d.Dp;
  // (two or four positions a lane on four wavefronts if their three hand-over arrays fit LDS: a
  // step costs a wavefront one log-sum-exp per position it owns, and the step is what a lattice
  // is bound by)
  const bool single_block = nblocks == 1;
  const int W = (single_block && cpl >= 4 && 3 * stride * sizeof(float) <= 144 * 1024) ? 4
                : (cpl >= 2 && stride * sizeof(float) <= 144 * 1024) ? 2 : 1;
  const size_t lds = W > 1 ? sizeof(float) * (size_t)(W - 1) * stride : 0;
  int* trouble = nullptr;
  RNNT_TRY(trouble_flag(&trouble));
  // one position a lane wherever 256 positions, or blocks of 256 side by side, cover the label axis
  // (B=8 T=10000, 401 positions: 84 ns a step; on one CU with two positions a lane 235)
  if (d.U <= 256 || alpha_blocks(d) > 1)
    return launch_alpha_walk(p, inLen, labLen, costs, d, s, trouble);
  for (int k = 0; k < nblocks; ++k) {  // lowest block first
    const float* ghin = k == 0 ? nullptr : p.hand[(k - 1) & 1];
    float* ghout = k == nblocks - 1 ? nullptr : p.hand[k & 1];
    const int u_base = k * 64 * cpl;
    switch ((nblocks > 1 ? 10000 : 0) + cpl / W * 100 + W) {
      CASE(4, 2, false) CASE(2, 4, false) CASE(4, 4, false)
      default:
        RNNT_TRY(launch_alpha_wide(p, inLen, labLen, costs, d, s, cpl / W, W, nblocks > 1, lds,
                                   trouble, u_base, ghin, ghout));
    }
    RNNT_LAUNCH_CHECK("alpha_kernel");
  }
  return kOk;
}
#endif

#if RNNT_IN_PART(2)
// eight or sixteen label positions a lane; several blocks are always 1024 positions each
int launch_alpha_wide(const Planes& p, const int* inLen, const int* labLen, float* costs,
                      const Dims& d, hipStream_t s, int C, int W, bool multi, size_t lds,
                      int* trouble, int u_base, const float* ghin, float* ghout) {
  const int stride = d.Dp;
  switch ((multi ? 10000 : 0) + C * 100 + W) {
    CASE(8, 1, false) CASE(16, 1, false) CASE(8, 2, false)
    CASE(16, 1, true) CASE(8, 2, true)
    default:
      return fail(kInvalid, "alpha: no kernel for %d label positions per lane", C);
  }
  return kOk;
}
#endif
#undef CASE

#if RNNT_IN_PART(0)
int launch_weights(const Planes& p, const int* inLen, const int* labLen, const Dims& d,
                   hipStream_t s) {
  if (d.B == 0 || d.T == 0 || d.U == 0) return kOk;
  hipLaunchKernelGGL(weights_kernel, dim3((d.Ua * (d.Dp / 4) + 255) / 256, 1, d.B), dim3(256), 0, s,
                     p, inLen, labLen, d);
  RNNT_LAUNCH_CHECK("weights_kernel");
  return kOk;
}

#endif

#if RNNT_IN_PART(3)
int launch_beta(const Planes& p, const int* labels, const int* inLen, const int* labLen,
                const Dims& d, hipStream_t s) {
  if (d.B == 0 || d.T == 0 || d.U == 0) return kOk;
  const int cpl = block_cells_per_lane(d), nblocks = label_blocks(d);
  // several positions a lane (2 or, from 513 positions on, 4): four wavefronts; there two or one if
  // only that many hand-over arrays fit LDS; one per block when the axis takes several launches
  const int stride = d.Dp;
  const bool single_block = nblocks == 1;
  const int W = !single_block ? 1
                : (cpl >= 4 && 3 * stride * sizeof(float) <= 144 * 1024) ? 4
                : (cpl >= 4 && stride * sizeof(float) <= 144 * 1024) ? 2 : 1;
  const size_t lds = W > 1 ? sizeof(float) * (size_t)(W - 1) * stride : 0;
  int* trouble = nullptr;
  RNNT_TRY(trouble_flag(&trouble));
  int waves = 0;
  const int n = beta_blocks(d, &waves);
  if (d.U <= 256 || n > 1) {
    unsigned long long* live = reinterpret_cast<unsigned long long*>(p.hand[0]);
    if (n > 1) {
      RNNT_TRY(clear_live(live, d, n, s));
      const dim3 grid(8 * n * ((d.B + 7) / 8));
      if (waves == 2)
        hipLaunchKernelGGL((beta_walk_kernel<2, true>), grid, dim3(192), 0, s, p, labels, inLen,
                           labLen, d, g_spin_limit, trouble, live, n);
      else
        hipLaunchKernelGGL((beta_walk_kernel<4, true>), grid, dim3(320), 0, s, p, labels, inLen,
                           labLen, d, g_spin_limit, trouble, live, n);
    } else if (d.U <= 64) {
      hipLaunchKernelGGL((beta_walk_kernel<1, false>), dim3(d.B), dim3(64), 0, s, p, labels, inLen,
                         labLen, d, g_spin_limit, trouble, live, 1);
    } else if (d.U <= 128) {
      hipLaunchKernelGGL((beta_walk_kernel<2, false>), dim3(d.B), dim3(128), 0, s, p, labels, inLen,
                         labLen, d, g_spin_limit, trouble, live, 1);
    } else {
      hipLaunchKernelGGL((beta_walk_kernel<4, false>), dim3(d.B), dim3(256), 0, s, p, labels, inLen,
                         labLen, d, g_spin_limit, trouble, live, 1);
    }
    RNNT_LAUNCH_CHECK("beta_walk_kernel");
    return kOk;
  }
  for (int k = nblocks - 1; k >= 0; --k) {  // highest block first
    const float* ghin = k == nblocks - 1 ? nullptr : p.hand[(k + 1) & 1];
    float* ghout = k == 0 ? nullptr : p.hand[k & 1];
    const int u_base = k * 64 * cpl;
    switch ((nblocks > 1 ? 10000 : 0) + cpl / W * 100 + W) {
#define CASE(C, W, M)                                                                       \
  case (M ? 10000 : 0) + C * 100 + W:                                                       \
    if (lds > 64 * 1024)                                                                    \
      RNNT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(beta_kernel<C, W, M>),     \
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));  \
    hipLaunchKernelGGL((beta_kernel<C, W, M>), dim3(d.B), dim3(64 * W), lds, s, p, labels, \
                       inLen, labLen, d, stride, u_base, ghin, ghout, g_spin_limit,        \
                       trouble);                                                            \
    break;
      CASE(2, 4, false) CASE(4, 4, false) CASE(8, 2, false) CASE(16, 1, false)
      CASE(16, 1, true)
#undef CASE
      default:
        return fail(kInvalid, "dalpha: no kernel for %d label positions per lane", cpl);
    }
    RNNT_LAUNCH_CHECK("beta_kernel");
  }
  return kOk;
}
#endif

#if RNNT_IN_PART(0)
int launch_sparse(const Planes& p, const float* bsum, const float* emT, float* egrads,
                  float* pgrads, const int* labels, const int* inLen, const int* labLen,
                  const float* scale, bool add, const Dims& d, hipStream_t s) {
  if (d.B == 0 || d.T == 0 || d.U == 0) return kOk;
  if (!bsum || !emT) return fail(kInvalid, "sparse terms: the per-frame terms were not formed");
  const int frames = 64 * (size_t)(d.V | 1) * sizeof(float) <= 64 * 1024 ? 64 : 32;
  const size_t rows_bytes = sizeof(float) * frames * (size_t)(d.V | 1);
  // (a small vocabulary also when the terms are to be stored: the arrays are zero-filled then,
  // and adding to zeros leaves the same bits -- B=8 T=10000 U=400 V=32: 1.67 ms with one
  // hardware add per term, all of them into 128 bytes a frame)
  if (rows_bytes <= 64 * 1024 && labels != nullptr) {
    hipLaunchKernelGGL(sparse_e_rows_kernel, dim3((d.T + frames - 1) / frames, d.B), dim3(256),
                       rows_bytes, s, bsum, emT, egrads, labels, inLen, labLen,
                       add ? scale : nullptr, d, frames);
    RNNT_LAUNCH_CHECK("sparse_e_rows_kernel");
  } else {
    hipLaunchKernelGGL(sparse_e_kernel, dim3((d.T + 255) / 256, d.B), dim3(256), 0, s, bsum, emT,
                       egrads, labels, inLen, labLen, scale, add ? 1 : 0, d);
    RNNT_LAUNCH_CHECK("sparse_e_kernel");
  }
  if (pgrads == nullptr) return kOk;  // the caller adds those terms itself
  hipLaunchKernelGGL(sparse_p_kernel, dim3((d.U + 255) / 256, d.B), dim3(256), 0, s, p, pgrads,
                     labels, inLen, labLen, scale, add ? 1 : 0, d);
  RNNT_LAUNCH_CHECK("sparse_p_kernel");
  return kOk;
}

int launch_post_beta(const Planes& p, const float* mE, const float* mP, float* Wn, float* Wt,
                     float* bsum, float* emT, const int* labels, const int* inLen,
                     const int* labLen, const Dims& d, hipStream_t s, const WImages& img) {
  if (d.B == 0 || d.T == 0 || d.U == 0) return kOk;
  const int Up = wplane_up(d.U), Tw = wplane_tw(d.T);
  if (img.e && Up > WImages::kCols)
    return fail(kInvalid, "W images hold at most %d label positions", WImages::kCols);
  // W tiles: 64 label positions x 64 anti-diagonals (all anti-diagonals below Tw + Up), or for
  // the images 64 label positions x 64 frames
  // (Wn == nullptr: no W at all, only the per-frame terms)
  const int wx = img.e ? Tw / 64 : (Tw + Up + 62) / 64, wy = (Up + 63) / 64;
  const int nw = (Wn || img.e) ? wx * wy * d.B : 0;
  if ((bsum == nullptr) != (emT == nullptr))
    return fail(kInvalid, "post_beta: the blank totals and the label-move terms come together");
  const int alone = (d.T + 4 * kBsFrames - 1) / (4 * kBsFrames);
  const bool shared = (long)alone * d.B <= 96;
  const int sx = shared ? (d.T + kBsFrames - 1) / kBsFrames : alone, ns = bsum ? sx * d.B : 0;
  if (nw + ns == 0) return kOk;
  if (shared)
    hipLaunchKernelGGL(post_beta_kernel<true>, dim3(nw + ns), dim3(256), 0, s, p, mE, mP, Wn, Wt,
                       bsum, emT, labels, inLen, labLen, d, Up, Tw, wx, wy, nw, sx, img);
  else
    hipLaunchKernelGGL(post_beta_kernel<false>, dim3(nw + ns), dim3(256), 0, s, p, mE, mP, Wn, Wt,
                       bsum, emT, labels, inLen, labLen, d, Up, Tw, wx, wy, nw, sx, img);
  RNNT_LAUNCH_CHECK("post_beta_kernel");
  return kOk;
}

// 0: lists where they can pay (maxplus_lists_pay) and a sample of the cells says they do; 1: every
// column for every cell; 2: lists wherever the shape allows (tests run small shapes through them)
static std::atomic<int> g_maxplus_mode{0};
void set_maxplus_mode(int mode) { g_maxplus_mode.store(mode); }
// Ranges of columns for maxplus_kernel<.., kParts>.
int maxplus_parts(const Dims& d) {
  const long tiles = (long)((d.T + kMpT - 1) / kMpT) * ((d.U + kMpU - 1) / kMpU) * d.B;
  const long all = (d.V + kMpK - 1) / kMpK;
  if (tiles == 0) return 1;
  const long n = std::min(std::min(kMpWanted / tiles, all / kMpMinChunks), (long)kMpMaxParts);
  return n < 1 ? 1 : (int)n;
}
size_t maxplus_parts_bytes(const Dims& d, int n) {
  return n > 1 ? (size_t)n * 2 * sizeof(float) * d.B * d.U * d.T : 0;
}

MaxplusPlan maxplus_plan(const Dims& d, size_t room) {
  const int mode = g_maxplus_mode.load();  // read once per call: the plan is what the call follows
  MaxplusPlan p;
  if (mode != 1 && maxplus_lists_possible(d)) p.lists = mode == 2 ? 2 : maxplus_lists_pay(d) ? 1 : 0;
  if (p.lists) {
    p.bytes = maxplus_lists_bytes(d);
  } else {
    p.parts = maxplus_parts(d);
    while (maxplus_parts_bytes(d, p.parts) > room) --p.parts;
    p.bytes = maxplus_parts_bytes(d, p.parts);
  }
  return p;
}

template <typename TIO>
static int maxplus_any(const TIO* E, const TIO* P, const int* inLen, const int* labLen,
                       float* best, int* arg, const Dims& d, hipStream_t s, void* scratch,
                       const MaxplusPlan& plan) {
  if (d.B == 0 || d.T == 0 || d.U == 0) return kOk;
  static_assert(kMpT == 128 && kMpU == 64, "the list pass counts failures per tile of this kernel");
  const int *tile_fail = nullptr, *lists_on = nullptr;
  if (plan.lists) {  // (the caller made the plan, and reserved what it says)
    RNNT_TRY(launch_maxplus_lists(E, P, inLen, labLen, best, arg, d, scratch, plan.lists == 2, s));
    maxplus_lists_counters(scratch, d, &tile_fail, &lists_on);
  }
  MaxplusParts parts;  // one range: the maxima and chunks wait in the table itself
  parts.n = plan.lists ? 1 : plan.parts;
  parts.top = parts.n > 1 ? static_cast<float*>(scratch) : best;
  parts.chunk = parts.n > 1
      ? reinterpret_cast<int*>(parts.top + (size_t)parts.n * d.B * d.U * d.T) : arg;
  const dim3 grid((d.T + kMpT - 1) / kMpT, (d.U + kMpU - 1) / kMpU, d.B * parts.n);
  const bool vec = d.V % 4 == 0 &&
                   ((reinterpret_cast<uintptr_t>(E) | reinterpret_cast<uintptr_t>(P)) &
                    (4 * sizeof(TIO) - 1)) == 0;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kMpThreads), 0, s, E, P, inLen, labLen, best, arg, d,
                       tile_fail, lists_on, maxplus_tile_limit(), parts);
  };
  if (plan.lists) {
    if (vec) launch(maxplus_kernel<true, false, TIO>);
    else launch(maxplus_kernel<false, false, TIO>);
    RNNT_LAUNCH_CHECK("maxplus_kernel");
  } else {
    if (vec) launch(maxplus_kernel<true, true, TIO>);
    else launch(maxplus_kernel<false, true, TIO>);
    RNNT_LAUNCH_CHECK("maxplus_kernel");
    const dim3 cells((d.T + 63) / 64, (d.U + 3) / 4, d.B);
    if (vec)
      hipLaunchKernelGGL((maxplus_index_kernel<true, TIO>), cells, dim3(256), 0, s, E, P, inLen,
                         labLen, best, arg, d, parts);
    else
      hipLaunchKernelGGL((maxplus_index_kernel<false, TIO>), cells, dim3(256), 0, s, E, P, inLen,
                         labLen, best, arg, d, parts);
    RNNT_LAUNCH_CHECK("maxplus_index_kernel");
  }
  if (tile_fail) RNNT_TRY(launch_maxplus_cells(E, P, inLen, labLen, best, arg, d, scratch, s));
  return kOk;
}
int launch_maxplus(const float* E, const float* P, const int* inLen, const int* labLen,
                   float* best, int* arg, const Dims& d, hipStream_t s, void* scratch,
                   const MaxplusPlan& plan) {
  return maxplus_any(E, P, inLen, labLen, best, arg, d, s, scratch, plan);
}
int launch_maxplus(const bf16_t* E, const bf16_t* P, const int* inLen, const int* labLen,
                   float* best, int* arg, const Dims& d, hipStream_t s, void* scratch,
                   const MaxplusPlan& plan) {
  return maxplus_any(E, P, inLen, labLen, best, arg, d, s, scratch, plan);
}
int launch_maxplus(const f16_t* E, const f16_t* P, const int* inLen, const int* labLen,
                   float* best, int* arg, const Dims& d, hipStream_t s, void* scratch,
                   const MaxplusPlan& plan) {
  return maxplus_any(E, P, inLen, labLen, best, arg, d, s, scratch, plan);
}
#endif

#if RNNT_IN_PART(4)
template <int W, bool kLive, bool kLdsBits>
static int viterbi_walk(const Planes& p, const float* bestS, const float* argS, unsigned* gcols,
                        const int* inLen, const int* labLen, int* labels_out, const Dims& d, int nw,
                        hipStream_t s, dim3 grid, size_t lds, int n) {
  int* trouble = nullptr;
  RNNT_TRY(trouble_flag(&trouble));
  unsigned long long* live = reinterpret_cast<unsigned long long*>(p.hand[0]);
  if (kLive) RNNT_TRY(clear_live(live, d, n, s));
  const auto kernel = viterbi_walk_kernel<W, kLive, kLdsBits>;
  if (lds > 48 * 1024)
    RNNT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  hipLaunchKernelGGL(kernel, grid, dim3(64 * (W + (kLive ? 1 : 0))), lds, s, p, bestS, argS, inLen,
                     labLen, gcols, labels_out, d, nw, g_spin_limit, trouble, live, n);
  RNNT_LAUNCH_CHECK("viterbi_walk_kernel");
  if (!kLdsBits) {
    hipLaunchKernelGGL(viterbi_trace_kernel, dim3(d.B), dim3(64), sizeof(int) * (size_t)d.U, s, argS,
                       inLen, labLen, gcols, labels_out, d, nw);
    RNNT_LAUNCH_CHECK("viterbi_trace_kernel");
  }
  return kOk;
}

// One position a lane: one workgroup up to 256 label positions, else blocks of 256 side by side.
// The decision columns stay in LDS if two workgroups of them fit a CU, or one where there is a CU
// for each; the path is then traced from there, without a launch of its own.
static int launch_viterbi_walk(const Planes& p, const float* bestS, const float* argS,
                               unsigned* gcols, const int* inLen, const int* labLen,
                               int* labels_out, const Dims& d, int nw, hipStream_t s) {
  const int W = d.U <= 64 ? 1 : d.U <= 128 ? 2 : 4, n = viterbi_blocks(d);
  const size_t lds = sizeof(int) * (((size_t)d.U + 3 & ~(size_t)3) + (size_t)64 * W * nw);
  const bool fits = n == 1 && lds <= (d.B <= 256 ? 140u : 60u) * 1024;
  const dim3 one(d.B);
#define WALK(W, LIVE, LDS, GRID, BYTES)                                                          \
  viterbi_walk<W, LIVE, LDS>(p, bestS, argS, gcols, inLen, labLen, labels_out, d, nw, s, GRID,   \
                             BYTES, n)
  if (n > 1) return WALK(4, true, false, dim3(8 * n * ((d.B + 7) / 8)), 0);
  if (W == 1) return fits ? WALK(1, false, true, one, lds) : WALK(1, false, false, one, 0);
  if (W == 2) return fits ? WALK(2, false, true, one, lds) : WALK(2, false, false, one, 0);
  return fits ? WALK(4, false, true, one, lds) : WALK(4, false, false, one, 0);
#undef WALK
}

int launch_viterbi(const Planes& p, const float* bestS, const float* argS,
                   unsigned long long* gbits, const int* inLen, const int* labLen,
                   int* labels_out, const Dims& d, hipStream_t s) {
  if (d.B == 0 || d.T == 0 || d.U <= 1) return kOk;
  unsigned* gcols = reinterpret_cast<unsigned*>(gbits);
  const int cpl = block_cells_per_lane(d), nblocks = label_blocks(d);
  const int stride = d.Dp;
  const int nw = viterbi_words(d);
  if (d.U <= 256 || viterbi_blocks(d) > 1)
    return launch_viterbi_walk(p, bestS, argS, gcols, inLen, labLen, labels_out, d, nw, s);
  // several positions a lane, on four wavefronts while their hand-over arrays fit
  const ViterbiOne one = viterbi_one(d);
  const int W = one.wavefronts;
  const bool use_lds = one.columns;
  const size_t lds = one.lds;
  if (lds > 150 * 1024)
    return fail(kInvalid, "viterbi: %d label positions and %d steps need %zu bytes of LDS", d.U,
                stride, lds);
  int* trouble = nullptr;
  RNNT_TRY(trouble_flag(&trouble));
  for (int k = 0; k < nblocks; ++k) {  // lowest block first; the last launch traces the path
    const float* ghin = k == 0 ? nullptr : p.hand[(k - 1) & 1];
    float* ghout = k == nblocks - 1 ? nullptr : p.hand[k & 1];
    const int u_base = k * 64 * cpl, traces = k == nblocks - 1 ? 1 : 0;
    switch ((nblocks > 1 ? 10000 : 0) + cpl / W * 100 + W) {
#define CASE(C, W)                                                                             \
  case C * 100 + W:                                                                            \
    if (use_lds)                                                                               \
      hipLaunchKernelGGL((viterbi_kernel<C, W, true, false>), dim3(d.B), dim3(64 * W), lds,   \
                         s, p, bestS, argS, inLen, labLen, gcols, labels_out, d, stride, nw,   \
                         g_spin_limit, trouble, u_base, ghin, ghout, traces);                  \
    else {                                                                                     \
      if (lds > 64 * 1024)                                                                     \
        RNNT_HIP(hipFuncSetAttribute(                                                          \
            reinterpret_cast<const void*>(viterbi_kernel<C, W, false, false>),                 \
            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                            \
      hipLaunchKernelGGL((viterbi_kernel<C, W, false, false>), dim3(d.B), dim3(64 * W), lds,  \
                         s, p, bestS, argS, inLen, labLen, gcols, labels_out, d, stride, nw,   \
                         g_spin_limit, trouble, u_base, ghin, ghout, traces);                  \
    }                                                                                          \
    break;
#define CASE_MULTI(C, W)                                                                       \
  case 10000 + C * 100 + W:                                                                    \
    if (lds > 64 * 1024)                                                                       \
      RNNT_HIP(hipFuncSetAttribute(                                                            \
          reinterpret_cast<const void*>(viterbi_kernel<C, W, false, true>),                    \
          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                              \
    hipLaunchKernelGGL((viterbi_kernel<C, W, false, true>), dim3(d.B), dim3(64 * W), lds, s,  \
                       p, bestS, argS, inLen, labLen, gcols, labels_out, d, stride, nw,        \
                       g_spin_limit, trouble, u_base, ghin, ghout, traces);                    \
    break;
      CASE(8, 1) CASE(16, 1) CASE(4, 2) CASE(8, 2) CASE(2, 4) CASE(4, 4)
      CASE_MULTI(16, 1) CASE_MULTI(8, 2)  // several blocks: always 1024 positions each
#undef CASE
#undef CASE_MULTI
      default:
        return fail(kInvalid, "viterbi: no kernel for %d label positions per lane", cpl);
    }
    RNNT_LAUNCH_CHECK("viterbi_kernel");
  }
  return kOk;
}

size_t viterbi_bits_bytes(const Dims& d) {
  return sizeof(unsigned) * (size_t)d.B * 64 * cells_per_lane(d.U) * viterbi_words(d);
}
#endif

}  // namespace rnnt
