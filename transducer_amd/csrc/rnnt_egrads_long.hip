// The dense gradient of the emissions over a label axis that egrads_stream_kernel (rnnt_grads.hip)
// would have to take in several launches: egrads[t,v] = X[t,v] sum_u W[t,u] Y[u,v] and the
// blank / label terms (transducer/torch_binding.py:85-87, transducer/test.h:82-113), in one.
//
// That kernel keeps a wavefront's columns of Y in registers, 112 label positions of them; a longer
// axis goes slice by slice, each of which writes, or reads and writes, all of egrads.  Here Y is
// streamed like the emissions' side of the log-normaliser: its three bf16 pieces are prepared once in
// the matrix instruction's operand order (yt_planes_kernel, 6 bytes per element of the predictions,
// in the memory that held the log-normaliser's Y pieces), a workgroup turns 128 frames x 32 label
// positions of W at a time into pieces in LDS, and a wavefront owns 32 columns and all 128 frames, so
// that E is read and egrads written once.  Where frames are few, the pieces are multiplied too few
// times to be worth writing and reading: a wavefront then forms them from the predictions as it
// goes, with tiles of 64 frames.
// Bound by the matrix instructions with the W pieces' staging beside them (B=8 T=10000 U=401
// V=1000: 384 GFLOP of bf16 products), then by E and egrads (0.64 GB).
#include <algorithm>
#include <type_traits>

#include "rnnt_internal.h"
#include "rnnt_io.h"
#include "rnnt_split.h"
#include "rnnt_grads.h"

namespace rnnt {

namespace {

constexpr int kElRows = 128;       // frames of a tile
constexpr int kElDirectRows = 64;  // ... where Y is not prepared
constexpr int kElDirect = 400;     // frames up to which it is not (launch_egrads_long)
constexpr int kElBlockPitch = 68;  // floats between columns of the block label terms add up in

inline int el_vblocks(const Dims& d) { return (d.V + 31) / 32; }
inline int el_steps(const Dims& d) { return 2 * ((d.U + 31) / 32); }  // of 16 label positions

// 16-byte slot of (row, c8 = which eight of the slab's 32 label positions) inside a piece plane
__device__ inline int wslot(int row, int c8) { return row * 4 + (c8 ^ ((row >> 2) & 3)); }

// Pieces of exp(P - mP): [b][block of 32 columns][step of 16 u][piece][lane][8 x bf16], lane
// 32 h + l holding column l, label positions 8 h .. 8 h + 7 of the step.  Zero outside.
template <typename TIO>
__global__ __launch_bounds__(256) void yt_planes_kernel(const TIO* __restrict__ P,
                                                        const float* __restrict__ mP,
                                                        uint4* __restrict__ Yt,
                                                        const int* __restrict__ labLen, Dims d,
                                                        int nvb, int nus) {
  const int b = blockIdx.z, vb = blockIdx.x, ks = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (ks >= nus) return;
  const int lane = threadIdx.x & 63, v = 32 * vb + (lane & 31), u0 = 16 * ks + 8 * (lane >> 5);
  int Ub = d.U;
  if (labLen) Ub = clampi(labLen[b], -1, d.U - 1) + 1;
  float y[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int u = u0 + i, uc = min(u, d.U - 1);
    const float e = ldf(P + ((size_t)b * d.U + uc) * d.V + min(v, d.V - 1));
    y[i] = u < Ub && v < d.V ? __expf(e - mP[(size_t)b * d.U + uc]) : 0.0f;
  }
  const Frag3 f = split8(y);
  uint4* dst = Yt + (((size_t)b * nvb + vb) * nus + ks) * 3 * 64 + lane;
  dst[0] = f.h;
  dst[64] = f.m;
  dst[128] = f.l;
}

// kDirect: Y is formed here, from the predictions (Yt is not there).
template <typename TIO, bool kDirect>
__global__ __launch_bounds__(256, 2) void egrads_long_kernel(
    const TIO* __restrict__ E, const TIO* __restrict__ P, const uint4* __restrict__ Yt,
    const float* __restrict__ mE, const float* __restrict__ mP, const float* __restrict__ Wn,
    const float* __restrict__ deltas, TIO* __restrict__ egrads, const int* __restrict__ inLen,
    const int* __restrict__ labLen, Dims d, int Up, int Tw, int nvb, int nus, int tile0,
    SparseTerms sp) {
  __shared__ __attribute__((aligned(16))) uint4 Xs[2][3][kElRows * 4];
  __shared__ float Ms[kElRows];                   // mE log2(e) of the tile's frames
  __shared__ unsigned short Match[4][kMaxLabels];  // per wavefront: labels among its columns
  constexpr int kTile = kDirect ? kElDirectRows : kElRows, kM = kTile / 32;  // blocks of 32 frames
  const int b = blockIdx.z, t0 = (tile0 + (int)blockIdx.y) * kTile;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, h = lane >> 5;
  int Tb, Ub;
  utt_extent(inLen, labLen, b, d.T, d.U, Tb, Ub);
  const int vcol0 = blockIdx.x * 128 + wave * 32, vcol = vcol0 + l32;
  const bool vok = vcol < d.V;
  TIO* out = egrads + (size_t)b * d.T * d.V;
  if (t0 >= Tb) {  // frames past the utterance: exactly zero
    for (int r = 0; r < kTile / 2; ++r) {
      const int t = t0 + 2 * r + h;
      if (t < d.T && vok) stf(out + (size_t)t * d.V + vcol, 0.0f);
    }
    return;
  }
  int nmatch = 0;
  if (sp.labels) {
    for (int u0 = 0; u0 < Ub - 1; u0 += 64) {
      const int u = u0 + lane;
      const int l = (u < Ub - 1) ? label_at(sp.labels, d, b, u) : -1;
      const bool hit = l >= vcol0 && l < vcol0 + 32 && l != d.blank;
      const unsigned long long m = __ballot(hit);
      if (hit) Match[wave][nmatch + __popcll(m & ((1ull << lane) - 1))] = (unsigned short)u;
      nmatch += __popcll(m);
    }
  }
  if (tid < kTile) Ms[tid] = mE[(size_t)b * d.T + min(t0 + tid, Tb - 1)] * kLog2e;

  // staging: rows srow and srow + 64 of the tile, label positions 8 c8 .. 8 c8 + 7 of the slab
  const int srow = tid >> 2, c8 = tid & 3;
  constexpr int kRowsEach = (kM + 1) / 2;
  const float* pw[kRowsEach];
  int slot[kRowsEach];
#pragma unroll
  for (int i = 0; i < kRowsEach; ++i) {
    const int row = srow + 64 * i;
    pw[i] = Wn + ((size_t)b * Tw + min(t0 + row, Tb - 1)) * Up;
    slot[i] = wslot(row, c8);
  }
  const uint4* yw = Yt + ((size_t)b * nvb + min(vcol0 >> 5, nvb - 1)) * nus * 3 * 64 + lane;
  // what a step's fragment of Y is made from, and the fragment (zero past the utterance)
  struct YRaw { float e[8], m[8]; };
  const TIO* Pv = P + (size_t)b * d.U * d.V + min(vcol, d.V - 1);
  const float* mPb = mP + (size_t)b * d.U;
  auto request_y = [&](int ks) {
    if constexpr (kDirect) {
      YRaw r;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int u = min(16 * ks + 8 * h + i, Ub - 1);
        r.e[i] = ldf(Pv + (size_t)u * d.V);
        r.m[i] = mPb[u];
      }
      return r;
    } else {
      const uint4* p = yw + (size_t)ks * 3 * 64;
      Frag3 y;
      y.h = p[0]; y.m = p[64]; y.l = p[128];
      return y;
    }
  };
  auto make_y = [&](const YRaw& r, int ks) -> Frag3 {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = 16 * ks + 8 * h + i < Ub ? __expf(r.e[i] - r.m[i]) : 0.0f;
    return split8(y);
  };
  int aslot[2][kM];
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int m = 0; m < kM; ++m) aslot[s][m] = wslot(32 * m + l32, 2 * s + h);

  // The instruction truncates what falls below its accumulator's last bit; every two slabs (24
  // instructions, 64 label positions) the sums go into a second set, rounded, and start again.
  floatx16 acc[kM], tot[kM];
#pragma unroll
  for (int m = 0; m < kM; ++m)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[m][r] = tot[m][r] = 0.0f;
  const int nk = (Ub + 31) >> 5;
  // The walk over the slabs with M blocks of 32 frames, one, two or four: what the utterance has left
  // for this tile (a last tile or a short utterance is multiplied at its own size).
  auto walk = [&](auto blocks) __attribute__((always_inline)) {
    constexpr int M = decltype(blocks)::value, kRows = (M + 1) / 2;  // (rows a thread stages)
    struct WRegs { float4 lo[kRows], hi[kRows]; };
    auto fetch = [&](int k) -> WRegs {  // (Up is a multiple of eight; Y is zero past the utterance)
      const int u = min(32 * k + 8 * c8, Up - 8);
      WRegs r;
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        r.lo[i] = *reinterpret_cast<const float4*>(pw[i] + u);
        r.hi[i] = *reinterpret_cast<const float4*>(pw[i] + u + 4);
      }
      return r;
    };
    auto stash = [&](int buf, const WRegs& r) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < kRows; ++i) {
        const float x[8] = {r.lo[i].x, r.lo[i].y, r.lo[i].z, r.lo[i].w,
                            r.hi[i].x, r.hi[i].y, r.hi[i].z, r.hi[i].w};
        const Frag3 f = split8(x);
        Xs[buf][0][slot[i]] = f.h;
        Xs[buf][1][slot[i]] = f.m;
        Xs[buf][2][slot[i]] = f.l;
      }
    };
    Frag3 y0, y1;
    YRaw n0, n1;  // (kDirect: the next slab's)
    // One slab, its order pinned as in the log-normaliser's: the second step's fragments are read under
    // the first step's instructions, a step's Y fragments are asked for again right after their last use.
    auto slab = [&](int kt, int cur) __attribute__((always_inline)) {
      const int ktn = min(kt + 1, nk - 1);
      const WRegs ws = fetch(ktn);
      if constexpr (kDirect) {
        y0 = make_y(n0, 2 * kt);
        y1 = make_y(n1, 2 * kt + 1);
        n0 = request_y(2 * ktn);
        n1 = request_y(2 * ktn + 1);
      }
      uint4 ah[M], am[M], al[M];
#pragma unroll
      for (int m = 0; m < M; ++m) al[m] = Xs[cur][2][aslot[0][m]];
#pragma unroll
      for (int m = 0; m < M; ++m) ah[m] = Xs[cur][0][aslot[0][m]];
#pragma unroll
      for (int m = 0; m < M; ++m) am[m] = Xs[cur][1][aslot[0][m]];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(al[m], y0.h, acc[m]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < M; ++m) al[m] = Xs[cur][2][aslot[1][m]];
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(ah[m], y0.l, acc[m]);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(am[m], y0.m, acc[m]);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(am[m], y0.h, acc[m]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < M; ++m) am[m] = Xs[cur][1][aslot[1][m]];
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(ah[m], y0.m, acc[m]);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(ah[m], y0.h, acc[m]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < M; ++m) ah[m] = Xs[cur][0][aslot[1][m]];
      if constexpr (!kDirect) y0 = request_y(2 * ktn);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(al[m], y1.h, acc[m]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(ah[m], y1.l, acc[m]);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(am[m], y1.m, acc[m]);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(am[m], y1.h, acc[m]);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(ah[m], y1.m, acc[m]);
#pragma unroll
      for (int m = 0; m < M; ++m) acc[m] = mfma_bf16(ah[m], y1.h, acc[m]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!kDirect) y1 = request_y(2 * ktn + 1);
      stash(cur ^ 1, ws);
      __syncthreads();
    };
    auto flush = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int r = 0; r < 16; ++r) { tot[m][r] += acc[m][r]; acc[m][r] = 0.0f; }
    };
    stash(0, fetch(0));
    if constexpr (kDirect) {
      n0 = request_y(0);
      n1 = request_y(1);
    } else {
      y0 = request_y(0);
      y1 = request_y(1);
    }
    __syncthreads();
    int kt = 0;
    for (; kt + 2 <= nk; kt += 2) {
      slab(kt, 0);
      slab(kt + 1, 1);
      flush();
    }
    if (kt < nk) {
      slab(kt, 0);
      flush();
    }
  };
  if (nk == 0) __syncthreads();
  else if (t0 + 32 >= Tb) walk(std::integral_constant<int, 1>{});
  else if (kDirect || t0 + 64 >= Tb) walk(std::integral_constant<int, 2>{});
  else walk(std::integral_constant<int, kM>{});

  // Write-out, 64 frames at a time: the tile's own scores are asked for, the label terms among this
  // wavefront's columns are added up in a block of LDS (a frame a lane, one label after the other, so
  // nothing collides), then X times the sums, less the terms.
  const float delta = deltas ? deltas[b] : 1.0f;
  const TIO* Eb = E + (size_t)b * d.T * d.V + min(vcol, d.V - 1);
  float* block = reinterpret_cast<float*>(&Xs[0][0][0]) + wave * (32 * kElBlockPitch);
  static_assert(4 * 32 * kElBlockPitch * sizeof(float) <= sizeof(Xs), "the blocks lie in the slabs' LDS");
  const bool terms = sp.labels != nullptr && Ub > 0;  // uniform
  const bool blank_here = terms && d.blank >= vcol0 && d.blank < vcol0 + 32;
  // (the last slab's barrier lies behind every read of the pieces)
#pragma unroll
  for (int p = 0; p < kM / 2; ++p) {
    if (t0 + 64 * p >= d.T) break;
    const int tl = t0 + 64 * p + lane;  // this lane's frame where lanes are frames
    float e[2][16];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int t = min(t0 + 64 * p + 32 * m + mfma_row(r, h), Tb - 1);
        e[m][r] = ldf(Eb + (size_t)t * d.V);
      }
    __builtin_amdgcn_sched_barrier(0);
    const bool any = nmatch > 0 || blank_here;  // uniform in the wavefront
    if (any) {
      const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
      for (int k = 0; k < 32 * kElBlockPitch / 4 / 64; ++k)
        reinterpret_cast<float4*>(block)[64 * k + lane] = zero;
      if (lane < 32 * kElBlockPitch / 4 % 64)
        reinterpret_cast<float4*>(block)[32 * kElBlockPitch / 4 / 64 * 64 + lane] = zero;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const float* em = sp.emT + (size_t)b * d.U * d.T + min(tl, Tb - 1);
      constexpr int kBatch = 8;
      for (int i0 = 0; i0 < nmatch; i0 += kBatch) {
        float term[kBatch];
        int col[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          const int u = Match[wave][min(i0 + k, nmatch - 1)];
          term[k] = em[(size_t)u * d.T];
          col[k] = label_at(sp.labels, d, b, u) - vcol0;
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k)
          if (i0 + k < nmatch) block[col[k] * kElBlockPitch + lane] -= term[k];
      }
      if (blank_here)
        block[(d.blank - vcol0) * kElBlockPitch + lane] += sp.bsum[(size_t)b * d.T + min(tl, Tb - 1)];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row0 = 32 * m + 8 * q + 4 * h;  // mfma_row(4 q, h) of the 64 frames
        float4 add = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (any) add = *reinterpret_cast<const float4*>(block + l32 * kElBlockPitch + row0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = 64 * p + row0 + i, t = t0 + row;
          const float x = exp_minus_scaled(e[m][4 * q + i], Ms[row]);
          const float g = x * tot[2 * p + m][4 * q + i] + f4at(add, i);
          if (t < d.T && vok) stf(out + (size_t)t * d.V + vcol, t < Tb ? delta * g : 0.0f);
        }
      }
    // (the block is cleared again by this wavefront only, after its own reads: LDS answers in order)
  }
}

template <typename TIO>
int egrads_long_any(const TIO* E, const TIO* P, const float* mE, const float* mP, const float* Wn,
                    const float* deltas, TIO* egrads, const int* inLen, const int* labLen,
                    const Dims& d, const SparseTerms& sparse, void* scratch, hipStream_t s) {
  if (sparse.labels && d.U - 1 > kMaxLabels)
    return fail(kInvalid, "egrads: blank/label terms can be folded in for at most %d labels",
                kMaxLabels);
  const int nvb = el_vblocks(d), nus = el_steps(d);
  const bool direct = d.T <= kElDirect;
  const int rows = direct ? kElDirectRows : kElRows, ttiles = (d.T + rows - 1) / rows, Up = wplane_up(d.U), Tw = wplane_tw(d.T);
  const uint4* Yt = static_cast<const uint4*>(scratch);
  if (direct) {
    hipLaunchKernelGGL((egrads_long_kernel<TIO, true>), dim3((d.V + 127) / 128, ttiles, d.B), dim3(256), 0,
                       s, E, P, Yt, mE, mP, Wn, deltas, egrads, inLen, labLen, d, Up, Tw, nvb, nus, 0,
                       sparse);
    RNNT_LAUNCH_CHECK("egrads_long_kernel");
    return kOk;
  }
  hipLaunchKernelGGL(yt_planes_kernel<TIO>, dim3(nvb, (nus + 3) / 4, d.B), dim3(256), 0, s, P, mP,
                     static_cast<uint4*>(scratch), labLen, d, nvb, nus);
  RNNT_LAUNCH_CHECK("yt_planes_kernel");
  for (int tile0 = 0; tile0 < ttiles; tile0 += 65535) {  // (what a grid's y holds)
    hipLaunchKernelGGL((egrads_long_kernel<TIO, false>),
                       dim3((d.V + 127) / 128, std::min(ttiles - tile0, 65535), d.B), dim3(256), 0, s,
                       E, P, Yt, mE, mP, Wn, deltas, egrads, inLen, labLen, d, Up, Tw, nvb, nus, tile0,
                       sparse);
    RNNT_LAUNCH_CHECK("egrads_long_kernel");
  }
  return kOk;
}

}  // namespace

// Where the streamed form takes more than one launch.  (us, that form and this one: B=8 T=10000 U=401
// V=1000, four slices 942 -> 515; T=2000 U=129 V=1000, two 88 -> 63; B=32 T=1000 U=150 V=5000
// 763 -> 569; B=1 T=1000 U=300 V=600 122 -> 37.  With one slice it is the streamed form, whose Y stays
// in registers: B=32 T=2000 U=101 V=10000 1190 against 1890, V=1000 190 against 222.)
// Y is prepared past 400 frames: with few frames the form that prepares it was slower than slices (B=64
// V=2500, ragged, slices, prepared, not: T=20 U=401 150, 232, 80; T=130 U=201 151, 180, 114; T=256
// U=201 220, 222, 177; T=400 U=401 627, 457, 401).  Time prepared over not, U=113 .. 700, V=100 .. 5000:
// up to 400 frames 0.92 .. 3.05, all below 1.03 where both take about 30 us; 600 frames 0.85 .. 1.52;
// from 1000 on mostly below 1 (2000: 0.75 .. 1.36, 10000: 0.66 .. 0.93).

int launch_egrads_long(const float* E, const float* P, const float* mE, const float* mP,
                       const float* Wn, const float* deltas, float* egrads, const int* inLen,
                       const int* labLen, const Dims& d, const SparseTerms& sparse, void* scratch,
                       hipStream_t s) {
  return egrads_long_any(E, P, mE, mP, Wn, deltas, egrads, inLen, labLen, d, sparse, scratch, s);
}
int launch_egrads_long(const bf16_t* E, const bf16_t* P, const float* mE, const float* mP,
                       const float* Wn, const float* deltas, bf16_t* egrads, const int* inLen,
                       const int* labLen, const Dims& d, const SparseTerms& sparse, void* scratch,
                       hipStream_t s) {
  return egrads_long_any(E, P, mE, mP, Wn, deltas, egrads, inLen, labLen, d, sparse, scratch, s);
}
int launch_egrads_long(const f16_t* E, const f16_t* P, const float* mE, const float* mP,
                       const float* Wn, const float* deltas, f16_t* egrads, const int* inLen,
                       const int* labLen, const Dims& d, const SparseTerms& sparse, void* scratch,
                       hipStream_t s) {
  return egrads_long_any(E, P, mE, mP, Wn, deltas, egrads, inLen, labLen, d, sparse, scratch, s);
}

}  // namespace rnnt
