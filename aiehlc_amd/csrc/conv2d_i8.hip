// int8 conv2d (NHWC x OHWI -> NHWC) with a per-output-channel requantize
// epilogue, as an im2col-free implicit GEMM on gfx950 MFMA.
//
// The reference's conv exists only as the generated control code of an AIE
// graph (thirdparty/adf/aie_control.cpp:854-1524: 8 `conv` kernels with
// ping/pong activation windows); no kernel source ships.  Semantics are the
// benchmark's: zero padding, stride, int32 accumulation, then
// y = sat_int8((acc + 2^(s_c-1)) >> s_c) per output channel c.
//
// Kernels: the row-block kernels (conv2d_i8_rows.hpp), conv2d_i8_taps,
// conv2d_i8_igemm, and conv2d_i8_flex for every other shape.
//
// GEMM view: rows = output pixels (n, ho, wo), columns = output channels,
// k = (r, s, ci).  A workgroup of conv2d_i8_igemm owns 64 consecutive pixels x 64 channels.
// Each of its 4 waves takes every 4th k-step of 32 (one (r, s, ci-block)),
// loading X and W fragments straight from global memory in MFMA operand
// layout (W rows are k-contiguous in OHWI; X pixels are ci-contiguous in
// NHWC), so no im2col buffer and no LDS staging of the operands.  The four
// partial 64x64 int32 tiles are summed through LDS, requantized and written
// as one contiguous 4 KiB run of NHWC output.
//
// Split K: when the tiles cover at most a third of the CUs (the deep layers
// of a CNN: few output pixels, long k = 9 * Cin), each tile's k-steps are divided
// among ksplit workgroups (grid.z), which write int32 partial sums to the
// context's workspace; conv2d_i8_splitk_reduce adds them and requantizes.
// The two kernels are ordered by the stream, so no atomics are involved and
// the sums are exact in any order.
#include <algorithm>

#include "conv2d_i8_rows.hpp"
#include "flex_tile.hpp"
#include "gfx950_ops.hpp"
#include "miaie_internal.hpp"

namespace {

namespace flex = miaie::flex;

__device__ __forceinline__ int requant1(int acc, int s) {
  int q = s ? (acc >> s) + ((acc >> (s - 1)) & 1) : acc;
  return min(max(q, -128), 127);
}

constexpr int PIX = 64;    // pixels per workgroup
constexpr int COB = 64;    // output channels per workgroup
constexpr int BATCH = 6;   // k-steps whose fragments are in flight per wave

// PARTIAL: k-steps [T z / ksplit, T (z+1) / ksplit) of the tile, z =
// blockIdx.z, summed into psum[z][pixel][channel] (int32, no requantize).
template <bool PARTIAL>
__global__ __launch_bounds__(256) void conv2d_i8_igemm(
    const int8_t* __restrict__ X, const int8_t* __restrict__ W, const uint8_t* __restrict__ shifts,
    int8_t* __restrict__ Y, int32_t* __restrict__ psum, int N, int H, int Wd, int Cin, int Cout, int R, int S,
    int stride, int pad, int Ho, int Wo, int ksplit) {
  __shared__ __attribute__((aligned(16))) int32_t part[4][PIX * COB];  // 64 KiB

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 31, fh = lane >> 5;
  const int P = N * Ho * Wo;
  const int p0 = blockIdx.x * PIX;
  const int co0 = blockIdx.y * COB;

  // the two pixels this lane feeds (one per 32-pixel block)
  int pn[2], phb[2], pwb[2];
  bool pvalid[2];
#pragma unroll
  for (int pb = 0; pb < 2; ++pb) {
    const int p = p0 + 32 * pb + fr;
    pvalid[pb] = p < P;
    const int pp = pvalid[pb] ? p : 0;
    const int wo = pp % Wo;
    const int t = pp / Wo;
    const int ho = t % Ho;
    pn[pb] = t / Ho;
    phb[pb] = ho * stride - pad;
    pwb[pb] = wo * stride - pad;
  }
  const int KW = R * S * Cin;  // weight row length (OHWI)
  const int8_t* wrow[2];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) wrow[cb] = W + (size_t)(co0 + 32 * cb + fr) * KW + 16 * fh;

  const int CBI = Cin / 32;
  const int T = R * S * CBI;
  const int tb = PARTIAL ? (int)((long long)T * blockIdx.z / ksplit) : 0;
  const int te = PARTIAL ? (int)((long long)T * (blockIdx.z + 1) / ksplit) : T;

  v16i acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = v16i{0};

  for (int t0 = tb + wave; t0 < te; t0 += 4 * BATCH) {
    v4i xf[BATCH][2], wf[BATCH][2];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const int t = t0 + 4 * u;
      if (t < te) {
        const int rs = t / CBI, cib = t - rs * CBI;
        const int r = rs / S, s = rs - r * S;
        const int koff = rs * Cin + cib * 32;
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) wf[u][cb] = MIAIE_LD(reinterpret_cast<const v4i*>(wrow[cb] + koff));
#pragma unroll
        for (int pb = 0; pb < 2; ++pb) {
          const int hi = phb[pb] + r, wi = pwb[pb] + s;
          const bool ok = pvalid[pb] && hi >= 0 && hi < H && wi >= 0 && wi < Wd;
          const int8_t* src = X + (((size_t)pn[pb] * H + hi) * Wd + wi) * Cin + cib * 32 + 16 * fh;
          xf[u][pb] = ok ? MIAIE_LD(reinterpret_cast<const v4i*>(src)) : v4i{0};
        }
      }
    }
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      if (t0 + 4 * u < te) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
          for (int pb = 0; pb < 2; ++pb)
            acc[cb][pb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[u][cb], xf[u][pb], acc[cb][pb], 0, 0, 0);
      }
    }
  }

  // acc[cb][pb][4g + t]: channel co = 32cb + 8g + 4*(lane/32) + t, pixel p = 32pb + lane%32.
  // Partial tile layout: [pixel][16-byte channel quad, XOR pixel%16].
  int32_t* mine = part[wave];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb)
#pragma unroll
    for (int pb = 0; pb < 2; ++pb)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int p = 32 * pb + fr;
        const int cq = (32 * cb + 8 * g + 4 * fh) >> 2;
        v4i v = {acc[cb][pb][4 * g], acc[cb][pb][4 * g + 1], acc[cb][pb][4 * g + 2], acc[cb][pb][4 * g + 3]};
        *reinterpret_cast<v4i*>(mine + p * COB + ((cq ^ (p & 15)) << 2)) = v;
      }
  __syncthreads();

  // thread -> pixel tid/4, channels 16*(tid%4) .. +16
  const int p = tid >> 2, c16 = (tid & 3) * 16;
  if (p0 + p >= P) return;
  int sum[16];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int cq = (c16 >> 2) + q;
    v4i s = v4i{0};
#pragma unroll
    for (int w = 0; w < 4; ++w) s += *reinterpret_cast<const v4i*>(part[w] + p * COB + ((cq ^ (p & 15)) << 2));
    sum[4 * q] = s[0];
    sum[4 * q + 1] = s[1];
    sum[4 * q + 2] = s[2];
    sum[4 * q + 3] = s[3];
  }
  if constexpr (PARTIAL) {
    int32_t* const dst = psum + ((size_t)blockIdx.z * P + p0 + p) * Cout + co0 + c16;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      MIAIE_ST(reinterpret_cast<v4i*>(dst + 4 * q), (v4i{sum[4 * q], sum[4 * q + 1], sum[4 * q + 2], sum[4 * q + 3]}));
    return;
  }
  uint32_t out[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t v = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int c = co0 + c16 + 4 * q + t;
      v |= (uint32_t)(requant1(sum[4 * q + t], MIAIE_LD(shifts + c)) & 0xFF) << (8 * t);
    }
    out[q] = v;
  }
  MIAIE_ST(reinterpret_cast<uint4*>(Y + (size_t)(p0 + p) * Cout + co0 + c16), make_uint4(out[0], out[1], out[2], out[3]));
}

// ------------------------------------------------------------ taps kernel
// LDS-staged implicit GEMM for Cin a multiple of 128 and Cout of 64 (the
// deep layers of a CNN, which the row-block kernel does not take).  The
// workgroup tile is 64 output pixels x 64 output channels, as in
// conv2d_i8_igemm, but the k loop runs over stages of one filter tap (r, s)
// and CK = 128 input channels, and each stage's two operands (the 64
// pixels' 128 channels at that tap, and the 64 channels' weights for it) are
// copied into an NS-stage LDS ring by global_load_lds_dwordx4 with eight
// lanes per 128-byte row: a copy instruction touches 8 cache lines, against
// 32 for a fragment loaded straight into MFMA layout.  The tap position is
// walked forward without division (a runtime division per stage cost more
// than the copies).  At Cin = 64 (two MFMAs per wave per stage) the per-stage
// barrier and waits outweigh this, and conv2d_i8_igemm is faster.  Positions
// outside the image are copied from a clamped address and their X fragments
// zeroed when read.  Each of the 4 waves owns 32 pixels x 32 channels (one
// v_mfma_i32_32x32x32_i8 accumulator), so there is no cross-wave reduction;
// with split K (grid.z) the tile's stages are divided among workgroups whose
// int32 partials conv2d_i8_splitk_reduce adds.
template <int TP, int TC>
struct TapsGeom {
  static constexpr int CK = 128;                    // input channels per stage
  static constexpr int NS = TP * TC > 64 * 64 ? 4 : 8;  // LDS stages in the ring
  static constexpr int CPR = CK / 16;               // 16-byte chunks per staged row
  static constexpr int XB = TP * CK, WB = TC * CK;  // the two operands of one stage
  static constexpr int STAGE = XB + WB;             // X rows, then W rows
  static constexpr int CPX = XB / 4096, CPW = WB / 4096;  // copies per thread per stage (256 x 16 bytes each)
  static constexpr int CPS = CPX + CPW;
  static constexpr int KS = CK / 32;                // 32-wide k-steps per stage
  static constexpr int NI = TP / 64, NJ = TC / 64;  // 32x32 blocks per wave (4 waves, 2 x 2)
  static constexpr int YP = TC / 2 + 16;            // epilogue: LDS pitch of a pixel's TC/2 output channels
  static constexpr int YW = TP / 2 * YP;            // one wave's output block
  static constexpr int LDS = NS * STAGE + 4 * YW;
  static_assert(CPX >= 1 && CPW >= 1 && NI >= 1 && NJ >= 1 && LDS <= 163840, "taps kernel staging");
  static_assert((NS - 2) * CPS <= 63, "copies in flight fit the vmcnt counter");
};

// Chunk swizzle of a staged 128-byte row: the 16 rows one half-wave
// fragment read touches land on distinct bank groups.
__device__ __forceinline__ int taps_swz(int row) { return (row >> 1) & 7; }

// Workgroup tile TP output pixels x TC output channels (64 x 64 for small
// grids, 128 x 128 otherwise); each wave owns TP/2 x TC/2, NI x NJ blocks of
// 32 x 32.
template <int TP, int TC, bool PARTIAL>
__global__ __launch_bounds__(256) void conv2d_i8_taps(
    const int8_t* __restrict__ X, const int8_t* __restrict__ W, const uint8_t* __restrict__ shifts,
    int8_t* __restrict__ Y, int32_t* __restrict__ psum, int N, int H, int Wd, int Cin, int Cout, int R, int S,
    int stride, int pad, int Ho, int Wo, int ksplit) {
  using G = TapsGeom<TP, TC>;
  constexpr int CK = G::CK, NI = G::NI, NJ = G::NJ;
  __shared__ __attribute__((aligned(1024))) int8_t lds[G::LDS];
  const uint32_t lds0 = miaie::dev::lds_addr(lds);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, fh = lane >> 5;
  const int pb = wave & 1, cb = wave >> 1;  // this wave's pixel half and channel half
  const int P = N * Ho * Wo;
  const int p0 = blockIdx.x * TP, co0 = blockIdx.y * TC;
  const int CB = Cin / CK, T = R * S * CB;
  const int sb = PARTIAL ? (int)((long long)T * blockIdx.z / ksplit) : 0;
  const int nst = (PARTIAL ? (int)((long long)T * (blockIdx.z + 1) / ksplit) : T) - sb;
  const int KW = R * S * Cin;

  // ---- copy geometry.  Copy i of wave w moves 1 KiB block q = 4i + w of an
  // operand: rows 8q + lane / 8, logical chunk (lane % 8) ^ swz(row), landing
  // at LDS byte 1024 q + 16 lane of the operand.
  int xhb[G::CPX], xwb[G::CPX];
  uint32_t xbase[G::CPX], wbase[G::CPW];
  const uint32_t rowx = (uint32_t)Wd * Cin;  // bytes per input row
#pragma unroll
  for (int i = 0; i < G::CPX; ++i) {
    const int row = (4 * i + wave) * 8 + lane / G::CPR;
    const int gc = (lane % G::CPR) ^ taps_swz(row);
    const int p = min(p0 + row, P - 1);  // rows past the last pixel copy a real one (never stored)
    const int wo = p % Wo, t = p / Wo;
    xhb[i] = (t % Ho) * stride - pad;
    xwb[i] = wo * stride - pad;
    xbase[i] = (uint32_t)((t / Ho) * H) * rowx + (uint32_t)(16 * gc);
  }
#pragma unroll
  for (int i = 0; i < G::CPW; ++i) {
    const int row = (4 * i + wave) * 8 + lane / G::CPR;
    wbase[i] = (uint32_t)((co0 + row) * KW + 16 * ((lane % G::CPR) ^ taps_swz(row)));
  }
  // this lane's fragment pixels (X rows TP/2 pb + 32 i + fr)
  bool pvalid[NI];
  int fhb[NI], fwb[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int pf = p0 + TP / 2 * pb + 32 * i + fr;
    pvalid[i] = pf < P;
    const int pp = pvalid[i] ? pf : 0;
    const int wo = pp % Wo, t = pp / Wo;
    fhb[i] = (t % Ho) * stride - pad;
    fwb[i] = wo * stride - pad;
  }

  // A stage position (filter row r, column s, channel chunk c) walked
  // forward without division.
  struct Tap {
    int r, s, c;
  };
  auto step = [&](Tap& t) {
    if (++t.c == CB) {
      t.c = 0;
      if (++t.s == S) {
        t.s = 0;
        ++t.r;
      }
    }
  };
  Tap at_issue, at_use;
  {
    const int rs = sb / CB;
    at_issue = Tap{rs / S, rs % S, sb % CB};
    at_use = at_issue;
  }
  const miaie::dbg::Span x_span = miaie::dbg::span_of(X), w_span = miaie::dbg::span_of(W);  // (debug build only)
  // copies of the stage at `t` into ring slot `slot`
  auto issue = [&](const Tap& t, int slot) {
    const uint32_t base = lds0 + slot * G::STAGE + 1024 * wave;
    const uint32_t wk = (uint32_t)((t.r * S + t.s) * Cin + t.c * CK), xk = (uint32_t)(t.c * CK);
    // X and W copies alternate (issuing all of one operand first measured 6%
    // slower at 64 x 64)
#pragma unroll
    for (int i = 0; i < (G::CPX > G::CPW ? G::CPX : G::CPW); ++i) {
      if (i < G::CPX) {
        const int hi = min(max(xhb[i] + t.r, 0), H - 1), wi = min(max(xwb[i] + t.s, 0), Wd - 1);
        miaie::dev::gload_lds16(X, xbase[i] + (uint32_t)hi * rowx + (uint32_t)wi * Cin + xk, base + 4096 * i, x_span);
      }
      if (i < G::CPW) miaie::dev::gload_lds16(W, wbase[i] + wk, base + G::XB + 4096 * i, w_span);
    }
  };

  v16i acc[NJ][NI];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[j][i] = v16i{0};
  const int8_t* const wfrag = lds + G::XB + (TC / 2 * cb + fr) * CK;
  const int8_t* const xfrag = lds + (TP / 2 * pb + fr) * CK;
  // the swizzle of rows r and r + 32 is the same: one per operand
  const int wsw = taps_swz(TC / 2 * cb + fr), xsw = taps_swz(TP / 2 * pb + fr);

#pragma unroll
  for (int i = 0; i < G::NS - 1; ++i)
    if (i < nst) {
      issue(at_issue, i);
      step(at_issue);
    }
  for (int s = 0; s < nst; ++s) {
    // this wave's copies of stage s have landed once only the stages issued
    // after it (at most NS - 2) are in flight; the barrier publishes everyone's
    // and frees the slot of stage s - 1 for stage s + NS - 1
    miaie::dev::wait_tiles_behind<G::CPS, G::NS - 1>(min(G::NS - 2, nst - 1 - s) + 1);
    miaie::dev::barrier();
    if (s + G::NS - 1 < nst) {
      issue(at_issue, (s + G::NS - 1) % G::NS);
      step(at_issue);
    }
    bool xin[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
      xin[i] = pvalid[i] && (unsigned)(fhb[i] + at_use.r) < (unsigned)H && (unsigned)(fwb[i] + at_use.s) < (unsigned)Wd;
    step(at_use);
    const int slot = (s % G::NS) * G::STAGE;
#pragma unroll
    for (int ks = 0; ks < G::KS; ++ks) {
      const int cw = ((2 * ks + fh) ^ wsw) << 4, cx = ((2 * ks + fh) ^ xsw) << 4;
      v4i wf[NJ], xf[NI];
#pragma unroll
      for (int j = 0; j < NJ; ++j) wf[j] = *reinterpret_cast<const v4i*>(wfrag + slot + 32 * CK * j + cw);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        xf[i] = *reinterpret_cast<const v4i*>(xfrag + slot + 32 * CK * i + cx);
        xf[i] = xin[i] ? xf[i] : v4i{0};
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < NI; ++i) acc[j][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[j], xf[i], acc[j][i], 0, 0, 0);
    }
  }

  // acc[j][i][4g + t]: channel TC/2 cb + 32j + 8g + 4fh + t, pixel TP/2 pb + 32i + fr
  if constexpr (PARTIAL) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int pf = p0 + TP / 2 * pb + 32 * i + fr;
      if (!pvalid[i]) continue;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        int32_t* const dst = psum + ((size_t)blockIdx.z * P + pf) * Cout + co0 + TC / 2 * cb + 32 * j + 4 * fh;
#pragma unroll
        for (int g = 0; g < 4; ++g)
          MIAIE_ST(reinterpret_cast<v4i*>(dst + 8 * g),
                   (v4i{acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]}));
      }
    }
    return;
  }
  // requantize into this wave's own LDS block (TP/2 pixels x TC/2 channels),
  // then 16-byte stores of whole pixel runs (an LDS wait, no workgroup barrier)
  int8_t* const yb = lds + G::NS * G::STAGE + wave * G::YW;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int cl = 32 * j + 4 * fh;  // channel within the wave's half
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint32_t sh = MIAIE_LD(reinterpret_cast<const uint32_t*>(shifts + co0 + TC / 2 * cb + cl + 8 * g));
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        uint32_t v = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t)
          v |= (uint32_t)(requant1(acc[j][i][4 * g + t], (sh >> (8 * t)) & 0xFF) & 0xFF) << (8 * t);
        *reinterpret_cast<uint32_t*>(yb + (32 * i + fr) * G::YP + cl + 8 * g) = v;
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS writes done
  __builtin_amdgcn_wave_barrier();
  constexpr int CPP = TC / 32;  // 16-byte chunks per pixel of the wave's half
#pragma unroll
  for (int it = 0; it < TP / 2 * CPP / 64; ++it) {
    const int flat = 64 * it + lane, sp = flat / CPP, ch = flat % CPP;
    const int p = p0 + TP / 2 * pb + sp;
    if (p < P) {
      const v4i v = *reinterpret_cast<const v4i*>(yb + sp * G::YP + 16 * ch);
      MIAIE_ST(reinterpret_cast<v4i*>(Y + (size_t)p * Cout + co0 + TC / 2 * cb + 16 * ch), v);
    }
  }
}

// The split-K epilogue: part[z][e] summed over z < ksplit for element e =
// pixel * Cout + channel, then the per-channel requantize.  One thread per 16
// channels of one pixel (Cout % 64 == 0).
__global__ __launch_bounds__(256) void conv2d_i8_splitk_reduce(const int32_t* __restrict__ part,
                                                               const uint8_t* __restrict__ shifts,
                                                               int8_t* __restrict__ Y, long long PC, int Cout,
                                                               int ksplit) {
  const long long e = ((long long)blockIdx.x * 256 + threadIdx.x) * 16;
  if (e >= PC) return;
  v4i s[4] = {v4i{0}, v4i{0}, v4i{0}, v4i{0}};
  for (int z = 0; z < ksplit; ++z) {
    const int32_t* src = part + (size_t)z * PC + e;
#pragma unroll
    for (int q = 0; q < 4; ++q) s[q] += MIAIE_LD(reinterpret_cast<const v4i*>(src + 4 * q));
  }
  const int c0 = (int)(e % Cout);
  uint32_t out[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t v = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t) v |= (uint32_t)(requant1(s[q][t], MIAIE_LD(shifts + c0 + 4 * q + t)) & 0xFF) << (8 * t);
    out[q] = v;
  }
  MIAIE_ST(reinterpret_cast<uint4*>(Y + e), make_uint4(out[0], out[1], out[2], out[3]));
}

// ------------------------------------------------------- register-staged kernel
// Workgroups per CU: the registers of eight (64 each) would spill.
template <class G>
constexpr int kPerCu = std::min(G::PER_CU, 6);

// Any shape, as an implicit GEMM on the register-staged tiles (flex_tile.hpp):
// rows are output pixels, columns output channels.  For one filter row r the
// S * Cin input bytes under the filter are one contiguous run of the image row
// hi = ho * stride - pad + r, and so are the weights' (r, :, :): k is taken as R such
// runs, each padded to whole 16-byte chunks (CPR per run).  The weights' chunks
// are zero past their run, so what the pixels' hold there does not matter
// (a neighbour's bytes); bytes outside the image row are zeroed.
struct RunShape {
  int H, Wd, Cin, R, Ho, Wo, stride, pad;
  int SC, CPR;                    // bytes per run (S * Cin), 16-byte chunks per run
  uint32_t cpr_inv, wo_inv, ho_inv;  // see div_small
};
// x / d with inv = floor(2^32 / d) + 1: exact for x * d < 2^32 and d > 1
__device__ __forceinline__ int div_small(int x, int d, uint32_t inv) { return d == 1 ? x : (int)__umulhi((uint32_t)x, inv); }

// chunk q = s * CH + ch of the k runs of pixels p0 + r0 + RPP i.  Byte
// offsets are 32-bit (the launcher keeps X below 2^31 bytes).
template <class G, int NL>
struct PixelLoader {
  const int8_t* X;
  const RunShape& k;
  int last;        // last offset a 16-byte load may start at
  int r0, ch;
  int n0, ho0, wo0;  // the thread's first pixel
  int hi0[NL];     // first input row under the filter (negative in the padding)
  int xb[NL];      // first byte of the run within its row (likewise)
  int at0[NL];     // its offset in X
  v4i v[NL];
  int keep[NL];    // valid bytes [keep & 255, keep >> 8)
  int moved[NL];   // distance a load was moved to stay inside X
  bool edge, shift;
  __device__ __forceinline__ PixelLoader(const int8_t* X_, const RunShape& k_, int total, int p0, int P, int tid)
      : X(X_), k(k_), last(total - 16), r0(tid / G::CH), ch(tid % G::CH), edge(false), shift(false) {
    const uint32_t p = (uint32_t)min(p0 + r0, P - 1), t = p / (uint32_t)k.Wo;
    wo0 = (int)(p - t * k.Wo);
    n0 = (int)(t / (uint32_t)k.Ho);
    ho0 = (int)t - n0 * k.Ho;
    rows();
  }
  // the tile dn images, dh rows and dw columns further (dh < Ho, dw < Wo)
  __device__ __forceinline__ void advance(int dn, int dh, int dw) {
    wo0 += dw;
    const int cw = wo0 >= k.Wo ? 1 : 0;
    wo0 -= cw ? k.Wo : 0;
    ho0 += dh + cw;
    const int chh = ho0 >= k.Ho ? 1 : 0;
    ho0 -= chh ? k.Ho : 0;
    n0 += dn + chh;
    rows();
  }
  // The thread's pixels from its first one: RPP i further, at most BM rows and
  // columns (small quotients).  Pixels past the last give offsets past the last
  // image, which load moves inside X: they are never stored.
  __device__ __forceinline__ void rows() {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int x = wo0 + G::RPP * i;
      const int dh = k.Wo > G::BM ? (int)(x >= k.Wo) : div_small(x, k.Wo, k.wo_inv);
      const int y = ho0 + dh, dn = k.Ho > G::BM ? (int)(y >= k.Ho) : div_small(y, k.Ho, k.ho_inv);
      hi0[i] = (y - dn * k.Ho) * k.stride - k.pad;
      xb[i] = ((x - dh * k.Wo) * k.stride - k.pad) * k.Cin;
      at0[i] = (int)((uint32_t)((n0 + dn) * k.H + hi0[i]) * (uint32_t)(k.Wd * k.Cin) + (uint32_t)xb[i]);
    }
  }
  __device__ __forceinline__ void load(int s) {
    const int q = s * G::CH + ch;
    int r = div_small(q, k.CPR, k.cpr_inv), c = q - r * k.CPR;
    if (r >= k.R) r = c = 0;  // past the last run (zero weights)
    const int row_bytes = k.Wd * k.Cin, step = r * row_bytes + 16 * c;
    bool e = false, m = false;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      // (a row outside the image is loaded from wherever the offset points,
      // moved inside X, and zeroed)
      const int at = (int)((uint32_t)at0[i] + (uint32_t)step), from = min(max(at, 0), last), b = xb[i] + 16 * c;
      v[i] = MIAIE_LD(reinterpret_cast<const flex::Any16*>(X + (uint32_t)from)).v;
      const int lo = min(max(-b, 0), 16);
      const int up = (unsigned)(hi0[i] + r) < (unsigned)k.H ? min(max(row_bytes - b, 0), 16) : 0;
      moved[i] = (int)((uint32_t)at - (uint32_t)from);
      keep[i] = lo | up << 8;
      e |= keep[i] != (16 << 8);
      m |= moved[i] != 0;
    }
    edge = __builtin_amdgcn_ballot_w64(e) != 0;
    shift = __builtin_amdgcn_ballot_w64(m) != 0;
  }
  __device__ __forceinline__ void put(int, int8_t* lds) {
    if (shift) {
#pragma unroll
      for (int i = 0; i < NL; ++i)
        v[i] = flex::shl_bytes(flex::shr_bytes(v[i], min(max(moved[i], 0), 16)), min(max(-moved[i], 0), 16));
    }
    if (edge) {
#pragma unroll
      for (int i = 0; i < NL; ++i) v[i] = v[i] & flex::byte_mask(keep[i] & 255, keep[i] >> 8);
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<v4i*>(lds + flex::row_off(G::KB, r0 + G::RPP * i, ch)) = v[i];
  }
};

// the same chunks of the weights of channels co0 + r0 + RPP i, zero past
// their run
template <class G, int NL>
struct WeightLoader {
  const int8_t* W;
  const RunShape& k;
  int last, r0, ch, valid;
  int at0[NL];
  v4i v[NL];
  int moved[NL];
  bool shift;
  __device__ __forceinline__ WeightLoader(const int8_t* W_, const RunShape& k_, int co0, int Cout, int tid)
      : W(W_), k(k_), last(Cout * k_.R * k_.SC - 16), r0(tid / G::CH), ch(tid % G::CH), valid(0), shift(false) {
#pragma unroll
    for (int i = 0; i < NL; ++i) at0[i] = min(co0 + r0 + G::RPP * i, Cout - 1) * (k.R * k.SC);
  }
  __device__ __forceinline__ void load(int s) {
    const int q = s * G::CH + ch;
    int r = div_small(q, k.CPR, k.cpr_inv), c = q - r * k.CPR;
    valid = r < k.R ? min(k.SC - 16 * c, 16) : 0;
    if (r >= k.R) r = c = 0;
    const int step = r * k.SC + 16 * c;
    bool m = false;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int at = at0[i] + step, from = min(at, last);
      v[i] = MIAIE_LD(reinterpret_cast<const flex::Any16*>(W + (uint32_t)from)).v;
      moved[i] = at - from;
      m |= moved[i] != 0;
    }
    shift = __builtin_amdgcn_ballot_w64(m) != 0;
  }
  __device__ __forceinline__ void put(int, int8_t* lds) {
    if (shift) {
#pragma unroll
      for (int i = 0; i < NL; ++i) v[i] = flex::shr_bytes(v[i], min(moved[i], 16));
    }
    const v4i mask = flex::byte_mask(0, valid);
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<v4i*>(lds + flex::row_off(G::KB, r0 + G::RPP * i, ch)) = v[i] & mask;
  }
};

// Bound by its vector instructions: the pixels' addresses, masks and the
// requantize outweigh the MFMAs.  8x48x48x96 -> 146, 5x5 (10 stages): 29 us,
// 19.9 ms with one thread per output.
template <class G>
__global__ __launch_bounds__(256, kPerCu<G>) void conv2d_i8_flex(const int8_t* __restrict__ X, const int8_t* __restrict__ W,
                                                         const uint8_t* __restrict__ shifts, int8_t* __restrict__ Y,
                                                         RunShape k, int x_bytes, int P, int Cout,
                                                         int8_t* __restrict__ work, int splits) {
  __shared__ __attribute__((aligned(1024))) int8_t lds[G::LDS];
  __shared__ int flag;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / G::WAVES_N, wn = wave % G::WAVES_N;
  int tm, tn;
  flex::tile_index<false>((P + G::BM - 1) / G::BM, (Cout + G::BN - 1) / G::BN, tm, tn);
  const int p0 = tm * G::BM, co0 = tn * G::BN;
  const int stages = (k.R * k.CPR + G::CH - 1) / G::CH, split = blockIdx.y;
  int s0, s1;
  flex::stage_range<G>(stages, split, splits, s0, s1);

  v4i acc[G::NI][G::NJ];
#pragma unroll
  for (int i = 0; i < G::NI; ++i)
#pragma unroll
    for (int j = 0; j < G::NJ; ++j) acc[i][j] = v4i{0};
  // this lane's channels' shifts, in flight during the main loop
  const int fr = lane & 15, fg = lane >> 4;
  int sh[G::NJ][4];
#pragma unroll
  for (int j = 0; j < G::NJ; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      sh[j][e] = MIAIE_LD(shifts + min(co0 + wn * G::WN + 16 * j + 4 * fg + e, Cout - 1));
  PixelLoader<G, G::NA> la(X, k, x_bytes, p0, P, tid);
  WeightLoader<G, G::NB> lb(W, k, co0, Cout, tid);
  flex::tile_loop<int8_t, G, false>(lds, la, lb, s0, s1, lane, wm, wn, acc);
  if (G::SPLITS && splits > 1 &&
      !flex::split_sum<int8_t, G>(acc, blockIdx.x, split, splits, work, miaie::ctx_counters(work), &flag, tid))
    return;

#pragma unroll
  for (int j = 0; j < G::NJ; ++j) {
    const int nl = wn * G::WN + 16 * j + 4 * fg;
#pragma unroll
    for (int i = 0; i < G::NI; ++i) {
      uint32_t y = 0;
      if (k.R * k.SC < (1 << 16)) {  // |acc| < 2^30: room for the rounding term
#pragma unroll
        for (int e = 0; e < 4; ++e)
          y |= (uint32_t)(min(max((acc[i][j][e] + (int)((1u << sh[j][e]) >> 1)) >> sh[j][e], -128), 127) & 0xFF) << (8 * e);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) y |= (uint32_t)(requant1(acc[i][j][e], sh[j][e]) & 0xFF) << (8 * e);
      }
      *reinterpret_cast<uint32_t*>(lds + (wm * G::WM + 16 * i + fr) * G::YP + nl) = y;
    }
  }
  __syncthreads();
  flex::store_y<G>(lds, Y, Cout, p0, co0, P, Cout, tid);
}

// The same for a k of one stage and more pixel tiles than workgroups that fit
// the GPU at once (a network's first layers): a workgroup keeps one channel
// tile, its weights in LDS and its shifts in registers, and walks over the
// pixel tiles first, first + step, ..., the next tile's loads in flight while
// this one is multiplied and stored.  grid.x: TN * step workgroups.
// 8x224x224x3 -> 64, 7x7, stride 2 (1568 tiles, k of 224 bytes): 11.3 us, 13.2 with
// a workgroup per tile, 919 with one thread per output; 16x224x224x1 -> 128, 3x3:
// 43.6 and 70.4 us; 8x201x201x96 -> 128, 1x1, stride 2: 9.2 and 11.8.
template <class G>
struct WalkGeom {
  static constexpr int LDS = G::A_BYTES + G::B_BYTES + G::BM * G::YP;
};
template <class G>
__global__ __launch_bounds__(256, kPerCu<G>) void conv2d_i8_flex_walk(
    const int8_t* __restrict__ X, const int8_t* __restrict__ W, const uint8_t* __restrict__ shifts,
    int8_t* __restrict__ Y, RunShape k, int x_bytes, int P, int Cout, int step, int dn, int dh, int dw) {
  __shared__ __attribute__((aligned(1024))) int8_t lds[WalkGeom<G>::LDS];
  int8_t* const bs = lds + G::A_BYTES;
  int8_t* const ys = bs + G::B_BYTES;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / G::WAVES_N, wn = wave % G::WAVES_N;
  const int TM = (P + G::BM - 1) / G::BM;
  const int tn = blockIdx.x / step, co0 = tn * G::BN;
  int tm = blockIdx.x - tn * step;
  const int fr = lane & 15, fg = lane >> 4;

  PixelLoader<G, G::NA> la(X, k, x_bytes, tm * G::BM, P, tid);
  WeightLoader<G, G::NB> lb(W, k, co0, Cout, tid);
  la.load(0);
  lb.load(0);
  int sh[G::NJ][4];
#pragma unroll
  for (int j = 0; j < G::NJ; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      sh[j][e] = MIAIE_LD(shifts + min(co0 + wn * G::WN + 16 * j + 4 * fg + e, Cout - 1));
  lb.put(0, bs);
  const int ksteps = (k.R * k.CPR + 3) / 4;  // 64-byte steps that hold any of k

  while (true) {
    la.put(0, lds);
    __syncthreads();  // (and the last tile's output rows have been read)
    const int next = tm + step;
    if (next < TM) {
      la.advance(dn, dh, dw);
      la.load(0);
    }
    v4i acc[G::NI][G::NJ];
#pragma unroll
    for (int i = 0; i < G::NI; ++i)
#pragma unroll
      for (int j = 0; j < G::NJ; ++j) acc[i][j] = v4i{0};
#pragma unroll
    for (int ks = 0; ks < G::KB / 64; ++ks) {
      if (ks >= ksteps) break;
      v4i a[G::NI], b[G::NJ];
#pragma unroll
      for (int i = 0; i < G::NI; ++i)
        a[i] = *reinterpret_cast<const v4i*>(lds + flex::row_off(G::KB, wm * G::WM + 16 * i + fr, 4 * ks + fg));
#pragma unroll
      for (int j = 0; j < G::NJ; ++j)
        b[j] = *reinterpret_cast<const v4i*>(bs + flex::row_off(G::KB, wn * G::WN + 16 * j + fr, 4 * ks + fg));
#pragma unroll
      for (int i = 0; i < G::NI; ++i)
#pragma unroll
        for (int j = 0; j < G::NJ; ++j) acc[i][j] = flex::Mma<int8_t>::mma(b[j], a[i], acc[i][j]);
    }
    // (k of one stage: |acc| < 2^22, room for the rounding term)
#pragma unroll
    for (int j = 0; j < G::NJ; ++j) {
      const int nl = wn * G::WN + 16 * j + 4 * fg;
#pragma unroll
      for (int i = 0; i < G::NI; ++i) {
        uint32_t y = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          y |= (uint32_t)(min(max((acc[i][j][e] + (int)((1u << sh[j][e]) >> 1)) >> sh[j][e], -128), 127) & 0xFF) << (8 * e);
        *reinterpret_cast<uint32_t*>(ys + (wm * G::WM + 16 * i + fr) * G::YP + nl) = y;
      }
    }
    __syncthreads();  // the output rows are whole, the pixels' LDS is free
    flex::store_y<G>(ys, Y, Cout, tm * G::BM, co0, P, Cout, tid);
    if (next >= TM) break;
    tm = next;
  }
}

// One thread per output element: a k of a few values (direct_us), operands of
// fewer than 16 bytes or above 2^31, and more tiles than a launch takes.
__global__ __launch_bounds__(256) void conv2d_i8_direct(const int8_t* __restrict__ X, const int8_t* __restrict__ W,
                                                        const uint8_t* __restrict__ shifts, int8_t* __restrict__ Y,
                                                        int N, int H, int Wd, int Cin, int Cout, int R, int S,
                                                        int stride, int pad, int Ho, int Wo) {
  const size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const size_t total = (size_t)N * Ho * Wo * Cout;
  if (idx >= total) return;
  const int co = (int)(idx % Cout);
  size_t t = idx / Cout;
  const int wo = (int)(t % Wo);
  t /= Wo;
  const int ho = (int)(t % Ho);
  const int n = (int)(t / Ho);
  uint32_t acc = 0;
  for (int r = 0; r < R; ++r) {
    const int hi = ho * stride + r - pad;
    if (hi < 0 || hi >= H) continue;
    for (int s = 0; s < S; ++s) {
      const int wi = wo * stride + s - pad;
      if (wi < 0 || wi >= Wd) continue;
      const int8_t* x = X + (((size_t)n * H + hi) * Wd + wi) * Cin;
      const int8_t* w = W + (((size_t)co * R + r) * S + s) * Cin;
      for (int ci = 0; ci < Cin; ++ci) acc += (uint32_t)((int)MIAIE_LD(x + ci) * (int)MIAIE_LD(w + ci));
    }
  }
  MIAIE_ST(Y + idx, (int8_t)requant1((int)acc, MIAIE_LD(shifts + co)));
}

}  // namespace

namespace miaie {

// Row-block shape: 4 output rows x 32 channels; 2 rows x 64 channels where
// Cout is a multiple of 64 and there are fewer than 8 output rows (a 4-row
// block would leave more of its rows empty).  Both shapes run the same
// number of workgroups; 4 x 32 stages 1.5 input rows per output row against
// 2, and half the weights, in fewer load instructions per workgroup, and
// measured 1-5% faster per launch at Cin 64 and 128 (56x56 and 112x112,
// Cout 64 and 128) and within 0.5% at Cin 32.
static bool rows_tall(int Ho, int Cout) { return Cout % 64 != 0 || Ho >= 8; }

template <int CIN>
static int launch_rows(miaie_ctx* ctx, const int8_t* X, const int8_t* W, const uint8_t* shifts, int8_t* Y, int N,
                       int H, int Wd, int Cout, int pad, int Ho, int Wo) {
  const hipError_t e =
      rows_tall(Ho, Cout)
          ? conv::launch_rows_as<CIN, 4, 32, false>(ctx->device, ctx->stream, X, W, shifts, Y, N, H, Wd, Cout, pad, Ho, Wo)
          : conv::launch_rows_as<CIN, 2, 64, false>(ctx->device, ctx->stream, X, W, shifts, Y, N, H, Wd, Cout, pad, Ho, Wo);
  return check_launch(ctx, e, "conv2d_i8_rows");
}

// Workgroups per tile of the implicit-GEMM kernels (1: no split).  Split
// when at least 3 workgroups per tile fit on the CUs (a 2-way split measured
// no faster: the reduce kernel's launch costs what the halved k-chain
// saves), into at most 8 and at most cus / tiles parts, each keeping at least
// min_per_split k-steps, with the partial sums inside the context's
// workspace of work_bytes.
static int conv_ksplit(size_t tiles, int T, int min_per_split, size_t elems, int cus, size_t work_bytes) {
  if (tiles * 3 > (size_t)cus) return 1;
  int ks = (int)std::min<size_t>((size_t)cus / tiles, 8);
  ks = std::min(ks, T / min_per_split);
  while (ks > 1 && (size_t)ks * elems * sizeof(int32_t) > work_bytes) --ks;
  return ks > 1 ? ks : 1;
}

// Estimated time of a launch (microseconds), for choosing between the
// chunked row-block kernel and the taps kernel: rounds of one workgroup per
// CU times a per-workgroup time fitted to back-to-back launches on MI355X
// (8x{56,28,14,7}^2 layers, Cin and Cout 256 and 512, 1x224^2x256 and
// 32x{28,14}^2 layers): a fixed start and end cost plus a cost per 64-channel
// chunk or per taps stage.
static double launch_rounds(size_t wgs, int cus) { return (double)((wgs + cus - 1) / cus); }

// conv2d_i8_rowsk<rows, 32*nj, nj, bw>: blocks of bw columns (64, or 32 for
// narrow layers) x rows = 256/bw rows, 8 waves of 32 pixels x 32*nj channels
struct RowsDeepTile {
  int nj, bw;
};
static double rows_deep_us(int N, int Ho, int Wo, int Cin, int Cout, RowsDeepTile t, int cus) {
  const int rows = 256 / t.bw;
  const size_t wgs = (size_t)N * ((Ho + rows - 1) / rows) * ((Wo + t.bw - 1) / t.bw) * (size_t)(Cout / (32 * t.nj));
  const int nk = Cin / 64;
  return launch_rounds(wgs, cus) * (t.nj == 2 ? 3.5 + 1.68 * nk : 2.8 + 1.0 * nk);
}

// Tile of the chunked row-block kernel with the lowest estimate: 32 x 64
// waves (two MFMAs per pixel fragment, 3/4 of the LDS reads per MAC) unless
// they leave so few workgroups that 32 x 32 finishes first; 32-column blocks
// where 64 would leave most columns empty (Wo <= 32, or just above 64).
static RowsDeepTile rows_deep_tile(int N, int Ho, int Wo, int Cin, int Cout, int cus) {
  RowsDeepTile best{1, 64};
  double best_us = rows_deep_us(N, Ho, Wo, Cin, Cout, best, cus);
  for (RowsDeepTile t : {RowsDeepTile{2, 64}, RowsDeepTile{2, 32}, RowsDeepTile{1, 32}}) {
    if (t.nj == 2 && Cout % 64) continue;
    const double us = rows_deep_us(N, Ho, Wo, Cin, Cout, t, cus);
    if (us < best_us) best = t, best_us = us;
  }
  return best;
}

// conv2d_i8_rows<3,3,128,...> (98 KiB of LDS at 4 rows x 32 channels, 116 KiB
// at 2 x 64: one workgroup per CU), 3.5-3.6 us per workgroup (8x112x112x128
// in 7 rounds, 24.4-25.1 us)
static double rows128_us(int N, int Ho, int Wo, int Cout, int cus) {
  const int rows = rows_tall(Ho, Cout) ? 4 : 2, wco = rows_tall(Ho, Cout) ? 32 : 64;
  const size_t wgs = (size_t)N * ((Ho + rows - 1) / rows) * ((Wo + conv::PB - 1) / conv::PB) * (size_t)(Cout / wco);
  return launch_rounds(wgs, cus) * 3.57;
}

// conv2d_i8_taps as its launcher runs it: 128 x 128 tiles when they fill a
// round of CUs, else 64 x 64 split over k; a stage is one tap x 128 channels.
static bool taps_big(size_t P, int Cout, int cus) {
  return Cout % 128 == 0 && ((P + 127) / 128) * (size_t)(Cout / 128) >= (size_t)cus;
}
static int taps_ksplit(size_t P, int Cin, int Cout, int R, int S, int cus, size_t work_bytes) {
  if (taps_big(P, Cout, cus)) return 1;
  return conv_ksplit(((P + 63) / 64) * (size_t)(Cout / 64), R * S * (Cin / 128), 4, P * Cout, cus, work_bytes);
}
static double taps_us(size_t P, int Cin, int Cout, int R, int S, int cus, size_t work_bytes) {
  const int stages = R * S * (Cin / 128);
  const size_t t128 = ((P + 127) / 128) * (size_t)(Cout / 128);
  if (taps_big(P, Cout, cus)) return launch_rounds(t128, cus) * (4.0 + 0.69 * stages);
  const size_t t64 = ((P + 63) / 64) * (size_t)(Cout / 64);
  const int ks = taps_ksplit(P, Cin, Cout, R, S, cus, work_bytes);
  return launch_rounds(t64 * ks, cus) * (2.5 + 0.41 * stages / ks) + (ks > 1 ? 3.0 : 0.0);
}

static int igemm_ksplit(size_t P, int Cin, int Cout, int R, int S, int cus, size_t work_bytes) {
  return conv_ksplit(((P + PIX - 1) / PIX) * (size_t)(Cout / COB), R * S * (Cin / 32), 4 * BATCH, P * Cout, cus, work_bytes);
}

// The kernel choice weighs estimated times on `cus` compute units: the
// context's count at launch (miaie_plan_set_cus or the device's), and an
// MI355X's 256 for miaie_plan_conv2d_i8, which has no context.  work_bytes:
// room for split-K partial sums (0: no split).
int conv2d_kernel_for(int N, int H, int Wd, int Cin, int Cout, int R, int S, int stride, int pad, bool aligned16,
                      bool shifts_aligned4, int cus, size_t work_bytes) {
  const int Ho = (H + 2 * pad - R) / stride + 1;
  const int Wo = (Wd + 2 * pad - S) / stride + 1;
  const size_t P = (size_t)N * Ho * Wo;
  // Row-block kernel (3x3, stride 1, Cin 32, 64 or 128; rows wider than 64
  // output columns in blocks of 64).  Its offsets are 32-bit: X, Y and W
  // (co0 * R*S*Cin) must each stay below 2^31 bytes, and the channel blocks
  // (>= 32 channels each) fit grid.y.
  const bool rows_ok = stride == 1 && R == 3 && S == 3 && (Cin == 32 || Cin == 64 || Cin == 128) && Cout % 32 == 0 &&
                       aligned16 && shifts_aligned4 && N <= 65535 &&
                       (size_t)N * H * Wd * Cin < ((size_t)1 << 31) && (size_t)N * Ho * Wo * Cout < ((size_t)1 << 31) &&
                       (size_t)Cout * R * S * Cin < ((size_t)1 << 31) && Cout / 32 <= 65535;
  // The same kernel over 64-channel chunks of a deeper Cin (the rounding
  // term in the accumulator start needs 9 * Cin * 2^14 < 2^30).
  const bool deep_ok = stride == 1 && R == 3 && S == 3 && Cin % 64 == 0 && Cin <= 4096 && Cout % 32 == 0 &&
                       aligned16 && shifts_aligned4 && N <= 65535 &&
                       (size_t)N * H * Wd * Cin < ((size_t)1 << 31) && (size_t)N * Ho * Wo * Cout < ((size_t)1 << 31) &&
                       (size_t)Cout * R * S * Cin < ((size_t)1 << 31) && Cout / 32 <= 65535;
  if (rows_ok) {
    // At Cin = 128 both apply: the chunked kernel's 32-column blocks leave
    // fewer empty columns on narrow layers, which pays where the row-block
    // kernel's grid takes more than one round of CUs
    if (Cin == 128 && deep_ok) {
      const RowsDeepTile t = rows_deep_tile(N, Ho, Wo, Cin, Cout, cus);
      if (rows_deep_us(N, Ho, Wo, Cin, Cout, t, cus) < rows128_us(N, Ho, Wo, Cout, cus))
        return MIAIE_CONV_ROWS_DEEP;
    }
    return MIAIE_CONV_ROWS;
  }
  // LDS-staged taps kernel (Cin a multiple of 128, Cout of 64): 32-bit copy
  // offsets, so X and W each stay below 2^31 bytes; 4-byte shift loads.
  const bool taps_ok = Cin % 128 == 0 && Cout % 64 == 0 && aligned16 && shifts_aligned4 &&
                       (size_t)N * H * Wd * Cin < ((size_t)1 << 31) && (size_t)Cout * R * S * Cin < ((size_t)1 << 31) &&
                       P < ((size_t)1 << 31) && Cout / 64 <= 65535;
  if (deep_ok && taps_ok) {
    const RowsDeepTile t = rows_deep_tile(N, Ho, Wo, Cin, Cout, cus);
    return rows_deep_us(N, Ho, Wo, Cin, Cout, t, cus) <=
                   taps_us(P, Cin, Cout, R, S, cus, work_bytes)
               ? MIAIE_CONV_ROWS_DEEP
               : MIAIE_CONV_TAPS;
  }
  if (deep_ok) return MIAIE_CONV_ROWS_DEEP;
  if (taps_ok) return MIAIE_CONV_TAPS;
  const bool fast = Cin % 32 == 0 && Cout % COB == 0 && aligned16 && P < ((size_t)1 << 31) &&
                    (P + PIX - 1) / PIX < ((size_t)1 << 31) && Cout / COB <= 65535;
  if (fast) return MIAIE_CONV_IGEMM;
  return MIAIE_CONV_DIRECT;
}

// The register-staged kernel: X and W of at least 16 bytes (one load) and
// below 2^31, with the padding around X included (offsets of runs that start
// in it are computed before they are moved inside).
static bool flex_ok(int N, int H, int Wd, int Cin, int Cout, int R, int S, int pad, size_t P) {
  const size_t sc = (size_t)S * Cin, cpr = (sc + 15) / 16, lim = ((size_t)1 << 31) - (1 << 12);
  const size_t row = ((size_t)Wd + 2 * (size_t)pad) * Cin + 16;
  return (size_t)N * H * Wd * Cin >= 16 && (size_t)Cout * R * sc >= 16 && row < lim &&
         ((size_t)N * H + 2 * (size_t)pad + R) * row < lim && (size_t)Cout * R * sc < lim && P < lim &&
         (R * cpr + 64) * cpr < ((size_t)1 << 32);
}

// its tile and split (bm = 0: more tiles than a launch takes).  64-byte stages
// (half the time of a 256-byte one for a k of 48 bytes and up to 64 channels) are
// left out where a walk over pixel tiles of longer stages is the faster one: for a
// k of two of them over more than four 64x64 tiles per CU (16x64x64x96->192, 1x1:
// 11.9 and 10.0 us), and of one over whole 128-column tiles and more than 64 per
// CU (8x224x224x64->256, 1x1: 47.9 and 43.6; at 24 per CU,
// 8x112x112x64->256: 12.6 and 15.6).
static flex::Plan flex_plan(miaie_ctx* ctx, long P, int Cin, int Cout, int R, int S) {
  const long k_bytes = 16l * R * ((S * Cin + 15) / 16), tiles64 = ((P + 63) / 64) * ((Cout + 63) / 64);
  const bool short_ok = k_bytes <= flex::Short::KB ? (Cout - 1) % 128 < 64 || tiles64 <= 64l * ctx->cus
                                                   : tiles64 <= 4l * ctx->cus;
  auto plan = [&](bool can_split) {
    return short_ok ? flex::plan(P, Cout, k_bytes, 1.5, ctx->cus, can_split, ctx->work_bytes)
                    : flex::plan_of<flex::Skinny, flex::Small, flex::Large>(P, Cout, k_bytes, 1.5, ctx->cus, can_split,
                                                                            ctx->work_bytes);
  };
  const flex::Plan f = plan(true);
  return f.splits > 1 && !may_split(ctx) ? plan(false) : f;
}

// Estimated time (us) of one thread per output: the chain of one output's loads,
// or the outputs' loads and address arithmetic over all CUs (fitted to 296
// layers of k <= 80 on 256 CUs; strided pixels cost more the deeper they are).
// A k of a few values leaves a tile's stage and MFMAs mostly empty: against the
// tile the register-staged kernel plans, 8x224x224x2 -> 1, 3x3: 7.6 and 13.2 us;
// 8x112x112x4 -> 4, 1x1: 3.3 and 5.1; on the other side of the line
// 8x224x224x3 -> 64, 7x7, stride 2: 919 and 11.3, 4x112x112x8 -> 8, 1x1: 4.6
// and 5.2.
static double direct_us(size_t outputs, int Cin, int R, int S, int cus) {
  const double taps = (double)R * S, k = taps * Cin;
  return 2.25 + std::max(0.1 * taps + 0.075 * k,
                         (double)outputs * 256e-6 / cus * (2.0 + 0.23 * taps + (0.46 + 0.02 * Cin) * k));
}

static int launch_flex(miaie_ctx* ctx, const flex::Plan& f, const int8_t* X, const int8_t* W, const uint8_t* shifts,
                       int8_t* Y, int N, int H, int Wd, int Cin, int Cout, int R, int S, int stride, int pad, int Ho,
                       int Wo) {
  RunShape k{H, Wd, Cin, R, Ho, Wo, stride, pad, S * Cin, (S * Cin + 15) / 16, 0, 0, 0};
  auto inverse = [](int d) { return (uint32_t)(((uint64_t)1 << 32) / (uint64_t)d + 1); };
  k.cpr_inv = inverse(k.CPR);
  k.wo_inv = inverse(Wo);
  k.ho_inv = inverse(Ho);
  const long P = (long)N * Ho * Wo;
  hipError_t e = hipSuccess;
  flex::with_geom(f, [&](auto g) {
    using G = typename decltype(g)::type;
    const long tn = (Cout + G::BN - 1) / G::BN, tm = f.tiles / tn;
    // one stage, and pixel tiles for more than one round of the workgroups
    // that fit (kPerCu: 4 per CU of 64x64, 2 of 128x128, 6 with 64-byte stages).
    // (Fewer workgroups, each with the same number of tiles: 12.7 us against 11.3 for
    // 8x224x224x3 -> 64, 7x7, stride 2.)
    const long step = std::max(1l, (long)kPerCu<G> * ctx->cus / tn);
    if (16 * R * k.CPR <= G::KB && tm > step) {
      const long pixels = step * G::BM;  // from one of a workgroup's tiles to its next
      e = launch<conv2d_i8_flex_walk<G>>(ctx->device, dim3((unsigned)(tn * step)), dim3(256), 0, ctx->stream, X, W,
                                         shifts, Y, k, N * H * Wd * Cin, (int)P, Cout, (int)step,
                                         (int)(pixels / Wo / Ho), (int)(pixels / Wo % Ho), (int)(pixels % Wo));
      return;
    }
    e = launch<conv2d_i8_flex<G>>(ctx->device, dim3((unsigned)f.tiles, (unsigned)f.splits), dim3(256), 0, ctx->stream, X,
                                  W, shifts, Y, k, N * H * Wd * Cin, (int)P, Cout, static_cast<int8_t*>(ctx->work), f.splits);
  });
  return check_launch(ctx, e, "conv2d_i8_flex");
}

int launch_conv2d_i8(miaie_ctx* ctx, const int8_t* X, const int8_t* W, const uint8_t* shifts, int8_t* Y,
                     int N, int H, int Wd, int Cin, int Cout, int R, int S, int stride, int pad) {
  const int Ho = (H + 2 * pad - R) / stride + 1;
  const int Wo = (Wd + 2 * pad - S) / stride + 1;
  const size_t P = (size_t)N * Ho * Wo;
  const bool al16 = aligned(X, 16) && aligned(W, 16) && aligned(Y, 16), al4 = aligned(shifts, 4);
  int kernel = conv2d_kernel_for(N, H, Wd, Cin, Cout, R, S, stride, pad, al16, al4, ctx->cus, ctx->work_bytes);
  int ks = kernel == MIAIE_CONV_TAPS    ? taps_ksplit(P, Cin, Cout, R, S, ctx->cus, ctx->work_bytes)
           : kernel == MIAIE_CONV_IGEMM ? igemm_ksplit(P, Cin, Cout, R, S, ctx->cus, ctx->work_bytes)
                                        : 1;
  if (ks > 1 && !may_split(ctx)) {  // planned again without the workspace
    kernel = conv2d_kernel_for(N, H, Wd, Cin, Cout, R, S, stride, pad, al16, al4, ctx->cus, 0);
    ks = 1;
  }
  if (kernel == MIAIE_CONV_ROWS) {
    if (Cin == 128) return launch_rows<128>(ctx, X, W, shifts, Y, N, H, Wd, Cout, pad, Ho, Wo);
    if (Cin == 64) return launch_rows<64>(ctx, X, W, shifts, Y, N, H, Wd, Cout, pad, Ho, Wo);
    return launch_rows<32>(ctx, X, W, shifts, Y, N, H, Wd, Cout, pad, Ho, Wo);
  }
  if (kernel == MIAIE_CONV_ROWS_DEEP) {
    const RowsDeepTile t = rows_deep_tile(N, Ho, Wo, Cin, Cout, ctx->cus);
    const int dev = ctx->device;
    hipError_t e;
    if (t.bw == 64 && t.nj == 2)
      e = conv::launch_rowsk_as<4, 64, 2, 64>(dev, ctx->stream, X, W, shifts, Y, N, H, Wd, Cin, Cout, pad, Ho, Wo);
    else if (t.bw == 64)
      e = conv::launch_rowsk_as<4, 32, 1, 64>(dev, ctx->stream, X, W, shifts, Y, N, H, Wd, Cin, Cout, pad, Ho, Wo);
    else if (t.nj == 2)
      e = conv::launch_rowsk_as<8, 64, 2, 32>(dev, ctx->stream, X, W, shifts, Y, N, H, Wd, Cin, Cout, pad, Ho, Wo);
    else
      e = conv::launch_rowsk_as<8, 32, 1, 32>(dev, ctx->stream, X, W, shifts, Y, N, H, Wd, Cin, Cout, pad, Ho, Wo);
    return check_launch(ctx, e, "conv2d_i8_rowsk");
  }
  if (kernel == MIAIE_CONV_TAPS) {
    // 128 x 128 tiles when they fill at least one round of CUs, else 64 x 64
    // (split over k when even those leave most CUs idle)
    const bool big = taps_big(P, Cout, ctx->cus);
    const int tp = big ? 128 : 64;
    const unsigned pxb = (unsigned)((P + tp - 1) / tp), chb = (unsigned)(Cout / tp);
    const int dev = ctx->device;
    if (big) {
      const hipError_t e = launch<conv2d_i8_taps<128, 128, false>>(dev, dim3(pxb, chb, 1), dim3(256), 0, ctx->stream,
                                                                   X, W, shifts, Y, nullptr, N, H, Wd, Cin, Cout, R,
                                                                   S, stride, pad, Ho, Wo, 1);
      return check_launch(ctx, e, "conv2d_i8_taps (128 x 128)");
    }
    if (ks > 1) {
      int32_t* const psum = static_cast<int32_t*>(ctx->work);
      hipError_t e = launch<conv2d_i8_taps<64, 64, true>>(dev, dim3(pxb, chb, (unsigned)ks), dim3(256), 0,
                                                          ctx->stream, X, W, shifts, Y, psum, N, H, Wd, Cin, Cout, R,
                                                          S, stride, pad, Ho, Wo, ks);
      if (int rc = check_launch(ctx, e, "conv2d_i8_taps (split K)")) return rc;
      const long long PC = (long long)(P * Cout);
      e = launch<conv2d_i8_splitk_reduce>(dev, dim3((unsigned)((PC / 16 + 255) / 256)), dim3(256), 0, ctx->stream,
                                          psum, shifts, Y, PC, Cout, ks);
      return check_launch(ctx, e, "conv2d_i8_splitk_reduce");
    }
    const hipError_t e = launch<conv2d_i8_taps<64, 64, false>>(dev, dim3(pxb, chb, 1), dim3(256), 0, ctx->stream, X,
                                                               W, shifts, Y, nullptr, N, H, Wd, Cin, Cout, R, S,
                                                               stride, pad, Ho, Wo, 1);
    return check_launch(ctx, e, "conv2d_i8_taps");
  }
  // From three 64x64 tiles per CU on, the register-staged kernel in place of the
  // implicit GEMM on fragments from memory, whose fragment loads touch 32 lines
  // each (4x112x112x96->256, 3x3: 38.1 against 33.2 us; 8x64x64x160->512, 1x1:
  // 25.9 against 15.5).  (Below three its workgroups start sooner:
  // 2x56x56x64->64, stride 2, 25 tiles: 4.7 against 6.8.)  But below six not for
  // larger filters of stride 1, whose pixels come from the L1 and L2 for each
  // further channel tile (32x28x28x96->128, 5x5, 3.1 tiles per CU: 26.1 against
  // 32.9; with one channel tile, 1x250x250x224->64, 3x3: 27.1 against 23.8), nor
  // over few channels (16x64x64x32->192, 7x7, stride 2: 15.6 against 19.6;
  // 16x64x64x320->192, 3x3, stride 2: 33.2 against 26.7); and not at all over 32
  // channels with half a 128x128 tile left over (8x112x112x32->192, 5x5: 50.7
  // against 55.8).
  const size_t tiles64 = ((P + 63) / 64) * (size_t)((Cout + 63) / 64), cus = (size_t)ctx->cus;
  const bool early = R * S == 1 || (stride > 1 ? Cin >= 96 : Cin >= 128 && Cout == 64);
  const bool big = tiles64 >= (early ? 3 : 6) * cus && !(R * S > 1 && stride == 1 && Cin == 32 && Cout % 128);
  flex::Plan f;
  if ((kernel != MIAIE_CONV_IGEMM || big) && flex_ok(N, H, Wd, Cin, Cout, R, S, pad, P))
    f = flex_plan(ctx, (long)P, Cin, Cout, R, S);
  if (kernel == MIAIE_CONV_IGEMM && !f.bm) {
    const unsigned pxb = (unsigned)((P + PIX - 1) / PIX), chb = (unsigned)(Cout / COB);
    if (ks > 1) {
      int32_t* const part = static_cast<int32_t*>(ctx->work);
      hipError_t e = launch<conv2d_i8_igemm<true>>(ctx->device, dim3(pxb, chb, (unsigned)ks), dim3(256), 0,
                                                   ctx->stream, X, W, shifts, Y, part, N, H, Wd, Cin, Cout, R, S,
                                                   stride, pad, Ho, Wo, ks);
      if (int rc = check_launch(ctx, e, "conv2d_i8_igemm (split K)")) return rc;
      const long long PC = (long long)(P * Cout);
      e = launch<conv2d_i8_splitk_reduce>(ctx->device, dim3((unsigned)((PC / 16 + 255) / 256)), dim3(256), 0,
                                          ctx->stream, part, shifts, Y, PC, Cout, ks);
      return check_launch(ctx, e, "conv2d_i8_splitk_reduce");
    }
    const hipError_t e = launch<conv2d_i8_igemm<false>>(ctx->device, dim3(pxb, chb), dim3(256), 0, ctx->stream, X, W,
                                                        shifts, Y, nullptr, N, H, Wd, Cin, Cout, R, S, stride, pad,
                                                        Ho, Wo, 1);
    return check_launch(ctx, e, "conv2d_i8_igemm");
  }
  // (the plan's estimates of one stage are a tenth low, those of a walk over pixel
  // tiles as much high or more)
  const bool tiny_k = Cin <= 16 && R * S <= 80 && R * S * Cin <= 80 && P * Cout < ((size_t)1 << 32) - 256;  // (threads)
  const double actual = f.kb > flex::Short::KB && f.tiles > 4l * ctx->cus ? 0.9 : 1.1;
  if (f.bm && !(tiny_k && direct_us(P * Cout, Cin, R, S, ctx->cus) < actual * f.us))
    return launch_flex(ctx, f, X, W, shifts, Y, N, H, Wd, Cin, Cout, R, S, stride, pad, Ho, Wo);
  const size_t total = P * Cout;
  const size_t blocks = (total + 255) / 256;
  if (blocks >= ((size_t)1 << 31)) return fail(ctx, MIAIE_EINVAL, "conv2d: output too large for the direct kernel");
  const hipError_t e = launch<conv2d_i8_direct>(ctx->device, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, X, W,
                                                shifts, Y, N, H, Wd, Cin, Cout, R, S, stride, pad, Ho, Wo);
  return check_launch(ctx, e, "conv2d_i8_direct");
}

}  // namespace miaie
