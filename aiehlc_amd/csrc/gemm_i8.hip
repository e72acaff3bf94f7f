// int8 x int8 -> int32 GEMM on gfx950 MFMA, with the fused requantize epilogue.
//
// Counterpart of the AIE `mm`/`perf` MAC loops (example/matrixmultiply/
// aieml_mm.cc:68-76, example/perf/aieml_perf.cc:69-82) generalised to int8
// operands and any M, N, K, and of the 64x64 sub-tiling that aiehlc's
// tiling prototype plans (src/mlir/mlirfront/tilinglinalg/tilinglinalg.cpp:101-103).
//
// Kernels:
//   gemm_i8_pipe    BM x BN x 64 workgroup tiles (256x256, 256x128, 128x128),
//                   4 waves of BM/2 x BN/2, v_mfma_i32_32x32x32_i8; a 4-stage
//                   LDS pipeline (the DMA ping-pong of aietypes.td:56-76 / the
//                   BD pairs of aie_control.cpp:854-875, generalised) filled
//                   by global_load_lds_dwordx4; the row-major (NN) B operand
//                   is transposed by ds_read_b64_tr_b8 on its way out of LDS.
//                   XCD-aware tile order.  K % 64 == 0, M >= BM, N >= BN;
//                   a tile that does not divide M (N) has its last tile row
//                   (column) moved back to end at M (N), overlapping the one
//                   before it (dev::tile_origin), which needs N % 16 == 0
//                   when BN does not divide N (16-byte column chunks).
//   gemm_i8_pipe16  256-row tiles with K % 128 == 0: the same pipeline with A
//                   staged two k-tiles at a time (A copies move whole cache
//                   lines), multiplied on v_mfma_i32_16x16x64_i8, which runs
//                   at a higher clock than the 32x32 form under the power
//                   limit; gemm_i8_pipe16_mixed puts 256x256 and 256x128
//                   tiles in one launch.
//   gemm_i8_flex    register-staged 16x128, 64x64 and 128x128 tiles
//                   (flex_tile.hpp) for every other shape, stride and
//                   alignment with K >= 16; K split over workgroups where
//                   tiles are few.
//   gemm_i8_tile64  64x64x64 tile, bounds-checked, for K < 16.
// The requantize epilogue (round, shift, saturate, optional ReLU) is fused
// into all of them.
//
// MFMA operand roles are swapped (srcA = B fragment, srcB = A fragment) so
// that each lane's accumulator holds 4 consecutive output columns of one row:
// one dword of int8 output or one 16-byte int32 vector per 4 values.
#include <type_traits>

#include "flex_tile.hpp"
#include "gemm_i8_kernels.hpp"
#include "gfx950_ops.hpp"
#include "miaie_internal.hpp"

namespace {

namespace dev = miaie::dev;
using namespace miaie::gemm;
using miaie::kernel_t;
using miaie::launch;
namespace flex = miaie::flex;

// ------------------------------------------------------------ 64x64 tile
// Bounds-checked fallback for K < 16 (and sizes of 2^30).
template <bool B_NT>
__global__ __launch_bounds__(256) void gemm_i8_tile64(const int8_t* __restrict__ A,
                                                      const int8_t* __restrict__ B,
                                                      int8_t* __restrict__ Y, int32_t* __restrict__ C,
                                                      int M, int N, int K, int lda, int ldb, int ldy,
                                                      int ldc, int shift, int relu) {
  __shared__ __attribute__((aligned(16))) int8_t as[64 * 64];
  __shared__ __attribute__((aligned(16))) int8_t bs[64 * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  const int wm = wave >> 1, wn = wave & 1;
  const int fr = lane & 31, fh = lane >> 5;

  v16i acc = v16i{0};
  for (int k0 = 0; k0 < K; k0 += 64) {
    // A (and NT B): thread -> row tid/4, 16-byte chunk tid%4
    {
      const int row = tid >> 2, ch = tid & 3;
      const int m = m0 + row, k = k0 + ch * 16;
      v4i v = v4i{0};
      if (m < M) {
        const int8_t* p = A + (size_t)m * lda + k;
        if (k + 16 <= K && miaie::aligned(p, 16)) {
          v = MIAIE_LD(reinterpret_cast<const v4i*>(p));
        } else {
          int8_t tmp[16];
#pragma unroll
          for (int t = 0; t < 16; ++t) tmp[t] = (k + t < K) ? MIAIE_LD(p + t) : 0;
          __builtin_memcpy(&v, tmp, 16);
        }
      }
      *reinterpret_cast<v4i*>(as + lds_off(row, ch)) = v;
    }
    if constexpr (B_NT) {
      const int row = tid >> 2, ch = tid & 3;
      const int n = n0 + row, k = k0 + ch * 16;
      v4i v = v4i{0};
      if (n < N) {
        const int8_t* p = B + (size_t)n * ldb + k;
        if (k + 16 <= K && miaie::aligned(p, 16)) {
          v = MIAIE_LD(reinterpret_cast<const v4i*>(p));
        } else {
          int8_t tmp[16];
#pragma unroll
          for (int t = 0; t < 16; ++t) tmp[t] = (k + t < K) ? MIAIE_LD(p + t) : 0;
          __builtin_memcpy(&v, tmp, 16);
        }
      }
      *reinterpret_cast<v4i*>(bs + lds_off(row, ch)) = v;
    } else {
      // thread -> column tid%64, k-chunk tid/64: 16 byte loads down the column
      const int col = tid & 63, ch = tid >> 6;
      const int n = n0 + col;
      int8_t tmp[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const int k = k0 + ch * 16 + t;
        tmp[t] = (n < N && k < K) ? MIAIE_LD(B + (size_t)k * ldb + n) : 0;
      }
      v4i v;
      __builtin_memcpy(&v, tmp, 16);
      *reinterpret_cast<v4i*>(bs + lds_off(col, ch)) = v;
    }
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const v4i af = *reinterpret_cast<const v4i*>(as + lds_off(wm * 32 + fr, 2 * ks + fh));
      const v4i bf = *reinterpret_cast<const v4i*>(bs + lds_off(wn * 32 + fr, 2 * ks + fh));
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf, af, acc, 0, 0, 0);
    }
    __syncthreads();
  }

  const int m = m0 + wm * 32 + fr;
  if (m >= M) return;
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int n = n0 + wn * 32 + 8 * (e >> 2) + 4 * fh + (e & 3);
    if (n < N) {
      if (C) MIAIE_ST(C + (size_t)m * ldc + n, acc[e]);
      if (Y) MIAIE_ST(Y + (size_t)m * ldy + n, (int8_t)requant1(acc[e], shift, relu));
    }
  }
}

// Register-staged tiles (flex_tile.hpp): any size, stride and alignment with
// K >= 16.  grid.x: output tiles, grid.y: the `splits` workgroups that divide a
// tile's K; mode: shift, relu << 8, splits << 16 (one
// argument: each costs the launch host time; what the loads need comes first,
// in the 14 dwords that arrive in SGPRs).  Bound by the latency of the stages'
// loads, and for few rows by reading B: 1000 x 2050 x 1000 NT (rows of 1000
// bytes) took 61.1 us in the byte-wise 64x64 kernel and takes 8.8; the MLP
// over 16 rows (4096 -> 11008 -> 4096, 90 MB of weights) 204.7 us in a
// vectorised 64x64 kernel without a split and 29.2 (27.3 with K split 8
// ways, 72 unsplit, on one box).
//
// ANY: 64-bit offsets, and a row-major B of any width (64x64 tiles alone):
// 4096x10x4096 10.5 us, 44.0 in a vectorised 64x64 kernel without a split.
template <class G, bool B_NT, bool ANY>
__global__ __launch_bounds__(256, G::PER_CU) void gemm_i8_flex(const int8_t* __restrict__ A, const int8_t* __restrict__ B, int M,
                                                       int N, int K, int lda, int ldb, uint32_t mode,
                                                       int8_t* __restrict__ Y, int32_t* __restrict__ C, int ldy, int ldc,
                                                       int8_t* __restrict__ work) {
  const int shift = mode & 31, relu = (mode >> 8) & 1, splits = mode >> 16;
  __shared__ __attribute__((aligned(1024))) int8_t lds[G::LDS];
  __shared__ int flag;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / G::WAVES_N, wn = wave % G::WAVES_N;
  int tm, tn;
  flex::tile_index<!B_NT && G::BN == 64>((M + G::BM - 1) / G::BM, (N + G::BN - 1) / G::BN, tm, tn);
  const int m0 = tm * G::BM, n0 = tn * G::BN;
  const int stages = (K + G::KB - 1) / G::KB, split = blockIdx.y;
  int s0, s1;
  flex::stage_range<G>(stages, split, splits, s0, s1);

  v4i acc[G::NI][G::NJ];
#pragma unroll
  for (int i = 0; i < G::NI; ++i)
#pragma unroll
    for (int j = 0; j < G::NJ; ++j) acc[i][j] = v4i{0};
  using Off = std::conditional_t<ANY, size_t, uint32_t>;
  flex::RowsLoader<G, G::NA, Off> la(A, m0, M, lda, K, tid);
  if constexpr (B_NT) {
    flex::RowsLoader<G, G::NB, Off> lb(B, n0, N, ldb, K, tid);
    flex::tile_loop<int8_t, G, false>(lds, la, lb, s0, s1, lane, wm, wn, acc);
  } else {
    std::conditional_t<ANY, flex::ColsLoaderAny<int8_t, G, false>, flex::ColsLoader<int8_t, G, false>> lb(B, n0, N, ldb,
                                                                                                     K, tid);
    flex::tile_loop<int8_t, G, true>(lds, la, lb, s0, s1, lane, wm, wn, acc);
  }
  if (G::SPLITS && splits > 1 &&
      !flex::split_sum<int8_t, G>(acc, blockIdx.x, split, splits, work, miaie::ctx_counters(work), &flag, tid))
    return;

  const int fr = lane & 15, fg = lane >> 4, lo = relu ? 0 : -128;
  const Requant rq{shift, shift ? 1 << (shift - 1) : 0, lo, 127};
#pragma unroll
  for (int i = 0; i < G::NI; ++i)
#pragma unroll
    for (int j = 0; j < G::NJ; ++j) {
      const int ml = wm * G::WM + 16 * i + fr, nl = wn * G::WN + 16 * j + 4 * fg;
      const v4i& a = acc[i][j];
      if (C) flex::store4(C, ldc, m0 + ml, n0 + nl, M, N, a);
      uint32_t y = 0;
      if (K < (1 << 16)) {  // |acc| + 2^30 < 2^31
        y = rq.pack4(a[0], a[1], a[2], a[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) y |= (uint32_t)(requant1(a[e], shift, relu) & 0xFF) << (8 * e);
      }
      *reinterpret_cast<uint32_t*>(lds + ml * G::YP + nl) = y;
    }
  if (!Y) return;
  __syncthreads();
  flex::store_y<G>(lds, Y, ldy, m0, n0, M, N, tid);
}

// keep_y: the caller reads Y right after (the MLP's H): ordinary stores that
// leave it in the caches (instantiated for NN B with ReLU, the MLP's form;
// other calls ignore it).
template <int BM, int BN, bool B_NT>
hipError_t launch_pipe(int device, hipStream_t st, const int8_t* A, const int8_t* B, int8_t* Y, int32_t* C, int M,
                       int N, int K, int lda, int ldb, int ldy, int ldc, int shift, int relu, bool keep_y) {
  // 128x128 tiles (small grids, where the power limit does not bind): two
  // waves per SIMD, so one wave's MFMAs run while the other waits at the
  // k-tile's barrier or for its LDS reads
  constexpr int NW = BM == 128 ? 8 : 4;
  dim3 grid(((M + BM - 1) / BM) * ((N + BN - 1) / BN)), block(64 * NW);
  const int yq = !Y ? Y_NONE : shift < 8 ? Y_MED3 : relu ? Y_HI_RELU : Y_HI;
  hipError_t e = hipSuccess;
  auto go = [&](auto k) {
    e = launch<decltype(k)::value>(device, grid, block, 0, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu);
  };
  auto go2 = [&](auto k) {
    e = launch<decltype(k)::value>(device, grid, block, 0, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu,
                                   nullptr);
  };
  // 256-row tiles with K a multiple of 128: A staged two k-tiles at a time,
  // 16x16x64 MFMAs (gemm_i8_pipe16).  128x128 tiles keep gemm_i8_pipe.
  if constexpr (BM == 256) {
    if (K % 128 == 0) {
      if constexpr (!B_NT) {
        if (keep_y && Y && !C && relu) {
          if (yq == Y_HI_RELU)
            go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, false, Y_HI_RELU, false, false, true>>{});
          else
            go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, false, Y_MED3, false, false, true>>{});
          return e;
        }
      }
      if (C) {
        switch (yq) {
          case Y_NONE: go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, B_NT, Y_NONE, true>>{}); break;
          case Y_MED3: go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, B_NT, Y_MED3, true>>{}); break;
          case Y_HI: go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, B_NT, Y_HI, true>>{}); break;
          default: go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, B_NT, Y_HI_RELU, true>>{}); break;
        }
      } else {
        switch (yq) {
          case Y_MED3: go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, B_NT, Y_MED3, false>>{}); break;
          case Y_HI: go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, B_NT, Y_HI, false>>{}); break;
          default: go2(kernel_t<gemm_i8_pipe16<BM, BN, NW, B_NT, Y_HI_RELU, false>>{}); break;
        }
      }
      return e;
    }
  }
  if (C) {
    switch (yq) {
      case Y_NONE: go(kernel_t<gemm_i8_pipe<BM, BN, NW, B_NT, Y_NONE, true>>{}); break;
      case Y_MED3: go(kernel_t<gemm_i8_pipe<BM, BN, NW, B_NT, Y_MED3, true>>{}); break;
      case Y_HI: go(kernel_t<gemm_i8_pipe<BM, BN, NW, B_NT, Y_HI, true>>{}); break;
      default: go(kernel_t<gemm_i8_pipe<BM, BN, NW, B_NT, Y_HI_RELU, true>>{}); break;
    }
  } else {
    switch (yq) {
      case Y_MED3: go(kernel_t<gemm_i8_pipe<BM, BN, NW, B_NT, Y_MED3, false>>{}); break;
      case Y_HI: go(kernel_t<gemm_i8_pipe<BM, BN, NW, B_NT, Y_HI, false>>{}); break;
      default: go(kernel_t<gemm_i8_pipe<BM, BN, NW, B_NT, Y_HI_RELU, false>>{}); break;
    }
  }
  return e;
}

template <bool B_NT>
hipError_t launch_pipe_mixed(int device, hipStream_t st, const int8_t* A, const int8_t* B, int8_t* Y, int32_t* C,
                             int M, int N, int K, int lda, int ldb, int ldy, int ldc, int shift, int relu, int nw,
                             bool keep_y) {
  const dim3 grid(((M + 255) / 256) * (nw + (N - 256 * nw + 127) / 128)), block(256);
  const int yq = !Y ? Y_NONE : shift < 8 ? Y_MED3 : relu ? Y_HI_RELU : Y_HI;
  hipError_t e = hipSuccess;
  auto go = [&](auto k) {
    e = launch<decltype(k)::value>(device, grid, block, 0, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu,
                                   nw);
  };
  if constexpr (!B_NT) {
    if (keep_y && Y && !C && relu) {
      if (yq == Y_HI_RELU)
        go(kernel_t<gemm_i8_pipe16_mixed<false, Y_HI_RELU, false, true>>{});
      else
        go(kernel_t<gemm_i8_pipe16_mixed<false, Y_MED3, false, true>>{});
      return e;
    }
  }
  if (C) {
    switch (yq) {
      case Y_NONE: go(kernel_t<gemm_i8_pipe16_mixed<B_NT, Y_NONE, true>>{}); break;
      case Y_MED3: go(kernel_t<gemm_i8_pipe16_mixed<B_NT, Y_MED3, true>>{}); break;
      case Y_HI: go(kernel_t<gemm_i8_pipe16_mixed<B_NT, Y_HI, true>>{}); break;
      default: go(kernel_t<gemm_i8_pipe16_mixed<B_NT, Y_HI_RELU, true>>{}); break;
    }
  } else {
    switch (yq) {
      case Y_MED3: go(kernel_t<gemm_i8_pipe16_mixed<B_NT, Y_MED3, false>>{}); break;
      case Y_HI: go(kernel_t<gemm_i8_pipe16_mixed<B_NT, Y_HI, false>>{}); break;
      default: go(kernel_t<gemm_i8_pipe16_mixed<B_NT, Y_HI_RELU, false>>{}); break;
    }
  }
  return e;
}

// Tiling planner for the pipelined kernel: picks the workgroup tile
// (BM x BN) among 256x256, 256x128 and 128x128 for an M x N x K product on
// `cus` compute units, or a mix of 256x256 and 256x128 tiles in one launch
// (gemm_i8_pipe16_mixed).  A tile's cost, in units of one 256x256x64 k-tile of
// MFMA work: its K/64 k-tiles plus about 6 units of prologue and epilogue,
// scaled by the tile's relative cost per k-tile (1 for 256x256; 0.55 for
// 256x128; 0.35 for 128x128, whose LDS reads per MFMA are twice those of
// 256x256).  A plan's cost is the finishing time of its tiles dealt in
// launch order to the CU that frees first (the dispatcher's order).
struct TileChoice {
  int bm, bn;
  double unit;
};
constexpr TileChoice kTiles[] = {{256, 256, 1.0}, {256, 128, 0.55}, {128, 128, 0.35}};

struct PipePlan {
  double cost = 0;  // units of one 256x256x64 k-tile
  int bm = 0, bn = 0;
  int nw = 0;  // > 0: mixed launch, 256-wide tiles over the first 256 nw columns, 256x128 after
};

// Finishing time of `n1` tasks of length d1 then `n2` of length d2, each
// dealt to the earliest-free of `cus` identical CUs.  CUs that free at the
// same time are kept as one group, so the loop runs once per group and round.
double list_makespan(long n1, double d1, long n2, double d2, int cus) {
  struct Grp {
    double t;
    long n;
  };
  Grp g[8];
  int ng = 1;
  g[0] = {0.0, cus};
  auto deal = [&](long tasks, double d) {
    while (tasks > 0) {
      int k = 0;  // earliest group
      for (int i = 1; i < ng; ++i)
        if (g[i].t < g[k].t) k = i;
      const long take = tasks < g[k].n ? tasks : g[k].n;
      tasks -= take;
      const double t_end = g[k].t + d;
      if (take == g[k].n) {
        g[k].t = t_end;
      } else {
        g[k].n -= take;
        int j = -1;  // merge with a group ending at the same time, else a new one
        for (int i = 0; i < ng; ++i)
          if (g[i].t == t_end) j = i;
        if (j >= 0)
          g[j].n += take;
        else if (ng < 8)
          g[ng++] = {t_end, take};
        else
          return false;
      }
    }
    return true;
  };
  if (!deal(n1, d1) || !deal(n2, d2)) return 1e300;  // (more than 8 distinct finishing times: not planned)
  double t = 0;
  for (int i = 0; i < ng; ++i) t = g[i].t > t ? g[i].t : t;
  return t;
}

PipePlan plan_pipe(int M, int N, int K, int cus) {
  PipePlan best;
  if (K % BK != 0 || cus < 1) return best;
  const double work = K / BK + 6.0;
  // lowest finishing time; among equal ones, the least total CU time (fewer
  // of the costlier narrow tiles, less energy under the power limit)
  double best_cost = 0, best_total = 0;
  auto consider = [&](double cost, double total, PipePlan p) {
    if (best.bm == 0 || cost < best_cost - 1e-9 || (cost < best_cost + 1e-9 && total < best_total - 1e-9)) {
      best_cost = cost;
      best_total = total;
      best = p;
      best.cost = cost;
    }
  };
  // A tile that does not divide M or N still takes the shape: the last
  // tile row or column overlaps its neighbour (dev::tile_origin), and is
  // planned as a whole tile.  A moved-back column tile starts on a 16-byte
  // chunk only when N % 16 == 0.
  auto cols_ok = [&](int n, int bn) { return n >= bn && (n % bn == 0 || N % 16 == 0); };
  for (const TileChoice& t : kTiles) {
    if (M < t.bm || !cols_ok(N, t.bn)) continue;
    const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    consider((double)((tiles + cus - 1) / cus) * t.unit * work, tiles * t.unit * work, PipePlan{0, t.bm, t.bn, 0});
  }
  // mixed 256x256 + 256x128 (the pair-staged kernel: K % 128 == 0)
  if (M >= 256 && K % 128 == 0) {
    const long tm = (M + 255) / 256;
    for (int nw = 1; cols_ok(N - 256 * nw, 128); ++nw) {
      const long wide = tm * nw, narrow = tm * ((N - 256 * nw + 127) / 128);
      const double dw = kTiles[0].unit * work, dn = kTiles[1].unit * work;
      consider(list_makespan(wide, dw, narrow, dn, cus), wide * dw + narrow * dn, PipePlan{0, 256, 256, nw});
    }
  }
  return best;
}

}  // namespace

namespace miaie {

// The pipelined kernel's operand conditions: 16-byte chunks (16-byte
// aligned operands and strides), per-lane offsets of up to 64 rows in 32
// bits, and the requant shortcut's K < 2^16.
static bool pipe_operands_ok(const int8_t* A, const int8_t* B, const int8_t* Y, const int32_t* C, int K, int lda,
                             int ldb, int ldy, int ldc) {
  return (K % BK == 0) && (!Y || K < (1 << 16)) && aligned(A, 16) && aligned(B, 16) && lda % 16 == 0 &&
         ldb % 16 == 0 && lda < (1 << 25) && ldb < (1 << 25) && (!Y || (aligned(Y, 16) && ldy % 16 == 0)) &&
         (!C || (aligned(C, 16) && ldc % 4 == 0));
}

// The register-staged kernel's operands: rows of at least 16 bytes and 32-bit
// offsets within a tile, or (Any) rows of A of 16 bytes alone.
enum class FlexOperands { None, Any, Rows };
static FlexOperands flex_operands(int N, int K, int lda, int ldb, int b_nt) {
  if (K < 16 || K >= (1 << 30) || N >= (1 << 30)) return FlexOperands::None;
  return (b_nt || N >= 16) && lda < (1 << 25) && ldb < (1 << 25) ? FlexOperands::Rows : FlexOperands::Any;
}

// How a product runs: pipelined tiles (pipe.bm > 0), register-staged ones
// (flex.bm > 0), or the 64x64 kernel.  Where both of the first two apply, the
// pipelined ones unless the others' estimate is well below theirs (a unit of
// plan_pipe takes about 0.5 us, 0.7 where B is too large for the caches to hold
// from the last call, plus 1.5 us): a handful of 128x128 tiles over a long K,
// which the register-staged kernel splits.  Pipelined against split:
// 128x4096x11008 49.2 and 20.0 us, 256x4096x11008 48.8 and 35.0, 512x512x8192 NT
// 29.4 and 12.6, 256x256x65472 NT 295 and 26; on the other side of the line
// 256x4096x4096 19.2 and 16.3 first time, 12.0 and 16.1 repeated, 256x1024x2048 NT
// 7.3 either way.
struct Route {
  PipePlan pipe;
  flex::Plan flex;
};
static Route route(miaie_ctx* ctx, int M, int N, int K, bool pipe_ok, FlexOperands ops, bool can_split) {
  Route r;
  if (pipe_ok) r.pipe = plan_pipe(M, N, K, ctx->cus);
  if (ops == FlexOperands::Any) {
    if (!r.pipe.bm) r.flex = flex::plan_any(M, N, K, ctx->cus, can_split, ctx->work_bytes);
    return r;
  }
  // (256-row tiles: enough of them that no split is better)
  if (r.pipe.bm != 256 && ops == FlexOperands::Rows) {
    r.flex = flex::plan(M, N, K, 1.0, ctx->cus, can_split, ctx->work_bytes);
    const double unit_us = (size_t)N * K > ((size_t)16 << 20) ? 0.7 : 0.5;
    if (r.pipe.bm && r.flex.bm && r.flex.us < 0.75 * (1.5 + unit_us * r.pipe.cost))
      r.pipe = PipePlan{};
    else if (r.pipe.bm)
      r.flex = flex::Plan{};
  }
  return r;
}

int plan_gemm_i8(miaie_ctx* ctx, int M, int N, int K, int dense_ok, miaie_gemm_plan* plan) {
  const Route r = route(ctx, M, N, K, dense_ok, flex_operands(N, K, K, N, false), true);
  const PipePlan& p = r.pipe;
  *plan = miaie_gemm_plan{};
  plan->threads = p.bm == 128 ? 512 : 256;
  if (p.bm && p.nw) {
    plan->kernel = MIAIE_KERNEL_PIPE_MIXED;
    plan->tile_m = 256;
    plan->tile_n = 256;
    plan->workgroups = ((M + 255) / 256) * (p.nw + (N - 256 * p.nw + 127) / 128);
  } else if (p.bm) {
    plan->kernel = MIAIE_KERNEL_PIPE;
    plan->tile_m = p.bm;
    plan->tile_n = p.bn;
    plan->workgroups = ((M + p.bm - 1) / p.bm) * ((N + p.bn - 1) / p.bn);
  } else if (r.flex.bm) {
    plan->kernel = MIAIE_KERNEL_TILE64;
    plan->tile_m = r.flex.bm;
    plan->tile_n = r.flex.bn;
    plan->workgroups = (int)(r.flex.tiles * r.flex.splits);
  } else {
    plan->kernel = MIAIE_KERNEL_TILE64;
    plan->tile_m = 64;
    plan->tile_n = 64;
    plan->workgroups = ((M + 63) / 64) * ((N + 63) / 64);
  }
  return MIAIE_OK;
}

// Chooses the kernel.  Y and/or C may be NULL (not both).
int launch_gemm_i8(miaie_ctx* ctx, const int8_t* A, const int8_t* B, int8_t* Y, int32_t* C, int M,
                   int N, int K, int lda, int ldb, int ldy, int ldc, int b_nt, int shift, int relu, bool keep_y) {
  const bool pipe_ok = pipe_operands_ok(A, B, Y, C, K, lda, ldb, ldy, ldc);
  const FlexOperands ops = flex_operands(N, K, lda, ldb, b_nt);
  Route r = route(ctx, M, N, K, pipe_ok, ops, true);
  if (r.flex.splits > 1 && !may_split(ctx)) r = route(ctx, M, N, K, pipe_ok, ops, false);
  const PipePlan& plan = r.pipe;
  const int dev = ctx->device;
  if (plan.bm && plan.nw) {
    const int nw = plan.nw;
    const hipError_t e =
        b_nt ? launch_pipe_mixed<true>(dev, ctx->stream, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu, nw, keep_y)
             : launch_pipe_mixed<false>(dev, ctx->stream, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu, nw,
                                        keep_y);
    return check_launch(ctx, e, "gemm_i8_pipe16_mixed");
  }
  if (plan.bm) {
    hipStream_t st = ctx->stream;
    const int bm = plan.bm, bn = plan.bn;
    hipError_t e;
    if (bm == 256 && bn == 256)
      e = b_nt ? launch_pipe<256, 256, true>(dev, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu, keep_y)
               : launch_pipe<256, 256, false>(dev, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu, keep_y);
    else if (bm == 256)
      e = b_nt ? launch_pipe<256, 128, true>(dev, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu, keep_y)
               : launch_pipe<256, 128, false>(dev, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu, keep_y);
    else
      e = b_nt ? launch_pipe<128, 128, true>(dev, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu, keep_y)
               : launch_pipe<128, 128, false>(dev, st, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc, shift, relu, keep_y);
    return check_launch(ctx, e, "gemm_i8_pipe");
  }
  dim3 grid((N + 63) / 64, (M + 63) / 64), block(256);
  if (grid.y > 65535) return fail(ctx, MIAIE_EINVAL, "gemm_i8: M too large for the 64x64 fallback");
  if (r.flex.bm) {
    const flex::Plan& f = r.flex;
    hipError_t e = hipSuccess;
    const dim3 fg((unsigned)f.tiles, (unsigned)f.splits);
    int8_t* const work = static_cast<int8_t*>(ctx->work);
    const uint32_t mode = (uint32_t)(shift | relu << 8 | f.splits << 16);
    auto go = [&](auto k) {
      e = launch<decltype(k)::value>(dev, fg, block, 0, ctx->stream, A, B, M, N, K, lda, ldb, mode, Y, C, ldy, ldc, work);
    };
    if (f.any)
      flex::with_geom_any(f, [&](auto g) {
        using G = typename decltype(g)::type;
        if (b_nt)
          go(kernel_t<gemm_i8_flex<G, true, true>>{});
        else
          go(kernel_t<gemm_i8_flex<G, false, true>>{});
      });
    else
      flex::with_geom(f, [&](auto g) {
        using G = typename decltype(g)::type;
        if (b_nt)
          go(kernel_t<gemm_i8_flex<G, true, false>>{});
        else
          go(kernel_t<gemm_i8_flex<G, false, false>>{});
      });
    return check_launch(ctx, e, "gemm_i8_flex");
  }
  const hipError_t e =
      b_nt ? launch<gemm_i8_tile64<true>>(dev, grid, block, 0, ctx->stream, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc,
                                          shift, relu)
           : launch<gemm_i8_tile64<false>>(dev, grid, block, 0, ctx->stream, A, B, Y, C, M, N, K, lda, ldb, ldy, ldc,
                                           shift, relu);
  return check_launch(ctx, e, "gemm_i8_tile64");
}

}  // namespace miaie
