// Register-staged MFMA tile for operands of any size, stride and alignment:
// device code shared by the int8 GEMM, the bf16 GEMM and the convolution.
//
// The pipelined kernels copy 16-byte chunks straight into LDS and so need
// 16-byte aligned rows and whole tiles.  Everything else (ragged sizes,
// unaligned rows, few rows, an image with 3 channels) runs here: the operands
// pass through registers, where a chunk that crosses the end of its row or of
// the image is shifted and masked.
//
// One workgroup of 4 waves owns a BM x BN output tile.  A stage is KB bytes of
// k (KB int8 or KB/2 bf16 values) of the BM rows and BN columns.  Each thread
// loads its 16-byte chunks of the next stage into registers (all in flight
// together) while the current stage, in LDS, is multiplied on
// v_mfma_i32_16x16x64_i8 / v_mfma_f32_16x16x32_bf16.  What bounds such small
// products is the latency of that chain of loads, so a stage is as deep as the
// registers allow (256 bytes of k: a product of K = 1000 is 4 stages), 2-8
// workgroups share a CU, and K is split over workgroups where tiles are few.
//
// Loads are 16 bytes wide from any byte address (gfx950's unaligned access
// mode).  A chunk that would reach past the end of its row (of a row-major
// operand's last column, of the image) is loaded from the last valid 16 bytes
// instead and shifted into place when it is written to LDS, so no load waits
// on a branch and none leaves the operand.
//
// The kernels take the number of splits as an argument: reading gridDim would
// add the 256 bytes of hidden arguments to each launch (0.15-0.3 us of host time).
//
// LDS layouts (both free of bank conflicts on the fragment reads, 16 lanes of
// which must cover 256 consecutive bytes of banks):
//   k-contiguous operand (A, B stored [N][K], conv weights and pixels):
//     [row][KB bytes], 16-byte chunk c of row r at c ^ (r mod 16), for KB = 128
//     c ^ (r / 2 mod 8)
//   B stored [K][N]: [k][BN values], chunk c of k-row k at c ^ kswz(k); the
//     fragments (16 bytes of consecutive k of one column) come from two
//     transposing reads (ds_read_b64_tr_b8 / _b16).
#pragma once

#include <algorithm>
#include <type_traits>

#include "gfx950_ops.hpp"
#include "miaie_internal.hpp"

namespace miaie {
namespace flex {

// 16 bytes at any address, and four 32-bit values at a 4-byte aligned one
struct __attribute__((packed, aligned(1))) Any16 {
  v4i v;
};
template <class V>
struct __attribute__((packed, aligned(4))) Dw4 {
  V v;
};

typedef uint32_t v4u __attribute__((ext_vector_type(4)));

template <int BM_, int BN_, int KB_, int WAVES_N_>
struct Geom {
  static constexpr int BM = BM_, BN = BN_, KB = KB_, WAVES_N = WAVES_N_;
  static constexpr int CH = KB / 16;                         // 16-byte chunks per row
  static constexpr int RPP = 256 / CH;                       // rows one pass of the workgroup covers
  static constexpr int WM = BM / (4 / WAVES_N), WN = BN / WAVES_N;
  static constexpr int NI = WM / 16, NJ = WN / 16;           // 16 x 16 blocks per wave
  static constexpr int A_BYTES = BM * KB, B_BYTES = BN * KB;
  static constexpr int NA = A_BYTES / 4096, NB = B_BYTES / 4096;  // chunks per thread per stage
  static constexpr int YP = BN + 16;                         // LDS pitch of an int8 output row
  static constexpr bool SPLITS = KB >= 128;  // whether its K is ever split
  static constexpr int PER_CU = BM >= 128 ? 2 : KB < 256 ? 8 : 4;  // workgroups whose registers and LDS fit a CU
  static constexpr int LDS = A_BYTES + B_BYTES > BM * YP ? A_BYTES + B_BYTES : BM * YP;
  static_assert(NA >= 1 && NB >= 1 && NI >= 1 && NJ >= 1, "tile too small for 4 waves");
};

// The tiles in use: a k of a few chunks; few rows; small and ragged products;
// large ones.  (A stage is loaded, written to LDS and multiplied whole: 16 to 128
// bytes of k in a 256-byte stage took 3.0 us where 2.5 suffice for 16x16x16 bf16,
// 5.4 against 3.7 for int8 65000x16x16 NT.)
using Short = Geom<64, 64, 64, 2>;
using Skinny = Geom<16, 128, 256, 4>;
using Small = Geom<64, 64, 256, 2>;
using Large = Geom<128, 128, 128, 2>;

// Output tile and workgroups per tile for an M x N product of k_bytes of k.
struct Plan {
  int bm = 0, bn = 0, kb = 0, splits = 1;
  bool any = false;  // rows of B below 16 bytes, or a pitch of 2^25 or more
  long tiles = 0;  // workgroups = tiles * splits
  double us = 0;   // estimated time
};

// The plan with the lowest estimated time.  A launch takes
//   t0 + max(latency * stages, rounds * (wg + stage * stages)) + (splits > 1 ? sum + sum_split * splits : 0)
// microseconds for `stages` stages per workgroup and rounds = workgroups per
// CU, rounded up: a single workgroup's chain of loads, or the CU's work when it
// has several.  Constants fitted to back-to-back launches on MI355X over 112
// GEMM and conv shapes (10 to 4e10 multiply-adds; 12% rms error; the plan
// picked is 1% slower than the best of all tiles and splits on average, 16% at
// worst), operands in the caches: weights streamed from memory take up to a third
// longer than estimated (16 x 11008 x 4096: 14.2 us, 11.2 estimated).  The
// 64-byte stage's constants: 2700 products of a short k, 11% rms.  A tile of
// 32 x 128 was never more than 2% better than these.
// `cost`: stage cost relative to the int8 GEMM's (conv 1.5: its loads compute
// their addresses).
// (No divisions: this runs on the host for every call.)
// bm is 0 where every tile makes too many workgroups for a launch.
template <class G>
inline void consider(Plan& best, double t0, double latency, double wg, double stage, double sum, double sum_split,
                     long M, long N, long k_bytes, double cost, int cus, double per_cu, bool can_split,
                     size_t work_bytes) {
  static constexpr int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16};
  static constexpr double kInverse[] = {1.0, 1.0 / 2, 1.0 / 3, 1.0 / 4, 1.0 / 6, 1.0 / 8, 1.0 / 12, 1.0 / 16};
  const long tiles = ((M + G::BM - 1) / G::BM) * ((N + G::BN - 1) / G::BN), stages = (k_bytes + G::KB - 1) / G::KB;
  if (tiles >= 1l << 24) return;  // tiles are grid.x, in which HIP takes fewer than 2^32 threads
  const size_t slot = (size_t)tiles * G::BM * G::BN * sizeof(int32_t);
  auto up = [](double x) { return (double)(long)(x + (1.0 - 1e-6)); };  // rounded up
  for (int i = 0; i < 8; ++i) {
    const int s = kSplits[i];
    // (more than four workgroups per CU never split)
    if (s > 1 && (!can_split || s > stages || tiles * s > 4l * cus || tiles > MIAIE_CTX_COUNTERS || slot * s > work_bytes))
      return;
    const double n = up((double)stages * kInverse[i]), rounds = up((double)(tiles * s) * per_cu);
    const double us = t0 + std::max(latency * cost * n, rounds * (wg + stage * cost * n)) + (s > 1 ? sum + sum_split * s : 0.0);
    if (best.bm == 0 || us < best.us) best = Plan{G::BM, G::BN, G::KB, s, false, tiles, us};
  }
}
template <class G>
inline void consider_tile(Plan& best, long M, long N, long k_bytes, double cost, int cus, bool can_split, size_t work_bytes) {
  const double per_cu = 1.0 / cus;
  if constexpr (std::is_same_v<G, Short>) {
    // (a k of three 64-byte stages at most: longer ones gain by deeper stages)
    if (k_bytes * cost <= 192)
      consider<G>(best, 2.35, 0.40, 0.18, 0.19, 0.0, 0.0, M, N, k_bytes, cost, cus, per_cu, false, work_bytes);
  } else if constexpr (std::is_same_v<G, Skinny>) {
    consider<G>(best, 1.7, 0.95, 0.90, 0.80, 1.6, 0.15, M, N, k_bytes, cost, cus, per_cu, can_split, work_bytes);
  } else if constexpr (std::is_same_v<G, Small>) {
    consider<G>(best, 2.4, 0.84, 0.55, 0.50, 1.5, 0.26, M, N, k_bytes, cost, cus, per_cu, can_split, work_bytes);
  } else {
    consider<G>(best, 3.5, 0.95, 1.20, 0.60, 1.5, 1.00, M, N, k_bytes, cost, cus, per_cu, can_split, work_bytes);
  }
}
template <class... G>
inline Plan plan_of(long M, long N, long k_bytes, double cost, int cus, bool can_split, size_t work_bytes) {
  Plan best;
  (consider_tile<G>(best, M, N, k_bytes, cost, cus, can_split, work_bytes), ...);
  return best;
}
inline Plan plan(long M, long N, long k_bytes, double cost, int cus, bool can_split, size_t work_bytes) {
  return plan_of<Short, Skinny, Small, Large>(M, N, k_bytes, cost, cus, can_split, work_bytes);
}
// The same for the loaders that take any operand (with_geom_any), on 64 x 64
// tiles alone.
inline Plan plan_any(long M, long N, long k_bytes, int cus, bool can_split, size_t work_bytes) {
  Plan p = plan_of<Short, Small>(M, N, k_bytes, 1.0, cus, can_split, work_bytes);
  p.any = p.bm != 0;
  return p;
}

// Calls go with the geometry a plan names, as a type.
template <class F>
void with_geom(const Plan& p, F&& go) {
  if (p.kb == Short::KB)
    go(type_t<Short>{});
  else if (p.bm == Skinny::BM)
    go(type_t<Skinny>{});
  else if (p.bm == Small::BM)
    go(type_t<Small>{});
  else
    go(type_t<Large>{});
}

template <class F>
void with_geom_any(const Plan& p, F&& go) {
  if (p.kb == Short::KB)
    go(type_t<Short>{});
  else
    go(type_t<Small>{});
}

__device__ __forceinline__ int row_off(int KB, int row, int chunk) {
  return row * KB + ((chunk ^ (KB >= 256 ? row & 15 : (row * KB / 256) & (KB / 16 - 1))) << 4);
}

// Chunk swizzle of k-row k of a [k][BN] operand with rows of PB bytes.  One
// 32-lane half of a transposing read takes, for int8, 16 bytes of k-rows
// jj + {0, 16} (jj < 8), and for bf16 32 bytes of k-rows jj + {0, 8} (jj < 4);
// with 256 / PB rows side by side in the banks, the remaining row bits choose
// the chunk.
template <class T, int PB>
__device__ __forceinline__ int kswz(int k) {
  if constexpr (sizeof(T) == 1) {
    static_assert(PB == 64 || PB == 128, "int8 columns per tile");
    return PB == 64 ? ((k >> 2) & 1) | (((k >> 4) & 1) << 1) : ((k >> 1) & 3) | (((k >> 4) & 1) << 2);
  } else {
    static_assert(PB == 128 || PB == 256, "bf16 columns per tile");
    return PB == 128 ? (((k >> 1) & 1) << 1) | (((k >> 3) & 1) << 2) : ((k & 3) << 1) | (((k >> 3) & 1) << 3);
  }
}

template <class T>
struct Mma;
template <>
struct Mma<int8_t> {
  using acc_t = v4i;
  static __device__ __forceinline__ acc_t mma(v4i a, v4i b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mma<uint16_t> {  // bf16 bits
  using acc_t = v4f;
  static __device__ __forceinline__ acc_t mma(v4i a, v4i b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  }
};

// v shifted down by n bytes (n >= 0, zeros shifted in; 0 from n = 16 on)
__device__ __forceinline__ v4i shr_bytes(v4i v, int n) {
  uint64_t lo = (uint32_t)v[0] | (uint64_t)(uint32_t)v[1] << 32, hi = (uint32_t)v[2] | (uint64_t)(uint32_t)v[3] << 32;
  const int s = 8 * (n & 7);
  if (n & 8) lo = hi, hi = 0;
  if (n >= 16) lo = hi = 0;
  lo = s ? (lo >> s) | (hi << (64 - s)) : lo;
  hi >>= s;
  return v4i{(int)lo, (int)(lo >> 32), (int)hi, (int)(hi >> 32)};
}
// v shifted up by n bytes
__device__ __forceinline__ v4i shl_bytes(v4i v, int n) {
  uint64_t lo = (uint32_t)v[0] | (uint64_t)(uint32_t)v[1] << 32, hi = (uint32_t)v[2] | (uint64_t)(uint32_t)v[3] << 32;
  const int s = 8 * (n & 7);
  if (n & 8) hi = lo, lo = 0;
  if (n >= 16) lo = hi = 0;
  hi = s ? (hi << s) | (lo >> (64 - s)) : hi;
  lo <<= s;
  return v4i{(int)lo, (int)(lo >> 32), (int)hi, (int)(hi >> 32)};
}
// ones in bytes [lo, hi), 0 <= lo, hi <= 16
__device__ __forceinline__ v4i byte_mask(int lo, int hi) {
  // low 32 bits of ~(~0 << 8n): n bytes of ones, n clamped to the dword
  auto below = [](int n) { return ~(uint32_t)(~0ull << (8 * min(max(n, 0), 4))); };
  v4i m;
#pragma unroll
  for (int w = 0; w < 4; ++w) m[w] = (int)(below(hi - 4 * w) & ~below(lo - 4 * w));
  return m;
}

// ------------------------------------------------------------- operand loaders
// load(s): this thread's chunks of stage s into registers.  put(s): the same
// chunks, set right where they reached past an end, into LDS.

// Rows of a k-contiguous operand: chunk ch of rows r0 + RPP i of the tile,
// zero past the last k.  k_bytes >= 16; with 32-bit offsets, pitch below 2^25.
template <class G, int NL, class Off = uint32_t>
struct RowsLoader {
  const int8_t* base;  // first row of the tile
  Off voff[NL];
  int k_bytes, r0, ch;
  v4i v[NL];
  // tile rows row0 .. of an operand of `rows` rows of k_bytes_ bytes, pitch ld
  // bytes (rows past the last repeat it: they are never stored)
  __device__ __forceinline__ RowsLoader(const int8_t* p, int row0, int rows, size_t ld, int k_bytes_, int tid)
      : base(p + (size_t)row0 * ld), k_bytes(k_bytes_), r0(tid / G::CH), ch(tid % G::CH) {
#pragma unroll
    for (int i = 0; i < NL; ++i) voff[i] = (Off)min(r0 + G::RPP * i, rows - 1 - row0) * (Off)ld;
  }
  __device__ __forceinline__ void load(int s) {
    const uint32_t at = (uint32_t)min(s * G::KB + 16 * ch, k_bytes - 16);
#pragma unroll
    for (int i = 0; i < NL; ++i) v[i] = MIAIE_LD(reinterpret_cast<const Any16*>(base + (voff[i] + at))).v;
  }
  __device__ __forceinline__ void put(int s, int8_t* lds) {
    if ((s + 1) * G::KB > k_bytes) {
      const int past = max(s * G::KB + 16 * ch - (k_bytes - 16), 0);
#pragma unroll
      for (int i = 0; i < NL; ++i) v[i] = shr_bytes(v[i], past);
    }
#pragma unroll
    for (int i = 0; i < NL; ++i) *reinterpret_cast<v4i*>(lds + row_off(G::KB, r0 + G::RPP * i, ch)) = v[i];
  }
};

// k-rows of a B stored [K][N]: chunk cb of k-rows k0 + KPP i of the stage.
// Rows past the last k are zero if ZERO, else they repeat it (A is zero
// there: enough for integers).  Columns past the last are anything (of the
// operand): they are never stored.  N * sizeof(T) >= 16, pitch below 2^25.
template <class T, class G, bool ZERO>
struct ColsLoader {
  static constexpr int PB = G::BN * (int)sizeof(T);  // bytes per k-row of the tile
  static constexpr int CB = PB / 16, KPP = 256 / CB;
  static constexpr int SK = G::KB / (int)sizeof(T);  // k-rows per stage
  const int8_t* base;
  size_t ld;
  uint32_t voff;
  int K, k0, cb, past;
  v4i v[G::NB];
  __device__ __forceinline__ ColsLoader(const int8_t* p, int n0, int N, size_t ld_, int K_, int tid)
      : base(p), ld(ld_), K(K_), k0(tid / CB), cb(tid % CB) {
    // a chunk that crosses the last column is loaded from the row's last 16 bytes
    const int want = n0 * (int)sizeof(T) + 16 * cb, at = min(want, N * (int)sizeof(T) - 16);
    past = want - at;
    voff = (uint32_t)k0 * (uint32_t)ld + (uint32_t)at;
  }
  __device__ __forceinline__ void load(int s) {
    if ((s + 1) * SK <= K) {
#pragma unroll
      for (int i = 0; i < G::NB; ++i)
        v[i] = MIAIE_LD(reinterpret_cast<const Any16*>(base + (size_t)(s * SK + KPP * i) * ld + voff)).v;
    } else {
      const uint32_t at = voff - (uint32_t)k0 * (uint32_t)ld;
#pragma unroll
      for (int i = 0; i < G::NB; ++i)
        v[i] = MIAIE_LD(reinterpret_cast<const Any16*>(base + (size_t)min(s * SK + k0 + KPP * i, K - 1) * ld + at)).v;
    }
  }
  __device__ __forceinline__ void put(int s, int8_t* lds) {
    if (__builtin_amdgcn_ballot_w64(past != 0)) {
#pragma unroll
      for (int i = 0; i < G::NB; ++i) v[i] = shr_bytes(v[i], past);
    }
    if (ZERO && (s + 1) * SK > K) {
#pragma unroll
      for (int i = 0; i < G::NB; ++i)
        if (s * SK + k0 + KPP * i >= K) v[i] = v4i{0};
    }
#pragma unroll
    for (int i = 0; i < G::NB; ++i) {
      const int k = k0 + KPP * i;
      *reinterpret_cast<v4i*>(lds + k * PB + ((cb ^ kswz<T, PB>(k)) << 4)) = v[i];
    }
  }
};

// The same for any N >= 1 and pitch, where the whole operand is 16 bytes or
// more: rows narrower than a load, too.  A chunk is loaded from where it starts
// (past the end of its row it holds the next one's values), or from the
// operand's last 16 bytes and shifted.
template <class T, class G, bool ZERO>
struct ColsLoaderAny {
  static constexpr int PB = G::BN * (int)sizeof(T);
  static constexpr int CB = PB / 16, KPP = 256 / CB;
  static constexpr int SK = G::KB / (int)sizeof(T);
  const int8_t* base;
  size_t ld, want, last;  // first byte of the chunk in its row, last offset a load may start at
  int K, k0, cb;
  v4i v[G::NB];
  int moved[G::NB];
  __device__ __forceinline__ ColsLoaderAny(const int8_t* p, int n0, int N, size_t ld_, int K_, int tid)
      : base(p), ld(ld_), want((size_t)n0 * sizeof(T) + 16 * (tid % CB)),
        last((size_t)(K_ - 1) * ld_ + (size_t)N * sizeof(T) - 16), K(K_), k0(tid / CB), cb(tid % CB) {}
  __device__ __forceinline__ void load(int s) {
#pragma unroll
    for (int i = 0; i < G::NB; ++i) {
      const size_t at = (size_t)min(s * SK + k0 + KPP * i, K - 1) * ld + want, from = at < last ? at : last;
      v[i] = MIAIE_LD(reinterpret_cast<const Any16*>(base + from)).v;
      moved[i] = at - from < 16 ? (int)(at - from) : 16;
    }
  }
  __device__ __forceinline__ void put(int s, int8_t* lds) {
#pragma unroll
    for (int i = 0; i < G::NB; ++i) {
      const int k = k0 + KPP * i;
      v[i] = ZERO && s * SK + k >= K ? v4i{0} : shr_bytes(v[i], moved[i]);
      *reinterpret_cast<v4i*>(lds + k * PB + ((cb ^ kswz<T, PB>(k)) << 4)) = v[i];
    }
  }
};

// ------------------------------------------------------------- the tile
// This workgroup's tile (grid.x).  Workgroups are dealt round-robin to the 8
// XCDs.  Where a tile takes half of each 128-byte line of a B stored [K][N]
// (PAIRS: 64 int8 columns) and B is read once (one tile row), the two tiles of
// a line go to one XCD, 8 workgroups apart, so that its L2 fetches the line
// once: the MLP 4096 -> 11008 -> 4096 over 40 rows 41.5 -> 34.9 us, 64 rows 42.3
// -> 37.1.  (A contiguous run of tiles per XCD: 38.6 and 40.4, and 5-9% slower
// for bf16, whose tiles take whole lines.)
template <bool PAIRS>
__device__ __forceinline__ void tile_index(int TM, int TN, int& tm, int& tn) {
  const int b = blockIdx.x;
  if (TN == 1) {  // (tile_coords' order, without its divisions)
    tm = TM % 8 == 0 ? (b & 7) * (TM >> 3) + (b >> 3) : b;
    tn = 0;
  } else if (PAIRS && TM == 1) {
    tm = 0;
    tn = (b | 15) < TN ? (b & ~15) + 2 * (b & 7) + ((b >> 3) & 1) : b;
  } else {
    dev::tile_coords<4>(b, TM, TN, tm, tn);
  }
}

// The stages [s0, s1) of one of the `splits` workgroups of a tile.  (32 bits
// hold 16 splits of 2^24 stages; in 64 bits the two divisions were 400 scalar
// instructions ahead of the first load.)
template <class G>
__device__ __forceinline__ void stage_range(int stages, int split, int splits, int& s0, int& s1) {
  s0 = 0;
  s1 = stages;
  if (G::SPLITS && splits > 1) {
    s0 = (int)((uint32_t)stages * (uint32_t)split / (uint32_t)splits);
    s1 = (int)((uint32_t)stages * (uint32_t)(split + 1) / (uint32_t)splits);
  }
}

// acc[i][j][e] += over stages [s0, s1): row wm*WM + 16i + lane%16, column
// wn*WN + 16j + 4*(lane/16) + e of the tile.  NN: B is [k][BN] in LDS.
template <class T, class G, bool NN, class LA, class LB>
__device__ __forceinline__ void tile_loop(int8_t* lds, LA& la, LB& lb, int s0, int s1, int lane, int wm, int wn,
                                          typename Mma<T>::acc_t (&acc)[G::NI][G::NJ]) {
  int8_t* const bs = lds + G::A_BYTES;
  const int fr = lane & 15, fg = lane >> 4;
  constexpr int PB = G::BN * (int)sizeof(T);
  la.load(s0);
  lb.load(s0);
  for (int s = s0; s < s1; ++s) {
    la.put(s, lds);
    lb.put(s, bs);
    __syncthreads();
    if (s + 1 < s1) {
      la.load(s + 1);
      lb.load(s + 1);
    }
#pragma unroll
    for (int ks = 0; ks < G::KB / 64; ++ks) {
      v4i a[G::NI], b[G::NJ];
#pragma unroll
      for (int i = 0; i < G::NI; ++i)
        a[i] = *reinterpret_cast<const v4i*>(lds + row_off(G::KB, wm * G::WM + 16 * i + fr, 4 * ks + fg));
#pragma unroll
      for (int j = 0; j < G::NJ; ++j) {
        if constexpr (!NN) {
          b[j] = *reinterpret_cast<const v4i*>(bs + row_off(G::KB, wn * G::WN + 16 * j + fr, 4 * ks + fg));
        } else if constexpr (sizeof(T) == 1) {
          // lane 16g + 2jj + h supplies k-row 64ks + 16g + 8r + jj, columns
          // 16j + 8h .. +8; lane 16g + c receives column c, k 16g + 8r .. +8
          const int kr = 64 * ks + 16 * fg + ((lane >> 1) & 7), c = wn * (G::WN / 16) + j;
          const int8_t* const p = bs + kr * PB + ((c ^ kswz<T, PB>(kr)) << 4) + 8 * (lane & 1);
          const miaie_v2i lo = dev::lds_read_tr8(p), hi = dev::lds_read_tr8(p + 8 * PB);
          b[j] = v4i{lo[0], lo[1], hi[0], hi[1]};
        } else {
          // lane 16g + 4jj + q supplies k-row 32ks + 8g + 4r + jj, columns
          // 16j + 4q .. +4; lane 16g + c receives column c, k 8g + 4r .. +4
          const int q = lane & 3, kr = 32 * ks + 8 * fg + ((lane >> 2) & 3), c = 2 * (wn * (G::WN / 16) + j) + (q >> 1);
          const int8_t* const p = bs + kr * PB + ((c ^ kswz<T, PB>(kr)) << 4) + 8 * (q & 1);
          const miaie_v2i lo = __builtin_bit_cast(miaie_v2i, dev::lds_read_tr16(p));
          const miaie_v2i hi = __builtin_bit_cast(miaie_v2i, dev::lds_read_tr16(p + 4 * PB));
          b[j] = v4i{lo[0], lo[1], hi[0], hi[1]};
        }
      }
#pragma unroll
      for (int i = 0; i < G::NI; ++i)
#pragma unroll
        for (int j = 0; j < G::NJ; ++j) acc[i][j] = Mma<T>::mma(b[j], a[i], acc[i][j]);
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------- split K
// Stores of partial sums go through this XCD's L2 to memory (device scope:
// the sc1 bit of a buffer store), where the other XCDs' caches read them from.
// With ordinary stores the workgroup would have to write its XCD's whole L2
// back before it may be counted (the release fence), which serialises at about
// 0.1 us per wave: 1056 workgroups took 129 us instead of 10.
constexpr int kDeviceScope = 16;  // cache policy operand: sc1
__device__ __forceinline__ __amdgpu_buffer_rsrc_t device_buffer(void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, bytes, 0x00020000);  // raw, 32-bit format
}

// A tile whose stages are divided among `splits` workgroups: each writes its
// accumulators to its slot of the context's workspace and counts itself in the
// tile's counter; the last to arrive adds all of them in split order (so
// floating-point sums do not depend on the order of arrival), sets the counter
// back to 0 for the next launch, and returns true: it alone stores the tile.  No
// workgroup waits for another.  A second launch
// for the sum costs the device about 2 us; this costs the last workgroup one
// round trip and its reads.
template <class T, class G>
__device__ __forceinline__ bool split_sum(typename Mma<T>::acc_t (&acc)[G::NI][G::NJ], int tile, int split, int splits,
                                          int8_t* work, uint32_t* counters, int* flag, int tid) {
  if constexpr (!G::SPLITS) return true;
  using acc_t = typename Mma<T>::acc_t;
  constexpr int TILE = G::BM * G::BN / 4;  // accumulator vectors per tile
  acc_t* const slots = reinterpret_cast<acc_t*>(work) + (size_t)tile * splits * TILE;
  auto at = [&](int s, int i, int j) { return slots + (size_t)s * TILE + (i * G::NJ + j) * 256 + tid; };
  const __amdgpu_buffer_rsrc_t buf = device_buffer(slots, splits * TILE * (int)sizeof(acc_t));
  auto off = [&](int s, int i, int j) { return (s * TILE + (i * G::NJ + j) * 256 + tid) * (int)sizeof(acc_t); };
#pragma unroll
  for (int i = 0; i < G::NI; ++i)
#pragma unroll
    for (int j = 0; j < G::NJ; ++j)
      if (MIAIE_CHECK(at(split, i, j), sizeof(acc_t), 1))
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, acc[i][j]), buf, off(split, i, j), 0, kDeviceScope);
  dev::waitcnt<0, 0>();  // this wave's partial sums have reached the device's memory ...
  __syncthreads();       // ... and so have the workgroup's, before it is counted
  if (tid == 0) {
    bool last = false;
    if (MIAIE_CHECK(counters + tile, sizeof(uint32_t), 1))
      last = __hip_atomic_fetch_add(counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
             (uint32_t)splits;
    *flag = last;
  }
  __syncthreads();
  if (!*flag) return false;
#pragma unroll
  for (int i = 0; i < G::NI; ++i)
#pragma unroll
    for (int j = 0; j < G::NJ; ++j) acc[i][j] = acc_t{};
  // 16 vectors in flight per thread
  constexpr int U = G::NI * G::NJ >= 16 ? 1 : 16 / (G::NI * G::NJ);
  for (int s = 0; s < splits; s += U) {
    acc_t p[U][G::NI][G::NJ];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < G::NI; ++i)
#pragma unroll
        for (int j = 0; j < G::NJ; ++j) {
          const int sp = min(s + u, splits - 1);
          p[u][i][j] = acc_t{};
          if (MIAIE_CHECK(at(sp, i, j), sizeof(acc_t), 0))
            p[u][i][j] =
                __builtin_bit_cast(acc_t, __builtin_amdgcn_raw_buffer_load_b128(buf, off(sp, i, j), 0, kDeviceScope));
        }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < splits) {
#pragma unroll
        for (int i = 0; i < G::NI; ++i)
#pragma unroll
          for (int j = 0; j < G::NJ; ++j) acc[i][j] += p[u][i][j];
      }
  }
  if (tid == 0) __hip_atomic_store(counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// ------------------------------------------------------------- output
// Four consecutive values of a row-major 32-bit output, the last ones of a row
// one by one.
template <class V, class E>
__device__ __forceinline__ void store4(E* out, size_t ld, int m, int n, int M, int N, V v) {
  if (m >= M) return;
  E* const p = out + (size_t)m * ld + n;
  if (n + 4 <= N) {
    MIAIE_ST(reinterpret_cast<Dw4<V>*>(p), Dw4<V>{v});
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) MIAIE_ST(p + e, v[e]);
  }
}

// Store the tile's int8 rows, staged in LDS with pitch G::YP: 16 bytes per
// thread, whole row pieces.
template <class G>
__device__ __forceinline__ void store_y(const int8_t* lds, int8_t* Y, size_t ld, long long m0, int n0, long long M,
                                        int N, int tid) {
  constexpr int CPR = G::BN / 16;
#pragma unroll
  for (int it = 0; it < (G::BM * CPR + 255) / 256; ++it) {
    const int flat = it * 256 + tid, r = flat / CPR, c = 16 * (flat % CPR);
    if (G::BM * CPR % 256 != 0 && flat >= G::BM * CPR) continue;
    if (m0 + r >= M || n0 + c >= N) continue;
    int8_t* const p = Y + (size_t)(m0 + r) * ld + n0 + c;
    const int8_t* const src = lds + r * G::YP + c;
    if (n0 + c + 16 <= N) {
      MIAIE_ST(reinterpret_cast<Any16*>(p), Any16{*reinterpret_cast<const v4i*>(src)});
    } else {
      for (int e = 0; n0 + c + e < N; ++e) MIAIE_ST(p + e, src[e]);
    }
  }
}

}  // namespace flex
}  // namespace miaie
