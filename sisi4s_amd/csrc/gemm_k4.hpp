// FP64 / FP32 product kernels over a family of block tiles (gemm.hip plans
// and launches them; gemm_k4_fp64.hip and gemm_k4_fp32.hip hold the
// instances).
#pragma once

#include "gemm_tile.hpp"

namespace sisi {

// Block tiles (four wave64s, 2 x 2).  The large one reads least per product;
// the small ones give a small product enough workgroups and a short chain: a
// wave's chunk takes 4096 cycles of FP64 MFMA at 128 x 128, 256 at 32 x 32.
// Oblong tiles (128 x 64, 128 x 32 and their transposes) were measured too
// and were best at no size by more than 5 %.
constexpr int kTiles[] = {128, 64, 32};
constexpr int kNumTiles = 3;
// first of them a complex product can take
constexpr int first_tile_z(int precision) { return precision == SISI_FP32 ? 1 : 0; }
// k per chunk: a wave of the 32 x 32 tile has four MFMAs per 16 k between two
// barriers, too few to cover the chain of store, barrier and reads; with 32 k
// 250^3 takes 8.9 -> 7.6 us, 500^3 14.9 -> 13.0, 777 x 640 x 1531 47 -> 40
// (FP32: 500^3 12.9 -> 10.2, 810^3 29 -> 22)
constexpr int tile_k(int tile) { return tile == 32 ? 32 : kTileK; }

// Load mappings: 0: A m-fast, B k-fast; +1: B n-fast; +2: A k-fast.
void launch_k4_fp64(int tile, int map, const GemmArgs &g, dim3 grid, hipStream_t s);
void launch_k4_fp32(int tile, int map, const GemmArgs &g, dim3 grid, hipStream_t s);
// The same for planar complex operands (g.cplx).
void launch_k4z_fp64(int tile, int map, const GemmArgs &g, dim3 grid, hipStream_t s);
void launch_k4z_fp32(int tile, int map, const GemmArgs &g, dim3 grid, hipStream_t s);
// Grouped launch of n products (batched solver): record p owns the blocks
// [start[p], start[p + 1]): tiles_m * tiles_n per k-split and batch entry.
// The systems of a grouped launch fill the device together, and one tile for
// all of them keeps their records in one launch.
constexpr int kTapeTile = 1;  // 64 x 64
void launch_k4_grouped_fp64(int map, const GemmArgs *const *args, const unsigned *start, int n,
                            unsigned total, hipStream_t s);
void launch_k4_grouped_fp32(int map, const GemmArgs *const *args, const unsigned *start, int n,
                            unsigned total, hipStream_t s);

#ifdef __HIPCC__

// FP32 sums over k in two levels: the accumulators of the 64 and 32 tiles are
// added into FP64 sums every kFlush k (the 128 tile has no registers for that:
// its chains are kept short by choose_tile), so a product that is split less
// along K than its few tiles would suggest has no longer FP32 chain than one
// split into parts of eight chunks.  Relative error against 64 bits in one
// chain, in such parts, and in two levels: 777 x 640 x 1531 7.0, 2.5, 2.0e-7;
// 250 x 250 x 8000 5.7, 2.2, 2.0e-7; of positive terms 5.3e-7, 6.8e-8, 5.0e-8
// and 1.7e-7, 2.4e-8, 2.2e-8.  FP64 sums stay one chain: in two levels they
// measured the same error and took 43.2 instead of 39.2 us at the first size.
constexpr int kFlush = 128;

// Output tile `pid`, k-split `ks`, batch entry `bz` of one product.  CPLX: the
// part bz (0 Re, 1 Im) of a planar complex product, its two plane products as
// one k loop (a separate launch and a read-modify-write of C for each of the
// four took a 9-orbital complex CCSD iteration 590 launches); in FP32 on the
// two-level tiles only.
template <int PREC, int TBM, int TBN, int WGM, int WGN, bool AK, bool BNF, bool CPLX = false>
__device__ __forceinline__ void gemm_k4_body(const GemmArgs &g, int pid, int ks, int bz) {
  using LT = typename TileTypes<PREC>::LT;
  using AT = typename TileTypes<PREC>::AT;
  constexpr int WM = TBM / WGM, WN = TBN / WGN, TI = WM / 16, TJ = WN / 16;
  static_assert(WGM * WGN == 4 && TI * 16 == WM && TJ * 16 == WN, "four waves, 16-multiples");
  constexpr int KC = tile_k(TBM);
  constexpr bool kTwoLevel = PREC == SISI_FP32 && TBM <= 64;
  static_assert(!CPLX || PREC == SISI_FP64 || kTwoLevel,
                "an FP32 sum over both plane products needs two levels");
  using LA = TileLds<TBM, AK, KC>;
  using LB = TileLds<TBN, !BNF, KC>;
  __shared__ __attribute__((aligned(16))) LT As[2][LA::kSize];
  __shared__ __attribute__((aligned(16))) LT Bs[2][LB::kSize];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  int tm, tn;
  tile_coords(g, pid, tm, tn);
  const int m0 = tm * TBM, n0 = tn * TBN;
  const int kbeg = ks * g.kchunk;
  const int kend = min(g.K, kbeg + g.kchunk);
  const int half = (kend - kbeg + KC - 1) / KC;  // chunks of one plane product
  const int chunks = CPLX ? 2 * half : half;
  const int wm = (wave % WGM) * WM, wn = (wave / WGM) * WN;
  // a wave whose sub-tile lies wholly outside the output skips its MFMAs
  const bool active = (m0 + wm < g.M) && (n0 + wn < g.N);

  TileLoader<LT, TBM, AK, KC> la;
  TileLoader<LT, TBN, !BNF, KC> lb;
  double scale = 1.0;  // of the chunk in the registers
  if constexpr (CPLX) {
    la.init(g.A, g.sam, g.sak, m0, g.M - 1, kbeg);
    lb.init(g.B + (bz ? g.zb : 0), g.sbn, g.sbk, n0, g.N - 1, kbeg);
    scale = bz ? g.sb : 1.0;
  } else {
    la.init(g.A + int64_t(bz) * g.bsa, g.sam, g.sak, m0, g.M - 1, kbeg);
    lb.init(g.B + int64_t(bz) * g.bsb, g.sbn, g.sbk, n0, g.N - 1, kbeg);
  }
  auto load = [&](int c) {
    if constexpr (CPLX) {
      if (c == half) {  // Im A with Im B (Re C) or Re B (Im C)
        la.init(g.A + g.za, g.sam, g.sak, m0, g.M - 1, kbeg);
        lb.init(g.B + (bz ? 0 : g.zb), g.sbn, g.sbk, n0, g.N - 1, kbeg);
        scale = bz ? g.sa : -g.sa * g.sb;
      }
      if (c >= half) c -= half;
    }
    const int nk = kend - kbeg - c * KC;
    if (nk >= KC) {
      la.load();
      lb.load();
    } else {
      la.load_tail(nk);
      lb.load_tail(nk);
    }
  };

  AT acc[TI][TJ];
  d4 sum[kTwoLevel ? TI : 1][kTwoLevel ? TJ : 1];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      acc[i][j] = AT{0, 0, 0, 0};
      if constexpr (kTwoLevel) sum[i][j] = d4{0, 0, 0, 0};
    }
  auto flush = [&]() {
    if constexpr (kTwoLevel) {
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
#pragma unroll
          for (int r = 0; r < 4; ++r) sum[i][j][r] += double(acc[i][j][r]);
          acc[i][j] = AT{0, 0, 0, 0};
        }
    }
  };
  auto result = [&](int i, int j, int r) -> double {
    if constexpr (kTwoLevel) return sum[i][j][r];
    else return double(acc[i][j][r]);
  };

  if (chunks > 0) {
    load(0);
    if (CPLX && scale != 1.0) la.scale(scale);
    la.store(As[0]);
    lb.store(Bs[0]);
    if (chunks > 1) load(1);
    __syncthreads();
    int left = kFlush / KC;  // chunks to the next addition into the sums
    for (int c = 0; c < chunks; ++c) {
      // buffer (c + 1) & 1 was last read before the barrier just passed
      if (c + 1 < chunks) {
        if (CPLX && scale != 1.0) la.scale(scale);
        la.store(As[(c + 1) & 1]);
        lb.store(Bs[(c + 1) & 1]);
        if (c + 2 < chunks) load(c + 2);
      }
      if (active)
        tile_mma<PREC, TI, TJ, LA::kRow, LA::kCol, LB::kRow, LB::kCol, KC>(
            As[c & 1] + wm * LA::kRow, Bs[c & 1] + wn * LB::kRow, lane, acc);
      if (kTwoLevel && --left == 0) {
        flush();
        left = kFlush / KC;
      }
      __syncthreads();
    }
    flush();
  }

  const int l16 = lane & 15, lk = lane >> 4;
  constexpr int LSTR = TileTypes<PREC>::kLane, RSTR = TileTypes<PREC>::kReg;
  if (g.ksplit == 1) {
    double *C = g.C + int64_t(bz) * g.bsc;
    // row offsets once per row, each column offset once per column (the
    // output splits cost divisions)
    int64_t om[TI];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const int m = m0 + wm + i * 16 + l16;
      om[i] = m < g.M ? out_off_m(g, m) : -1;
    }
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + wn + j * 16 + LSTR * lk + RSTR * r;
        if (n >= g.N) continue;
        const int64_t on = out_off_n(g, n);
#pragma unroll
        for (int i = 0; i < TI; ++i) {
          if (om[i] < 0) continue;
          const int64_t o = om[i] + on;
          double v = g.alpha * result(i, j, r);
          if (g.beta != 0.0) v += g.beta * C[o];
          C[o] = v;
        }
      }
  } else {
    double *W = g.work + (int64_t(bz) * g.ksplit + ks) * int64_t(g.M) * g.N;
#pragma unroll
    for (int i = 0; i < TI; ++i) {
      const int m = m0 + wm + i * 16 + l16;
      if (m >= g.M) continue;
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int n = n0 + wn + j * 16 + LSTR * lk + RSTR * r;
          if (n < g.N) W[m + int64_t(n) * g.M] = result(i, j, r);
        }
    }
  }
}

template <int PREC, int TBM, int TBN, int WGM, int WGN, bool AK, bool BNF, bool CPLX>
__global__ __launch_bounds__(256, 2) void gemm_k4_kernel(GemmArgs g) {
  gemm_k4_body<PREC, TBM, TBN, WGM, WGN, AK, BNF, CPLX>(g, blockIdx.x, blockIdx.y, blockIdx.z);
}

template <int PREC, int TBM, int TBN, int WGM, int WGN, bool AK, bool BNF>
__global__ __launch_bounds__(256, 2) void gemm_k4_grouped(const GemmArgs *const *args,
                                                          const unsigned *__restrict__ start,
                                                          int n) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= blockIdx.x) lo = mid;
    else hi = mid - 1;
  }
  // the record is read in place (a copy kept the whole struct live in
  // registers and made the kernel spill)
  const GemmArgs &g = *args[lo];
  const int tiles = g.tiles_m * g.tiles_n;
  const int local = int(blockIdx.x - start[lo]);
  const int r = local / tiles;
  gemm_k4_body<PREC, TBM, TBN, WGM, WGN, AK, BNF>(g, local % tiles, r % g.ksplit, r / g.ksplit);
}

template <int PREC, bool CPLX>
void launch_k4_tiles(int tile, int map, const GemmArgs &g, dim3 grid, hipStream_t s) {
  switch (tile * 4 + map) {
#define SISI_K4_ONE(T, MAP, AK_, BNF_)                                                          \
  case T * 4 + MAP:                                                                             \
    if constexpr (CPLX && T < first_tile_z(PREC))                                                     \
      throw Error(SISI_ERR_INVALID, "gemm: no such tile of a complex product");                 \
    else                                                                                        \
      hipLaunchKernelGGL((gemm_k4_kernel<PREC, kTiles[T], kTiles[T], 2, 2, AK_, BNF_, CPLX>),   \
                         grid, dim3(256), 0, s, g);                                             \
    break;
#define SISI_K4_ALL(T)             \
  SISI_K4_ONE(T, 0, false, false)  \
  SISI_K4_ONE(T, 1, false, true)   \
  SISI_K4_ONE(T, 2, true, false)   \
  SISI_K4_ONE(T, 3, true, true)
    SISI_K4_ALL(0)
    SISI_K4_ALL(1)
    SISI_K4_ALL(2)
#undef SISI_K4_ALL
#undef SISI_K4_ONE
    default: throw Error(SISI_ERR_INVALID, "gemm: unknown tile");
  }
  SISI_HIP(hipGetLastError());
}

template <int PREC>
void launch_k4_grouped_maps(int map, const GemmArgs *const *args, const unsigned *start, int n,
                            unsigned total, hipStream_t s) {
  constexpr int T = kTiles[kTapeTile];
  switch (map) {
#define SISI_K4_ONE(MAP, AK_, BNF_)                                                        \
  case MAP:                                                                                \
    hipLaunchKernelGGL((gemm_k4_grouped<PREC, T, T, 2, 2, AK_, BNF_>), dim3(total),        \
                       dim3(256), 0, s, args, start, n);                                   \
    break;
    SISI_K4_ONE(0, false, false)
    SISI_K4_ONE(1, false, true)
    SISI_K4_ONE(2, true, false)
    SISI_K4_ONE(3, true, true)
#undef SISI_K4_ONE
    default: throw Error(SISI_ERR_INVALID, "grouped gemm: unknown load mapping");
  }
  SISI_HIP(hipGetLastError());
}

#endif  // __HIPCC__

}  // namespace sisi
