// Segmented MFMA GEMM: C = alpha * sum_s scale_s A_s B_s + beta * C with up
// to four products of different K, operands and layouts accumulated in the
// same registers, so a sum of contractions into one output costs one launch
// and one epilogue pass instead of one read-modify-write of C per product.
//
// FP64 / FP32: the tile core of gemm_tile.hpp.  On-the-fly BF16x3: block
// tile, LDS staging and MFMA forms of the kernel in gemm.hip, the operand
// load mapping (m- or k-fast A, k- or n-fast B) chosen per segment at run
// time.
#include <cstdlib>

#include "engine.hpp"
#include "gemm.hpp"
#include "gemm_tile.hpp"

namespace sisi {

namespace {

// Block tile 64 x 64 of four waves of 32 x 32, every operand k-fast.  The
// chunk pipeline is the one of gemm_k4.hpp; a chunk of the next segment is
// fetched while the last one of this segment is multiplied, so the segments
// run as one k loop.
//
// FP64 MFMA bounds it.  The tile: four workgroups share a CU (37 KB of LDS,
// 94 registers), which hides the chains of a k loop of only ~30 chunks and
// the read-modify-write of C at its end.  A (T) pass in FP64 with tiles of 64
// x 64, 80 x 128, 96 x 128, 128 x 128: No = 12, Nv = 240 287, 324, 356, 316
// ms; No = 14, Nv = 288 869, 1032, 891, 1118; No = 7, Nv = 95 7.1, 9.7, 10.4,
// 12.4.  The kernel before it (element loads with bounds checks, two barriers
// per chunk, 80 x 128 and 128 x 128 tiles) took 370, 1387 and 14.5 ms.
constexpr int kSegTile = 64;

template <int PREC>
__global__ __launch_bounds__(256, 2) void gemm_seg_k4_kernel(SegGemmArgs a) {
  using LT = typename TileTypes<PREC>::LT;
  using AT = typename TileTypes<PREC>::AT;
  constexpr int TBM = kSegTile, TBN = kSegTile, WGM = 2, WGN = 2;
  constexpr int WM = TBM / WGM, WN = TBN / WGN, TI = WM / 16, TJ = WN / 16;
  using LA = TileLds<TBM, true>;
  using LB = TileLds<TBN, true>;
  __shared__ __attribute__((aligned(16))) LT As[2][LA::kSize];
  __shared__ __attribute__((aligned(16))) LT Bs[2][LB::kSize];
  const GemmArgs &g = a.g;
  // the segments are indexed at run time: read from the argument block where
  // it lies (a copy of it in scratch made every field a per-lane value)
  using Args = __attribute__((address_space(4))) const SegGemmArgs;
  Args *ka = (Args *)__builtin_amdgcn_kernarg_segment_ptr();

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  int tm, tn;
  tile_coords(g, blockIdx.x, tm, tn);
  const int m0 = tm * TBM, n0 = tn * TBN;

  TileLoader<LT, TBM, true> la;
  TileLoader<LT, TBN, true> lb;
  int chunks = 0;
  for (int i = 0; i < a.nseg; ++i) chunks += (ka->seg[i].K + kTileK - 1) / kTileK;
  int s = -1, left = 0;  // segment of the next chunk, and k left in it
  double scale = 1.0;    // of the chunk in the registers
  auto fetch = [&]() {
    if (left <= 0) {
      ++s;
      la.init(ka->seg[s].A, ka->seg[s].sam, 1, m0, g.M - 1, 0);
      lb.init(ka->seg[s].B, ka->seg[s].sbn, 1, n0, g.N - 1, 0);
      scale = ka->seg[s].scale;
      left = ka->seg[s].K;
    }
    if (left >= kTileK) {
      la.load();
      lb.load();
    } else {
      la.load_tail(left);
      lb.load_tail(left);
    }
    left -= kTileK;
  };

  AT acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j) acc[i][j] = AT{0, 0, 0, 0};

  const int wm = (wave % WGM) * WM, wn = (wave / WGM) * WN;
  const bool active = (m0 + wm < g.M) && (n0 + wn < g.N);

  // chunk c is multiplied in iteration c >= 0; iteration -1 fills the pipeline
  fetch();
  for (int c = -1; c < chunks; ++c) {
    if (c + 1 < chunks) {
      if (scale != 1.0) la.scale(scale);
      la.store(As[(c + 1) & 1]);
      lb.store(Bs[(c + 1) & 1]);
      if (c + 2 < chunks) fetch();
    }
    if (active && c >= 0)
      tile_mma<PREC, TI, TJ, LA::kRow, LA::kCol, LB::kRow, LB::kCol>(
          As[c & 1] + wm * LA::kRow, Bs[c & 1] + wn * LB::kRow, lane, acc);
    __syncthreads();
  }

  // row offsets once per row, each column offset once per column (the
  // output splits cost divisions)
  const int l16 = lane & 15, lk = lane >> 4;
  constexpr int LSTR = TileTypes<PREC>::kLane, RSTR = TileTypes<PREC>::kReg;
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
        double v = g.alpha * double(acc[i][j][r]);
        if (g.beta != 0.0) v += g.beta * g.C[o];
        g.C[o] = v;
      }
    }
}

__device__ __forceinline__ GemmSeg seg_at(const SegGemmArgs &a, int s) {
  return s == 0 ? a.seg[0] : s == 1 ? a.seg[1] : s == 2 ? a.seg[2] : a.seg[3];
}

__device__ __forceinline__ int seg_k(const SegGemmArgs &a, int s) {
  return s == 0 ? a.seg[0].K : s == 1 ? a.seg[1].K : s == 2 ? a.seg[2].K : a.seg[3].K;
}

__global__ __launch_bounds__(256, 2) void gemm_seg_b3_kernel(SegGemmArgs a) {
  constexpr int BK = 32;
  constexpr int RS = BK + 8;  // row stride in bf16 (keeps 16-byte alignment)
  __shared__ __attribute__((aligned(16))) __bf16 Ah[BM * RS];
  __shared__ __attribute__((aligned(16))) __bf16 Al[BM * RS];
  __shared__ __attribute__((aligned(16))) __bf16 Bh[BN * RS];
  __shared__ __attribute__((aligned(16))) __bf16 Bl[BN * RS];
  const GemmArgs &g = a.g;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar branches
  int tm, tn;
  tile_coords(g, blockIdx.x, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  double ra[16], rb[16];
  int lak = 0, lbnf = 0;
  // Out-of-range elements load from a clamped (in-range) address (no
  // branch) and are zeroed at the LDS store, one chunk later.
  const int mlast = g.M - 1, nlast = g.N - 1;
  int lk0 = 0, lK = 0;
  double lsc = 1.0;
  auto load = [&](int s, int k0) {
    const GemmSeg sg = seg_at(a, s);
    const int klast = sg.K - 1;
    lak = sg.ak;
    lbnf = sg.bnf;
    lk0 = k0;
    lK = sg.K;
    lsc = sg.scale;
    if (!sg.ak) {  // m fastest: 32 threads x 4 m, 8 k rows, 4 passes
      const int mm = (tid & 31) * 4, kk = tid >> 5;
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int k = k0 + kk + 8 * h;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int m = m0 + mm + j;
          ra[h * 4 + j] = sg.A[int64_t(min(m, mlast)) * sg.sam + int64_t(min(k, klast)) * sg.sak];
        }
      }
    } else {  // k fastest: 32 threads along k, m = t/32 + 8 j
      const int kk = tid & 31, mm = tid >> 5;
      const int k = k0 + kk;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int m = m0 + mm + 8 * j;
        ra[j] = sg.A[int64_t(min(m, mlast)) * sg.sam + int64_t(min(k, klast)) * sg.sak];
      }
    }
    if (sg.bnf) {
      const int nn = (tid & 31) * 4, kk = tid >> 5;
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const int k = k0 + kk + 8 * h;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int n = n0 + nn + j;
          rb[h * 4 + j] = sg.B[int64_t(min(k, klast)) * sg.sbk + int64_t(min(n, nlast)) * sg.sbn];
        }
      }
    } else {
      const int kk = tid & 31, nn = tid >> 5;
      const int k = k0 + kk;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int n = n0 + nn + 8 * j;
        rb[j] = sg.B[int64_t(min(k, klast)) * sg.sbk + int64_t(min(n, nlast)) * sg.sbn];
      }
    }
  };
  auto store = [&]() {
    __bf16 h, l;
    if (!lak) {
      const int mm = (tid & 31) * 4, kk = tid >> 5;
#pragma unroll
      for (int hh = 0; hh < 4; ++hh)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          split_bf16(ra[hh * 4 + j] * ((m0 + mm + j <= mlast && lk0 + kk + 8 * hh < lK) ? lsc : 0.0), h, l);
          Ah[(mm + j) * RS + kk + 8 * hh] = h;
          Al[(mm + j) * RS + kk + 8 * hh] = l;
        }
    } else {
      const int kk = tid & 31, mm = tid >> 5;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        split_bf16(ra[j] * ((m0 + mm + 8 * j <= mlast && lk0 + kk < lK) ? lsc : 0.0), h, l);
        Ah[(mm + 8 * j) * RS + kk] = h;
        Al[(mm + 8 * j) * RS + kk] = l;
      }
    }
    if (lbnf) {
      const int nn = (tid & 31) * 4, kk = tid >> 5;
#pragma unroll
      for (int hh = 0; hh < 4; ++hh)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          split_bf16(rb[hh * 4 + j] * ((n0 + nn + j <= nlast && lk0 + kk + 8 * hh < lK) ? 1.0 : 0.0), h, l);
          Bh[(nn + j) * RS + kk + 8 * hh] = h;
          Bl[(nn + j) * RS + kk + 8 * hh] = l;
        }
    } else {
      const int kk = tid & 31, nn = tid >> 5;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        split_bf16(rb[j] * ((n0 + nn + 8 * j <= nlast && lk0 + kk < lK) ? 1.0 : 0.0), h, l);
        Bh[(nn + 8 * j) * RS + kk] = h;
        Bl[(nn + 8 * j) * RS + kk] = l;
      }
    }
  };

  f4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f4{0, 0, 0, 0};
  const int wm = (wave & 1) * 64, wn = (wave >> 1) * 64;
  const int l16 = lane & 15, lk = lane >> 4;

  int s = 0, k0 = 0;
  bool have = a.nseg > 0;
  if (have) load(0, 0);
  while (have) {
    store();
    __syncthreads();
    int s1 = s, k1 = k0 + BK;
    if (k1 >= seg_k(a, s)) {
      s1 = s + 1;
      k1 = 0;
    }
    const bool more = s1 < a.nseg;
    if (more) load(s1, k1);
    bf8 ah[4], al[4], bh[4], bl[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = wm + i * 16 + l16;
      ah[i] = *reinterpret_cast<const bf8 *>(&Ah[row * RS + 8 * lk]);
      al[i] = *reinterpret_cast<const bf8 *>(&Al[row * RS + 8 * lk]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int col = wn + j * 16 + l16;
      bh[j] = *reinterpret_cast<const bf8 *>(&Bh[col * RS + 8 * lk]);
      bl[j] = *reinterpret_cast<const bf8 *>(&Bl[col * RS + 8 * lk]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bl[j], ah[i], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[j], al[i], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bh[j], ah[i], acc[i][j], 0, 0, 0);
    __syncthreads();
    s = s1;
    k0 = k1;
    have = more;
  }

  int64_t om[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + wm + i * 16 + l16;
    om[i] = m < g.M ? out_off_m(g, m) : -1;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = n0 + wn + j * 16 + 4 * lk + r;
      if (n >= g.N) continue;
      const int64_t on = out_off_n(g, n);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (om[i] < 0) continue;
        const int64_t o = om[i] + on;
        double v = g.alpha * double(acc[i][j][r]);
        if (g.beta != 0.0) v += g.beta * g.C[o];
        g.C[o] = v;
      }
    }
}

}  // namespace

void gemm_segments(Engine &eng, int precision, SegGemmArgs a) {
  GemmArgs &g = a.g;
  if (g.M <= 0 || g.N <= 0) return;
  SISI_REQUIRE(a.nseg >= 1 && a.nseg <= kMaxSegs, SISI_ERR_INVALID,
               "gemm_segments: 1 to 4 segments");
  SISI_REQUIRE(precision == SISI_FP64 || precision == SISI_FP32 || precision == SISI_BF16X3,
               SISI_ERR_INVALID, "gemm_segments: unknown precision");
  double flops = 0.0;
  for (int s = 0; s < a.nseg; ++s) {
    GemmSeg &sg = a.seg[s];
    SISI_REQUIRE(sg.K > 0 && sg.A && sg.B, SISI_ERR_INVALID,
                 "gemm_segments: every segment needs K > 0 and operands");
    // the flags only choose which index consecutive threads walk
    sg.bnf = (sg.sbn == 1 && sg.sbk != 1) ? 1 : 0;
    sg.ak = (sg.sak == 1 && sg.sam != 1) ? 1 : 0;
    flops += 2.0 * double(g.M) * double(g.N) * double(sg.K);
  }
  g.batch = 1;
  g.ksplit = 1;
  g.kchunk = 0;
  g.split_out = !(g.dm0 >= g.M && g.dn0 >= g.N);
  {
    static const int env_group = getenv("SISI_GEMM_GROUP") ? atoi(getenv("SISI_GEMM_GROUP")) : 8;
    g.group = env_group > 0 ? env_group : 8;
  }
  if (precision == SISI_BF16X3) {
    g.tiles_m = (g.M + BM - 1) / BM;
    g.tiles_n = (g.N + BN - 1) / BN;
    g.xcd_map = 1;
    const int64_t tiles = int64_t(g.tiles_m) * g.tiles_n;
    SISI_REQUIRE(tiles < (int64_t(1) << 31), SISI_ERR_INVALID, "gemm_segments: too many tiles");
    Timed t(*eng.timers, Kind::GemmB3, flops);
    hipLaunchKernelGGL(gemm_seg_b3_kernel, dim3(unsigned(tiles), 1u, 1u), dim3(256), 0,
                       eng.stream, a);
    SISI_HIP(hipGetLastError());
    return;
  }
  for (int i = 0; i < a.nseg; ++i)
    SISI_REQUIRE(a.seg[i].sak == 1 && a.seg[i].sbk == 1, SISI_ERR_INVALID,
                 "gemm_segments: FP64 and FP32 segments are k-fast");
  g.tiles_m = (g.M + kSegTile - 1) / kSegTile;
  g.tiles_n = (g.N + kSegTile - 1) / kSegTile;
  g.xcd_map = 1;
  const int64_t tiles = int64_t(g.tiles_m) * g.tiles_n;
  SISI_REQUIRE(tiles < (int64_t(1) << 31), SISI_ERR_INVALID, "gemm_segments: too many tiles");
  Timed t(*eng.timers, precision == SISI_FP64 ? Kind::Gemm64 : Kind::Gemm32, flops);
  const dim3 grid(unsigned(tiles), 1u, 1u);
  if (precision == SISI_FP64)
    hipLaunchKernelGGL(gemm_seg_k4_kernel<SISI_FP64>, grid, dim3(256), 0, eng.stream, a);
  else
    hipLaunchKernelGGL(gemm_seg_k4_kernel<SISI_FP32>, grid, dim3(256), 0, eng.stream, a);
  SISI_HIP(hipGetLastError());
}

}  // namespace sisi
