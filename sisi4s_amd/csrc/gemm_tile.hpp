// Device core of the FP64 / FP32 MFMA products (gemm_k4.hpp, gemm_seg.hip):
// operand tiles staged through a double-buffered LDS chunk of 16 k.
//
// What bounds it: the FP64 MFMA pipe (v_mfma_f64_16x16x4 takes 64 cycles, a
// 64 x 64 wave tile 4096 cycles per chunk); everything else has to stay out
// of its way.  So the main loop holds no bounds checks and no conversions: a
// chunk that is whole in k loads 16 bytes per instruction from pointers
// computed once (rows past the edge read a clamped row, whose products are
// never stored), the next chunk's loads fly during the current chunk's MFMAs,
// and one barrier per chunk separates the two LDS buffers.  Only the last,
// partial chunk of k selects zeros.
#pragma once

#include "gemm_device.hpp"

namespace sisi {

typedef double d2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
// two doubles at any element address (odd leading dimensions)
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int kTileK = 16;  // k per chunk, where not stated otherwise

// LDS layout of R rows by KC k: k-fast rows of KC + 2 elements (144 bytes: the
// 16 rows of a fragment read fall on distinct banks) or m-fast rows of R + 4.
// Both measure no bank conflicts at 2560^3 (m-fast rows of R + 16 cost four
// cycles per fragment read).
template <int R, bool KF, int KC = kTileK>
struct TileLds {
  static constexpr int kRow = KF ? KC + 2 : 1;
  static constexpr int kCol = KF ? 1 : R + 4;
  static constexpr int kSize = KF ? R * (KC + 2) : KC * (R + 4);
};

// One operand's tile rows [r0, r0 + R): global loads of a KC-k chunk into
// registers, and the store into LDS.  KF: k is the index the threads walk.
template <typename LT, int R, bool KF, int KC = kTileK>
struct TileLoader {
  static constexpr int kGran = R * KC / 2;  // two-element granules per chunk
  static constexpr int kQ = (kGran + 255) / 256;
  static constexpr bool kWhole = kGran % 256 == 0;
  using L2 = typename std::conditional<sizeof(LT) == 8, d2, f2>::type;

  const double *base = nullptr;  // uniform, moved by one chunk per load
  int64_t step = 0;              // elements per chunk
  int64_t sr = 1, sk = 0;
  int64_t off[kQ];
  int last = 0;  // last valid row, relative to r0
  bool vec = false;
  d2 v[kQ];

  static __device__ __forceinline__ void place(int e, int &row, int &k) {
    row = KF ? e / (KC / 2) : 2 * (e % (R / 2));
    k = KF ? 2 * (e % (KC / 2)) : e / (R / 2);
  }

  __device__ __forceinline__ void init(const double *p, int64_t s_row, int64_t s_k, int r0,
                                       int rlast, int k0) {
    sr = s_row;
    sk = s_k;
    base = p + int64_t(r0) * sr + int64_t(k0) * sk;
    step = KC * sk;
    last = rlast - r0;
    // 16-byte loads need the walked index at unit stride; along the rows
    // also every row of the tile in range
    vec = KF ? sk == 1 : (sr == 1 && last >= R - 1);
#pragma unroll
    for (int q = 0; q < kQ; ++q) {
      int row, k;
      place(int(threadIdx.x) + 256 * q, row, k);
      off[q] = int64_t(min(row, last)) * sr + int64_t(k) * sk;
    }
  }

  // a chunk whole in k
  __device__ __forceinline__ void load() {
    if (vec) {
#pragma unroll
      for (int q = 0; q < kQ; ++q)
        if (kWhole || int(threadIdx.x) + 256 * q < kGran)
          v[q] = *reinterpret_cast<const d2u *>(base + off[q]);
    } else {
#pragma unroll
      for (int q = 0; q < kQ; ++q)
        if (kWhole || int(threadIdx.x) + 256 * q < kGran) {
          int row, k;
          place(int(threadIdx.x) + 256 * q, row, k);
          const int64_t d = KF ? sk : (row < last ? sr : 0);
          v[q].x = base[off[q]];
          v[q].y = base[off[q] + d];
        }
    }
    base += step;
  }

  // the last chunk, nk < KC: elements past nk are zero (loaded from a clamped k)
  __device__ __forceinline__ void load_tail(int nk) {
#pragma unroll
    for (int q = 0; q < kQ; ++q)
      if (kWhole || int(threadIdx.x) + 256 * q < kGran) {
        int row, k;
        place(int(threadIdx.x) + 256 * q, row, k);
        const int64_t r = int64_t(min(row, last)) * sr;
        if (KF) {
          const double x = base[r + int64_t(min(k, nk - 1)) * sk];
          const double y = base[r + int64_t(min(k + 1, nk - 1)) * sk];
          v[q].x = k < nk ? x : 0.0;
          v[q].y = k + 1 < nk ? y : 0.0;
        } else {
          const int64_t o = r + int64_t(min(k, nk - 1)) * sk;
          const double x = base[o];
          const double y = base[o + (row < last ? sr : 0)];
          v[q].x = k < nk ? x : 0.0;
          v[q].y = k < nk ? y : 0.0;
        }
      }
  }

  __device__ __forceinline__ void scale(double s) {
#pragma unroll
    for (int q = 0; q < kQ; ++q) v[q] *= s;
  }

  __device__ __forceinline__ void store(LT *lds) const {
#pragma unroll
    for (int q = 0; q < kQ; ++q)
      if (kWhole || int(threadIdx.x) + 256 * q < kGran) {
        int row, k;
        place(int(threadIdx.x) + 256 * q, row, k);
        L2 w;
        w.x = LT(v[q].x);
        w.y = LT(v[q].y);
        *reinterpret_cast<L2 *>(
            lds + row * TileLds<R, KF, KC>::kRow + k * TileLds<R, KF, KC>::kCol) = w;
      }
  }
};

template <int PREC>
struct TileTypes {
  using LT = typename std::conditional<PREC == SISI_FP64, double, float>::type;
  using AT = typename std::conditional<PREC == SISI_FP64, d4, f4>::type;
  // result layout of the 16x16 tile: row (here n) = kLane*(lane/16) + kReg*reg
  // (v_mfma_f64_16x16x4f64: lane/16 + 4*reg; the f32 form: 4*(lane/16) + reg)
  static constexpr int kLane = PREC == SISI_FP64 ? 1 : 4;
  static constexpr int kReg = PREC == SISI_FP64 ? 4 : 1;
};

// One LDS chunk into a wave's accumulators.  a and b point at the wave's
// first row of each operand.
template <int PREC, int TI, int TJ, int AROW, int ACOL, int BROW, int BCOL, int KC = kTileK>
__device__ __forceinline__ void tile_mma(const typename TileTypes<PREC>::LT *a,
                                         const typename TileTypes<PREC>::LT *b, int lane,
                                         typename TileTypes<PREC>::AT (&acc)[TI][TJ]) {
  using LT = typename TileTypes<PREC>::LT;
  const int l16 = lane & 15, lk = lane >> 4;
  const LT *pa = a + l16 * AROW + lk * ACOL, *pb = b + l16 * BROW + lk * BCOL;
#pragma unroll
  for (int kq = 0; kq < KC / 4; ++kq) {
    LT av[TI], bv[TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i) av[i] = pa[i * 16 * AROW + kq * 4 * ACOL];
#pragma unroll
    for (int j = 0; j < TJ; ++j) bv[j] = pb[j * 16 * BROW + kq * 4 * BCOL];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j) {
        if constexpr (PREC == SISI_FP64)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j], av[i], acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[j], av[i], acc[i][j], 0, 0, 0);
      }
  }
}

}  // namespace sisi
