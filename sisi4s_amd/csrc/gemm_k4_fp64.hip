// FP64 instances of the tiled product kernels (gemm_k4.hpp).
#include "gemm_k4.hpp"

namespace sisi {

void launch_k4_fp64(int tile, int map, const GemmArgs &g, dim3 grid, hipStream_t s) {
  launch_k4_tiles<SISI_FP64, false>(tile, map, g, grid, s);
}

void launch_k4_grouped_fp64(int map, const GemmArgs *const *args, const unsigned *start, int n,
                            unsigned total, hipStream_t s) {
  launch_k4_grouped_maps<SISI_FP64>(map, args, start, n, total, s);
}

}  // namespace sisi
