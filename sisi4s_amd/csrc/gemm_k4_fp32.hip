// FP32 instances of the tiled product kernels (gemm_k4.hpp).
#include "gemm_k4.hpp"

namespace sisi {

void launch_k4_fp32(int tile, int map, const GemmArgs &g, dim3 grid, hipStream_t s) {
  launch_k4_tiles<SISI_FP32, false>(tile, map, g, grid, s);
}

void launch_k4_grouped_fp32(int map, const GemmArgs *const *args, const unsigned *start, int n,
                            unsigned total, hipStream_t s) {
  launch_k4_grouped_maps<SISI_FP32>(map, args, start, n, total, s);
}

}  // namespace sisi
