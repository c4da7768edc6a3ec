// FP64 instances of the tiled product kernels on planar complex operands
// (gemm_k4.hpp).
#include "gemm_k4.hpp"

namespace sisi {

void launch_k4z_fp64(int tile, int map, const GemmArgs &g, dim3 grid, hipStream_t s) {
  launch_k4_tiles<SISI_FP64, true>(tile, map, g, grid, s);
}

}  // namespace sisi
