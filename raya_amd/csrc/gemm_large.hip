// The GEMM kernel's large tiles (gemm_kernel.hpp), in a unit of their own to compile beside the others.
#define RAYA_GEMM_INSTANTIATE
#include "gemm_kernel.hpp"

namespace raya {
namespace gemm {

template hipError_t launch_tile<Tile256, false>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile256, true>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile256x128, false>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile256x128, true>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile128, false>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile128, true>(const GemmLaunch &, unsigned, hipStream_t);

}  // namespace gemm
}  // namespace raya
