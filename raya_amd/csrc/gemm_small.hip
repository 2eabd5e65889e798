// The GEMM kernel's small tiles (gemm_kernel.hpp), in a unit of their own to compile beside the others.
#define RAYA_GEMM_INSTANTIATE
#include "gemm_kernel.hpp"

namespace raya {
namespace gemm {

template hipError_t launch_tile<Tile64x128, false>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile64x128, true>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile64, false>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile64, true>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile32, false>(const GemmLaunch &, unsigned, hipStream_t);
template hipError_t launch_tile<Tile32, true>(const GemmLaunch &, unsigned, hipStream_t);

}  // namespace gemm
}  // namespace raya
