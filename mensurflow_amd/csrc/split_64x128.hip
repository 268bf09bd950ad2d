// The split kernel on the 64x128 tile (split_kernel.hpp).
#include "split.hpp"
#include "split_kernel.hpp"

namespace mfr::gemm {

void launch_split_64x128(const GemmParams& p, bool ak, bool bk, unsigned blocks, hipStream_t s) {
    launch_split_tile<64, 128, 32, 2, 2>(p, ak, bk, blocks, s);
}

} // namespace mfr::gemm
