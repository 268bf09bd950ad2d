// The split kernel on the 256x256 tile (split_kernel.hpp).
#include "split.hpp"
#include "split_kernel.hpp"

namespace mfr::gemm {

void launch_split_256x256(const GemmParams& p, bool ak, bool bk, unsigned blocks, hipStream_t s) {
    launch_split_tile<256, 256, 16, 2, 4>(p, ak, bk, blocks, s);
}

} // namespace mfr::gemm
