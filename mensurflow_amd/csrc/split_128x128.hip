// The split kernel on the 128x128 tile (split_kernel.hpp).
#include "split.hpp"
#include "split_kernel.hpp"

namespace mfr::gemm {

void launch_split_128x128(const GemmParams& p, bool ak, bool bk, unsigned blocks, hipStream_t s) {
    launch_split_tile<128, 128, 32, 2, 4>(p, ak, bk, blocks, s);
}

} // namespace mfr::gemm
