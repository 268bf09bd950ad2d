// The split kernel's register form on the 64x64 tile (split_kernel.hpp).
#include "split.hpp"
#include "split_kernel.hpp"

namespace mfr::gemm {

void launch_split_regs_64x64(const GemmParams& p, bool ak, bool bk, unsigned blocks,
                             hipStream_t s) {
    launch_split_regs_tile<64, 64, 8, 1>(p, ak, bk, blocks, s);
}

void launch_split_regs_32x64(const GemmParams& p, bool ak, bool bk, unsigned blocks,
                             hipStream_t s) {
    launch_split_regs_tile<32, 64, 8, 2>(p, ak, bk, blocks, s);
}

} // namespace mfr::gemm
