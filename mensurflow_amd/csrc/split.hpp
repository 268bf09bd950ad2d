// Launches of the split tile kernel (split_kernel.hpp), one translation unit per tile shape.
#pragma once

#include "gemm_kernel.hpp"

namespace mfr::gemm {

// p's tile fields are filled for the tile; ak, bk: A and B are read along k.
void launch_split_256x256(const GemmParams& p, bool ak, bool bk, unsigned blocks, hipStream_t s);
void launch_split_128x128(const GemmParams& p, bool ak, bool bk, unsigned blocks, hipStream_t s);
void launch_split_128x64(const GemmParams& p, bool ak, bool bk, unsigned blocks, hipStream_t s);
void launch_split_64x128(const GemmParams& p, bool ak, bool bk, unsigned blocks, hipStream_t s);
// No LDS in the depth loop; M/N-major lines as regs_reach (regs_reach.hpp) allows.
void launch_split_regs_64x64(const GemmParams& p, bool ak, bool bk, unsigned blocks,
                             hipStream_t s);
// Likewise, on 64x64 tiles of which at most 32 rows are inside the matrix.
void launch_split_regs_32x64(const GemmParams& p, bool ak, bool bk, unsigned blocks,
                             hipStream_t s);
void launch_split_64x64(const GemmParams& p, bool ak, bool bk, unsigned blocks, hipStream_t s);

} // namespace mfr::gemm
