// The GEMM register form's dispatch rule against its address arithmetic (csrc/regs_reach.hpp):
// for every stride that regs_reach takes, step_offset is the 64-bit place of each lane, and its
// byte offset stays below 2^32.
#include "regs_reach.hpp"

#include <cstdio>
#include <initializer_list>

int main() {
    using namespace mfr::gemm;
    int failed = 0, taken = 0;
    for (const int64_t size : {int64_t{0}, int64_t{1}, int64_t{63}, int64_t{256}, int64_t{4099},
                               int64_t{1} << 20, kFarLines - 1, kFarLines, kFarLines + 1,
                               int64_t{1} << 31, int64_t{1} << 40}) {
        for (const int64_t line : {size, -size}) {
            bool holds = true;
            for (int half = 0; half < 2; ++half) {
                for (int row : {0, 1, 63}) {
                    const int64_t place = 8 * half * line + row;
                    holds = holds && static_cast<int64_t>(step_offset(line, half, row)) == place &&
                            4 * place < (int64_t{1} << 32);
                }
            }
            taken += regs_reach(line);
            if (regs_reach(line) && !holds) {
                std::printf("a stride of %lld is taken but not held\n", static_cast<long long>(line));
                ++failed;
            }
        }
    }
    // The strides of ordinary matrices are taken (0 counts twice above).
    if (taken < 8 || !regs_reach(256) || !regs_reach(kFarLines - 1) || regs_reach(-256)) {
        std::printf("regs_reach takes %d strides\n", taken);
        ++failed;
    }
    if (failed == 0) {
        std::printf("gemm_reach_test passed\n");
    }
    return failed;
}
