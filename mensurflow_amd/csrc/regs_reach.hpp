// What the register form of the split GEMM (split_kernel.hpp) can address: its lanes hold an
// M/N-major operand's place in a 16-deep step as 32 bits from the step's first depth line. No HIP
// header, so that the CPU tests check the two functions against each other.
#pragma once

#include <cstdint>

namespace mfr::gemm {

// Floats from a step's first depth line to `row` of the lane half's first depth (8 half lines on),
// `line` floats between depth lines.
constexpr uint32_t step_offset(int64_t line, int half, int row) {
    return static_cast<uint32_t>(8 * half * line + row);
}

// Whether step_offset holds every place of a step whose depth lines are `line` floats apart: it is
// added as an unsigned number, so lines must not run backwards, and byte offsets of less than
// 2^31 keep the load's own address arithmetic within 32 bits.
constexpr int64_t kFarLines = int64_t{1} << 26;
constexpr bool regs_reach(int64_t line) { return line >= 0 && line < kFarLines; }

} // namespace mfr::gemm
