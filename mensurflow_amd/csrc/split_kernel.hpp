// The fp32 GEMM tile on the bf16 matrix cores: each fp32 operand element is cut exactly into three
// bf16 parts (8 bits each) and the product is summed from the six part products that reach fp32
// precision (the method of Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", ARITH 2019). The three left out are at
// most 2^-24 of |a b| together and 1.4e-8 of it root mean square, and each 16 depths that hold
// anything but zeros round the sum six times, where the fp32 matrix cores round it once per depth
// and their products not at all. A sum of k products whose nonzero ones lie in s steps of 16 depths
// is so within (2 + 6 s) 2^-24 of sum |a b| of the exact one, against k 2^-24.
//
// On dense operands that is nearer (2-norm error at a depth of 64 / 1024 / 4096: uniform 1.1e-7 /
// 4.6e-7 / 9.2e-7 against 1.5e-7 / 5.8e-7 / 1.03e-6 on the fp32 matrix cores; normal 1.1e-7 / 4.9e-7 /
// 9.8e-7 against 1.4e-7 / 5.8e-7 / 1.1e-6; positive 8.4e-8 / 2.8e-7 / 5.2e-7 against 1.1e-7 / 4.3e-7 /
// 8.9e-7). On sparse or widely scaled rows it is further off: with 1 / 4 / 16 / 32 nonzeros in rows
// of 512 / 512 / 1024 / 4096 3.5e-8 / 5.6e-8 / 9.1e-8 / 1.2e-7 against 2.5e-8 / 4.2e-8 / 5.9e-8 /
// 6.9e-8, half zeros (1024 deep) 2.3e-7 against 2.1e-7, exp(2 N) times normal 2.4e-7 against 2.1e-7.
// Included by the split_*.hip translation units (launches) through split.hpp; see gemm.hip for the
// tiles, regions and splits around it.
#pragma once

#include "regs_reach.hpp"
#include "split_parts.hpp"

namespace mfr::gemm {

// ---- where the part products do not stand for the fp32 products --------------------------------
//
// The parts hold an element exactly from 2^-100 to the largest bf16, and a part product is at
// least 2^-126 for elements from 2^-49. Outside that a tile's sums may be wrong, and they show it:
//   - they are not finite (an infinite or NaN element has NaN parts whatever they meet, one above
//     the largest bf16 an infinite part; or fp32 products would overflow as well), or
//   - they are small next to what can have been lost: at most 2^-126 in each part of an element,
//     times the largest element it meets, and in each of the six part products, over the depth.
//     2^26 times as much would stay under the sums' own rounding.
// A wavefront whose sums are finite and clear of that bound is done (sums_bound: 2^-74 for 4096
// depths of a million normal values).
// Where a few sums are not clear (a sum that happens to be 0), the wavefront reads their rows and
// columns again for their smallest nonzero magnitude; with more of them (padding rows), the
// workgroup reads its operands again. A wavefront runs its blocks on the fp32 matrix cores
// (plain_blocks) where that is under 2^-49 or a sum is not finite. So zeros cost a second read
// only where sums are zero too (1024^3 with zero rows in A 20 -> 31 us, 2048^3 94 -> 121, 4096^3 570 ->
// 680), and a few tiny elements among others (softmax weights) nothing.
// (Keeping the least magnitude beside the squares instead cost 7 % at 4096^3: every operation
// per element cut adds to a loop that is bound by issue and by power.)

constexpr uint32_t kSmallest = (127u - 49u) << 23; // 2^-49
constexpr int kFewLines = 4;

// What a sum of kk products has to reach to be clear: `squares` is the sum of the squares of the
// tile's elements, whose root is at least the largest.
__device__ __forceinline__ float sums_bound(float squares, int64_t kk) {
    return 2.0f * (1.0f + sqrtf(squares)) * static_cast<float>(kk) * 0x1p-97f;
}

enum class Sums { kClear, kUnclear, kNotFinite };

// How the sums of the wavefront's blocks stand.
template <int FM, int FN>
__device__ __forceinline__ Sums judge(const floatx16 (&acc)[FM][FN], float bound) {
    float zero = 0.0f;
    float least = __builtin_inff();
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                zero = fmaf(acc[i][j][e], 0.0f, zero); // NaN once a sum is not finite
                least = fminf(least, __builtin_fabsf(acc[i][j][e]));
            }
        }
    }
    if (!__all(zero == 0.0f)) {
        return Sums::kNotFinite;
    }
    return __all(least >= bound) ? Sums::kClear : Sums::kUnclear;
}

// The smallest nonzero magnitude in a line of kk elements, as float bits - 1 (zero wraps past
// every other value), in every lane.
__device__ __forceinline__ uint32_t smallest_in_line(const float* line, int64_t stride, int64_t kk,
                                                     int lane) {
    uint32_t least = 0xffffffffu;
    for (int64_t k = lane; k < kk; k += 256) {
        // Four loads in flight; past the end the line's first element again.
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            v[u] = line[k + 64 * u < kk ? (k + 64 * u) * stride : 0];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            least = min(least, (__float_as_uint(v[u]) & 0x7fffffffu) - 1);
        }
    }
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) {
        least = min(least, static_cast<uint32_t>(__shfl_xor(static_cast<int>(least), m, 64)));
    }
    return least;
}

// Whether the operands of a wavefront's unclear sums (not at least `bound`, which is infinite or NaN
// where an element of the tile is) hold an element under 2^-49: 1 or 0, or -1 when more than kFewLines rows or columns are concerned. a, b: element (row 0,
// depth 0) of the wavefront's blocks; rows and columns past the matrix repeat the last.
template <int FM, int FN>
__device__ __forceinline__ int few_underflow(const floatx16 (&acc)[FM][FN], float bound,
                                             const float* a, int64_t a_rs, int64_t a_cs, int rows,
                                             const float* b, int64_t b_cs, int64_t b_rs, int cols,
                                             int64_t kk, int lane) {
    uint32_t col_mask[FN];
    uint32_t row_mask[FM];
    int lines = 0;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        bool low = false;
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                low = low || !(__builtin_fabsf(acc[i][j][e]) >= bound);
            }
        }
        const uint64_t lanes = __ballot(low);
        col_mask[j] = static_cast<uint32_t>(lanes) | static_cast<uint32_t>(lanes >> 32);
        lines += __popc(col_mask[j]);
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        row_mask[i] = 0;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            bool low = false;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                low = low || !(__builtin_fabsf(acc[i][j][e]) >= bound);
            }
            const uint64_t lanes = __ballot(low);
            const int row = 8 * (e / 4) + e % 4;
            row_mask[i] |= (static_cast<uint32_t>(lanes) != 0 ? 1u : 0u) << row;
            row_mask[i] |= (static_cast<uint32_t>(lanes >> 32) != 0 ? 1u : 0u) << (row + 4);
        }
        lines += __popc(row_mask[i]);
    }
    if (lines > 2 * kFewLines) {
        return -1;
    }
    uint32_t least = 0xffffffffu;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        for (uint32_t m = row_mask[i]; m != 0; m &= m - 1) {
            const int row = min(32 * i + __ffs(static_cast<int>(m)) - 1, rows - 1);
            least = min(least, smallest_in_line(a + row * a_rs, a_cs, kk, lane));
        }
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        for (uint32_t m = col_mask[j]; m != 0; m &= m - 1) {
            const int col = min(32 * j + __ffs(static_cast<int>(m)) - 1, cols - 1);
            least = min(least, smallest_in_line(b + col * b_cs, b_rs, kk, lane));
        }
    }
    return least < kSmallest - 1 ? 1 : 0;
}

typedef float native4 __attribute__((ext_vector_type(4)));

// One operand's depth slice: ROWS rows (M for A, N for B) by KT depths, taken from memory to
// registers in units of 8 depths of one row, cut there and written to LDS as three bf16 planes
// [plane][depth / 8][row][8], so an MFMA fragment (8 depths of a row per lane, 32 rows per half
// wavefront) is one 16-byte LDS read from consecutive addresses.
//
// KMAJ: a unit is two 16-byte loads (4-byte aligned suffices); consecutive threads take a row's
// units, so a wave-instruction reads whole runs of KT floats, and the padded pitch of a plane's
// depth group keeps their LDS writes off each other's banks. Otherwise: a unit is eight 4-byte
// loads, one per depth line, the threads of a wavefront along the line.
template <int ROWS, int KT, bool KMAJ, int THREADS> struct SplitLoader {
    static constexpr int kGroups = KT / 8;
    static constexpr int kUnits = ROWS * kGroups;
    static constexpr int kPerThread = kUnits / THREADS;
    static_assert(kUnits % THREADS == 0, "every thread takes the same number of units");
    static_assert(ROWS % 64 == 0, "a wavefront's units lie in one depth group");
    static constexpr int kPad = KMAJ ? 8 / kGroups : 0;
    static constexpr int kPitch = ROWS + kPad;             // 16-byte pieces per depth group
    static constexpr int kPieces = 3 * kGroups * kPitch;   // per slice

    float reg[kPerThread][8];
    const float* at[KMAJ ? kPerThread : 1]; // K-major: this thread's unit in the next slice
    const float* line;                      // M/N-major: the next slice's first depth line
    int64_t stride;                         // M/N-major: floats between depth lines
    uint32_t row_of[KMAJ ? 1 : kPerThread];

    __device__ __forceinline__ static int unit_row(int i) {
        const int u = static_cast<int>(threadIdx.x) + i * THREADS;
        return KMAJ ? u / kGroups : u % ROWS;
    }

    __device__ __forceinline__ static int unit_group(int i) {
        const int u = static_cast<int>(threadIdx.x) + i * THREADS;
        return KMAJ ? u % kGroups : __builtin_amdgcn_readfirstlane(u / ROWS);
    }

    // base: element (row 0, depth 0) of the tile's first slice. Rows past the matrix repeat its
    // last row (their sums are never stored).
    __device__ __forceinline__ SplitLoader(const float* base, int64_t row_stride, int64_t k_stride,
                                           int rows_inside) {
        line = base;
        stride = k_stride;
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            const int row = unit_row(i) < rows_inside ? unit_row(i) : rows_inside - 1;
            if constexpr (KMAJ) {
                at[i] = base + row * row_stride + 8 * unit_group(i);
            } else {
                row_of[i] = static_cast<uint32_t>(row);
            }
        }
    }

    // Loads the next slice's units: a whole slice, or one of which k_left depths exist.
    template <bool WHOLE> __device__ __forceinline__ void load(int64_t k_left) {
        if constexpr (WHOLE) {
#pragma unroll
            for (int i = 0; i < kPerThread; ++i) {
                if constexpr (KMAJ) {
                    typedef native4 __attribute__((aligned(4))) loose4;
                    const native4 lo = *reinterpret_cast<const loose4*>(at[i]);
                    const native4 hi = *reinterpret_cast<const loose4*>(at[i] + 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        reg[i][e] = lo[e];
                        reg[i][4 + e] = hi[e];
                    }
                } else {
                    const float* l = line + 8 * unit_group(i) * stride;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        reg[i][e] = l[row_of[i]];
                        l += stride;
                    }
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < kPerThread; ++i) {
                const int k0 = 8 * unit_group(i);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    reg[i][e] = 0.0f;
                    if (k0 + e < k_left) {
                        reg[i][e] = KMAJ ? at[KMAJ ? i : 0][e]
                                         : line[(k0 + e) * stride + row_of[KMAJ ? 0 : i]];
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < (KMAJ ? kPerThread : 0); ++i) {
            at[i] += KT;
        }
        line += KMAJ ? 0 : KT * stride;
    }

    // Cuts the loaded units into the planes.
    __device__ __forceinline__ void cut_and_store(uint4* planes, float& squares) const {
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            uint32_t part[3][4];
            cut_eight(reg[i], part, squares);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                planes[(q * kGroups + unit_group(i)) * kPitch + unit_row(i)] =
                    make_uint4(part[q][0], part[q][1], part[q][2], part[q][3]);
            }
        }
    }

    // The smallest nonzero magnitude in the loaded units, as bits - 1 (zero wraps past all).
    __device__ __forceinline__ uint32_t smallest() const {
        uint32_t least = 0xffffffffu;
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                least = min(least, (__float_as_uint(reg[i][e]) & 0x7fffffffu) - 1);
            }
        }
        return least;
    }

    // The fragment of row `row` (the lane's) for 16-deep step `step` of a slice, part `q`.
    __device__ __forceinline__ static bf16x8 fragment(const uint4* planes, int q, int step,
                                                      int half, int row) {
        return __builtin_bit_cast(bf16x8,
                                  planes[(q * kGroups + 2 * step + half) * kPitch + row]);
    }
};

// Eight depths of a row, from `at` on.
template <bool KMAJ>
__device__ __forceinline__ void load_eight(float (&v)[8], const float* at, int64_t stride) {
    if constexpr (KMAJ) {
        typedef native4 __attribute__((aligned(4))) loose4;
        const native4 lo = *reinterpret_cast<const loose4*>(at);
        const native4 hi = *reinterpret_cast<const loose4*>(at + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = lo[e];
            v[4 + e] = hi[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = *at;
            at += stride;
        }
    }
}

// The wavefront's blocks on the fp32 matrix cores, straight from global memory: what a tile runs
// again where the part products do not stand for its products. Rows past the matrix repeat
// its last row. Lanes 0-31 take eight depths of their rows at a time, lanes 32-63 the next eight
// (2048^3 with one infinite element 570 -> 247 us against one depth each, 1024^3 121 -> 56); not
// for the 256x256 tile's 8 blocks, where the compiler then orders the main loop's loads and cuts
// another way (4096^3 608 -> 622 us, the MLP 188 -> 197).
template <int FM, int FN, bool AK, bool BK>
__device__ __forceinline__ void plain_blocks(floatx16 (&acc)[FM][FN], const float* a_base,
                                             const float* b_base, const GemmParams& p, int64_t kk,
                                             int rows_a, int rows_b, int row0, int col0, int half,
                                             int r32) {
    const float* pa[FM];
    const float* pb[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int row = row0 + 32 * i + r32 < rows_a ? row0 + 32 * i + r32 : rows_a - 1;
        pa[i] = a_base + row * p.a_rs;
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int col = col0 + 32 * j + r32 < rows_b ? col0 + 32 * j + r32 : rows_b - 1;
        pb[j] = b_base + col * p.b_cs;
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] = 0.0f;
            }
        }
    }
    int64_t k = 0;
    if constexpr (FM * FN <= 2) {
#pragma unroll 1
        for (; k + 16 <= kk; k += 16) {
            const int64_t d = k + 8 * half;
            float fa[FM][8], fb[FN][8];
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                load_eight<AK>(fa[i], pa[i] + d * p.a_cs, p.a_cs);
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                load_eight<BK>(fb[j], pb[j] + d * p.b_rs, p.b_rs);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
#pragma unroll
                for (int i = 0; i < FM; ++i) {
#pragma unroll
                    for (int j = 0; j < FN; ++j) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][e], fb[j][e],
                                                                         acc[i][j], 0, 0, 0);
                    }
                }
            }
        }
    }
#pragma unroll 1
    for (; k < kk; k += 2) {
        const int64_t d = k + half;
        const bool inside = d < kk;
        float fa[FM], fb[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            fa[i] = inside ? pa[i][d * p.a_cs] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            fb[j] = inside ? pb[j][d * p.b_rs] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
            }
        }
    }
}

// The tile through LDS. Bound at 4096^3 (256x256 tiles, one per CU) by the matrix cores' power:
// they are busy 71 % of the cycles at 1.84 GHz; 555-607 us by box and clock, 226-247 TFLOP/s of
// fp32 product, 1.36-1.48 PFLOP/s of bf16, against 961 us on the fp32 matrix cores. Smaller tiles
// are bound by LDS reads (three planes of each fragment) and by the cuts, 11 vector operations a
// pair of elements, which a tile of B rows and columns spreads over B products each.
//   - 256x256: 8 wavefronts of 128x64 (2 per SIMD), 16-deep slices: 48 KiB a buffer. With 64x64
//     wavefronts LDS reads would take a third more.
//   - 128x128: 8 wavefronts of 64x32 on 32-deep slices (2048^3 89 us; 4 wavefronts of 64x64, one
//     per SIMD, 2048 x 2048 x 1024 58 against 46 us).
//   - the others: 4 wavefronts, 32-deep slices, 2 or 3 workgroups per CU.
// Cutting as the slice passes through registers costs each element once per tile; cutting it per
// wavefront after LDS would cost four times that.
// Two slices in flight in registers instead of one (2048^3 92 against 92 us), an explicit
// MFMA / vector operation interleave (4096^3 578-591 against 574 us) and subtracting the parts
// with the two-product dot instruction (four operations fewer a pair; 595 against 563 us) were no
// faster.
template <int BM, int BN, int KT, int WAVES_M, int WAVES_N, bool AK, bool BK>
__global__ __launch_bounds__(WAVES_M * WAVES_N * 64) void sgemm_split_kernel(GemmParams p) {
    constexpr int THREADS = WAVES_M * WAVES_N * 64;
    constexpr int WM = BM / WAVES_M;
    constexpr int WN = BN / WAVES_N;
    constexpr int FM = WM / 32;
    constexpr int FN = WN / 32;
    static_assert(KT % 16 == 0 && WM % 32 == 0 && WN % 32 == 0, "tile shape");
    using LoadA = SplitLoader<BM, KT, AK, THREADS>;
    using LoadB = SplitLoader<BN, KT, BK, THREADS>;
    // One LDS object per buffer, so the compiler sees that the writes of the next slice and the
    // reads of this one do not meet.
    __shared__ uint4 tile_a0[LoadA::kPieces];
    __shared__ uint4 tile_a1[LoadA::kPieces];
    __shared__ uint4 tile_b0[LoadB::kPieces];
    __shared__ uint4 tile_b1[LoadB::kPieces];
    // The tanh gelu's exp table, and what the end of the tile exchanges.
    __shared__ double gelu_table[64];
    __shared__ float squares_of[WAVES_M * WAVES_N];
    __shared__ uint32_t unclear, smallest;
    if (p.act == MFR_ACT_GELU_TANH && threadIdx.x < 64) {
        gelu_table[threadIdx.x] = gelu_math::kExp2Table[threadIdx.x];
    }

    if (threadIdx.x == 0) {
        unclear = 0;
        smallest = 0xffffffffu;
    }

    const TileWork w = tile_work<BM, BN>(p);
    const float* a_base = p.a + w.off_a + w.m0 * p.a_rs + w.k_begin * p.a_cs;
    const float* b_base = p.b + w.off_b + w.n0 * p.b_cs + w.k_begin * p.b_rs;
    const int lane = threadIdx.x % 64;
    const int wave = threadIdx.x / 64;
    const int wave_m = wave / WAVES_N;
    const int wave_n = wave % WAVES_N;
    const int half = lane / 32;
    const int r32 = lane % 32;

    floatx16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] = 0.0f;
            }
        }
    }

    LoadA la(a_base, p.a_rs, p.a_cs, w.rows_a);
    LoadB lb(b_base, p.b_cs, p.b_rs, w.rows_b);
    float squares = 0.0f;
    const int64_t kk = w.kk;
    const int64_t slices = kk > 0 ? (kk + KT - 1) / KT : 0;

    const auto load = [&](int64_t s) __attribute__((always_inline)) {
        const int64_t k_left = kk - s * KT;
        if (k_left >= KT) {
            la.template load<true>(k_left);
            lb.template load<true>(k_left);
        } else if (k_left > 0) {
            la.template load<false>(k_left);
            lb.template load<false>(k_left);
        }
    };
    // Slice s: its MFMAs from (sa, sb), with slice s + 1 (loaded a slice ago) cut into (na, nb) and
    // slice s + 2 loaded (whole: it is a whole one).
    const auto slice = [&](auto whole, int64_t s, const uint4* sa, const uint4* sb, uint4* na,
                           uint4* nb) __attribute__((always_inline)) {
        la.cut_and_store(na, squares);
        lb.cut_and_store(nb, squares);
        if constexpr (decltype(whole)::value) {
            la.template load<true>(KT);
            lb.template load<true>(KT);
        } else {
            load(s + 2);
        }
#pragma unroll
        for (int step = 0; step < KT / 16; ++step) {
            bf16x8 fb[FN][3];
#pragma unroll
            for (int j = 0; j < FN; ++j) {
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    fb[j][q] = LoadB::fragment(sb, q, step, half, wave_n * WN + 32 * j + r32);
                }
            }
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                bf16x8 fa[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    fa[q] = LoadA::fragment(sa, q, step, half, wave_m * WM + 32 * i + r32);
                }
#pragma unroll
                for (int t = 0; t < 6; ++t) {
#pragma unroll
                    for (int j = 0; j < FN; ++j) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            fa[kPartA[t]], fb[j][kPartB[t]], acc[i][j], 0, 0, 0);
                    }
                }
            }
        }
        lds_barrier();
    };
    if (slices == 0) {
        lds_barrier(); // no depth, so no other: the gelu table is written
    }
    if (slices > 0) {
        load(0);
        la.cut_and_store(tile_a0, squares);
        lb.cut_and_store(tile_b0, squares);
        load(1);
        lds_barrier();
    }
    int64_t s = 0;
    for (; (s + 4) * KT <= kk; s += 2) {
        slice(std::true_type{}, s, tile_a0, tile_b0, tile_a1, tile_b1);
        slice(std::true_type{}, s + 1, tile_a1, tile_b1, tile_a0, tile_b0);
    }
    for (; s < slices; s += 2) {
        slice(std::false_type{}, s, tile_a0, tile_b0, tile_a1, tile_b1);
        if (s + 1 < slices) {
            slice(std::false_type{}, s + 1, tile_a1, tile_b1, tile_a0, tile_b0);
        }
    }
    if (slices > 0) {
        constexpr int kWaves = WAVES_M * WAVES_N;
        squares = mfr::dev::butterfly_sum(squares);
        if (lane == 0) {
            squares_of[wave] = squares;
        }
        lds_barrier();
        float all_squares = 0.0f;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
            all_squares += squares_of[i];
        }
        const float bound = sums_bound(all_squares, kk);
        const Sums stand = judge(acc, bound);
        int under = 0;
        if (stand == Sums::kUnclear) {
            under = few_underflow(acc, bound, a_base + wave_m * WM * p.a_rs, p.a_rs, p.a_cs,
                                  w.rows_a - wave_m * WM, b_base + wave_n * WN * p.b_cs, p.b_cs,
                                  p.b_rs, w.rows_b - wave_n * WN, kk, lane);
            if (under < 0 && lane == 0) {
                unclear = 1;
            }
        }
        lds_barrier();
        if (__builtin_amdgcn_readfirstlane(unclear) != 0) {
            LoadA ra(a_base, p.a_rs, p.a_cs, w.rows_a);
            LoadB rb(b_base, p.b_cs, p.b_rs, w.rows_b);
            uint32_t found = 0xffffffffu;
            int64_t k_left = kk;
            for (; k_left >= KT; k_left -= KT) {
                ra.template load<true>(k_left);
                rb.template load<true>(k_left);
                found = min(found, min(ra.smallest(), rb.smallest()));
            }
            if (k_left > 0) {
                ra.template load<false>(k_left);
                rb.template load<false>(k_left);
                found = min(found, min(ra.smallest(), rb.smallest()));
            }
            atomicMin(&smallest, found);
            lds_barrier();
            if (under < 0) {
                under = smallest < kSmallest - 1 ? 1 : 0;
            }
        }
        if (__builtin_amdgcn_readfirstlane(stand == Sums::kNotFinite || under > 0) != 0) {
            plain_blocks<FM, FN, AK, BK>(acc, a_base, b_base, p, kk, w.rows_a, w.rows_b,
                                         wave_m * WM, wave_n * WN, half, r32);
        }
    }
    finish_tile<BM, BN, WM, WN, FM, FN>(acc, p, w, wave_m, wave_n, half, r32, gelu_table);
}

// ---- the register form ------------------------------------------------------------------------

// One operand's share of a 16-deep step for a wavefront of the register form: F blocks of 32 rows,
// lane l the 8 depths 8 (l / 32) .. of row l % 32 of each, which are its MFMA fragments.
template <int F, bool KMAJ, int SETS = 1> struct StepLoader {
    float reg[SETS][F][8]; // a step in flight each
    const float* at[KMAJ ? F : 1]; // K-major: this lane's depths in the wavefront's next step
    const float* line;             // M/N-major: the next step's first depth line
    int64_t stride;
    uint32_t offset[KMAJ ? 1 : F]; // M/N-major: this lane's float within the step (32 bits)

    // base: element (row 0 of the wavefront's blocks, depth 0) of the tile's depth range;
    // rows_inside: rows from there inside the matrix (rows past them repeat the last one, or row
    // 0 of a wavefront wholly outside, which lies inside through `base`).
    __device__ __forceinline__ StepLoader(const float* base, int64_t row_stride, int64_t k_stride,
                                          int rows_inside, int first_step, int half, int r32) {
        line = base + 16 * first_step * k_stride;
        stride = k_stride;
#pragma unroll
        for (int f = 0; f < F; ++f) {
            const int row = 32 * f + r32 < rows_inside ? 32 * f + r32 : rows_inside - 1;
            if constexpr (KMAJ) {
                at[f] = base + row * row_stride + 16 * first_step + 8 * half;
            } else {
                offset[f] = step_offset(k_stride, half, row);
            }
        }
    }

    // Loads a step (whole, or k_left depths of it) and moves on by `steps` steps.
    template <bool WHOLE> __device__ __forceinline__ void load(int set, int64_t k_left,
                                                               int steps, int half) {
#pragma unroll
        for (int f = 0; f < F; ++f) {
            if constexpr (WHOLE && KMAJ) {
                typedef native4 __attribute__((aligned(4))) loose4;
                const native4 lo = *reinterpret_cast<const loose4*>(at[f]);
                const native4 hi = *reinterpret_cast<const loose4*>(at[f] + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    reg[set][f][e] = lo[e];
                    reg[set][f][4 + e] = hi[e];
                }
            } else if constexpr (WHOLE) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    reg[set][f][e] = (line + e * stride)[offset[f]];
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    reg[set][f][e] = 0.0f;
                    if (8 * half + e < k_left) {
                        reg[set][f][e] = KMAJ ? at[KMAJ ? f : 0][e]
                                         : (line + e * stride)[offset[KMAJ ? 0 : f]];
                    }
                }
            }
        }
#pragma unroll
        for (int f = 0; f < (KMAJ ? F : 0); ++f) {
            at[f] += 16 * steps;
        }
        line += KMAJ ? 0 : 16 * steps * stride;
    }

    __device__ __forceinline__ void cut(int set, bf16x8 (&part)[F][3],
                                        float& squares) const {
#pragma unroll
        for (int f = 0; f < F; ++f) {
            uint32_t words[3][4];
            cut_eight(reg[set][f], words, squares);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                part[f][q] = __builtin_bit_cast(
                    bf16x8, make_uint4(words[q][0], words[q][1], words[q][2], words[q][3]));
            }
        }
    }

    __device__ __forceinline__ uint32_t smallest() const {
        uint32_t least = 0xffffffffu;
#pragma unroll
        for (int f = 0; f < F; ++f) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                least = min(least, (__float_as_uint(reg[0][f][e]) & 0x7fffffffu) - 1);
            }
        }
        return least;
    }
};

// The tile with no LDS in its depth loop: WAVES_K sets of one wavefront take every WAVES_K-th
// 16-deep step of the whole BM x BN tile, its operands straight from memory to registers in the
// fragments' own layout and cut there. The sets' sums are then added through LDS in set order, the
// first BM BN / 1024 sets finishing one 32x32 block each.
//
// The same cuts and MFMAs as the LDS form, but no barrier holds the wavefronts in step and every
// MFMA has independent ones beside it, which counts where a CU has one workgroup: 1024^3 24.8 ->
// 20.7 us. With several workgroups per CU the LDS form is faster (2048 x 2048 x 1024: 58.8 us
// against 67 with 4 sets and 76 with 8). SETS steps are in flight in registers: 1 for 64x64, 2 for
// 32x64 (the first 32 rows of a 64x64 tile: a few rows against a large matrix, 32 x 4096 x 4096
// 25.3 -> 22.6 us). 32-deep steps (a whole 128-byte line of a K-major row each) took 1024^3 from
// 19.7 to 25.3 us, and 32x32 tiles of 16 sets over the whole depth, which need no reduce, 35.8 us
// at 32 x 4096 x 4096.
template <int BM, int BN, int WAVES_K, int SETS, bool AK, bool BK>
__global__ __launch_bounds__(WAVES_K * 64) void sgemm_split_regs_kernel(GemmParams p) {
    constexpr int FM = BM / 32, FN = BN / 32;
    constexpr int kBlocks = FM * FN;
    static_assert(kBlocks <= WAVES_K && WAVES_K * kBlocks <= 32, "a block a set; 128 KiB of LDS");
    __shared__ float sums[WAVES_K][kBlocks][16][64];
    __shared__ double gelu_table[64];
    __shared__ float squares_of[WAVES_K];
    __shared__ uint32_t unclear, smallest;
    if (p.act == MFR_ACT_GELU_TANH && threadIdx.x < 64) {
        gelu_table[threadIdx.x] = gelu_math::kExp2Table[threadIdx.x];
    }
    if (threadIdx.x == 0) {
        unclear = 0;
        smallest = 0xffffffffu;
    }

    const TileWork w = tile_work<BM, BN>(p);
    const float* a_base = p.a + w.off_a + w.m0 * p.a_rs + w.k_begin * p.a_cs;
    const float* b_base = p.b + w.off_b + w.n0 * p.b_cs + w.k_begin * p.b_rs;
    const int lane = threadIdx.x % 64;
    const int set = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));
    const int half = lane / 32;
    const int r32 = lane % 32;
    const int64_t kk = w.kk;
    const int64_t steps = kk > 0 ? (kk + 15) / 16 : 0;

    floatx16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] = 0.0f;
            }
        }
    }
    float squares = 0.0f;
    {
        StepLoader<FM, AK, SETS> la(a_base, p.a_rs, p.a_cs, w.rows_a, set, half, r32);
        StepLoader<FN, BK, SETS> lb(b_base, p.b_cs, p.b_rs, w.rows_b, set, half, r32);
        const auto load = [&](int into, int64_t t) __attribute__((always_inline)) {
            const int64_t k_left = kk - 16 * t;
            if (k_left >= 16) {
                la.template load<true>(into, k_left, WAVES_K, half);
                lb.template load<true>(into, k_left, WAVES_K, half);
            } else if (k_left > 0) {
                la.template load<false>(into, k_left, WAVES_K, half);
                lb.template load<false>(into, k_left, WAVES_K, half);
            }
        };
        // Step t, loaded into register set `from`, which then takes step t + SETS WAVES_K.
        const auto step = [&](auto whole, int from, int64_t t) __attribute__((always_inline)) {
            bf16x8 fa[FM][3], fb[FN][3];
            la.cut(from, fa, squares);
            lb.cut(from, fb, squares);
            if constexpr (decltype(whole)::value) {
                la.template load<true>(from, 16, WAVES_K, half);
                lb.template load<true>(from, 16, WAVES_K, half);
            } else {
                load(from, t + SETS * WAVES_K);
            }
#pragma unroll
            for (int q = 0; q < 6; ++q) {
#pragma unroll
                for (int i = 0; i < FM; ++i) {
#pragma unroll
                    for (int j = 0; j < FN; ++j) {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            fa[i][kPartA[q]], fb[j][kPartB[q]], acc[i][j], 0, 0, 0);
                    }
                }
            }
        };
        int64_t t = set;
#pragma unroll
        for (int i = 0; i < SETS; ++i) {
            load(i, t + i * WAVES_K);
        }
        for (; 16 * (t + (2 * SETS - 1) * WAVES_K + 1) <= kk; t += SETS * WAVES_K) {
#pragma unroll
            for (int i = 0; i < SETS; ++i) {
                step(std::true_type{}, i, t + i * WAVES_K);
            }
        }
        for (; t < steps; t += SETS * WAVES_K) {
#pragma unroll
            for (int i = 0; i < SETS; ++i) {
                if (t + i * WAVES_K < steps) {
                    step(std::false_type{}, i, t + i * WAVES_K);
                }
            }
        }
    }
    squares = mfr::dev::butterfly_sum(squares);
    if (lane == 0) {
        squares_of[set] = squares;
    }
    // Every set parks its blocks; set b adds block b over the sets, in set order.
#pragma unroll
    for (int b = 0; b < kBlocks; ++b) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            sums[set][b][e][lane] = acc[b / FN][b % FN][e];
        }
    }
    lds_barrier();
    const bool has = set < kBlocks;
    const int row0 = 32 * (set / FN);
    const int col0 = 32 * (set % FN);
    floatx16 mine[1][1];
    float all_squares = 0.0f;
    if (has) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            float v = sums[0][set][e][lane];
#pragma unroll
            for (int k = 1; k < WAVES_K; ++k) {
                v += sums[k][set][e][lane];
            }
            mine[0][0][e] = v;
        }
    }
#pragma unroll
    for (int i = 0; i < WAVES_K; ++i) {
        all_squares += squares_of[i];
    }
    const float bound = sums_bound(all_squares, kk);
    Sums stand = Sums::kClear;
    int under = 0;
    if (has && steps > 0) {
        stand = judge(mine, bound);
        if (stand == Sums::kUnclear) {
            under = few_underflow(mine, bound, a_base + row0 * p.a_rs, p.a_rs, p.a_cs,
                                  w.rows_a - row0, b_base + col0 * p.b_cs, p.b_cs, p.b_rs,
                                  w.rows_b - col0, kk, lane);
            if (under < 0 && lane == 0) {
                unclear = 1;
            }
        }
    }
    lds_barrier();
    if (__builtin_amdgcn_readfirstlane(unclear) != 0) {
        StepLoader<FM, AK> ra(a_base, p.a_rs, p.a_cs, w.rows_a, set, half, r32);
        StepLoader<FN, BK> rb(b_base, p.b_cs, p.b_rs, w.rows_b, set, half, r32);
        uint32_t found = 0xffffffffu;
        int64_t k_left = kk - 16 * set;
#pragma unroll 4
        for (; k_left >= 16; k_left -= 16 * WAVES_K) { // several steps' loads in flight
            ra.template load<true>(0, k_left, WAVES_K, half);
            rb.template load<true>(0, k_left, WAVES_K, half);
            found = min(found, min(ra.smallest(), rb.smallest()));
        }
        if (k_left > 0) {
            ra.template load<false>(0, k_left, WAVES_K, half);
            rb.template load<false>(0, k_left, WAVES_K, half);
            found = min(found, min(ra.smallest(), rb.smallest()));
        }
        atomicMin(&smallest, found);
        lds_barrier();
        if (under < 0) {
            under = smallest < kSmallest - 1 ? 1 : 0;
        }
    }
    if (!has) {
        return;
    }
    if (__builtin_amdgcn_readfirstlane(stand == Sums::kNotFinite || under > 0) != 0) {
        plain_blocks<1, 1, AK, BK>(mine, a_base, b_base, p, kk, w.rows_a, w.rows_b, row0, col0,
                                   half, r32);
    }
    finish_tile<BM, BN, 32, 32, 1, 1>(mine, p, w, set / FN, set % FN, half, r32, gelu_table);
}

template <int BM, int BN, int KT, int WAVES_M, int WAVES_N>
void launch_split_tile(const GemmParams& p, bool ak, bool bk, unsigned blocks,
                       hipStream_t stream) {
    constexpr unsigned threads = WAVES_M * WAVES_N * 64;
    if (ak && bk) {
        sgemm_split_kernel<BM, BN, KT, WAVES_M, WAVES_N, true, true>
            <<<blocks, threads, 0, stream>>>(p);
    } else if (ak) {
        sgemm_split_kernel<BM, BN, KT, WAVES_M, WAVES_N, true, false>
            <<<blocks, threads, 0, stream>>>(p);
    } else if (bk) {
        sgemm_split_kernel<BM, BN, KT, WAVES_M, WAVES_N, false, true>
            <<<blocks, threads, 0, stream>>>(p);
    } else {
        sgemm_split_kernel<BM, BN, KT, WAVES_M, WAVES_N, false, false>
            <<<blocks, threads, 0, stream>>>(p);
    }
}

template <int BM, int BN, int WAVES_K, int SETS>
void launch_split_regs_tile(const GemmParams& p, bool ak, bool bk, unsigned blocks,
                            hipStream_t stream) {
    constexpr unsigned threads = WAVES_K * 64;
    if (ak && bk) {
        sgemm_split_regs_kernel<BM, BN, WAVES_K, SETS, true, true><<<blocks, threads, 0, stream>>>(p);
    } else if (ak) {
        sgemm_split_regs_kernel<BM, BN, WAVES_K, SETS, true, false><<<blocks, threads, 0, stream>>>(p);
    } else if (bk) {
        sgemm_split_regs_kernel<BM, BN, WAVES_K, SETS, false, true><<<blocks, threads, 0, stream>>>(p);
    } else {
        sgemm_split_regs_kernel<BM, BN, WAVES_K, SETS, false, false><<<blocks, threads, 0, stream>>>(p);
    }
}

} // namespace mfr::gemm
