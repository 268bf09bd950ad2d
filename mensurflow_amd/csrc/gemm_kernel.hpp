// Device code of the GEMM: the parameters, the output tile's place and write-out that every tile
// kernel shares, and the fp32 MFMA tile kernel of short depths with its operand loader. See
// gemm.hip for the design.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace mfr::gemm {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// Word 3 of a raw buffer resource on gfx9 (32-bit dword format, no swizzle): the buffer unit
// checks each access against the resource's size in bytes, returning zeros for loads past it and
// dropping stores past it.
constexpr int kBufferWord3 = 0x00020000;

struct GemmParams {
    const float* a;
    const float* b;
    float* c;
    const float* c0;
    const float* bias;
    int64_t m, n, k;
    int64_t a_rs, a_cs, b_rs, b_cs, c_rs, c0_rs;
    int64_t batch[MFR_MAX_BATCH_DIMS];
    int64_t a_bs[MFR_MAX_BATCH_DIMS], b_bs[MFR_MAX_BATCH_DIMS];
    int64_t c_bs[MFR_MAX_BATCH_DIMS], c0_bs[MFR_MAX_BATCH_DIMS];
    int32_t batch_dims;
    int32_t act;
    int64_t batch_count;
    int32_t tiles_m, tiles_n;
    int32_t group_m;
    float alpha, beta;
    // Split-K: the depth is cut into `splits` ranges of k_per_split (a multiple of the depth
    // slice; the last may be shorter). With splits > 1 each workgroup writes its raw fp32 sums to
    // partial[split][batch][m][n] (dense, batch in linear order) instead of running the
    // epilogue; split_reduce_kernel then adds the splits and applies it.
    int64_t k_per_split;
    int32_t splits;
    float* partial;
    // Nonzero: C is written with non-temporal (streaming) stores on interior tiles without C0 or
    // an activation. Set for outputs larger than the last-level cache whose rows all start on
    // 128-byte lines (partial lines would be merged in L2 otherwise).
    int32_t stream_c;
    // Nonzero: C(i, j) = -inf for j > i in every batch matrix (MFR_GEMM_CAUSAL; panel path only).
    int32_t causal;
};

// Global -> register -> LDS copy of one operand slice: ROWS rows (M for A, N for B) by KT depth.
// KMAJ: unit stride along the depth (element (r, p) at base + r*row_stride + p).
// otherwise: unit stride along the rows (element (r, p) at base + p*k_stride + r).
// V: 4 = 16-byte loads along the unit-stride dimension (its extent and the other stride are
// multiples of 4, the base 16-byte aligned), 1 = 4-byte loads.
template <int ROWS, int KT, bool KMAJ, int V, int THREADS> struct SliceLoader {
    static constexpr int kUnits = ROWS * KT / V;        // loads per slice
    static constexpr int kPerThread = kUnits / THREADS;
    static_assert(kUnits % THREADS == 0, "slice must split evenly over the workgroup");
    // LDS row pitch: [ROWS][KT+4] (K-major) or [KT][ROWS+8].
    static constexpr int kPitch = KMAJ ? KT + 4 : ROWS + 8;
    static constexpr int kFloats = KMAJ ? ROWS * (KT + 4) : KT * (ROWS + 8);

    using Vec = typename std::conditional<V == 4, float4, float>::type;
    Vec reg[kPerThread];

    // (row, depth) of this thread's i-th load, in elements.
    __device__ __forceinline__ static void coords(int i, int& r, int& p) {
        const int u = static_cast<int>(threadIdx.x) + i * THREADS;
        if constexpr (KMAJ) {
            constexpr int per_row = KT / V;
            r = u / per_row;
            p = (u % per_row) * V;
        } else {
            constexpr int per_depth = ROWS / V;
            p = u / per_depth;
            r = (u % per_depth) * V;
        }
    }

    // base points at element (row 0, depth k0) of the slice. rows_left / k_left: how many rows
    // and depths of the slice are inside the matrix (>= ROWS / KT for an interior slice).
    __device__ __forceinline__ void load(const float* base, int64_t row_stride, int64_t k_stride,
                                         int rows_left, int k_left) {
        const bool full = rows_left >= ROWS && k_left >= KT;
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            int r, p;
            coords(i, r, p);
            const float* src = KMAJ ? base + r * row_stride + p : base + p * k_stride + r;
            if (full || (r < rows_left && p < k_left)) {
                if constexpr (V == 4) {
                    reg[i] = *reinterpret_cast<const float4*>(src);
                } else {
                    reg[i] = *src;
                }
            } else {
                if constexpr (V == 4) {
                    reg[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                } else {
                    reg[i] = 0.f;
                }
            }
        }
    }

    __device__ __forceinline__ void store(float* lds) const {
#pragma unroll
        for (int i = 0; i < kPerThread; ++i) {
            int r, p;
            coords(i, r, p);
            float* dst = KMAJ ? lds + r * kPitch + p : lds + p * kPitch + r;
            if constexpr (V == 4) {
                *reinterpret_cast<float4*>(dst) = reg[i];
            } else {
                *dst = reg[i];
            }
        }
    }

    // The four MFMA-step values of fragment row `row` (0..ROWS-1) for depth group g (8 depths):
    // lanes 0-31 (half 0) take depths 8g+0..3, lanes 32-63 (half 1) depths 8g+4..7.
    __device__ __forceinline__ static void fragment(const float* lds, int row, int g, int half,
                                                    float out[4]) {
        if constexpr (KMAJ) {
            const float4 v = *reinterpret_cast<const float4*>(lds + row * kPitch + 8 * g + 4 * half);
            out[0] = v.x;
            out[1] = v.y;
            out[2] = v.z;
            out[3] = v.w;
        } else {
            // One per-lane address; the depth offsets are constants the LDS reads carry as
            // immediates (per-depth addresses would each take a register across the depth loop).
            const float* column = lds + 4 * half * kPitch + row;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                out[s] = column[(8 * g + s) * kPitch];
            }
        }
    }
};

// Writes a wavefront's accumulators: block (i, j), element e is C(row0 + 32i + 8(e/4) + e%4,
// col0 + 32j), as
//   C = act(fl(fl(fl(alpha * acc) + fl(beta * C0)) + bias))      (RAW: C = acc),
// the C0 term only when c0 is non-null, so the roundings are the reference's. Without a bias, -0
// is added (x + -0 is x for every x, -0 included), which spares a test per element. alpha * acc
// is exact for alpha == 1. INTERIOR: every row and column is
// inside C (no checks). C0 == kC0Batched: c0 is non-null and a row-block's C0 values are all
// loaded before any is used, so the loads overlap; kC0None: no C0; kC0Checked: c0 checked per
// element (one copy of the code for both cases). STREAM: non-temporal stores.
enum { kC0None = 0, kC0Batched = 1, kC0Checked = 2 };
// ROWS_PAST_M: a tile whose columns are all inside C and whose rows may run past m; every element
// is computed and stored through a buffer resource of m rows, which drops the stores to rows past
// m (no per-element test; the caller checks that (m + 256) * c_rs * 4 fits 32 bits).
template <int FM, int FN, int ACT, bool INTERIOR, bool RAW, int C0, bool STREAM = false,
          bool ROWS_PAST_M = false>
__device__ __forceinline__ void write_tile(const floatx16 (&acc)[FM][FN], float* c, int64_t c_rs,
                                           const float* c0, int64_t c0_rs, const GemmParams& p,
                                           int64_t row0, int64_t col0,
                                           const double* exp_table = nullptr) {
    static_assert(!ROWS_PAST_M || (!INTERIOR && C0 == kC0None && !STREAM), "row-edge copy");
    // Byte offsets into C within the resource (32 bits by the caller's check).
    // The record count is a 32-bit unsigned field; the caller keeps 4 (m + 256) c_rs below 2^32.
    const __amdgpu_buffer_rsrc_t c_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        c, 0, ROWS_PAST_M ? static_cast<int>(static_cast<uint32_t>(4 * p.m * c_rs)) : 0,
        kBufferWord3);
    // Kernel parameters read once: per element, the compiler would reload them after each store.
    const float alpha = p.alpha;
    const float beta = p.beta;
    const float* const bias_base = RAW ? nullptr : p.bias;
    // The bias of each column block, loaded before any store and waited for at once (the empty
    // asm reads it): a first use inside a predicated element would leave the load pending on the
    // paths that skip it, and every later element would wait for the memory counter, which also
    // counts the stores issued since.
    float bias_of[FN];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int64_t col = col0 + 32 * j;
        bias_of[j] = bias_base != nullptr && (INTERIOR || col < p.n) ? bias_base[col] : -0.0f;
        asm volatile("" ::"v"(bias_of[j]));
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int64_t row_i = row0 + 32 * i;
        float* c_i = c + row_i * c_rs + col0;
        float c0v[FN][16];
        if constexpr (C0 == kC0Batched) {
            const float* c0_i = c0 + row_i * c0_rs + col0;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int dr = 8 * (e / 4) + e % 4;
                    const bool inside = INTERIOR || (col0 + 32 * j < p.n && row_i + dr < p.m);
                    c0v[j][e] = inside ? c0_i[dr * c0_rs + 32 * j] : 0.0f;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int64_t col = col0 + 32 * j;
            if (!INTERIOR && !ROWS_PAST_M && col >= p.n) {
                continue;
            }
            const float bias = bias_of[j];
            // Elements outside C (rows past m) are computed all the same and only the loads and
            // stores are predicated, so no branch separates them.
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int dr = 8 * (e / 4) + e % 4;
                const bool row_ok = INTERIOR || ROWS_PAST_M || row_i + dr < p.m;
                float v = acc[i][j][e];
                if constexpr (!RAW) {
                    v = alpha * v;
                    if constexpr (C0 == kC0Batched) {
                        const float scaled = beta * c0v[j][e];
                        v = v + scaled;
                    } else if constexpr (C0 == kC0Checked) {
                        if (c0 != nullptr) {
                            const float c0_value = row_ok ? c0[(row_i + dr) * c0_rs + col] : 0.0f;
                            const float scaled = beta * c0_value;
                            v = v + scaled;
                        }
                    }
                    v = v + bias; // -0 without a bias: x + -0 is x
                    if constexpr (ACT == MFR_ACT_GELU_TANH) {
                        v = gelu_math::gelu_tanh(v, exp_table);
                    } else if constexpr (ACT != MFR_ACT_NONE) {
                        v = mfr::dev::gelu(v, ACT);
                    }
                }
                if constexpr (ROWS_PAST_M) {
                    const uint32_t offset =
                        static_cast<uint32_t>(4 * ((row_i + dr) * c_rs + col0 + 32 * j));
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), c_rsrc,
                                                          offset, 0, 0);
                } else if (row_ok) {
                    if constexpr (STREAM) {
                        __builtin_nontemporal_store(v, &c_i[dr * c_rs + 32 * j]);
                    } else {
                        c_i[dr * c_rs + 32 * j] = v;
                    }
                }
            }
        }
    }
}

// The epilogue for activation ACT. Without one it is dispatched on C0 and on whether the tile is
// interior. The tanh gelu has three copies without C0 (the MLP's case): interior tiles, tiles
// whose rows alone run past m (stores through a buffer resource that drops those rows), and other
// edges. With C0 tested and loaded between the elements, each element would wait for the memory
// counter, which also counts the stores before it. Every other gelu epilogue is one checked copy.
template <int FM, int FN, int ACT>
__device__ __forceinline__ void epilogue(const floatx16 (&acc)[FM][FN], float* c, int64_t c_rs,
                                         const float* c0, int64_t c0_rs, const GemmParams& p,
                                         int64_t row0, int64_t col0, bool interior,
                                         bool rows_only_edge, const double* exp_table) {
    if constexpr (ACT == MFR_ACT_GELU_TANH) {
        if (interior && c0 == nullptr) {
            write_tile<FM, FN, ACT, true, false, kC0None>(acc, c, c_rs, c0, c0_rs, p, row0, col0,
                                                          exp_table);
        } else if (rows_only_edge && c0 == nullptr) {
            write_tile<FM, FN, ACT, false, false, kC0None, false, true>(acc, c, c_rs, c0, c0_rs, p,
                                                                        row0, col0, exp_table);
        } else if (c0 == nullptr) {
            write_tile<FM, FN, ACT, false, false, kC0None>(acc, c, c_rs, c0, c0_rs, p, row0, col0,
                                                           exp_table);
        } else {
            write_tile<FM, FN, ACT, false, false, kC0Checked>(acc, c, c_rs, c0, c0_rs, p, row0,
                                                              col0, exp_table);
        }
    } else if constexpr (ACT != MFR_ACT_NONE) {
        write_tile<FM, FN, ACT, false, false, kC0Checked>(acc, c, c_rs, c0, c0_rs, p, row0, col0);
    } else if (c0 != nullptr) {
        if (interior) {
            write_tile<FM, FN, ACT, true, false, kC0Batched>(acc, c, c_rs, c0, c0_rs, p, row0,
                                                             col0);
        } else {
            write_tile<FM, FN, ACT, false, false, kC0Batched>(acc, c, c_rs, c0, c0_rs, p, row0,
                                                              col0);
        }
    } else {
        if (interior && p.stream_c) {
            write_tile<FM, FN, ACT, true, false, kC0None, true>(acc, c, c_rs, c0, c0_rs, p, row0,
                                                                col0);
        } else if (interior) {
            write_tile<FM, FN, ACT, true, false, kC0None>(acc, c, c_rs, c0, c0_rs, p, row0, col0);
        } else {
            write_tile<FM, FN, ACT, false, false, kC0None>(acc, c, c_rs, c0, c0_rs, p, row0,
                                                           col0);
        }
    }
}

// Which output tile a workgroup computes: the XCD-aware remap of the hardware workgroup index,
// grouped row-major order within the batch, the depth split outermost; and the operand offsets
// of its batch entry.
struct TileWork {
    int64_t split, batch_linear, m0, n0;
    int64_t off_a, off_b, off_c, off_c0;
    int rows_a, rows_b; // rows of A (M) and of B (N) inside the matrix, capped at the tile
    int64_t k_begin, kk; // depth range [k_begin, k_begin + kk)
};

template <int BM, int BN> __device__ __forceinline__ TileWork tile_work(const GemmParams& p) {
    TileWork w;
    // Every index here is below the launch's workgroup count, which the host keeps under 2^31,
    // so the decomposition runs in 32-bit unsigned arithmetic: a 64-bit division is a long
    // scalar instruction sequence, and every wavefront of every workgroup runs these (about a
    // thousand instructions before a small tile's first load in 64 bits).
    const uint32_t tiles_m = static_cast<uint32_t>(p.tiles_m);
    const uint32_t tiles_n = static_cast<uint32_t>(p.tiles_n);
    const uint32_t tiles_per_batch = tiles_m * tiles_n;
    const uint32_t tiles_per_split = tiles_per_batch * static_cast<uint32_t>(p.batch_count);
    const uint32_t total = tiles_per_split * static_cast<uint32_t>(p.splits);
    const uint32_t hw = blockIdx.x;
    const uint32_t per_xcd = total / 8;
    const uint32_t logical_all = hw < per_xcd * 8 ? (hw % 8) * per_xcd + hw / 8 : hw;
    const uint32_t split = logical_all / tiles_per_split;
    const uint32_t logical = logical_all - split * tiles_per_split;
    const uint32_t batch_linear = logical / tiles_per_batch;
    const uint32_t t = logical - batch_linear * tiles_per_batch;
    // Groups of group_m tile-rows; a group taller than the matrix is the matrix (the same order,
    // and group_tiles stays within the batch's tile count).
    const uint32_t gm = static_cast<uint32_t>(p.group_m) < tiles_m
                            ? static_cast<uint32_t>(p.group_m)
                            : tiles_m;
    const uint32_t group_tiles = gm * tiles_n;
    const uint32_t group = t / group_tiles;
    const uint32_t first_m = group * gm;
    const uint32_t rows_in_group = tiles_m - first_m < gm ? tiles_m - first_m : gm;
    const uint32_t in_group = t - group * group_tiles;
    const int64_t tile_m = first_m + in_group % rows_in_group;
    const int64_t tile_n = in_group / rows_in_group;
    w.split = split;
    w.batch_linear = batch_linear;
    uint32_t batch_index = batch_linear;
    w.off_a = w.off_b = w.off_c = w.off_c0 = 0;
    for (int d = p.batch_dims - 1; d >= 0; --d) {
        const uint32_t extent = static_cast<uint32_t>(p.batch[d]);
        const int64_t idx = batch_index % extent;
        batch_index /= extent;
        w.off_a += idx * p.a_bs[d];
        w.off_b += idx * p.b_bs[d];
        w.off_c += idx * p.c_bs[d];
        w.off_c0 += idx * p.c0_bs[d];
    }
    w.m0 = tile_m * BM;
    w.n0 = tile_n * BN;
    w.rows_a = p.m - w.m0 < BM ? static_cast<int>(p.m - w.m0) : BM;
    w.rows_b = p.n - w.n0 < BN ? static_cast<int>(p.n - w.n0) : BN;
    w.k_begin = w.split * p.k_per_split;
    w.kk = p.k - w.k_begin < p.k_per_split ? p.k - w.k_begin : p.k_per_split;
    return w;
}

// One depth slice of MFMAs from the LDS tiles sa, sb: the wavefront's FM x FN 32x32 blocks.
template <typename LoadA, typename LoadB, int KT, int FM, int FN, int WM, int WN>
__device__ __forceinline__ void slice_mfma(floatx16 (&acc)[FM][FN], const float* sa,
                                           const float* sb, int wave_m, int wave_n, int half,
                                           int r32) {
#pragma unroll
    for (int g = 0; g < KT / 8; ++g) {
        float fa[FM][4];
        float fb[FN][4];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            LoadA::fragment(sa, wave_m * WM + i * 32 + r32, g, half, fa[i]);
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            LoadB::fragment(sb, wave_n * WN + j * 32 + r32, g, half, fb[j]);
        }
#pragma unroll
        for (int st = 0; st < 4; ++st) {
#pragma unroll
            for (int i = 0; i < FM; ++i) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][st], fb[j][st],
                                                                      acc[i][j], 0, 0, 0);
                }
            }
        }
    }
}

// The end of a tile: split-K partial sums, or the epilogue with the activation chosen once.
template <int BM, int BN, int WM, int WN, int FM, int FN>
__device__ __forceinline__ void finish_tile(const floatx16 (&acc)[FM][FN], const GemmParams& p,
                                            const TileWork& w, int wave_m, int wave_n, int half,
                                            int r32, const double* exp_table) {
    // Accumulator e of block (i, j) is C(row, col) with row = 32i + 8(e/4) + 4*half + e%4,
    // col = 32j + lane%32 (the layout of every 32x32 MFMA).
    const int64_t row0 = w.m0 + wave_m * WM + 4 * half;
    const int64_t col0 = w.n0 + wave_n * WN + r32;
    const bool interior = w.m0 + BM <= p.m && w.n0 + BN <= p.n;
    // Rows past m only, and C's byte offsets (rows past m included) within 32 bits.
    const bool rows_only_edge = !interior && w.n0 + BN <= p.n &&
                                (p.m + BM) * p.c_rs * 4 < (int64_t{1} << 32);
    if (p.partial != nullptr) {
        // Split-K: raw sums only, to partial[split][batch] (dense m x n).
        float* part = p.partial + (w.split * p.batch_count + w.batch_linear) * p.m * p.n;
        if (interior) {
            write_tile<FM, FN, MFR_ACT_NONE, true, true, kC0None>(
                acc, part, p.n, nullptr, 0, p, row0, col0);
        } else {
            write_tile<FM, FN, MFR_ACT_NONE, false, true, kC0None>(
                acc, part, p.n, nullptr, 0, p, row0, col0);
        }
        return;
    }
    float* c_base = p.c + w.off_c;
    const float* c0_base = p.c0 != nullptr && p.beta != 0.0f ? p.c0 + w.off_c0 : nullptr;
    // One activation per branch (uniform), so each epilogue is straight-line code: unrolled
    // over every accumulator, the three would not fit the instruction cache together.
    if (p.act == MFR_ACT_NONE) {
        epilogue<FM, FN, MFR_ACT_NONE>(acc, c_base, p.c_rs, c0_base, p.c0_rs, p, row0, col0,
                                       interior, rows_only_edge, exp_table);
    } else if (p.act == MFR_ACT_GELU_TANH) {
        epilogue<FM, FN, MFR_ACT_GELU_TANH>(acc, c_base, p.c_rs, c0_base, p.c0_rs, p, row0, col0,
                                            interior, rows_only_edge, exp_table);
    } else {
        epilogue<FM, FN, MFR_ACT_GELU_ERF>(acc, c_base, p.c_rs, c0_base, p.c0_rs, p, row0, col0,
                                           interior, rows_only_edge, exp_table);
    }
}

template <int BM, int BN, int KT, int WAVES_M, int WAVES_N, bool AK, bool BK, int VA, int VB>
__global__ __launch_bounds__(WAVES_M * WAVES_N * 64) void sgemm_kernel(GemmParams p) {
    constexpr int THREADS = WAVES_M * WAVES_N * 64;
    constexpr int WM = BM / WAVES_M;
    constexpr int WN = BN / WAVES_N;
    constexpr int FM = WM / 32; // 32x32 accumulator blocks per wavefront, along M
    constexpr int FN = WN / 32;
    static_assert(KT % 8 == 0 && WM % 32 == 0 && WN % 32 == 0, "tile shape");
    using LoadA = SliceLoader<BM, KT, AK, VA, THREADS>;
    using LoadB = SliceLoader<BN, KT, BK, VB, THREADS>;
    __shared__ float smem[2 * (LoadA::kFloats + LoadB::kFloats)];
    // Buffer `which` (0 or 1) of each operand's double-buffered slice.
    auto lds_a = [&](int which) { return smem + which * LoadA::kFloats; };
    auto lds_b = [&](int which) { return smem + 2 * LoadA::kFloats + which * LoadB::kFloats; };

    const TileWork w = tile_work<BM, BN>(p);
    const float* a_base = p.a + w.off_a + w.m0 * p.a_rs + w.k_begin * p.a_cs;
    const float* b_base = p.b + w.off_b + w.n0 * p.b_cs + w.k_begin * p.b_rs;
    // Per slice the bases advance by KT depths.
    const int64_t a_step = KT * p.a_cs;
    const int64_t b_step = KT * p.b_rs;

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

    const int64_t kk = w.kk;
    const int64_t slices = kk > 0 ? (kk + KT - 1) / KT : 0;
    LoadA la;
    LoadB lb;
    if (slices > 0) {
        const int k_left = kk < KT ? static_cast<int>(kk) : KT;
        la.load(a_base, p.a_rs, p.a_cs, w.rows_a, k_left);
        lb.load(b_base, p.b_cs, p.b_rs, w.rows_b, k_left);
        la.store(lds_a(0));
        lb.store(lds_b(0));
        __syncthreads();
    }
    for (int64_t s = 0; s < slices; ++s) {
        const int cur = static_cast<int>(s & 1);
        const bool more = s + 1 < slices;
        if (more) {
            const int64_t k_next = (s + 1) * KT;
            const int k_left = kk - k_next < KT ? static_cast<int>(kk - k_next) : KT;
            la.load(a_base + (s + 1) * a_step, p.a_rs, p.a_cs, w.rows_a, k_left);
            lb.load(b_base + (s + 1) * b_step, p.b_cs, p.b_rs, w.rows_b, k_left);
        }
        slice_mfma<LoadA, LoadB, KT, FM, FN, WM, WN>(acc, lds_a(cur), lds_b(cur), wave_m, wave_n,
                                                     half, r32);
        if (more) {
            la.store(lds_a(cur ^ 1));
            lb.store(lds_b(cur ^ 1));
        }
        __syncthreads();
    }

    finish_tile<BM, BN, WM, WN, FM, FN>(acc, p, w, wave_m, wave_n, half, r32,
                                        gelu_math::kExp2Table);
}

} // namespace mfr::gemm
