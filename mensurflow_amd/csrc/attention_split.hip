// Fused attention on the bf16 matrix cores: q, k, v and the softmax weights cut exactly into three
// bf16 parts each, both products summed in fp32 from the six part products that reach fp32
// precision (split_kernel.hpp has their error), the online softmax of attention.hip between them.
//
// The fp32 matrix cores bound the tile kernels of attention.hip (8 x 16 x 1024 x 64 causal: 73 % of
// their peak). Here a 64-key block of 32 queries at d = 64 is 96 MFMAs of 32 cycles instead of 128
// of 64, and the cuts: k and v once per workgroup as the tiles pass through registers, q once, the
// weights once (32 per lane and block).
//
// Layout: a wavefront owns 32 queries and computes S^T = K Q^T (lane: one query, 16 keys per 32),
// so its weights are already the B operand of O^T += V^T P^T. In a 16-key step, lane half h holds
// the keys 4h .. 4h+3 and 8+4h .. 8+4h+3 of the step; the V tile is stored so that the 16 bytes a
// lane reads for a depth are those 8 keys. K: [plane][depth / 8][key][8], V: [plane][8-key
// group][depth][8], one 16-byte LDS read per fragment from consecutive addresses.
//
// Measured (us; before on the fp32 matrix cores, 32 or 16 queries per wavefront): 8 x 16 x 1024
// causal, d = 32 / 64 / 96 / 128: 90 -> 65, 150 -> 112, 241 -> 153, 319 -> 198; 8 x 16 x 1024 x 64
// non-causal 284 -> 187; 4 x 16 x 1000 x 128 with padded keys 334 -> 184, the mask as one ballot
// per 32 keys (a word per query and 4 keys, loaded ahead of the scores, spilled: 277). The error
// against 64 bits falls too (3.3e-7 -> 2.8e-7 and 6.4e-7 -> 5.3e-7).
#include "attention.hpp"
#include "split_parts.hpp"

namespace {

using mfr::attn::AttnParams;
using mfr::attn::block_work;
using mfr::attn::BlockWork;
using namespace mfr::gemm;

constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float exp2_native(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float max_halves(float v) {
    float a, b;
    mfr::dev::swap_pair<true>(v, a, b);
    return fmaxf(a, b);
}

__device__ __forceinline__ float sum_halves(float v) {
    float a, b;
    mfr::dev::swap_pair<true>(v, a, b);
    return a + b;
}

// The running softmax of a wavefront's 32 queries (lane: query lane % 32, half its keys).
struct Running {
    float top = -INFINITY; // of base-2 scores
    float sum = 0.0f;      // this lane's share
};

// How a kernel reads the mask: not at all, one row for all queries (padded keys), or a row each.
enum MaskForm { kNoMask, kOneRow, kRows };

// The mask of a 32-key sub-block from key k0 as bits: bit r is key k0 + r + 4 half (so element e
// of the scores is bit 8 (e / 4) + e % 4), 0 past the last key. One row: a byte per lane and a
// ballot. A row per query (mask_row, the lane's): a word per 4 keys where they are adjacent.
template <MaskForm MASK>
__device__ __forceinline__ uint32_t mask_bits(const AttnParams& p, const uint8_t* mask_row,
                                              int64_t k0, int half, int r32) {
    if constexpr (MASK == kOneRow) {
        const bool keep = k0 + r32 < p.lk && mask_row[(k0 + r32) * p.mask_cs] != 0;
        return static_cast<uint32_t>(__ballot(keep)) >> (4 * half);
    } else {
        uint32_t bits = 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int64_t first = k0 + 8 * g + 4 * half;
            uint32_t word = 0;
            if (p.mask_cs == 1 && first + 3 < p.lk) {
                typedef uint32_t __attribute__((aligned(1))) loose_word;
                word = *reinterpret_cast<const loose_word*>(mask_row + first);
            } else {
#pragma unroll 1
                for (int e = 0; e < 4; ++e) {
                    if (first + e < p.lk) {
                        word |= static_cast<uint32_t>(mask_row[(first + e) * p.mask_cs])
                                << (8 * e);
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                bits |= (word & (0xffu << (8 * e))) != 0 ? 1u << (8 * g + e) : 0u;
            }
        }
        return bits;
    }
}

// One 32-key sub-block's masking: element e is key k0 + 8 (e / 4) + 4 half + e % 4.
template <MaskForm MASK>
__device__ __forceinline__ void mask_scores(floatx16& s, const AttnParams& p, uint32_t bits,
                                            int64_t k0, int64_t query, int half) {
    const int64_t keys_left = p.lk - k0;
    const int64_t diag = query - k0; // causal keeps relative keys <= diag
    const int lim_k = static_cast<int>(keys_left < 32 ? (keys_left < 0 ? 0 : keys_left) : 32) -
                      4 * half;
    const int lim_q = static_cast<int>(!p.causal || diag >= 32 ? 32 : diag < -1 ? -1 : diag) -
                      4 * half;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int rel = 8 * (e / 4) + e % 4; // minus 4 half, as the limits
        bool keep = rel < lim_k && rel <= lim_q;
        if constexpr (MASK != kNoMask) {
            keep = keep && (bits & (1u << rel)) != 0;
        }
        s[e] = keep ? s[e] : -INFINITY;
    }
}

// The online softmax of one block: scores become weights; the output so far is rescaled where a
// maximum moved.
template <int SUB, int DB>
__device__ __forceinline__ void softmax_step(floatx16 (&s)[SUB], floatx16 (&o)[DB], Running& run) {
    float most = -INFINITY;
#pragma unroll
    for (int b = 0; b < SUB; ++b) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            most = fmaxf(most, s[b][e]);
        }
    }
    most = fmaxf(run.top, max_halves(most));
    const float reference = most == -INFINITY ? 0.0f : most;
    if (__any(most != run.top)) {
        const float shrink = exp2_native(run.top - reference);
        run.top = most;
        run.sum *= shrink;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                o[b][e] *= shrink;
            }
        }
    }
#pragma unroll
    for (int b = 0; b < SUB; ++b) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            s[b][e] = exp2_native(s[b][e] - reference);
            run.sum += s[b][e];
        }
    }
}

// ---- where the part products do not stand for the fp32 products --------------------------------
//
// A wavefront runs its queries again on the fp32 matrix cores (plain_queries) when
//   - a result is not finite: an infinite or NaN operand has NaN parts whatever it meets, one above
//     the largest bf16 (or a query that its scale takes there) infinite ones;
//   - its scores may have lost something: parts and part products under 2^-126 count as lost, so a
//     score misses at most 2^-126 (sqrt(d) (|q| + |k|) + 6 d), an absolute error of its base-2
//     exponent. With the squares of the workgroup's keys and of the lane's query (both as cut)
//     summing to less than 2^126, that is under 2^-58;
//   - an output may have: its terms lose at most 2^-126 (6 + |v|) a key. 2^26 times as much, with a
//     little room (the bound at the kernel's end, with the root of the sum of all squares for the
//     largest value), stays under the output's own rounding. A smaller output is run again, but one
//     of exactly 0 only where values under 2^-49 were met: without them its products are zeros, or
//     under 2^-126 each, of weights below 2^-77.
// So zero values, and a few tiny ones among others, cost nothing.
//
// Magnitudes are compared as float bits without the sign, times two, minus 1: one operation an
// element, zero wraps past every other value.
__device__ __forceinline__ uint32_t magnitude(float v) { return (__float_as_uint(v) << 1) - 1; }
constexpr uint32_t kSmallestValue = ((127u - 49u) << 24) - 1; // 2^-49
constexpr float kMostSquares = 0x1p126f;

// The wavefront's queries on the fp32 matrix cores, straight from global memory, scaled after their
// products as the kernel of attention.hip scales them.
template <int D, MaskForm MASK>
__device__ __forceinline__ void plain_queries(const AttnParams& p, const BlockWork& work,
                                              const uint8_t* mask_row, int64_t wq0, int64_t k_end,
                                              int half, int r32, floatx16 (&o)[D / 32],
                                              Running& run) {
    constexpr int DB = D / 32;
    const int64_t query = wq0 + r32;
    const float* q_row = p.q + work.off_q + (query < p.lq ? query : p.lq - 1) * p.q_rs;
    // Causal: no key past the wavefront's own queries (k_end is the workgroup's), whose value might
    // be infinite or NaN.
    k_end = p.causal && k_end > wq0 + 32 ? wq0 + 32 : k_end;
    run = Running{};
#pragma unroll
    for (int b = 0; b < DB; ++b) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            o[b][e] = 0.0f;
        }
    }
#pragma unroll 1
    for (int64_t k0 = 0; k0 < k_end; k0 += 32) {
        floatx16 s[1];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            s[0][e] = 0.0f;
        }
        const int64_t key = k0 + r32 < p.lk ? k0 + r32 : p.lk - 1;
        const float* k_row = p.k + work.off_k + key * p.k_rs;
#pragma unroll 2
        for (int depth = 0; depth < D; depth += 2) {
            s[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(k_row[depth + half], q_row[depth + half],
                                                        s[0], 0, 0, 0);
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            s[0][e] = p.scale * s[0][e] * kLog2e;
        }
        uint32_t bits = 0;
        if constexpr (MASK != kNoMask) {
            bits = mask_bits<MASK>(p, mask_row, k0, half, r32);
        }
        mask_scores<MASK>(s[0], p, bits, k0, query, half);
        softmax_step<1, DB>(s, o, run);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            // Element e is key 8 (e / 4) + 4 half + e % 4 of both operands; keys past the end
            // have weight 0 and read as zeros.
            const int64_t at = k0 + 8 * (e / 4) + 4 * half + e % 4;
            const float* v_row = p.v + work.off_v + (at < p.lk ? at : p.lk - 1) * p.v_rs;
#pragma unroll
            for (int b = 0; b < DB; ++b) {
                const float v = at < p.lk ? v_row[32 * b + r32] : 0.0f;
                o[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, s[0][e], o[b], 0, 0, 0);
            }
        }
    }
}

// D: head size. BK: keys per block. 2 wavefronts per SIMD (256 registers) with 8 wavefronts.
template <int D, int BK, MaskForm MASK, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void attention_split_kernel(
    AttnParams p) {
    constexpr int THREADS = WAVES * 64;
    constexpr int BLOCK_Q = 32 * WAVES;
    constexpr int STEPS = D / 16; // depth steps of K Q^T
    constexpr int SUB = BK / 32;  // 32-key sub-blocks
    constexpr int DB = D / 32;    // 32-depth blocks of the output
    // Tiles in 16-byte pieces; the K pitch keeps a row's pieces off each other's banks as the
    // threads of a row store them.
    constexpr int kPitchK = BK + 1, kPitchV = D;
    constexpr int kGroupsK = D / 8, kGroupsV = BK / 8;
    constexpr int kPiecesK = 3 * kGroupsK * kPitchK, kPiecesV = 3 * kGroupsV * kPitchV;
    constexpr int kUnits = BK * D / 8; // 8-element units of a K tile, and of a V tile
    constexpr int kPer = (kUnits + THREADS - 1) / THREADS;
    __shared__ uint4 k_tile0[kPiecesK], k_tile1[kPiecesK];
    __shared__ uint4 v_tile0[kPiecesV], v_tile1[kPiecesV];
    __shared__ uint32_t smallest, large_keys;
    __shared__ float4 v_squares_of[WAVES / 4];
    if (threadIdx.x == 0) {
        smallest = 0xffffffffu;
        large_keys = 0;
    }

    const BlockWork work = block_work(p);
    const int lane = threadIdx.x % 64;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));
    const int half = lane / 32;
    const int r32 = lane % 32;
    const int64_t q0 = work.qb * BLOCK_Q;
    const int64_t wq0 = q0 + wave * 32;
    const int64_t query = wq0 + r32;
    const bool wave_live = wq0 < p.lq;
    const uint8_t* mask_row = nullptr;
    if constexpr (MASK != kNoMask) {
        mask_row = p.mask + work.off_m + (query < p.lq ? query : 0) * p.mask_rs;
    }

    // q times scale log2 e, cut: depth 16 step + 8 half + j of the lane's query.
    bf16x8 qf[STEPS][3];
    float q_squares = 0.0f, k_squares = 0.0f, v_squares = 0.0f;
    {
        const float scale = p.scale * kLog2e;
        const float* q_row = p.q + work.off_q + (query < p.lq ? query : p.lq - 1) * p.q_rs;
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            const float4 lo = *reinterpret_cast<const float4*>(q_row + 16 * st + 8 * half);
            const float4 hi = *reinterpret_cast<const float4*>(q_row + 16 * st + 8 * half + 4);
            const float x[8] = {lo.x * scale, lo.y * scale, lo.z * scale, lo.w * scale,
                                hi.x * scale, hi.y * scale, hi.z * scale, hi.w * scale};
            uint32_t part[3][4];
            cut_eight(x, part, q_squares);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                qf[st][i] = __builtin_bit_cast(
                    bf16x8, make_uint4(part[i][0], part[i][1], part[i][2], part[i][3]));
            }
        }
    }

    // Keys this workgroup needs: all of them, or (causal) up to its last query.
    int64_t k_end = p.lk;
    if (p.causal) {
        const int64_t last_query = (q0 + BLOCK_Q < p.lq ? q0 + BLOCK_Q : p.lq) - 1;
        k_end = last_query + 1 < k_end ? last_query + 1 : k_end;
    }
    const int64_t blocks = (k_end + BK - 1) / BK;

    // The tiles' units in flight. K unit u: key u / (D / 8), depths 8 (u % (D / 8)) ..; V unit u:
    // depth u % D, group u / D = 2 t + h: keys 16 t + 4 h + 0 .. 3 and 16 t + 8 + 4 h + 0 .. 3.
    float k_reg[kPer][8], v_reg[kPer][8];
    const float* k_base = p.k + work.off_k;
    const float* v_base = p.v + work.off_v;
    uint32_t least = 0xffffffffu; // the smallest nonzero value's magnitude
    const auto load = [&](int64_t blk) __attribute__((always_inline)) {
        const int64_t k0 = blk * BK;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int u = static_cast<int>(threadIdx.x) + THREADS * i;
            if (kUnits % THREADS != 0 && u >= kUnits) {
                break;
            }
            // Keys past the end repeat the last one; their weights are 0.
            const int64_t key = k0 + u / kGroupsK < p.lk ? k0 + u / kGroupsK : p.lk - 1;
            const float* k_at = k_base + key * p.k_rs + 8 * (u % kGroupsK);
            const float4 lo = *reinterpret_cast<const float4*>(k_at);
            const float4 hi = *reinterpret_cast<const float4*>(k_at + 4);
            k_reg[i][0] = lo.x;
            k_reg[i][1] = lo.y;
            k_reg[i][2] = lo.z;
            k_reg[i][3] = lo.w;
            k_reg[i][4] = hi.x;
            k_reg[i][5] = hi.y;
            k_reg[i][6] = hi.z;
            k_reg[i][7] = hi.w;
            const int g = u / D;
            const int64_t first = k0 + 16 * (g / 2) + 4 * (g % 2);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int64_t at = first + (j < 4 ? j : j + 4);
                v_reg[i][j] = v_base[(at < p.lk ? at : p.lk - 1) * p.v_rs + u % D];
            }
        }
    };
    const auto cut = [&](uint4* k_tile, uint4* v_tile) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int u = static_cast<int>(threadIdx.x) + THREADS * i;
            if (kUnits % THREADS != 0 && u >= kUnits) {
                break;
            }
            uint32_t part[3][4];
            cut_eight(k_reg[i], part, k_squares);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                k_tile[(q * kGroupsK + u % kGroupsK) * kPitchK + u / kGroupsK] =
                    make_uint4(part[q][0], part[q][1], part[q][2], part[q][3]);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                least = min(least, magnitude(v_reg[i][j]));
            }
            cut_eight(v_reg[i], part, v_squares);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                v_tile[(q * kGroupsV + u / D) * kPitchV + u % D] =
                    make_uint4(part[q][0], part[q][1], part[q][2], part[q][3]);
            }
        }
    };

    Running run;
    floatx16 oacc[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            oacc[b][e] = 0.0f;
        }
    }
    const auto block = [&](int64_t kb, const uint4* k_tile, const uint4* v_tile, uint4* k_next,
                           uint4* v_next) __attribute__((always_inline)) {
        const bool more = kb + 1 < blocks;
        if (more) {
            load(kb + 1);
        }
        if (wave_live && (!p.causal || kb * BK <= wq0 + 31)) {
            // The mask is read ahead of the scores.
            uint32_t bits[SUB] = {};
            if constexpr (MASK != kNoMask) {
#pragma unroll
                for (int b = 0; b < SUB; ++b) {
                    bits[b] = mask_bits<MASK>(p, mask_row, kb * BK + 32 * b, half, r32);
                }
            }
            floatx16 s[SUB];
#pragma unroll
            for (int b = 0; b < SUB; ++b) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    s[b][e] = 0.0f;
                }
            }
#pragma unroll
            for (int st = 0; st < STEPS; ++st) {
                bf16x8 kf[SUB][3];
#pragma unroll
                for (int b = 0; b < SUB; ++b) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        kf[b][q] = __builtin_bit_cast(
                            bf16x8,
                            k_tile[(q * kGroupsK + 2 * st + half) * kPitchK + 32 * b + r32]);
                    }
                }
#pragma unroll
                for (int t = 0; t < 6; ++t) {
#pragma unroll
                    for (int b = 0; b < SUB; ++b) {
                        s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            kf[b][kPartA[t]], qf[st][kPartB[t]], s[b], 0, 0, 0);
                    }
                }
            }
            if (MASK != kNoMask || kb * BK + BK > p.lk || (p.causal && kb * BK + BK - 1 > wq0)) {
#pragma unroll
                for (int b = 0; b < SUB; ++b) {
                    mask_scores<MASK>(s[b], p, bits[b], kb * BK + 32 * b, query, half);
                }
            }
            softmax_step<SUB, DB>(s, oacc, run);
#pragma unroll
            for (int t = 0; t < BK / 16; ++t) {
                bf16x8 pf[3];
                {
                    float w[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        w[j] = s[t / 2][8 * (t % 2) + j];
                    }
                    uint32_t part[3][4];
                    float unused = 0.0f;
                    cut_eight(w, part, unused);
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        pf[q] = __builtin_bit_cast(
                            bf16x8, make_uint4(part[q][0], part[q][1], part[q][2], part[q][3]));
                    }
                }
#pragma unroll
                for (int b = 0; b < DB; ++b) {
                    bf16x8 vf[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        vf[q] = __builtin_bit_cast(
                            bf16x8,
                            v_tile[(q * kGroupsV + 2 * t + half) * kPitchV + 32 * b + r32]);
                    }
#pragma unroll
                    for (int i = 0; i < 6; ++i) {
                        oacc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            vf[kPartA[i]], pf[kPartB[i]], oacc[b], 0, 0, 0);
                    }
                }
            }
        }
        if (more) {
            cut(k_next, v_next);
        }
        lds_barrier();
    };
    if (blocks > 0) {
        load(0);
        cut(k_tile0, v_tile0);
        lds_barrier();
    }
    for (int64_t kb = 0; kb < blocks; kb += 2) {
        block(kb, k_tile0, v_tile0, k_tile1, v_tile1);
        if (kb + 1 < blocks) {
            block(kb + 1, k_tile1, v_tile1, k_tile0, v_tile0);
        }
    }

    if (__any(least < kSmallestValue)) {
        atomicMin(&smallest, least);
    }
    if (!(k_squares < kMostSquares / THREADS)) {
        large_keys = 1;
    }
    v_squares = mfr::dev::butterfly_sum(v_squares);
    if (lane == 0) {
        reinterpret_cast<float*>(v_squares_of)[wave] = v_squares;
    }
    lds_barrier();
    if (!wave_live) {
        return;
    }
    v_squares = 0.0f;
#pragma unroll
    for (const float4& four : v_squares_of) {
        v_squares += (four.x + four.y) + (four.z + four.w);
    }
    float total = sum_halves(run.sum);
    float zero = total * 0.0f; // NaN once a result is not finite
    float least_out = __builtin_inff();
#pragma unroll
    for (int b = 0; b < DB; ++b) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            zero = fmaf(oacc[b][e], 0.0f, zero);
            least_out = fminf(least_out, __builtin_fabsf(oacc[b][e]));
        }
    }
    const float bound = static_cast<float>(k_end) * 0x1p-97f *
                        (8.0f + fminf(__builtin_amdgcn_sqrtf(v_squares), 0x1p127f));
    bool again = zero != 0.0f || !(q_squares < kMostSquares) || large_keys != 0;
    if (__any(least_out < bound) && !__any(again)) {
        // The least output that is not 0.
        uint32_t nonzero = 0xffffffffu;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                nonzero = min(nonzero, magnitude(oacc[b][e]));
            }
        }
        again = nonzero < magnitude(bound) || (least_out == 0.0f && smallest < kSmallestValue);
    }
    if (__any(again)) {
        plain_queries<D, MASK>(p, work, mask_row, wq0, k_end, half, r32, oacc, run);
        total = sum_halves(run.sum);
    }
    // A row whose every key was removed has total == 0 and gives zeros; a NaN score makes total
    // NaN and so the whole row.
    const float inv = total == 0.0f ? 0.0f : 1.0f / total;
    if (query < p.lq) {
        float* out = p.out + work.off_o + query * p.out_rs + 4 * half;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                *reinterpret_cast<float4*>(out + 32 * b + 8 * g) =
                    make_float4(oacc[b][4 * g] * inv, oacc[b][4 * g + 1] * inv,
                                oacc[b][4 * g + 2] * inv, oacc[b][4 * g + 3] * inv);
            }
        }
    }
}

template <int D, int BK, int WAVES>
void launch_masked(const AttnParams& p, unsigned blocks, hipStream_t stream) {
    if (p.mask == nullptr) {
        attention_split_kernel<D, BK, kNoMask, WAVES><<<blocks, WAVES * 64, 0, stream>>>(p);
    } else if (p.mask_rs == 0 || p.lq == 1) {
        attention_split_kernel<D, BK, kOneRow, WAVES><<<blocks, WAVES * 64, 0, stream>>>(p);
    } else {
        attention_split_kernel<D, BK, kRows, WAVES><<<blocks, WAVES * 64, 0, stream>>>(p);
    }
}

} // namespace

namespace mfr::attn {

void launch_split(const AttnParams& p, int64_t d, int waves, unsigned blocks, hipStream_t stream) {
    if (d == 32) {
        launch_masked<32, 64, 4>(p, blocks, stream);
    } else if (d == 64 && waves == 8) {
        launch_masked<64, 64, 8>(p, blocks, stream);
    } else if (d == 64) {
        launch_masked<64, 32, 4>(p, blocks, stream);
    } else if (d == 96 && waves == 8) {
        launch_masked<96, 32, 8>(p, blocks, stream);
    } else if (d == 96) {
        launch_masked<96, 32, 4>(p, blocks, stream);
    } else if (waves == 8) {
        launch_masked<128, 32, 8>(p, blocks, stream);
    } else {
        launch_masked<128, 32, 4>(p, blocks, stream);
    }
}

} // namespace mfr::attn
