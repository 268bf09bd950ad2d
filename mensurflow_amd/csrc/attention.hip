// Fused scaled dot-product attention (include/mfr_rocm.h, mfr_attention). One kernel computes
// softmax(scale * q k^T, masked) v without writing the [.., lq, lk] scores to memory; the
// reference composes the same op from a batched GEMM, where(), softmax and a second batched GEMM
// (src/ops/attention.cpp:48-98). d = 32, 64, 96 and 128 run on the bf16 matrix cores
// (attention_split.hip) and 1 to 4 queries mostly in the decode form (attention_decode.hip); this file
// holds the entry point and the fp32 matrix core kernel of d = 16, 48, 80 and 112.
//
// Design (a workgroup of 4 wavefronts of 32 queries; keys in blocks of BK):
//   - Scores are computed transposed, S^T = K Q^T, with v_mfma_f32_32x32x2_f32: the accumulator
//     of a 32-key x 32-query block puts one query in each lane column (lanes l and l+32 hold
//     query l % 32, 16 keys each). Every per-query quantity of the softmax (running maximum,
//     running sum, rescale factor) is then lane-local, with one exchange between the two lane
//     halves per key block for the maximum.
//   - The output is also computed transposed, O^T += V^T P^T. Its B operand P^T needs, in lane l
//     at step s of depth group g, the weight of query l % 32 and key 8g + 4(l / 32) + s, which is
//     exactly accumulator element 4g + s of that lane in S^T: the probabilities feed the second
//     product straight from registers, with no shuffle and no trip through LDS.
//   - q's fragments stay in registers for the whole key loop. K and V tiles are double-buffered
//     in LDS through the GEMM's slice loader: K [keys][d+4] (K-major, 16-byte fragment reads),
//     V [keys][d+8] (read as V^T fragments, four 4-byte reads).
//   - Causal attention skips, per wavefront, every key block lying wholly above its queries'
//     diagonal, and the key loop stops at the workgroup's last query. Workgroups are
//     issued longest first (the last query blocks of every batch entry) so the short ones fill
//     the tail.
//   - The result is scaled by the reciprocal of the row sum, staged through LDS and stored as
//     16-byte rows.
#include "attention.hpp"
#include "gemm_kernel.hpp"

#include <cmath>

namespace {

using mfr::gemm::floatx16;
using mfr::gemm::SliceLoader;

constexpr int kWaves = 4; // wavefronts of 32 queries per workgroup

// Wavefronts per workgroup for one launch: 8 for d = 64, 96 and 128, where one K/V tile then
// serves 256 queries, except 4 when workgroups of 8 would leave fewer than two per CU (causal,
// whose work grows with the query block, so the longest decides the time) or idle CUs; and for
// d = 64 where 128 queries and 512 keys are all there are and every CU has two heads (half of 8
// wavefronts would be idle, and three workgroups of 4 fit a CU where one of 8 does: 1000 x 16
// causal 23.2 -> 11.7 us, 1000 x 128 causal 50 -> 36; from 1024 keys on 4 are up to 7 % slower, with
// one head per CU 28 %, at d = 96 and 128 always 5-25 %).
int waves_used(int64_t d, int64_t lq, int64_t lk, int64_t batch_count, bool causal, int cus) {
    if (d == 32 || d % 32 != 0 ||
        (d == 64 && lq <= 128 && lk <= 512 && batch_count >= 2 * static_cast<int64_t>(cus))) {
        return kWaves;
    }
    const int64_t blocks = batch_count * ((lq + 255) / 256);
    return blocks < (causal ? 2 : 1) * static_cast<int64_t>(cus) ? kWaves : 8;
}
constexpr float kLog2e = 1.4426950408889634f;

using mfr::attn::AttnParams;

using mfr::attn::block_work;
using mfr::attn::BlockWork;

// max / sum of the values in lanes l and l ^ 32, in every lane, through the vector ALU's lane swaps (mfr::dev::swap_pair), not an LDS-crossbar permute and its
// wait on the softmax's critical path; every lane of a pair gets the same bits.
using mfr::dev::swap_pair;
__device__ inline float max_halves(float x) {
    float a, b;
    swap_pair<true>(x, a, b);
    return fmaxf(a, b);
}
__device__ inline float sum_halves(float x) {
    float a, b;
    swap_pair<true>(x, a, b);
    return a + b;
}

// exp(x - m) through the hardware's 2^x (v_exp_f32, 1 ulp; results below 2^-126 may flush to
// zero, which is below the rounding of any row sum, whose largest term is exp(0) = 1). m is
// never -inf here (the caller substitutes 0), so x = -inf gives exp2(-inf) = 0 without a NaN.
__device__ inline float weight(float x, float m) {
    return __builtin_amdgcn_exp2f((x - m) * kLog2e);
}

// MASKED: a mask tensor is given (read for every score). Without it only the key count and the
// causal diagonal remove scores, and only blocks that reach past either are checked. WAVES
// wavefronts of 32 queries per workgroup; MIN_WAVES is the occupancy the compiler must allow
// (wavefronts per SIMD).
template <int D, int BK, bool MASKED, int WAVES = kWaves, int MIN_WAVES = 2>
__global__ __launch_bounds__(WAVES * 64, MIN_WAVES) void attention_kernel(AttnParams p) {
    constexpr int THREADS = WAVES * 64;
    constexpr int BLOCK_Q = WAVES * 32;
    constexpr int SUB = BK / 32; // 32-key sub-blocks per key block
    // d need not be a multiple of 32: the output side runs on DP = d rounded up to 32, whose V
    // rows past d load as zeros, so those output columns are zero and never stored.
    static_assert(D % 16 == 0, "d is a multiple of 16");
    constexpr int DP = (D + 31) / 32 * 32;
    constexpr int DB = DP / 32;  // 32-wide output column blocks
    constexpr int G = D / 8;     // depth groups of q . k
    constexpr int kStagePitch = DP + 4;
    using LoadK = SliceLoader<BK, D, true, 4, THREADS>;   // rows = keys, depth = d
    using LoadV = SliceLoader<DP, BK, false, 4, THREADS>; // rows = d (DP), depth = keys
    // Double-buffered K and V tiles; after the key loop the same memory stages the output.
    constexpr int kTileFloats = 2 * (LoadK::kFloats + LoadV::kFloats);
    constexpr int kStageFloats = WAVES * 32 * kStagePitch;
    __shared__ float smem[kTileFloats > kStageFloats ? kTileFloats : kStageFloats];
    auto lds_k = [&](int which) { return smem + which * LoadK::kFloats; };
    auto lds_v = [&](int which) { return smem + 2 * LoadK::kFloats + which * LoadV::kFloats; };

    // ---- which (batch entry, query block): the longest (last) query blocks first ----
    const BlockWork work = block_work(p);
    const int64_t qb = work.qb;
    const int64_t off_q = work.off_q, off_k = work.off_k, off_v = work.off_v,
                  off_o = work.off_o, off_m = work.off_m;

    const int lane = threadIdx.x % 64;
    // Uniform across the wavefront; read into a scalar register so that the branches on it
    // (active sub-blocks, edge blocks) are scalar branches.
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));
    const int half = lane / 32;
    const int r32 = lane % 32;
    const int64_t q0 = qb * BLOCK_Q;
    const int64_t wq0 = q0 + wave * 32; // first query of this wavefront
    const int64_t query = wq0 + r32;    // this lane's query
    const bool wave_live = wq0 < p.lq;

    // q fragments: B operand of S^T = K Q^T, depth 8g + 4*half + s at step s of group g.
    float qf[G][4];
    {
        const float* qrow = p.q + off_q + query * p.q_rs + 4 * half;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (query < p.lq) {
                v = *reinterpret_cast<const float4*>(qrow + 8 * g);
            }
            qf[g][0] = v.x;
            qf[g][1] = v.y;
            qf[g][2] = v.z;
            qf[g][3] = v.w;
        }
    }
    const uint8_t* mask_row = nullptr;
    if constexpr (MASKED) {
        mask_row = p.mask + off_m + (query < p.lq ? query : 0) * p.mask_rs;
    }

    // Keys this workgroup needs: all of them, or (causal) up to its last query.
    int64_t k_end = p.lk;
    if (p.causal) {
        const int64_t last_query = (q0 + BLOCK_Q < p.lq ? q0 + BLOCK_Q : p.lq) - 1;
        k_end = last_query + 1 < k_end ? last_query + 1 : k_end;
    }
    const int64_t blocks = (k_end + BK - 1) / BK;

    float m_run = -INFINITY; // running maximum of this lane's query
    float l_run = 0.0f;      // this lane's share of the running sum (its 16 keys per sub-block)
    floatx16 oacc[DB];
#pragma unroll
    for (int b = 0; b < DB; ++b) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            oacc[b][e] = 0.0f;
        }
    }

    const float* k_base = p.k + off_k;
    const float* v_base = p.v + off_v;

    // Keys of block `blk` inside the matrix, and whether this wavefront needs the block at all
    // (uniform across the wavefront: causal attention skips blocks lying wholly above its
    // queries' diagonal). Inside a needed block every MFMA runs unconditionally (masking removes
    // what is not wanted), which keeps the accumulators in place.
    auto keys_in = [&](int64_t blk) {
        const int64_t left = p.lk - blk * BK;
        return left < BK ? static_cast<int>(left) : BK;
    };
    auto needed = [&](int64_t blk) { return wave_live && (!p.causal || blk * BK <= wq0 + 31); };

    // ---- S^T = K Q^T for one block, the sub-blocks' accumulator chains interleaved ----
    auto scores = [&](const float* sk, floatx16(&sacc)[SUB]) {
#pragma unroll
        for (int sb = 0; sb < SUB; ++sb) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                sacc[sb][e] = 0.0f;
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float kf[SUB][4];
#pragma unroll
            for (int sb = 0; sb < SUB; ++sb) {
                LoadK::fragment(sk, 32 * sb + r32, g, half, kf[sb]);
            }
#pragma unroll
            for (int st = 0; st < 4; ++st) {
#pragma unroll
                for (int sb = 0; sb < SUB; ++sb) {
                    sacc[sb] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[sb][st], qf[g][st],
                                                                     sacc[sb], 0, 0, 0);
                }
            }
        }
    };

    // ---- scale, mask and the online softmax of the block starting at key k0: sacc becomes
    //      the weights exp(s - m) (per lane: query `query`, 16 keys per sub-block) ----
    auto softmax = [&](int64_t k0, floatx16(&sacc)[SUB]) {
        // Key of element e of sub-block sb, relative to k0: 32*sb + 8*(e/4) + e%4 + 4*half.
        // A block needs checking when it reaches past the last key or (causal) past the
        // wavefront's first query; both tests are uniform across the wavefront.
        const bool edge = k0 + BK > p.lk || (p.causal && k0 + BK - 1 > wq0);
        if (MASKED || edge) {
            const int64_t keys_left = p.lk - k0;
            const int64_t diag = query - k0; // causal keeps relative keys <= diag
            const int lim_k = static_cast<int>(keys_left < BK ? keys_left : BK) - 4 * half;
            const int lim_q = static_cast<int>(!p.causal || diag >= BK ? BK
                                               : diag < -1 ? -1
                                                           : diag) -
                              4 * half;
#pragma unroll
            for (int sb = 0; sb < SUB; ++sb) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int rel = 32 * sb + 8 * (e / 4) + e % 4; // minus 4*half (above)
                    bool keep = rel < lim_k && rel <= lim_q;
                    if constexpr (MASKED) {
                        if (keep) {
                            keep = mask_row[(k0 + rel + 4 * half) * p.mask_cs] != 0;
                        }
                    }
                    sacc[sb][e] = keep ? p.scale * sacc[sb][e] : -INFINITY;
                }
            }
        } else {
#pragma unroll
            for (int sb = 0; sb < SUB; ++sb) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    sacc[sb][e] = p.scale * sacc[sb][e];
                }
            }
        }
        float block_max = -INFINITY;
#pragma unroll
        for (int sb = 0; sb < SUB; ++sb) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                block_max = fmaxf(block_max, sacc[sb][e]);
            }
        }
        block_max = max_halves(block_max);
        const float m_new = fmaxf(m_run, block_max);
        const float m_use = m_new == -INFINITY ? 0.0f : m_new;
        const float rescale = weight(m_run, m_use); // exactly 1 where the maximum stayed
        m_run = m_new;
        l_run *= rescale;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                oacc[b][e] *= rescale;
            }
        }
#pragma unroll
        for (int sb = 0; sb < SUB; ++sb) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float w = weight(sacc[sb][e], m_use);
                sacc[sb][e] = w;
                l_run += w;
            }
        }
    };

    // ---- O^T += V^T P^T: P^T's fragments are the S^T accumulators themselves ----
    auto accumulate = [&](const float* sv, const floatx16(&sacc)[SUB]) {
#pragma unroll
        for (int sb = 0; sb < SUB; ++sb) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float vf[DB][4];
#pragma unroll
                for (int b = 0; b < DB; ++b) {
                    LoadV::fragment(sv, 32 * b + r32, 4 * sb + g, half, vf[b]);
                }
#pragma unroll
                for (int st = 0; st < 4; ++st) {
#pragma unroll
                    for (int b = 0; b < DB; ++b) {
                        oacc[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                            vf[b][st], sacc[sb][4 * g + st], oacc[b], 0, 0, 0);
                    }
                }
            }
        }
    };

    LoadK lk_;
    LoadV lv_;
    if (blocks > 0) {
        lk_.load(k_base, p.k_rs, 1, keys_in(0), D);
        lv_.load(v_base, 1, p.v_rs, D, keys_in(0));
        lk_.store(lds_k(0));
        lv_.store(lds_v(0));
        __syncthreads();
    }
    // One barrier per block: the next block's tiles are loaded into registers while this one is
    // computed, then written to the other buffers.
    for (int64_t kb = 0; kb < blocks; ++kb) {
        const int cur = static_cast<int>(kb & 1);
        const bool more = kb + 1 < blocks;
        if (more) {
            lk_.load(k_base + (kb + 1) * BK * p.k_rs, p.k_rs, 1, keys_in(kb + 1), D);
            lv_.load(v_base + (kb + 1) * BK * p.v_rs, 1, p.v_rs, D, keys_in(kb + 1));
        }
        if (needed(kb)) {
            floatx16 sacc[SUB];
            scores(lds_k(cur), sacc);
            softmax(kb * BK, sacc);
            accumulate(lds_v(cur), sacc);
        }
        if (more) {
            lk_.store(lds_k(cur ^ 1));
            lv_.store(lds_v(cur ^ 1));
        }
        __syncthreads();
    }

    // ---- normalise, stage [32 queries][D] per wavefront in LDS, store 16-byte rows ----
    const float l_total = sum_halves(l_run);
    // A row whose every key was removed has l_total == 0 and gives zeros; a NaN score makes
    // l_total NaN and so the whole row.
    const float inv = l_total == 0.0f ? 0.0f : 1.0f / l_total;
    float* stage = smem + wave * 32 * kStagePitch;
    __syncthreads();
#pragma unroll
    for (int b = 0; b < DB; ++b) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int col = 32 * b + 8 * (e / 4) + 4 * half + e % 4;
            stage[r32 * kStagePitch + col] = oacc[b][e] * inv;
        }
    }
    __syncthreads();
    float* out_base = p.out + off_o;
    constexpr int kRowUnits = D / 4;
#pragma unroll
    for (int i = 0; i < 32 * kRowUnits / 64; ++i) {
        const int u = lane + 64 * i;
        const int row = u / kRowUnits;
        const int c4 = u % kRowUnits;
        const int64_t qrow = wq0 + row;
        if (qrow < p.lq) {
            *reinterpret_cast<float4*>(out_base + qrow * p.out_rs + 4 * c4) =
                *reinterpret_cast<const float4*>(stage + row * kStagePitch + 4 * c4);
        }
    }
}

template <bool MASKED>
void launch(int64_t d, const AttnParams& p, unsigned grid, hipStream_t st) {
    switch (d) {
    case 16: attention_kernel<16, 64, MASKED, 4><<<grid, 4 * 64, 0, st>>>(p); break;
    case 48: attention_kernel<48, 64, MASKED, 4><<<grid, 4 * 64, 0, st>>>(p); break;
    case 80: attention_kernel<80, 64, MASKED, 4><<<grid, 4 * 64, 0, st>>>(p); break;
    default: attention_kernel<112, 64, MASKED, 4><<<grid, 4 * 64, 0, st>>>(p); break;
    }
}

bool aligned_rows(const void* base, int64_t row_stride, const int64_t* bs, int dims) {
    if (!mfr::aligned16(base) || row_stride % 4 != 0) {
        return false;
    }
    for (int d = 0; d < dims; ++d) {
        if (bs[d] % 4 != 0) {
            return false;
        }
    }
    return true;
}

void run_attention(mfr_stream& s, const mfr_attention_desc& d) {
    using mfr::require;
    require(d.lq >= 0 && d.lk >= 0 && d.d >= 0, "attention: negative dimension");
    require(d.batch_dims >= 0 && d.batch_dims <= MFR_MAX_BATCH_DIMS,
            "attention: batch_dims out of range");
    int64_t batch_count = 1;
    for (int i = 0; i < d.batch_dims; ++i) {
        require(d.batch[i] >= 0, "attention: negative batch size");
        batch_count *= d.batch[i];
    }
    if (d.lq == 0 || batch_count == 0) {
        return;
    }
    if (d.d <= 0 || d.d > 128 || d.d % 16 != 0) {
        throw mfr::Error(MFR_E_UNSUPPORTED,
                         "attention: fused kernel takes d = 16, 32, ..., 128 (a multiple of 16)");
    }
    require(d.q != nullptr && d.out != nullptr, "attention: null q or out");
    require(d.lk == 0 || (d.k != nullptr && d.v != nullptr), "attention: null k or v");
    require(d.q_rs >= d.d && d.out_rs >= d.d, "attention: row stride smaller than d");
    const bool aligned =
        aligned_rows(d.q, d.q_rs, d.q_bs, d.batch_dims) &&
        aligned_rows(d.out, d.out_rs, d.out_bs, d.batch_dims) &&
        (d.lk == 0 || (aligned_rows(d.k, d.k_rs, d.k_bs, d.batch_dims) &&
                       aligned_rows(d.v, d.v_rs, d.v_bs, d.batch_dims)));
    if (!aligned) {
        throw mfr::Error(MFR_E_UNSUPPORTED,
                         "attention: fused kernel needs 16-byte aligned rows and strides");
    }
    AttnParams p{};
    p.q = d.q;
    p.k = d.k;
    p.v = d.v;
    p.out = d.out;
    p.mask = d.mask;
    p.lq = d.lq;
    // Causal query i keeps keys 0 .. i: no form reads those past the last query.
    p.lk = d.causal != 0 && d.lq < d.lk ? d.lq : d.lk;
    p.q_rs = d.q_rs;
    p.k_rs = d.k_rs;
    p.v_rs = d.v_rs;
    p.out_rs = d.out_rs;
    p.mask_rs = d.mask != nullptr ? d.mask_rs : 0;
    p.mask_cs = d.mask != nullptr ? d.mask_cs : 0;
    p.batch_dims = d.batch_dims;
    for (int i = 0; i < d.batch_dims; ++i) {
        p.batch[i] = d.batch[i];
        p.q_bs[i] = d.q_bs[i];
        p.k_bs[i] = d.k_bs[i];
        p.v_bs[i] = d.v_bs[i];
        p.out_bs[i] = d.out_bs[i];
        p.mask_bs[i] = d.mask != nullptr ? d.mask_bs[i] : 0;
    }
    p.batch_count = batch_count;
    p.causal = d.causal != 0;
    p.scale = d.scale != 0.0f ? d.scale
                              : static_cast<float>(1.0 / std::sqrt(static_cast<double>(d.d)));
    if (mfr::attn::decode_takes(p.lq, p.lk, d.d, batch_count, s.compute_units)) {
        mfr::attn::run_decode(s, p, d.d);
        return;
    }
    const int waves = waves_used(d.d, p.lq, p.lk, batch_count, d.causal != 0, s.compute_units);
    const int64_t block_q = 32 * waves; // queries per workgroup
    const int64_t q_blocks = (d.lq + block_q - 1) / block_q;
    const int64_t blocks = q_blocks * batch_count;
    require(mfr::one_launch(blocks, 64 * waves), "attention: problem too large for one launch");
    p.q_blocks = static_cast<int32_t>(q_blocks);
    const unsigned grid = static_cast<unsigned>(blocks);
    if (d.d % 32 == 0) {
        mfr::attn::launch_split(p, d.d, waves, grid, s.stream);
    } else if (d.mask != nullptr) {
        launch<true>(d.d, p, grid, s.stream);
    } else {
        launch<false>(d.d, p, grid, s.stream);
    }
    mfr::check_launch("attention_kernel");
}

} // namespace

extern "C" int mfr_attention(mfr_stream_t stream, const mfr_attention_desc* desc) {
    return mfr::guarded([&] {
        auto& s = mfr::stream_of(stream);
        mfr::require(desc != nullptr, "attention: null descriptor");
        run_attention(s, *desc);
    });
}
