// What the fused attention kernels share: their parameters, and the decode form's launch.
#pragma once

#include "common.hpp"

namespace mfr::attn {

struct AttnParams {
    const float* q;
    const float* k;
    const float* v;
    float* out;
    const uint8_t* mask;
    int64_t lq, lk;
    int64_t q_rs, k_rs, v_rs, out_rs, mask_rs, mask_cs;
    int64_t batch[MFR_MAX_BATCH_DIMS];
    int64_t q_bs[MFR_MAX_BATCH_DIMS], k_bs[MFR_MAX_BATCH_DIMS], v_bs[MFR_MAX_BATCH_DIMS];
    int64_t out_bs[MFR_MAX_BATCH_DIMS], mask_bs[MFR_MAX_BATCH_DIMS];
    int64_t batch_count;
    int32_t batch_dims;
    int32_t causal;
    int32_t q_blocks;
    float scale;
};

// Which (batch entry, query block) workgroup blockIdx.x computes, and that entry's element
// offsets into q, k, v, out and the mask. Query blocks are issued longest first (the last ones of
// every batch entry).
struct BlockWork {
    int64_t qb;
    int64_t off_q, off_k, off_v, off_o, off_m;
};

// The indices are below the workgroup count (under 2^31), so the decomposition runs in 32-bit
// unsigned arithmetic: a 64-bit division is a long scalar instruction sequence that every
// wavefront of the workgroup runs before its first load.
__device__ inline BlockWork block_work(const AttnParams& p) {
    const uint32_t bid = blockIdx.x;
    const uint32_t batch_count = static_cast<uint32_t>(p.batch_count);
    const uint32_t q_blocks = static_cast<uint32_t>(p.q_blocks);
    const uint32_t level = bid / batch_count;
    BlockWork w{};
    w.qb = q_blocks - 1 - level;
    uint32_t bi = bid - level * batch_count;
    for (int d = p.batch_dims - 1; d >= 0; --d) {
        const uint32_t extent = static_cast<uint32_t>(p.batch[d]);
        const int64_t idx = bi % extent;
        bi /= extent;
        w.off_q += idx * p.q_bs[d];
        w.off_k += idx * p.k_bs[d];
        w.off_v += idx * p.v_bs[d];
        w.off_o += idx * p.out_bs[d];
        w.off_m += idx * p.mask_bs[d];
    }
    return w;
}

// The most queries the decode form takes.
constexpr int64_t kDecodeMaxQueries = 4;

// A few queries against many keys (attention_decode.hip): p filled but for its block fields,
// 1 <= lq <= kDecodeMaxQueries, lk >= 1, rows as mfr_attention requires.
void run_decode(mfr_stream& s, const AttnParams& p, int64_t d);

// The split form (attention_split.hip): bf16 parts on the bf16 matrix cores, d = 32, 64, 96, 128.
// p filled for workgroups of `waves` (4, or 8 but for d = 32) wavefronts of 32 queries.
void launch_split(const AttnParams& p, int64_t d, int waves, unsigned blocks, hipStream_t stream);

} // namespace mfr::attn
