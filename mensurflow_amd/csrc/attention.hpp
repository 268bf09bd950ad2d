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
    // Issue order of the query blocks: longest first, or (paired) the longer half longest first,
    // then the shorter half shortest first.
    int32_t paired;
    float scale;
};

// The most queries the decode form takes.
constexpr int64_t kDecodeMaxQueries = 4;

// A few queries against many keys (attention_decode.hip): p filled but for its block fields,
// 1 <= lq <= kDecodeMaxQueries, lk >= 1, rows as mfr_attention requires.
void run_decode(mfr_stream& s, const AttnParams& p, int64_t d);

} // namespace mfr::attn
