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
    int64_t lq, lk; // causal: lk is at most lq
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

// Whether the decode form takes 1 to 4 queries against lk keys. It reads K and V once at the HBM's
// rate and cuts long key counts over the chip, but each query is vector work for every lane, and
// joining the lane groups of 4 queries costs 4 us at d = 32.
// Times of the tile kernels over the decode form's (2 to 20000 heads, 4 to 16384 keys):
//   - 1 query: 0.97 to 26 everywhere;
//   - 2 queries: 1.0 to 22, but d = 16 below 256 keys 0.45-0.8, d = 32 below 128 keys 0.75-1.0;
//   - 3 or 4, d a multiple of 32: 1.05 to 8.7 where the heads leave half the chip idle, from 128
//     keys (d = 32: 256, d = 128: 64) on; with 256 heads or more 0.25-1.0 (20000 x 4 x 16 x 32: 185
//     us against 668), but d = 32 from 2048 keys on, 1.0 to 1.7;
//   - 3 or 4, d = 16 and 48: 1.2 to 16 for as long key counts as below, 0.15-0.9 under them;
//     d = 80 and 112: 1.1 to 16 everywhere.
inline bool decode_takes(int64_t lq, int64_t lk, int64_t d, int64_t batch_count, int cus) {
    if (lq < 1 || lq > kDecodeMaxQueries || lk < 1) {
        return false;
    }
    if (lq == 1) {
        return true;
    }
    if (lq == 2) {
        return d >= 48 || lk >= (d == 16 ? 256 : 128);
    }
    const bool idle = 2 * batch_count <= cus;
    if (d % 32 == 0) {
        return lk >= (d == 32 ? 256 : d == 128 ? 64 : 128) && (idle || (d == 32 && lk >= 2048));
    }
    if (d == 16) {
        return lk >= 4096 || (idle && lk >= 1024);
    }
    return d > 48 || lk >= 1024 || (lk >= 256 && batch_count <= cus);
}

// A few queries against many keys (attention_decode.hip): p filled but for its block fields,
// 1 <= lq <= kDecodeMaxQueries, lk >= 1, rows as mfr_attention requires.
void run_decode(mfr_stream& s, const AttnParams& p, int64_t d);

// The split form (attention_split.hip): bf16 parts on the bf16 matrix cores, d = 32, 64, 96, 128.
// p filled for workgroups of `waves` (4, or 8 but for d = 32) wavefronts of 32 queries.
void launch_split(const AttnParams& p, int64_t d, int waves, unsigned blocks, hipStream_t stream);

} // namespace mfr::attn
