// Attention of a few queries (at most 4) against many keys, the decode step of a generating
// program: bound by reading K and V once from HBM.
//
// The tile kernels (attention.hip) give every workgroup 128 or 256 queries of one head, so one
// query a head left 1 lane in 32 with work and one workgroup per head walking all its keys: 8 x 16
// heads, 4096 keys of 64 took 340 us, 0.8 TB/s. Here the keys of a head are cut into ranges, a
// workgroup each (about 4 per CU), and every lane holds 4 depths of the queries: G = d / 4 lanes
// (rounded up to a power of two) share a key, 64 / G keys per wavefront and load, kKeys loads of
// K and of V in flight. Each such lane group keeps its own running maximum, sum and weighted
// values (online softmax in base 2, as the tile kernels), joined through LDS at the end; the
// ranges' results are joined by a second kernel.
#include "attention.hpp"

#include <algorithm>

namespace {

using mfr::attn::AttnParams;

constexpr int kWaves = 4;  // wavefronts per workgroup
constexpr int kKeys = 8;   // keys per lane group and iteration
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float exp2_native(float x) { return __builtin_amdgcn_exp2f(x); }

// The sum of v over the G lanes of a lane group, in every lane of it.
template <int G> __device__ __forceinline__ float group_sum(float v) {
    if constexpr (G >= 32) {
        float a, b;
        mfr::dev::swap_pair<false>(v, a, b);
        v = a + b;
    }
    if constexpr (G >= 16) {
        v += mfr::dev::xor_lane<8>(v);
    }
    if constexpr (G >= 8) {
        v += mfr::dev::xor_lane<4>(v);
    }
    v += mfr::dev::xor_lane<2>(v);
    v += mfr::dev::xor_lane<1>(v);
    return v;
}

// exp2(m - top), 0 for an empty part (m = -inf, also where every part is empty).
__device__ __forceinline__ float part_weight(float m, float top) {
    return m == -INFINITY ? 0.0f : exp2_native(m - top);
}

// One range of `range` keys of one batch entry: blockIdx.x = entry * ranges + range index. With
// ranges == 1 the output rows; else the part (maximum, sum, weighted values) of each query to
// parts[(entry * lq + query) * ranges + range index][d + 2].
template <int G, int QN>
__global__ __launch_bounds__(kWaves * 64) void attention_decode_kernel(AttnParams p, int d,
                                                                       int ranges, int64_t range,
                                                                       float* parts) {
    constexpr int kGroups = 64 / G;              // lane groups per wavefront
    constexpr int kParts = kWaves * kGroups;     // lane groups per workgroup
    __shared__ float values[kParts][4 * G + 4];
    __shared__ float top_of[kParts], sum_of[kParts];
    const uint32_t entry = blockIdx.x / static_cast<uint32_t>(ranges);
    const int index = static_cast<int>(blockIdx.x - entry * static_cast<uint32_t>(ranges));
    int64_t off_q = 0, off_k = 0, off_v = 0, off_o = 0, off_m = 0;
    uint32_t rest = entry;
    for (int b = p.batch_dims - 1; b >= 0; --b) {
        const uint32_t extent = static_cast<uint32_t>(p.batch[b]);
        const int64_t at = rest % extent;
        rest /= extent;
        off_q += at * p.q_bs[b];
        off_k += at * p.k_bs[b];
        off_v += at * p.v_bs[b];
        off_o += at * p.out_bs[b];
        off_m += at * p.mask_bs[b];
    }
    const int lane = threadIdx.x % 64;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / 64));
    const int group = lane / G;
    const int depth = 4 * (lane % G);
    const bool live = depth < d; // lanes past d / 4 of a group hold zeros
    const int64_t first = index * range;
    const int64_t end = first + range < p.lk ? first + range : p.lk;

    // Scores are scaled after their products (as the tile kernels' are where it matters), so that
    // only they can overflow, and are base-2 exponents.
    float4 q[QN], acc[QN];
    float top[QN], sum[QN];
#pragma unroll
    for (int i = 0; i < QN; ++i) {
        q[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (live && i < p.lq) {
            q[i] = *reinterpret_cast<const float4*>(p.q + off_q + i * p.q_rs + depth);
        }
        acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        top[i] = -INFINITY;
        sum[i] = 0.0f;
    }
    const float* k_base = p.k + off_k + depth;
    const float* v_base = p.v + off_v + depth;
    for (int64_t block = first + wave * kKeys * kGroups; block < end;
         block += kWaves * kKeys * kGroups) {
        float4 k[kKeys], v[kKeys];
#pragma unroll
        for (int u = 0; u < kKeys; ++u) {
            const int64_t key = block + u * kGroups + group;
            k[u] = v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (live && key < end) {
                k[u] = mfr::dev::load_streaming(k_base + key * p.k_rs);
                v[u] = mfr::dev::load_streaming(v_base + key * p.v_rs);
            }
        }
#pragma unroll
        for (int i = 0; i < QN; ++i) {
            float score[kKeys];
            float most = top[i];
#pragma unroll
            for (int u = 0; u < kKeys; ++u) {
                const int64_t key = block + u * kGroups + group;
                float s = q[i].x * k[u].x;
                s = fmaf(q[i].y, k[u].y, s);
                s = fmaf(q[i].z, k[u].z, s);
                s = fmaf(q[i].w, k[u].w, s);
                s = p.scale * group_sum<G>(s) * kLog2e;
                bool keep = key < end && i < p.lq && (p.causal == 0 || key <= i);
                if (keep && p.mask != nullptr) {
                    keep = p.mask[off_m + i * p.mask_rs + key * p.mask_cs] != 0;
                }
                score[u] = keep ? s : -INFINITY;
                most = fmaxf(most, score[u]);
            }
            // Nothing kept yet: any finite reference gives weights of 0.
            const float reference = most == -INFINITY ? 0.0f : most;
            const float shrink = exp2_native(top[i] - reference);
            top[i] = most;
            sum[i] *= shrink;
            acc[i].x *= shrink;
            acc[i].y *= shrink;
            acc[i].z *= shrink;
            acc[i].w *= shrink;
#pragma unroll
            for (int u = 0; u < kKeys; ++u) {
                const float w = exp2_native(score[u] - reference);
                sum[i] += w;
                acc[i].x = fmaf(w, v[u].x, acc[i].x);
                acc[i].y = fmaf(w, v[u].y, acc[i].y);
                acc[i].z = fmaf(w, v[u].z, acc[i].z);
                acc[i].w = fmaf(w, v[u].w, acc[i].w);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < QN; ++i) {
        if (i > 0) {
            __syncthreads(); // the query before has been read
        }
        const int part = wave * kGroups + group;
        *reinterpret_cast<float4*>(&values[part][depth]) = acc[i];
        if (depth == 0) {
            top_of[part] = top[i];
            sum_of[part] = sum[i];
        }
        __syncthreads();
        if (i < p.lq && static_cast<int>(threadIdx.x) < d) {
            float most = -INFINITY;
#pragma unroll
            for (int g = 0; g < kParts; ++g) {
                most = fmaxf(most, top_of[g]);
            }
            float total = 0.0f, value = 0.0f;
#pragma unroll
            for (int g = 0; g < kParts; ++g) {
                const float w = part_weight(top_of[g], most);
                total = fmaf(w, sum_of[g], total);
                value = fmaf(w, values[g][threadIdx.x], value);
            }
            if (ranges == 1) {
                const float inv = total == 0.0f ? 0.0f : 1.0f / total;
                p.out[off_o + i * p.out_rs + threadIdx.x] = value * inv;
            } else {
                float* to = parts + ((static_cast<int64_t>(entry) * p.lq + i) * ranges + index) *
                                        (d + 2);
                to[2 + threadIdx.x] = value;
                if (threadIdx.x == 0) {
                    to[0] = most;
                    to[1] = total;
                }
            }
        }
    }
}

// Joins the ranges of one query (blockIdx.x = entry * lq + query), thread = depth.
__global__ __launch_bounds__(128) void attention_join_kernel(AttnParams p, int d, int ranges,
                                                             const float* parts) {
    const uint32_t lq = static_cast<uint32_t>(p.lq);
    const uint32_t entry = blockIdx.x / lq;
    const uint32_t query = blockIdx.x - entry * lq;
    int64_t off_o = 0;
    uint32_t rest = entry;
    for (int b = p.batch_dims - 1; b >= 0; --b) {
        const uint32_t extent = static_cast<uint32_t>(p.batch[b]);
        off_o += static_cast<int64_t>(rest % extent) * p.out_bs[b];
        rest /= extent;
    }
    if (static_cast<int>(threadIdx.x) >= d) {
        return;
    }
    const float* from = parts + static_cast<int64_t>(blockIdx.x) * ranges * (d + 2);
    float most = -INFINITY;
    for (int r = 0; r < ranges; ++r) {
        most = fmaxf(most, from[r * (d + 2)]);
    }
    float total = 0.0f, value = 0.0f;
#pragma unroll 8
    for (int r = 0; r < ranges; ++r) {
        const float* part = from + r * (d + 2);
        const float w = part_weight(part[0], most);
        total = fmaf(w, part[1], total);
        value = fmaf(w, part[2 + threadIdx.x], value);
    }
    const float inv = total == 0.0f ? 0.0f : 1.0f / total;
    p.out[off_o + query * p.out_rs + threadIdx.x] = value * inv;
}

template <int G>
void launch_queries(const AttnParams& p, int d, int ranges, int64_t range, float* parts,
                    unsigned grid, hipStream_t stream) {
    if (p.lq == 1) {
        attention_decode_kernel<G, 1><<<grid, kWaves * 64, 0, stream>>>(p, d, ranges, range, parts);
    } else if (p.lq == 2) {
        attention_decode_kernel<G, 2><<<grid, kWaves * 64, 0, stream>>>(p, d, ranges, range, parts);
    } else {
        attention_decode_kernel<G, 4><<<grid, kWaves * 64, 0, stream>>>(p, d, ranges, range, parts);
    }
}

} // namespace

namespace mfr::attn {

void run_decode(mfr_stream& s, const AttnParams& p, int64_t d) {
    static_assert(kDecodeMaxQueries == 4, "launch_queries covers every count");
    // Ranges of at least 256 keys, for about 4 workgroups per CU; one range needs no workspace.
    constexpr int64_t kLeastKeys = 256;
    constexpr int64_t kMostRanges = 64;
    const int64_t wanted = (4 * static_cast<int64_t>(s.compute_units) + p.batch_count - 1) /
                           p.batch_count;
    int64_t ranges = std::min({wanted, (p.lk + kLeastKeys - 1) / kLeastKeys, kMostRanges});
    int64_t range = (p.lk + ranges - 1) / ranges;
    ranges = (p.lk + range - 1) / range;
    std::unique_lock<std::mutex> hold(s.workspace_mutex, std::defer_lock);
    float* parts = nullptr;
    if (ranges > 1) {
        // Held until both kernels are queued: another thread's reserve() may not free `parts`.
        hold.lock();
        const size_t bytes =
            static_cast<size_t>(p.batch_count * p.lq * ranges * (d + 2)) * sizeof(float);
        // Under stream capture one range: a graph would keep the workspace's address, which a later
        // call may free to grow it, and its replays may run beside calls that use it.
        // (The default stream cannot be asked while another captures: one range then, too.)
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(s.stream, &capture) != hipSuccess) {
            (void)hipGetLastError();
        } else if (capture == hipStreamCaptureStatusNone) {
            try {
                parts = static_cast<float*>(s.reserve(bytes));
            } catch (const mfr::Error&) {
                (void)hipGetLastError(); // without the memory: one range
            }
        }
        if (parts == nullptr) {
            ranges = 1;
            range = p.lk;
        }
    }
    const int64_t blocks = p.batch_count * ranges;
    mfr::require(mfr::one_launch(blocks, kWaves * 64) &&
                     (ranges == 1 || mfr::one_launch(p.batch_count * p.lq, 128)),
                 "attention: problem too large for one launch");
    const unsigned grid = static_cast<unsigned>(blocks);
    const int depth = static_cast<int>(d);
    const int count = static_cast<int>(ranges);
    if (d <= 16) {
        launch_queries<4>(p, depth, count, range, parts, grid, s.stream);
    } else if (d <= 32) {
        launch_queries<8>(p, depth, count, range, parts, grid, s.stream);
    } else if (d <= 64) {
        launch_queries<16>(p, depth, count, range, parts, grid, s.stream);
    } else {
        launch_queries<32>(p, depth, count, range, parts, grid, s.stream);
    }
    mfr::check_launch("attention_decode_kernel");
    if (ranges > 1) {
        attention_join_kernel<<<static_cast<unsigned>(p.batch_count * p.lq), 128, 0, s.stream>>>(
            p, depth, count, parts);
        mfr::check_launch("attention_join_kernel");
    }
}

} // namespace mfr::attn
