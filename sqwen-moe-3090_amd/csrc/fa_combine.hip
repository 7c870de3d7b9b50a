// fa_combine.hip - merges the split-KV partials of the decode and prefill
// attention kernels: out = sum_s acc_s e^(m_s - M) / sum_s l_s e^(m_s - M), with
// M = max_s m_s (the log-sum-exp rule), optionally times sigmoid(gate) (the
// output gate of src/model/attn.rs:282-283 in the reference). The weights
// e^(m_s - M) <= 1 come from the hardware exp2 (about 1 ulp; a weight below
// 2^-126, negligible beside the largest one of 1, may read as 0). Partials:
// acc [n_splits][rows][256] unnormalised, ml [n_splits][rows][2] = (m, l) with m
// in natural-log units of the scaled logits.
#include "common.hpp"

namespace sqa {
namespace {

constexpr float kLog2e = 1.4426950408889634f;

// x of lane ^ 16 and of lane ^ 32 through gfx950's row swaps (VALU, no LDS
// round trip): a swap of x with itself leaves x in one result and the
// partner's x in the other
__device__ __forceinline__ float lane_xor16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float((threadIdx.x & 16) ? r[0] : r[1]);
}
__device__ __forceinline__ float lane_xor32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float((threadIdx.x & 32) ? r[0] : r[1]);
}

// Merge of up to kMaxSplits (256) split partials with one memory latency on the
// path. Grid: (rows, 16 chunks of 16 dims); 256 threads = 16 dims x 16 split
// groups. Each thread issues the loads of its 16 splits' acc values and (m, l)
// pairs at once; the maximum, the weights and the sums then follow from
// registers, with cross-lane reductions inside a wavefront and one LDS exchange
// per quantity across the 4 wavefronts.
static_assert(kMaxSplits == 256, "16 split groups x 16 splits per thread");
__global__ __launch_bounds__(256) void fa_combine_kernel(const float *__restrict__ part_acc,
                                                              const float *__restrict__ part_ml,
                                                              int n_splits, int rows_total,
                                                              float *__restrict__ dst, const char *gate,
                                                              int64_t gate_nb1, int64_t gate_nb2, int H) {
    __shared__ float xm[4], xo[4][16], xl[4];
    const int row = blockIdx.x;
    const int tid = threadIdx.x;
    const int dl = tid & 15, sg = tid >> 4, wv = tid >> 6;
    const int d = blockIdx.y * 16 + dl;
    const int64_t sstride = (int64_t)rows_total * 256;
    const float *pa = part_acc + (int64_t)row * 256 + d;
    const float2 *pm = reinterpret_cast<const float2 *>(part_ml) + row;
    float acc[16];
    float2 ml[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int sp = sg + 16 * j;
        const bool ok = sp < n_splits;
        acc[j] = ok ? pa[sp * sstride] : 0.0f;
        ml[j] = ok ? pm[(int64_t)sp * rows_total] : make_float2(-INFINITY, 0.0f);
    }
    // M: maximum over all splits (lanes 16 apart hold other split groups)
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < 16; ++j) m = fmaxf(m, ml[j].x);
    m = fmaxf(m, lane_xor16(m));
    m = fmaxf(m, lane_xor32(m));
    if ((tid & 63) == 0) xm[wv] = m;
    __syncthreads();
    const float M = fmaxf(fmaxf(xm[0], xm[1]), fmaxf(xm[2], xm[3]));
    float o = 0.0f, l = 0.0f;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        // a prefill split in which the row sees no key (m = -inf) has left its acc
        // unwritten: whatever the workspace holds there (0 * NaN) must not enter
        const bool dead = ml[j].x == -INFINITY;
        const float w = dead ? 0.0f : __builtin_amdgcn_exp2f((ml[j].x - M) * kLog2e);
        o = dead ? o : fmaf(acc[j], w, o);
        l = fmaf(ml[j].y, w, l);
    }
    o += lane_xor16(o);
    o += lane_xor32(o);
    l += lane_xor16(l);
    l += lane_xor32(l);
    if ((tid & 63) < 16) xo[wv][dl] = o;
    if ((tid & 63) == 0) xl[wv] = l;
    __syncthreads();
    if (tid < 16) {
        const float ot = (xo[0][dl] + xo[1][dl]) + (xo[2][dl] + xo[3][dl]);
        const float L = (xl[0] + xl[1]) + (xl[2] + xl[3]);
        float r = (L == 0.0f) ? 0.0f : ot * (1.0f / L);
        if (gate) {
            const int t = row / H, h = row % H;
            const float gv = reinterpret_cast<const float *>(gate + t * gate_nb2 + h * gate_nb1)[d];
            r = r * (1.0f / (1.0f + expf(-gv)));
        }
        dst[(int64_t)row * 256 + d] = r;
    }
}

// The same merge for many rows (prefill): WPR wavefronts per row, a float4 of
// the row per lane. Lane s first reads the (m, l) pair of split s (one load per
// 64 splits), takes the row's maximum and its split's weight; the partials are
// then read kBatch splits at a time, only those of nonzero weight: a split in
// which the row sees no key (m = -inf) has left its acc unwritten. With WPR = 4
// wavefront w takes splits w, w + 4, ... and the four sums meet in LDS.
// Bound by the partials' bytes, its launch and two memory latencies. 592 rows x
// 40 splits (24 MB): 16.8 us in the kernel above (16 blocks per row, 64 bytes of
// a partial at a time), 7.4 us here at 42 splits; 8192 rows x 4 splits (33 MB):
// 8.0 us with every thread walking the splits' pairs by itself, 8.4 us here.
constexpr int kBatch = 4;
constexpr int kRowsMin = 256;
constexpr int kRowsOneWaveSplits = 8;
template <int WPR>
__global__ __launch_bounds__(256) void fa_combine_rows_kernel(const float *__restrict__ part_acc,
                                                              const float *__restrict__ part_ml,
                                                              int n_splits, int rows_total,
                                                              float *__restrict__ dst, const char *gate,
                                                              int64_t gate_nb1, int64_t gate_nb2, int H) {
    constexpr int kW = kMaxSplits / 64;  // splits per lane
    __shared__ float4 xo[WPR > 1 ? 4 : 1][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = threadIdx.x & 63;
    const int row = WPR > 1 ? (int)blockIdx.x : (int)blockIdx.x * 4 + wave;
    if (row >= rows_total) return;  // whole wavefronts; with WPR > 1 the grid is rows_total
    const float2 *pm = reinterpret_cast<const float2 *>(part_ml) + row;
    const int n_w = (n_splits + 63) >> 6;
    const int64_t sstride = (int64_t)rows_total * 256;
    const float *pa = part_acc + (int64_t)row * 256 + 4 * c;
    // the first batch is on its way before the weights are known (what an
    // unwritten partial holds is never used: its weight is 0)
    float4 a[kBatch];
    const int w0 = WPR > 1 ? wave : 0;
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
        const int sp = w0 + WPR * j;
        a[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (sp < n_splits) a[j] = *reinterpret_cast<const float4 *>(pa + sp * sstride);
    }
    float2 ml[kW];
    float M = -INFINITY;
#pragma unroll
    for (int k = 0; k < kW; ++k) {
        const int sp = 64 * k + c;
        ml[k] = k < n_w && sp < n_splits ? pm[(int64_t)sp * rows_total] : make_float2(-INFINITY, 0.0f);
        M = fmaxf(M, ml[k].x);
    }
#pragma unroll
    for (int o = 1; o <= 8; o <<= 1) M = fmaxf(M, __shfl_xor(M, o));
    M = fmaxf(M, lane_xor16(M));
    M = fmaxf(M, lane_xor32(M));
    float w[kW], L = 0.0f;
#pragma unroll
    for (int k = 0; k < kW; ++k) {
        w[k] = ml[k].x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((ml[k].x - M) * kLog2e);
        L = fmaf(ml[k].y, w[k], L);
    }
#pragma unroll
    for (int o = 1; o <= 8; o <<= 1) L += __shfl_xor(L, o);
    L += lane_xor16(L);
    L += lane_xor32(L);
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < kW; ++k) {
        if (k >= n_w) break;
        const int end = n_splits - 64 * k < 64 ? n_splits - 64 * k : 64;
        for (int s0 = w0; s0 < end; s0 += WPR * kBatch) {
            float wt[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int sp = s0 + WPR * j;
                wt[j] = sp < end ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w[k]), sp)) : 0.0f;
                if (64 * k + s0 != w0 && wt[j] != 0.0f)
                    a[j] = *reinterpret_cast<const float4 *>(pa + (64 * k + sp) * sstride);
            }
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                if (wt[j] == 0.0f) continue;
                o.x = fmaf(a[j].x, wt[j], o.x);
                o.y = fmaf(a[j].y, wt[j], o.y);
                o.z = fmaf(a[j].z, wt[j], o.z);
                o.w = fmaf(a[j].w, wt[j], o.w);
            }
        }
    }
    if (WPR > 1) {
        xo[wave][c] = o;
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int j = 1; j < 4; ++j) {
            const float4 a = xo[j][c];
            o.x += a.x, o.y += a.y, o.z += a.z, o.w += a.w;
        }
    }
    const float inv = L == 0.0f ? 0.0f : 1.0f / L;
    float r[4] = {o.x * inv, o.y * inv, o.z * inv, o.w * inv};
    if (gate) {
        const int t = row / H, h = row % H;
        const float *gp = reinterpret_cast<const float *>(gate + t * gate_nb2 + h * gate_nb1) + 4 * c;
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = r[j] * (1.0f / (1.0f + expf(-gp[j])));
    }
    *reinterpret_cast<float4 *>(dst + (int64_t)row * 256 + 4 * c) = make_float4(r[0], r[1], r[2], r[3]);
}

}  // namespace

int launch_fa_combine(const float *part_acc, const float *part_ml, int n_splits, int rows_total,
                      float *dst, const sqa_tensor *gate, int H, hipStream_t s) {
    const char *g = gate ? (const char *)gate->data : nullptr;
    const int64_t g1 = gate ? (int64_t)gate->nb[1] : 0, g2 = gate ? (int64_t)gate->nb[2] : 0;
    if (n_splits > kMaxSplits)
        return set_error(SQA_ERR_UNSUPPORTED, "fa_combine: %d splits > %d", n_splits, kMaxSplits);
    const int prof = profile_start("fa_combine", s);
    // Few rows (decode, verify, the smallest chunks) need the 16 blocks per row of
    // the first kernel to fill the chip; from kRowsMin rows on, one block or a
    // quarter of one per row does, and reads 1 KB of a partial at a time.
    if (rows_total >= kRowsMin && n_splits <= kRowsOneWaveSplits) {
        fa_combine_rows_kernel<1><<<dim3((unsigned)((rows_total + 3) / 4)), dim3(256), 0, s>>>(
            part_acc, part_ml, n_splits, rows_total, dst, g, g1, g2, H);
    } else if (rows_total >= kRowsMin) {
        fa_combine_rows_kernel<4><<<dim3((unsigned)rows_total), dim3(256), 0, s>>>(
            part_acc, part_ml, n_splits, rows_total, dst, g, g1, g2, H);
    } else {
        fa_combine_kernel<<<dim3((unsigned)rows_total, 16), dim3(256), 0, s>>>(part_acc, part_ml, n_splits,
                                                                            rows_total, dst, g, g1, g2, H);
    }
    profile_stop(prof, s);
    return hip_status(hipGetLastError(), "fa_combine launch");
}

}  // namespace sqa
