// out_proj.hip - the W_o projection that closes the full-attention layer:
//   dst = W . (x * sigmoid(gate))        (src/model/attn.rs:281-285 in the
// reference: ggml_sigmoid + ggml_mul, then ggml_mul_mat(attn_output, gated))
// with W = attn_output.weight in ggml's Q4_K format, ne = [K, N] (K = n_head *
// head_dim = 4096 here, N = n_embd), x and gate F32 [K, M] (M tokens), dst F32
// [N, M].
//
// Q4_K super-block (256 values, 144 bytes): fp16 d and dmin, twelve bytes of
// 6-bit (scale, min) pairs for the 8 sub-blocks of 32, then 128 bytes of 4-bit
// codes (byte l of 32-byte group j: value 64j + l in the low nibble, value
// 64j + 32 + l in the high one). A value is d*scale*code - dmin*min.
//
// Up to 4 tokens (decode, verify) one kernel, op_gemv (below); more tokens two:
//   op_prep   xg = x * sigmoid(gate) in fp32, written as an fp16 hi + lo pair (xg
//             = hi + lo to ~22 bits) in the order of the MFMA's B operand, and
//             the sub-block sums S = sum xg as the B operand of the min term
//   op_gemm   16x16x32 f16 MFMAs over the raw codes: every product exact, then d
//             and dmin per super-block in fp32. Two forms by the amount of work:
//             op_gemm (K split over the wavefronts, no barrier) while one of its
//             tiles leaves a CU at most one workgroup, else op_gemm2 (operands
//             shared through LDS)
//
// MFMA operand layouts (lane = 16*g + n):
//   16x16x32 f16: A[n][8g..8g+7]   B[8g..8g+7][n]   C[4g..4g+3][n]
#include <mutex>

#include "common.hpp"

namespace sqa {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kQK = 256;           // values per Q4_K super-block
constexpr int kBlockBytes = 144;   // bytes per super-block
constexpr int kGemvTokens = 4;     // token counts up to this take op_gemv
constexpr int64_t kPrepPairs = 2048;  // 8 wavefronts per CU, see op_prep

__device__ __forceinline__ float h2f(uint32_t bits) {
    _Float16 h;
    const uint16_t b = (uint16_t)bits;
    __builtin_memcpy(&h, &b, 2);
    return (float)h;
}

// ---------------------------------------------------------------- op_prep
// One wavefront per 16 tokens and SUBS 32-value sub-blocks of K (1, or a pair): lane
// 16q + n takes values 8q .. 8q + 7 of token n and writes xg = x * sigmoid(gate) as
// fp16 hi and lo in the order in which op_gemm reads them, 1 KB per load. Its time is
// one chain of load, exp and store while there are few wavefronts: one sub-block
// each then (us per call of the whole projection, pairs / this: 33 tokens, N = 5120,
// K = 2048 17.3 / 14.6, 100, 8192, 2048 20.1 / 19.2, 300, 4096, 4096 46.6 / 46.0), and
// its stores from kPrepPairs pairs on (512, 2048, 4096 32.3 / 32.5, 2048 of them 105.8 /
// 106.1).
// B operand (c, e) of super-block s, c < 4, e < 2, holds in lane 16g + n
// the values 64g + 32e + 8c .. + 7 of token n: an MFMA then takes from each lane
// group another code group (64 values, 32 bytes of a weight row), so a lane needs
// 32 consecutive weight bytes and two of the 8 scales. hi and lo of tile T at
// ((T * K/256 + s) * 8 + 2c + e) * 2 KB. The sub-block sums S go out as three bf16
// parts each (24 bits, fp32's range): the B operand of the min MFMA of
// super-block s, 1 KB at (T * K/256 + s), where lane 16g + n holds S of sub-blocks
// 2g, 2g + 1 as {s0, s1} of part 0, of part 1, of part 2, and two zeros. Tokens
// M.. of the last tile are zeros. x (and gate) rows are 16-byte aligned when VEC.
__device__ __forceinline__ float xsum16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float xsum32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <bool GATE, bool VEC, int SUBS>
__global__ __launch_bounds__(256) void op_prep_kernel(const char *__restrict__ x, int64_t x_nb1,
                                                      const char *__restrict__ gate, int64_t g_nb1, int K, int M,
                                                      int tiles, uint4 *__restrict__ xb, uint16_t *__restrict__ sb) {
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const int subs = K / 32, per = subs / SUBS;
    const int64_t wid = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wid >= (int64_t)tiles * per) return;
    const int T = (int)(wid / per), sub0 = (int)(wid - (int64_t)T * per) * SUBS;
    const int pr = sub0 >> 1;  // sub-block pair (64 values)
    const int t = 16 * T + n;
    uint32_t sw[SUBS][3];  // the three parts of S
#pragma unroll
    for (int u = 0; u < SUBS; ++u) {
        const int sub = sub0 + u;
        float v[8], gv[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = gv[j] = 0.0f;
        if (t < M) {
            const float *xr = reinterpret_cast<const float *>(x + t * x_nb1) + 32 * sub + 8 * g;
            const float *gr = GATE ? reinterpret_cast<const float *>(gate + t * g_nb1) + 32 * sub + 8 * g : nullptr;
            if (VEC) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const float4 a = reinterpret_cast<const float4 *>(xr)[c];
                    v[4 * c] = a.x, v[4 * c + 1] = a.y, v[4 * c + 2] = a.z, v[4 * c + 3] = a.w;
                    if (GATE) {
                        const float4 b = reinterpret_cast<const float4 *>(gr)[c];
                        gv[4 * c] = b.x, gv[4 * c + 1] = b.y, gv[4 * c + 2] = b.z, gv[4 * c + 3] = b.w;
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    v[j] = xr[j];
                    if (GATE) gv[j] = gr[j];
                }
            }
            if (GATE) {
#pragma unroll
                for (int j = 0; j < 8; ++j) v[j] = v[j] * (1.0f / (1.0f + expf(-gv[j])));
            }
        }
        float sum = 0.0f;
        uint16_t hb[8], lb[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            sum += v[j];
            float a = v[j];
            // opaque: one fp32 value feeds both the stored hi and the hi subtracted for lo
            asm volatile("" : "+v"(a));
            const _Float16 h = (_Float16)a;
            const _Float16 l = (_Float16)(a - (float)h);
            __builtin_memcpy(&hb[j], &h, 2);
            __builtin_memcpy(&lb[j], &l, 2);
        }
        uint4 a, b;
        __builtin_memcpy(&a, hb, 16);
        __builtin_memcpy(&b, lb, 16);
        uint4 *o = xb + ((int64_t)T * subs + 8 * (pr >> 2) + 2 * g + (sub & 1)) * 128 + 16 * (pr & 3) + n;
        o[0] = a;
        o[64] = b;
        // S = its leading 8 bits (truncated) + those of the rest, twice: each
        // difference is exact
        float r = xsum32(xsum16(sum));
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const uint32_t top = __float_as_uint(r) & 0xFFFF0000u;
            sw[u][c] = top >> 16;
            r -= __uint_as_float(top);
        }
    }
    if (g == (pr & 3)) {
        uint16_t *s = sb + (((int64_t)T * (subs / 8) + (pr >> 2)) * 64 + lane) * 8;
        if constexpr (SUBS == 2) {
            *reinterpret_cast<uint4 *>(s) =
                make_uint4(sw[0][0] | (sw[1][0] << 16), sw[0][1] | (sw[1][1] << 16), sw[0][2] | (sw[1][2] << 16), 0u);
        } else {
            s += sub0 & 1;
#pragma unroll
            for (int c = 0; c < 3; ++c) s[2 * c] = (uint16_t)sw[0][c];
            s[6] = 0;
        }
    }
}

// ---------------------------------------------------------------- op_gemm
// What a lane (g, n) keeps of the super-block header of row n: scales and mins of
// sub-blocks 2g and 2g + 1 (ggml's get_scale_min_k4, branch-free: sub-blocks 0-3
// have 6 bits in bytes s and s + 4 of the 12, 4-7 four bits in byte s + 4 and two
// on top of bytes s - 4 and s), and d | dmin of the row.
struct OpHead {
    uint32_t sc0, sc1, mins, d;
};
__device__ __forceinline__ OpHead op_head(uint4 hd, int g) {
    const uint32_t sh = 16u * (uint32_t)(g & 1);
    const uint32_t q0 = hd.y >> sh, q1 = hd.z >> sh, q2 = hd.w >> sh;  // bytes of 2g, 2g + 1 (mod 4)
    const bool top = g >= 2;
    const uint32_t sc = top ? (q2 & 0x0F0Fu) | ((q0 >> 2) & 0x3030u) : q0 & 0x3F3Fu;
    const uint32_t mn = top ? ((q2 >> 4) & 0x0F0Fu) | ((q1 >> 2) & 0x3030u) : q1 & 0x3F3Fu;
    OpHead h;
    h.sc0 = sc & 0xFFu;
    h.sc1 = sc >> 8;
    // bf16 of the integers: their fp32 bits end in zeros
    h.mins = (__float_as_uint((float)(mn & 0xFFu)) >> 16) | (__float_as_uint((float)(mn >> 8)) & 0xFFFF0000u);
    h.d = hd.x;
    return h;
}

// A operands of a step: 8 code bytes, low nibbles (sub-block 2g) and high (2g + 1)
// as code * scale * 2^-24 (see op_gemm)
__device__ __forceinline__ void op_a_operand(const OpHead &h, uint32_t qx, uint32_t qy, half8 &alo, half8 &ahi) {
    uint32_t sp[4];  // bytes 2m, 2m+1 spread to the two halves of dword m
    sp[0] = __builtin_amdgcn_perm(0u, qx, 0x0c010c00u);
    sp[1] = __builtin_amdgcn_perm(0u, qx, 0x0c030c02u);
    sp[2] = __builtin_amdgcn_perm(0u, qy, 0x0c010c00u);
    sp[3] = __builtin_amdgcn_perm(0u, qy, 0x0c030c02u);
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        lo[m] = __umul24(sp[m] & 0x000F000Fu, h.sc0);
        hi[m] = __umul24((sp[m] >> 4) & 0x000F000Fu, h.sc1);
    }
    __builtin_memcpy(&alo, lo, 16);
    __builtin_memcpy(&ahi, hi, 16);
}

// acc += d 2^24 C - dmin * (mins . S) of one super-block and row tile
template <int TT>
__device__ __forceinline__ void op_scale_add(const OpHead &h, int g, const floatx4 (&C)[TT], const uint4 (&sv)[TT],
                                             floatx4 (&acc)[TT]) {
    const uint32_t aw[4] = {h.mins, h.mins, h.mins, 0u};
    bf16x8 am;
    __builtin_memcpy(&am, aw, 16);
    float d[4], dm[4];  // d 2^24 and dmin of C rows 4g..4g+3
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = (uint32_t)__shfl((int)h.d, 4 * g + i);
        d[i] = h2f(w & 0xffffu) * 16777216.0f;
        dm[i] = h2f(w >> 16);
    }
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        bf16x8 bm;
        __builtin_memcpy(&bm, &sv[tt], 16);
        const floatx4 cm = __builtin_amdgcn_mfma_f32_16x16x32_bf16(am, bm, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[tt][i] = fmaf(-dm[i], cm[i], fmaf(d[i], C[tt][i], acc[tt][i]));
    }
}

struct GemmParams {
    const uint8_t *w;
    int64_t w_nb1;
    const uint4 *xb, *sb;  // B operands, see op_prep
    int K, N, M, tiles;    // tiles of 16 tokens
    int row_blocks, token_groups;  // workgroups along N, along the tokens
    bool rows_first;       // order of the workgroups, see place_of
    float *dst;
    int64_t d_nb1;
};

// Workgroups go round-robin to the 8 XCDs: the row block and token group of
// workgroup lin such that each XCD takes a contiguous run of them, either of token
// groups (every row block of them: its L2 then serves their operands to all row
// blocks, and all XCDs read all weights) or, with rows_first, of row blocks.
struct Place {
    int row_block, token_group;
};
__device__ __forceinline__ Place place_of(const GemmParams &p) {
    const int lin = (int)blockIdx.x, nb = (int)gridDim.x;
    const int x = lin & 7, per = nb >> 3, rem = nb & 7;
    const int id = x * per + (x < rem ? x : rem) + (lin >> 3);
    return p.rows_first ? Place{id / p.token_groups, id % p.token_groups} : Place{id % p.row_blocks, id / p.row_blocks};
}

// A workgroup of KS wavefronts owns 16 RT rows of W and 16 TT tokens; wavefront w
// takes super-blocks w, w + KS, ... of K, reading weights and operands straight
// from memory (no barrier in the loop), and the KS partial sums meet in LDS.
//   * The A operand is code * scale of the code's sub-block as an fp16 subnormal: an
//     integer of at most 15 * 63 = 945, i.e. exactly code * scale * 2^-24 (one
//     v_mul_u32_u24 scales the two codes of a dword, as the halves cannot carry
//     into each other). The super-block accumulates into one MFMA chain C = 2^-24
//     sum_k scale * code * x against x hi and lo, and acc += d 2^24 C once per
//     super-block.
//   * The min term is one bf16 MFMA per super-block: A = the mins (integers up to
//     63, exact) of sub-blocks 2g, 2g + 1 three times over, B = the three parts
//     of their S; acc -= dmin * its sum.
// What bounds it is traffic into the CUs, (N / 16 RT) * M * K * 4 bytes of
// operands at 64 bytes a clock and CU, and the VALU that builds A, paid once per
// TT token tiles.
template <int KS, int RT, int TT>
__global__ __launch_bounds__(64 * KS) void op_gemm_kernel(GemmParams p) {
    __shared__ float red[KS][RT * TT][4][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const Place at = place_of(p);
    const int r0 = at.row_block * 16 * RT;
    const int T0 = at.token_group * TT;
    const int nsb = p.K / kQK;

    floatx4 acc[RT][TT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) acc[rt][tt] = floatx4{0.f, 0.f, 0.f, 0.f};
    const uint8_t *wrow[RT];  // rows past N read the last one and are never stored
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int r = r0 + 16 * rt + n;
        wrow[rt] = p.w + (int64_t)(r < p.N ? r : p.N - 1) * p.w_nb1;
    }
    const uint4 *xt[TT], *st[TT];  // token tiles past the last one read it and are never stored
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        const int T = T0 + tt < p.tiles ? T0 + tt : p.tiles - 1;
        xt[tt] = p.xb + (int64_t)T * (p.K / 32) * 128 + lane;
        st[tt] = p.sb + (int64_t)T * nsb * 64 + lane;
    }

    for (int s = wave; s < nsb; s += KS) {
        OpHead hd[RT];
        uint4 q[RT][2];  // code group g: 8 bytes per step
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const uint8_t *blk = wrow[rt] + (int64_t)s * kBlockBytes;
            hd[rt] = op_head(*reinterpret_cast<const uint4 *>(blk), g);
#pragma unroll
            for (int k = 0; k < 2; ++k) q[rt][k] = *reinterpret_cast<const uint4 *>(blk + 16 + 32 * g + 16 * k);
        }
        uint4 sv[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) sv[tt] = st[tt][(int64_t)s * 64];
        floatx4 C[RT][TT];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) C[rt][tt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            half8 b[TT][4];  // operands (j, 0) hi, lo, (j, 1) hi, lo
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const uint4 v = xt[tt][((int64_t)s * 8 + 2 * j) * 128 + 64 * c];
                    __builtin_memcpy(&b[tt][c], &v, 16);
                }
            half8 a[RT][2];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const uint4 w = q[rt][j >> 1];
                op_a_operand(hd[rt], j & 1 ? w.z : w.x, j & 1 ? w.w : w.y, a[rt][0], a[rt][1]);
            }
            // the four MFMAs of a C tile apart: each waits for the one before
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt)
                        C[rt][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[rt][c >> 1], b[tt][c], C[rt][tt], 0, 0, 0);
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) op_scale_add<TT>(hd[rt], g, C[rt], sv, acc[rt]);
    }

    // ---- the KS partial sums through LDS; wavefront w finishes tiles w, w + KS, ...
    if (KS > 1) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int i = 0; i < 4; ++i) red[wave][rt * TT + tt][i][lane] = acc[rt][tt][i];
        __syncthreads();
    }
#pragma unroll
    for (int u0 = 0; u0 < RT * TT; u0 += KS) {
        const int u = u0 + wave;
        if (u >= RT * TT) break;
        const int r = r0 + 16 * (u / TT), t = 16 * (T0 + u % TT) + n;
        float o[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float a = 0.0f;
#pragma unroll
            for (int w = 0; w < KS; ++w) a += red[w][u][i][lane];
            o[i] = a;
        }
        if (r < p.N && t < p.M)
            *reinterpret_cast<float4 *>(reinterpret_cast<char *>(p.dst) + (int64_t)t * p.d_nb1 + 4 * (r + 4 * g)) =
                make_float4(o[0], o[1], o[2], o[3]);
    }
}

// ---------------------------------------------------------------- op_gemm2
// More tokens: a workgroup of 8 wavefronts owns 128 rows of W (wavefront w: rows
// 16w..16w+15) and 32 tokens; the arithmetic is op_gemm's. Everything comes HBM ->
// LDS by DMA, double buffered: the operands of half a super-block (two steps, 2
// tiles, hi and lo: 16 KB, shared by the eight wavefronts), the 128 weight rows'
// super-block (18 KB) and the S operands (2 KB). 512 tokens, N = 2048, K = 4096:
// 28 us; each wavefront reads every operand, 16 KB a half and wavefront, and
// those LDS reads (128 bytes a clock) cost more than the MFMAs they feed. Measured
// and slower: 64 tokens a workgroup (48 us with op_prep, 33 this form: half the
// CUs idle; equal from 1024 tokens), activations two halves ahead in three buffers
// (34, and 64 against 55 at 1024 tokens: one workgroup per CU), 64 rows (36 at
// 512), two row tiles per wavefront with the K halves on two sets of four
// wavefronts and the weights straight to registers (37: the wait for the weights).
constexpr int kG2Rows = 128;
constexpr int kG2Waves = kG2Rows / 16;            // 8: two wavefronts per SIMD
constexpr int kG2WBytes = kG2Rows * kBlockBytes;  // 18432
constexpr int kG2WInst = kG2WBytes / 1024;        // 18 DMA instructions
constexpr int kG2WPer = (kG2WInst + kG2Waves - 1) / kG2Waves;
constexpr int kG2TT = 2;                          // token tiles
constexpr int kG2Half = 4 * kG2TT * 2 * 1024;     // [step, nibble half][tile][hi, lo] of 1 KB
constexpr int kG2XInst = kG2Half / 1024 / kG2Waves;  // activation DMA instructions per wavefront
constexpr int kG2SBytes = kG2TT * 1024;
// 73728 bytes of dynamic LDS: two workgroups per CU
constexpr int kG2Lds = 2 * (kG2Half + kG2WBytes + kG2SBytes);
static_assert(kG2WBytes % 1024 == 0, "weight stage in whole DMA instructions");

// 16 bytes per lane from sbase + voff into LDS at m0 + 16 * lane, asynchronously
// (the caller waits with s_waitcnt vmcnt); sbase and m0 are wave-uniform.
__device__ __forceinline__ void dma16(uint32_t voff, const void *sbase, uint32_t m0v) {
    const uint64_t b = (uint64_t)(uintptr_t)sbase;
    const uint64_t bs = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(b >> 32)) << 32) |
                        (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    const uint32_t ms = (uint32_t)__builtin_amdgcn_readfirstlane((int)m0v);
    // m0 as an operand: the compiler writes it and knows it holds the LDS base
    asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(bs), "{m0}"(ms) : "memory");
}

__global__ __launch_bounds__(64 * kG2Waves) void op_gemm2_kernel(GemmParams p) {
    constexpr int TT = kG2TT;
    extern __shared__ __align__(16) uint8_t lds[];
    uint8_t(*xs)[kG2Half] = reinterpret_cast<uint8_t(*)[kG2Half]>(lds);
    uint8_t(*wb)[kG2WBytes] = reinterpret_cast<uint8_t(*)[kG2WBytes]>(lds + 2 * kG2Half);
    uint8_t(*ss)[kG2SBytes] = reinterpret_cast<uint8_t(*)[kG2SBytes]>(lds + 2 * (kG2Half + kG2WBytes));
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63, g = lane >> 4, n = lane & 15;
    const Place at = place_of(p);
    const int row0 = at.row_block * kG2Rows;
    const int T0 = at.token_group * TT;
    const int nsb = p.K / kQK;
    const uint32_t xs0 = (uint32_t)(uintptr_t)&xs[0][0], wb0 = (uint32_t)(uintptr_t)&wb[0][0];
    const uint32_t ss0 = (uint32_t)(uintptr_t)&ss[0][0];

    // ---- DMA plans (wave-uniform bases, per-lane offsets) ----
    // a token tile past the last one reads it and is never stored
    auto tile = [&](int tt) { return T0 + tt < p.tiles ? T0 + tt : p.tiles - 1; };
    // operand i = kG2XInst * wave + r of half h: sub-block, tile, hi or lo
    auto issue_x = [&](int h, int buf) {
#pragma unroll
        for (int r = 0; r < kG2XInst; ++r) {
            const int i = kG2XInst * wave + r;
            dma16(16u * lane, p.xb + ((int64_t)tile((i >> 1) % TT) * (8 * nsb) + 4 * h + (i >> 1) / TT) * 128 + 64 * (i & 1),
                  xs0 + (uint32_t)(buf * kG2Half + 1024 * i));
        }
    };
    // weights: chunk id = 64 * i + lane -> row id / 9, chunk id % 9 (rows past N
    // read the last one and are never stored)
    uint32_t wrow[kG2WPer], wch[kG2WPer];
#pragma unroll
    for (int r = 0; r < kG2WPer; ++r) {
        const int i = kG2Waves * r + wave;
        const int c = 64 * (i < kG2WInst ? i : 0) + lane, row = row0 + c / 9;
        wrow[r] = (uint32_t)((int64_t)((row < p.N ? row : p.N - 1) - row0) * p.w_nb1);
        wch[r] = 16u * (uint32_t)(c % 9);
    }
    const uint8_t *w0 = p.w + (int64_t)row0 * p.w_nb1;
    auto issue_w = [&](int sb, int buf) {
#pragma unroll
        for (int r = 0; r < kG2WPer; ++r) {
            const int i = kG2Waves * r + wave;
            if (i < kG2WInst)
                dma16(wrow[r] + wch[r], w0 + (int64_t)sb * kBlockBytes, wb0 + (uint32_t)(buf * kG2WBytes + 1024 * i));
        }
        if (wave < TT)
            dma16(16u * lane, p.sb + ((int64_t)tile(wave) * nsb + sb) * 64, ss0 + (uint32_t)(buf * kG2SBytes + 1024 * wave));
    };

    floatx4 acc[TT];
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) acc[tt] = floatx4{0.f, 0.f, 0.f, 0.f};
    issue_w(0, 0);
    issue_x(0, 0);
    for (int sb = 0; sb < nsb; ++sb) {
        const uint8_t *hrow = &wb[sb & 1][0] + (16 * wave + n) * kBlockBytes;
        OpHead hd;
        floatx4 C[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) C[tt] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            const int h = 2 * sb + hh;
            // this wavefront's DMAs have landed (those of half h were the last it
            // issued); the barrier publishes every wavefront's and retires the buffers
            // that the next DMAs overwrite
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (hh == 0 && sb + 1 < nsb) issue_w(sb + 1, (sb + 1) & 1);
            if (h + 1 < 2 * nsb) issue_x(h + 1, (h + 1) & 1);
            if (hh == 0) hd = op_head(*reinterpret_cast<const uint4 *>(hrow), g);
            const uint4 w = *reinterpret_cast<const uint4 *>(hrow + 16 + 32 * g + 16 * hh);
            const uint8_t *xb = &xs[h & 1][0] + 16 * lane;
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) {
                half8 a[2], b[TT][4];  // step 2 hh + jj
                op_a_operand(hd, jj ? w.z : w.x, jj ? w.w : w.y, a[0], a[1]);
#pragma unroll
                for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        b[tt][c] = *reinterpret_cast<const half8 *>(
                            xb + (((2 * jj + (c >> 1)) * TT + tt) * 2 + (c & 1)) * 1024);
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt)
                        C[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[c >> 1], b[tt][c], C[tt], 0, 0, 0);
            }
        }
        uint4 sv[TT];
#pragma unroll
        for (int tt = 0; tt < TT; ++tt)
            sv[tt] = *reinterpret_cast<const uint4 *>(&ss[sb & 1][0] + 1024 * tt + 16 * lane);
        op_scale_add<TT>(hd, g, C, sv, acc);
    }
    const int r = row0 + 16 * wave;
    if (r >= p.N) return;
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
        const int t = 16 * (T0 + tt) + n;
        if (t < p.M)
            *reinterpret_cast<float4 *>(reinterpret_cast<char *>(p.dst) + (int64_t)t * p.d_nb1 + 4 * (r + 4 * g)) =
                make_float4(acc[tt][0], acc[tt][1], acc[tt][2], acc[tt][3]);
    }
}

// ---------------------------------------------------------------- op_gemv
// Decode and verify (M <= 4 tokens, MT = 1, 2 or 4 slots): one workgroup of
// kGemvThreads threads takes kGemvRows rows of W. Thread t owns the 8
// activations k = 8t .. 8t + 7 (and the same slice of every further
// 8 * kGemvThreads values of K) for all of those rows, so it loads its slice of
// x and gate once and, for each row, the slice's 8 code bytes, all before it
// uses any of them: one memory latency, then arithmetic, then one reduction.
// The four threads of a lane quad share one 32-value sub-block: each loads and
// unpacks the super-block headers of two of the 8 rows, and the quad
// broadcasts the rows' scales.
//   Value 64j + 16h2 + i of a super-block sits in byte 32j + 16(h2 & 1) + i of
//   its codes, low nibble for h2 < 2, high for h2 >= 2; sub-block 2j + (h2 >> 1).
// Per row and token: out += d * scale * sum(code * xg) - dmin * min * sum(xg).
// The codes enter v_fma_mix as fp16 subnormals, two per v_and, against the
// fp32 activations, so every product is exact: a low nibble left in bits 0-3
// of an fp16 is code * 2^-24, a high nibble left in bits 4-7 is code * 2^-20,
// and the 2^24 or 2^20 goes into the scale. The gate's sigmoid is 1/(1 + 2^(-g
// log2 e)) from the hardware exp2 and reciprocal (about 2 ulp). The partial
// sums of the (row, token) pairs are added by recursive halving inside each
// wavefront (lane swaps and DPP moves, each lane ending with one pair's sum),
// then across the wavefronts through LDS. VEC: x (and gate) rows are 16-byte
// aligned and read four floats at a time.
// Lane K of each quad's x in all four lanes of the quad (quad_perm [K,K,K,K]).
template <int K>
__device__ __forceinline__ float quad_bcast(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), K * 0x55, 0xf, 0xf, false));
}

// One halving step of the GEMV's wavefront sum (below): values a[0 .. 2N) to
// a[0 .. N), the lane with `up` clear keeping the lower half, plus the
// partner's copy of the kept half moved by the DPP control CTRL.
template <int N, int CTRL>
__device__ __forceinline__ void halve_dpp(float *a, bool up) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const float keep = up ? a[N + j] : a[j];
        const float give = up ? a[j] : a[N + j];
        a[j] = keep + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(give), CTRL, 0xf, 0xf, false));
    }
}

constexpr int kGemvRows = 8;
constexpr int kGemvThreads = 512;
template <int MT, bool VEC>
__global__ __launch_bounds__(kGemvThreads) void op_gemv_kernel(const uint8_t *__restrict__ w, int64_t w_nb1,
                                                               const char *__restrict__ x, int64_t x_nb1,
                                                               const char *__restrict__ gate, int64_t g_nb1, int K,
                                                               int N, int M, float *__restrict__ dst, int64_t d_nb1) {
    constexpr int R = kGemvRows, W = kGemvThreads / 64;
    __shared__ float red[W][R * MT];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row0 = blockIdx.x * R;
    float acc[R][MT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = 0.0f;
    // x * code + acc, the code in the low (SEL 0) or high (SEL 1) fp16 half of c
#define SQA_MIX(ACC, X, C, SEL)                                                                           \
    asm("v_fma_mix_f32 %0, %1, %2, %0 op_sel:[0," #SEL ",0] op_sel_hi:[0,1,0]" : "+v"(ACC) : "v"(X), "v"(C))
    for (int k0 = 8 * tid; k0 < K; k0 += 8 * kGemvThreads) {
        const int sb = k0 >> 8, v = k0 & 255, j = v >> 6, h2 = (v >> 4) & 3;
        const bool hi_nib = h2 >= 2;
        const uint32_t nib = hi_nib ? 0x00F000F0u : 0x000F000Fu;  // codes of bytes 0, 2 of a dword
        const float cscale = hi_nib ? 1048576.0f : 16777216.0f;     // 2^20 or 2^24
        const int s = 2 * j + (h2 >> 1);                            // sub-block
        const int cb = 16 + 32 * j + 16 * (h2 & 1) + (v & 8);       // the slice's first code byte
        // weights first (8 code bytes of every row; the super-block headers of
        // rows 2 qd and 2 qd + 1 only, see below), then the activations
        const int qd = lane & 3;  // the lane quad shares one sub-block (32 values)
        uint4 hdr[2];
        uint2 q[R];
#pragma unroll
        for (int u = 0; u < 2; ++u)
            hdr[u] = *reinterpret_cast<const uint4 *>(w + (int64_t)(row0 + 2 * qd + u) * w_nb1 +
                                                      (int64_t)sb * kBlockBytes);
#pragma unroll
        for (int r = 0; r < R; ++r)
            q[r] = *reinterpret_cast<const uint2 *>(w + (int64_t)(row0 + r) * w_nb1 + (int64_t)sb * kBlockBytes + cb);
        float xg[MT][8];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const bool ok = t < M;
            const float *xr = reinterpret_cast<const float *>(x + (ok ? t : 0) * x_nb1) + k0;
            const float *gr = gate ? reinterpret_cast<const float *>(gate + (ok ? t : 0) * g_nb1) + k0 : nullptr;
            float gv[8];
            if (VEC) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const float4 a = reinterpret_cast<const float4 *>(xr)[c];
                    xg[t][4 * c] = a.x, xg[t][4 * c + 1] = a.y, xg[t][4 * c + 2] = a.z, xg[t][4 * c + 3] = a.w;
                    if (gr) {
                        const float4 b = reinterpret_cast<const float4 *>(gr)[c];
                        gv[4 * c] = b.x, gv[4 * c + 1] = b.y, gv[4 * c + 2] = b.z, gv[4 * c + 3] = b.w;
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    xg[t][i] = xr[i];
                    if (gr) gv[i] = gr[i];
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (gr)
                    xg[t][i] *= __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * gv[i]));
                xg[t][i] = ok ? xg[t][i] : 0.0f;
            }
        }
        // d * scale * 2^24 (or 2^20) and dmin * min of sub-block s for the 8 rows:
        // the four lanes of a quad share s, so lane qd unpacks rows 2 qd and
        // 2 qd + 1 (ggml's get_scale_min_k4, branch-free) and the quad
        // broadcasts them (quad_perm [k,k,k,k])
        float dsu[2], dmu[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t q0 = hdr[u].y, q1 = hdr[u].z, q2 = hdr[u].w;
            const uint32_t lo_sh = 8u * (uint32_t)(s & 3);
            const uint32_t sc_lo = (q0 >> lo_sh) & 63u, mn_lo = (q1 >> lo_sh) & 63u;
            const uint32_t sc_hi = ((q2 >> lo_sh) & 15u) | (((q0 >> (lo_sh + 6u)) & 3u) << 4);
            const uint32_t mn_hi = ((q2 >> (lo_sh + 4u)) & 15u) | (((q1 >> (lo_sh + 6u)) & 3u) << 4);
            const uint32_t sc = s < 4 ? sc_lo : sc_hi, mn = s < 4 ? mn_lo : mn_hi;
            dsu[u] = h2f(hdr[u].x & 0xffffu) * (float)sc * cscale;
            dmu[u] = h2f(hdr[u].x >> 16) * (float)mn;
        }
        float ds[R], dm[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int k = r >> 1;
            ds[r] = k == 0 ? quad_bcast<0>(dsu[r & 1]) : k == 1 ? quad_bcast<1>(dsu[r & 1])
                  : k == 2 ? quad_bcast<2>(dsu[r & 1]) : quad_bcast<3>(dsu[r & 1]);
            dm[r] = k == 0 ? quad_bcast<0>(dmu[r & 1]) : k == 1 ? quad_bcast<1>(dmu[r & 1])
                  : k == 2 ? quad_bcast<2>(dmu[r & 1]) : quad_bcast<3>(dmu[r & 1]);
        }
        float sx[MT];  // sum of this slice's activations (the min term)
#pragma unroll
        for (int t = 0; t < MT; ++t)
            sx[t] = ((xg[t][0] + xg[t][1]) + (xg[t][2] + xg[t][3])) + ((xg[t][4] + xg[t][5]) + (xg[t][6] + xg[t][7]));
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const uint32_t qw[2] = {q[r].x, q[r].y};
            float dot[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) dot[t] = 0.0f;
#pragma unroll
            for (int m = 0; m < 2; ++m) {  // bytes 4m .. 4m+3 of the slice: values 4m .. 4m+3
                const uint32_t c02 = qw[m] & nib;         // values 4m, 4m + 2
                const uint32_t c13 = (qw[m] >> 8) & nib;  // values 4m + 1, 4m + 3
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    SQA_MIX(dot[t], xg[t][4 * m], c02, 0);
                    SQA_MIX(dot[t], xg[t][4 * m + 1], c13, 0);
                    SQA_MIX(dot[t], xg[t][4 * m + 2], c02, 1);
                    SQA_MIX(dot[t], xg[t][4 * m + 3], c13, 1);
                }
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) acc[r][t] = fmaf(-dm[r], sx[t], fmaf(ds[r], dot[t], acc[r][t]));
        }
    }
#undef SQA_MIX
    // Sum of the V = R * MT values (index r * MT + t) over the wavefront by
    // recursive halving: each step pairs lanes that differ in one bit; the lane
    // with the bit clear keeps the lower half of its values, the other the
    // upper half, each adding its partner's copy of the half it keeps. Lane bits
    // 5 and 4 swap halves between rows (permlane32 / permlane16 swaps, which
    // exchange the upper 32 lanes of the first operand with the lower 32 of the
    // second and the odd rows of the first with the even rows of the second: a
    // swap and an add per pair), bit 3 pairs lane ^ 8 (row_ror:8), bit 2 lane ^ 7
    // (row_half_mirror: the same bits above 2), bit 1 lane ^ 2 (quad_perm), and
    // the bits left over are summed in place. Lane l then holds the full sum of
    // index l >> (6 - log2 V): V - 1 swaps or DPP moves instead of 6 V.
    constexpr int V = R * MT;
    static_assert(V == 8 || V == 16 || V == 32, "halving steps below");
    float a[V];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) a[r * MT + t] = acc[r][t];
#pragma unroll
    for (int j = 0; j < V / 2; ++j) {  // bit 5
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[j]), __float_as_uint(a[V / 2 + j]), false, false);
        a[j] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    }
#pragma unroll
    for (int j = 0; j < V / 4; ++j) {  // bit 4
        const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[j]), __float_as_uint(a[V / 4 + j]), false, false);
        a[j] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    }
    halve_dpp<V / 8, 0x128>(a, (lane & 8) != 0);                   // bit 3, lane ^ 8 (row_ror:8)
    if constexpr (V >= 16) halve_dpp<V / 16, 0x141>(a, (lane & 4) != 0);  // bit 2, lane ^ 7 (row_half_mirror)
    if constexpr (V >= 32) halve_dpp<V / 32, 0x4e>(a, (lane & 2) != 0);   // bit 1, lane ^ 2 (quad_perm [2,3,0,1])
    float s = a[0];
    s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0xb1, 0xf, 0xf, false));  // lane ^ 1
    if constexpr (V <= 16) s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x4e, 0xf, 0xf, false));
    if constexpr (V <= 8) s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x141, 0xf, 0xf, false));
    constexpr int kSpan = 64 / V;  // lanes that share an index
    if ((lane & (kSpan - 1)) == 0) red[wave][lane / kSpan] = s;
    __syncthreads();
    if (tid < R * MT) {
        const int r = tid / MT, t = tid - r * MT;
        float o = 0.0f;
#pragma unroll
        for (int wv = 0; wv < W; ++wv) o += red[wv][tid];
        if (t < M && row0 + r < N) reinterpret_cast<float *>(reinterpret_cast<char *>(dst) + t * d_nb1)[row0 + r] = o;
    }
}

// Workspace of the GEMM path (see op_prep): 2 KB of x operands per 16 tokens and
// sub-block, 1 KB of S operands per 16 tokens and super-block.
struct OpLayout {
    int64_t tiles;
    size_t sb, total;
};
OpLayout op_layout(int64_t K, int64_t M) {
    OpLayout l;
    l.tiles = (M + 15) / 16;
    l.sb = (size_t)(l.tiles * (K / 32)) * 2048;
    l.total = l.sb + (size_t)(l.tiles * (K / kQK)) * 1024 + 256;
    return l;
}

}  // namespace

size_t out_proj_workspace(int64_t K, int64_t M) {
    if (M <= kGemvTokens) return 0;  // the decode path keeps its operands in registers
    return op_layout(K, M).total;
}

int launch_out_proj(const sqa_tensor &w, const sqa_tensor &x, const sqa_tensor *gate, const sqa_tensor &dst,
                    void *ws, size_t ws_bytes, hipStream_t s) {
    const int64_t K = w.ne[0], N = w.ne[1], M = x.ne[1];
    if (M == 0 || N == 0) return SQA_OK;
    if (M <= kGemvTokens) {
        const int mt = M == 1 ? 1 : (M == 2 ? 2 : 4);
        const int prof = profile_start("out_proj", s);
        const uint8_t *wd = (const uint8_t *)w.data;
        const char *xd = (const char *)x.data, *gd = gate ? (const char *)gate->data : nullptr;
        const int64_t wn = (int64_t)w.nb[1], xn = (int64_t)x.nb[1], gn = gate ? (int64_t)gate->nb[1] : 0;
        float *dd = (float *)dst.data;
        const int64_t dn = (int64_t)dst.nb[1];
        const dim3 grid((unsigned)(N / kGemvRows));
        const bool vec = (uintptr_t)xd % 16 == 0 && xn % 16 == 0 && (!gd || ((uintptr_t)gd % 16 == 0 && gn % 16 == 0));
#define SQA_GEMV(MTV)                                                                                          \
    (vec ? op_gemv_kernel<MTV, true> : op_gemv_kernel<MTV, false>)<<<grid, dim3(kGemvThreads), 0, s>>>(        \
        wd, wn, xd, xn, gd, gn, (int)K, (int)N, (int)M, dd, dn)
        if (mt == 1)
            SQA_GEMV(1);
        else if (mt == 2)
            SQA_GEMV(2);
        else
            SQA_GEMV(4);
#undef SQA_GEMV
        profile_stop(prof, s);
        return hip_status(hipGetLastError(), "out_proj launch");
    }
    const OpLayout L = op_layout(K, M);
    const size_t need = L.total;
    if (!ws || ws_bytes < need)
        return set_error(SQA_ERR_WORKSPACE, "out_proj: workspace %zu bytes < %zu needed", ws_bytes, need);
    uint8_t *base = reinterpret_cast<uint8_t *>(((uintptr_t)ws + 255) & ~(uintptr_t)255);
    uint4 *xb = reinterpret_cast<uint4 *>(base);
    uint16_t *sb = reinterpret_cast<uint16_t *>(base + L.sb);
    static std::once_flag g2_once;
    static hipError_t g2_err = hipSuccess;
    std::call_once(g2_once, [] {
        g2_err = hipFuncSetAttribute((const void *)op_gemm2_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kG2Lds);
    });
    if (g2_err != hipSuccess) return hip_status(g2_err, "out_proj LDS attribute");

    const int prof = profile_start("out_proj", s);
    const bool vec = (uintptr_t)x.data % 16 == 0 && x.nb[1] % 16 == 0 &&
                     (!gate || ((uintptr_t)gate->data % 16 == 0 && gate->nb[1] % 16 == 0));
    const char *xd = (const char *)x.data, *gd = gate ? (const char *)gate->data : nullptr;
    const int64_t xn = (int64_t)x.nb[1], gn = gate ? (int64_t)gate->nb[1] : 0;
    const int Ki = (int)K, Mi = (int)M, tl = (int)L.tiles;
    const int subs = L.tiles * (K / 64) >= kPrepPairs ? 2 : 1;
    const dim3 pg((unsigned)((L.tiles * (K / 32) / subs + 3) / 4));
#define SQA_PREP(GATE, VEC)                                                                       \
    (subs == 2 ? op_prep_kernel<GATE, VEC, 2> : op_prep_kernel<GATE, VEC, 1>)<<<pg, dim3(256), 0, s>>>( \
        xd, xn, gd, gn, Ki, Mi, tl, xb, sb)
    if (gate && vec)
        SQA_PREP(true, true);
    else if (gate)
        SQA_PREP(true, false);
    else if (vec)
        SQA_PREP(false, true);
    else
        SQA_PREP(false, false);
#undef SQA_PREP
    GemmParams p;
    p.w = (const uint8_t *)w.data;
    p.w_nb1 = (int64_t)w.nb[1];
    p.xb = xb;
    p.sb = reinterpret_cast<const uint4 *>(sb);
    p.K = Ki;
    p.N = (int)N;
    p.M = Mi;
    p.tiles = tl;
    p.dst = (float *)dst.data;
    p.d_nb1 = (int64_t)dst.nb[1];
    p.rows_first = false;
#define SQA_GEMM(KS, RT, TT)                                                                                   \
    do {                                                                                                       \
        p.row_blocks = (int)((N + 16 * RT - 1) / (16 * RT));                                                   \
        p.token_groups = (tl + TT - 1) / TT;                                                                   \
        op_gemm_kernel<KS, RT, TT><<<dim3((unsigned)(p.row_blocks * p.token_groups)), dim3(64 * KS), 0, s>>>(p); \
    } while (0)
    // The smallest workgroup tile of op_gemm that still leaves at most one workgroup
    // per CU (with two the time grows by half or doubles), counted with the tokens and
    // rows that fill a tile up; for one token tile also two per CU of the smallest, as the
    // second tile of the others would be thrown away; else op_gemm2. us at N = 2048, K =
    // 4096 with op_prep, op_gemm <16, 1, 1> / <16, 1, 2> / <16, 2, 2> / <8, 4, 2> /
    // op_gemm2: 23 tokens 9.9 / 12.3 / 14.3 / 20.5 / 28.1, 64 tokens 13.8 / 13.0 / 14.4 /
    // 20.5 / 28.2, 128 tokens 23.1 / 20.4 / 15.4 / 20.9 / 28.6, 256 tokens 39 / 36 / 27.6 /
    // 23.6 / 30.6, 300 tokens 46 / 43 / 36 / 38 / 31.9, 512 tokens 70 / 62 / 46 / 41 / 32.8.
    // (With a pre-pass 0.5 to 1 us slower than this one: 23 tokens are 9.1 now.)
    // K = 4096, <16, 1, 1> / <16, 1, 2> / <16, 2, 2> / <8, 4, 2>: 16 tokens, N = 5120 12.5 /
    // 16.9 / 13.3 / 19.2, 48 tokens, 2720 13.0 / 18.2 / 13.9 / 20.0, 48 tokens, 5120 21.3 /
    // 24.1 / 21.9 / 19.7. K does not enter: at K = 1024, where 12 of the 16 wavefronts have
    // no super-block, 48 tokens with N = 2720 take 8.7 / 11.6 / 9.9 / 11.4. op_gemm2's DMA
    // addresses its 128 rows with 32-bit offsets.
    const int64_t cus = device_cu_count(), row_tiles = N / 16;
    auto groups = [&](int64_t rt, int64_t tt) { return (row_tiles + rt - 1) / rt * ((L.tiles + tt - 1) / tt); };
    if (groups(1, 1) <= (L.tiles == 1 ? 2 : 1) * cus) {
        SQA_GEMM(16, 1, 1);
    } else if (groups(1, 2) <= cus) {
        SQA_GEMM(16, 1, 2);
    } else if (groups(2, 2) <= cus) {
        SQA_GEMM(16, 2, 2);
    } else if (groups(4, 2) <= cus || (uint64_t)kG2Rows * w.nb[1] >= (1ull << 32)) {
        SQA_GEMM(8, 4, 2);
    } else {
        p.row_blocks = (int)((N + kG2Rows - 1) / kG2Rows);
        p.token_groups = (tl + kG2TT - 1) / kG2TT;
        // Every XCD reads all of one, weights or operands, and its share of the other:
        // row blocks first where the weights are clearly the larger. us per call, token
        // groups / row blocks first: 100 tokens, N = 8192, K = 2048 (weights 10 times the
        // operands) 19.2 / 17.3, 200 of them 28.3 / 27.0, 300, 4096, 4096 (1.9) 46.1 / 44.1,
        // 1000, 8192, 2048 (1.14) 100.8 / 102.6, 512, 2048, 4096 (0.56) 33.4 / 34.3.
        // op_gemm's calls are all better with token groups first (128 tokens 13.8 / 15.5).
        p.rows_first = 2 * (uint64_t)N * (K / kQK) * kBlockBytes > 3 * (uint64_t)L.sb;
        op_gemm2_kernel<<<dim3((unsigned)(p.row_blocks * p.token_groups)), dim3(64 * kG2Waves), kG2Lds, s>>>(p);
    }
#undef SQA_GEMM
    profile_stop(prof, s);
    return hip_status(hipGetLastError(), "out_proj launch");
}

}  // namespace sqa
