// fa_prefill.hip - FlashAttention for prefill chunks (more than 16 query rows
// per KV head, or more than 4 positions): the ubatch node of
// src/model/attn.rs:228-251 in the reference (n_q = 512 or 2048 over a q4_0
// cache of 16K-133K keys).
//
// Two short pre-passes in one launch, then one MFMA kernel:
//   kvprep K, V q4_0 -> per 32-key tile and KV head: Kc fp16 codes (nib - 8)
//                 [32 keys][256] and Dk fp16 scales [8 blocks][32 keys]; Vc
//                 fp16 codes [256 dims][32 keys] and Dv fp16 scales [8 blocks]
//                 [32 keys]; per KV head the largest |d_v|
//   qprep  Q f32 -> q8_0 with ggml's x86 rounding (d = amax/127, codes =
//                 rint(x * 127/amax)), then Q' = code * fp16(d) * scale *
//                 log2(e) as an fp16 hi + lo pair [n_q*H][256] each (Q' has at
//                 most 7 + 24 significant bits; hi + lo hold 22 of them)
// A tile of one KV head is a contiguous 33792-byte record [Kc | Dk | Vc | Dv]
// laid out exactly as the main kernel wants it in LDS (rows permuted, chunks
// swizzled, see below), so its K and V halves move HBM -> LDS as straight
// copies. Keys past n_kv are zero.
//
// fa_prefill_kernel: a workgroup takes 128 (or 64) query rows of ONE KV head (GQA
// packed: row r is position r / G, head kvh*G + r % G) and streams 32-key
// tiles. Its 8 wavefronts (2 per SIMD) split the work by kind (rows and registers
// for 128 query rows, half of both for 64):
//   score wave w (0..3), rows 32w..32w+31, holds their Q' hi and lo (128
//     registers): S^T = sum over q4_0 blocks b of d_k[b] * (Kc_b.Q'h_b +
//     Kc_b.Q'l_b), the products on v_mfma_f32_16x16x32_f16 (all exact in
//     fp32: a code has at most 3 significant bits) and the d_k scaling as an
//     fp32 FMA with the fp16 scale as operand; then the mask and the
//     online softmax in fp32 (base 2, with a lazy reference maximum that moves
//     only when a logit passes it by more than a slack of ks binades, so
//     P <= 2^ks and most tiles need no rescale of O; ks = 8 unless V is large,
//     below). P (as an fp16 hi + lo pair) and the rescale factors go to LDS.
//   value wave 4 + w, the same 32 rows, holds their O (128 registers) one tile
//     behind: O = alpha O + P V per block b (alpha only when a maximum moved)
//     with A = P d_v as an fp16 hi + lo pair built by packed fp16 ops (two
//     MFMAs, ~22 bits) and B = the exact V codes, so every product is exact in
//     fp32. P carries 2^ep, one power of two per KV head, and l, summed from
//     the same P, carries the same factor. ep and ks follow the largest |d_v|
//     of the head so that A = P 2^ep d_v stays below 2^15 for every finite V
//     while P 2^ep stays as far from the fp16 subnormals as that allows.
//     The d_v and V operands of a tile are read ahead of the MFMAs that use them.
//   A masked key contributes exactly 0 even over NaN/Inf block scales (as ggml's
//   CPU loop, which skips it): a -inf mask entry replaces the logit, and the
//   pre-pass reads NaN/Inf V scales as 0.
// Computing S^T (keys as rows) leaves each lane with 8 logits of one query row
// in the A-operand layout of the P*V MFMA. K rows sit in LDS in the order
// r -> key sigma(r) = 8*((r>>2)&3) + 4*(r>>4) + (r&3), which makes a lane's 8
// logits keys 8g..8g+7, so its V operand is one 16-byte run of a Vc row.
//
// LDS reads are ds_read_b64 (16 lanes a pass). To keep them conflict free,
// 16-byte chunk c of K row r is stored at chunk c ^ (r & 7) with its 8-byte
// halves swapped when r & 8, and chunk c of Vc row d at c ^ ((d >> 1) & 3),
// halves swapped when d & 8.
//
// Tiles move HBM -> LDS with global_load_lds_dwordx4, issued by the value waves: in
// iteration t the K half (and mask rows) of tile t + 1 and the V half of tile t
// are in flight while the score waves work on tile t and the value waves on tile
// t - 1; one barrier per iteration.
//
// Operand layout of the 16x16x32 MFMAs (64 lanes, lane = 16*g + n):
//   A: A[row n][k = 8g..8g+7]   B: B[k = 8g..8g+7][col n]   C: C[rows 4g..4g+3][col n]
#include <mutex>

#include "common.hpp"

namespace sqa {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

constexpr int kPK = 32;                  // keys per tile
constexpr int kScoreWaves = 4;           // 32 rows each
constexpr int kValueWaves = 4;           // 32 rows each
constexpr int kWaves = kScoreWaves + kValueWaves;
constexpr int kThreads = 64 * kWaves;
constexpr int kMaxRG = 2;                // 16-row groups per score wave: 1 or 2 (kRG in the kernel)
constexpr int rows_per_wg(int rg) { return kScoreWaves * rg * 16; }  // 64 or 128 query rows
constexpr int kOffDk = kPK * 512;        // inside the K half: Dk after Kc
constexpr int kKHalf = kOffDk + 8 * kPK * 2;  // Kc + Dk: 16896 bytes
constexpr int kOffDv = kHeadDim * kPK * 2;  // inside the V half: Dv after Vc
constexpr int kVHalf = kOffDv + 8 * kPK * 2;  // Vc + Dv: 16896 bytes
constexpr int kTileBytes = kKHalf + kVHalf;   // one tile record
constexpr int kKInst = (kKHalf + 1023) / 1024;  // 17 DMA instructions, the last one 512 bytes
constexpr int kVInst = (kVHalf + 1023) / 1024;  // 17, the last one 512 bytes
constexpr int kKStage = kKInst * 1024, kVStage = kVInst * 1024;
// LDS map (sized for kMaxRG): 2 K stages | 2 V stages | 2 P buffers | 2 rescale buffers | 2 mask stages
constexpr int kLdsV = 2 * kKStage;
constexpr int kLdsP = kLdsV + 2 * kVStage;        // [4 waves][kRG][2 halves][64 lanes][16 B]
constexpr int kPBuf = kScoreWaves * kMaxRG * 2 * 1024;
constexpr int kLdsA = kLdsP + 2 * kPBuf;          // [4 waves][kRG][16 rows] f32
constexpr int kABuf = kScoreWaves * kMaxRG * 16 * 4;
constexpr int kLdsMask = kLdsA + 2 * kABuf;       // [qb positions][32 keys] f16
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kSlack = 8;  // log2 of the largest P the lazy rescale admits (V not large)
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

static_assert(kTileBytes == 33792 && kTileBytes % 256 == 0, "tile record");
static_assert(kKHalf == kVHalf && kKInst == 17 && kVInst == 17, "both halves: 16 DMA instructions and a half");
constexpr int kLdsMaxBytes = kLdsMask + 2 * 128 * kPK * 2;  // with the mask stages of G = 1
static_assert(kLdsMaxBytes <= 160 * 1024, "LDS budget");

__device__ __forceinline__ float h2f(uint32_t bits) {
    const uint16_t b = (uint16_t)bits;
    _Float16 f;
    __builtin_memcpy(&f, &b, 2);
    return (float)f;
}

__device__ __forceinline__ uint4 swap_halves(uint4 v, bool swap) {
    return swap ? make_uint4(v.z, v.w, v.x, v.y) : v;
}

// max(x, x of lane ^ 16) and max(x, x of lane ^ 32) with gfx950's row swaps (no
// LDS round trip): each swap returns the two halves of a lane pair's values.
__device__ __forceinline__ float xmax16(float x) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xmax32(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// LDS/record row of key k (0..31) of a tile: the inverse of sigma.
__device__ __forceinline__ int key_row(int k) { return 16 * ((k >> 2) & 1) + 4 * (k >> 3) + (k & 3); }

// ---------------------------------------------------------------- pre-passes

// One workgroup per (64 keys, KV head): the 64 q4_0 rows of K and of V are
// staged in LDS with 16-byte loads (zeros past n_kv), then
//   K: thread t takes blocks (key, b) = t and t + 256 (key = idx / 8, b = idx % 8):
//      its 32 codes as fp16 (4 swizzled 16-byte chunks of the key's row) and its
//      scale into the Dk row of block b;
//   V: thread t writes the Vc row of dim t (32 codes, 64 bytes) of both tiles;
//      the first wavefront writes the Dv rows and the group's largest |d_v|
//      (fp16 magnitude bits) into dvmax[head][group].
// N dwords of a q4_0 block's qs bytes starting at byte off (2 mod 4 for even
// blocks, 0 mod 4 for odd ones) of an LDS row: aligned reads, shifted by
// alignbit. Every read stays inside the row's 144 bytes.
template <int N = 4>
__device__ __forceinline__ void qs_dwords(const uint8_t *row, int off, uint32_t *q) {
    const uint32_t *p = reinterpret_cast<const uint32_t *>(row + (off & ~3));
    const uint32_t sh = 8u * (uint32_t)(off & 3);
    uint32_t a = p[0];
#pragma unroll
    for (int m = 0; m < N; ++m) {
        const uint32_t b = p[sh ? m + 1 : (m + 1 < N ? m + 1 : m)];
        q[m] = __builtin_amdgcn_alignbit(b, a, sh);
        a = b;
    }
}

// Two 4-bit codes n (bits 0-3 and 16-19 of x) as the packed fp16 pair n - 8:
// 0x6400 | n is exactly 1024 + n, and 1024 + n - 1032 is exact.
__device__ __forceinline__ uint32_t codes_f16(uint32_t x) {
    const uint32_t y = (x & 0x000F000Fu) | 0x64006400u;
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    h2 v;
    __builtin_memcpy(&v, &y, 4);
    const h2 d = v + h2{(_Float16)-1032.0f, (_Float16)-1032.0f};
    uint32_t r;
    __builtin_memcpy(&r, &d, 4);
    return r;
}

struct KvPrep {
    const uint8_t *k, *v;
    int64_t k_nb1, k_nb2, v_nb1, v_nb2;
    int64_t n_kv, kv_tiles;
    int hkv, groups;   // KV heads; 64-key groups per head
    uint8_t *kv;
    uint32_t *dvmax;   // [hkv][groups]
};

__device__ __forceinline__ void kvprep(const KvPrep &p, int group, int h) {
    __shared__ __align__(16) uint8_t sk[64 * kHeadRowBytes], sv[64 * kHeadRowBytes];
    const int t = threadIdx.x;
    const int64_t k0 = (int64_t)group * 64;
    const uint8_t *k = p.k, *v = p.v;
    uint8_t *kv = p.kv;
    const int64_t k_nb1 = p.k_nb1, k_nb2 = p.k_nb2, v_nb1 = p.v_nb1, v_nb2 = p.v_nb2, n_kv = p.n_kv,
                  kv_tiles = p.kv_tiles;
    for (int idx = t; idx < 64 * 9; idx += 256) {  // 9 x 16 bytes per 144-byte row
        const int key = idx / 9, c = idx - 9 * key;
        uint4 a = make_uint4(0, 0, 0, 0), b = make_uint4(0, 0, 0, 0);
        if (k0 + key < n_kv) {
            a = *reinterpret_cast<const uint4 *>(k + (k0 + key) * k_nb1 + h * k_nb2 + 16 * c);
            b = *reinterpret_cast<const uint4 *>(v + (k0 + key) * v_nb1 + h * v_nb2 + 16 * c);
        }
        *reinterpret_cast<uint4 *>(sk + kHeadRowBytes * key + 16 * c) = a;
        *reinterpret_cast<uint4 *>(sv + kHeadRowBytes * key + 16 * c) = b;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int idx = t + 256 * i;
        const int key = idx >> 3, b = idx & 7;
        const uint16_t *src = reinterpret_cast<const uint16_t *>(sk + kHeadRowBytes * key + 18 * b);
        // the block's 16 qs bytes as 4 dwords (they start 2 bytes off a dword for
        // even b); codes 2j, 2j+1 (low nibbles) and 16 + 2j, 17 + 2j (high) as fp16
        uint32_t q[4];
        qs_dwords(sk + kHeadRowBytes * key, 18 * b + 2, q);
        uint32_t out[16];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const uint32_t x0 = __builtin_amdgcn_perm(0u, q[m], 0x0c010c00u);  // bytes 4m, 4m+1
            const uint32_t x1 = __builtin_amdgcn_perm(0u, q[m], 0x0c030c02u);  // bytes 4m+2, 4m+3
            out[2 * m] = codes_f16(x0);
            out[2 * m + 1] = codes_f16(x1);
            out[8 + 2 * m] = codes_f16(x0 >> 4);
            out[8 + 2 * m + 1] = codes_f16(x1 >> 4);
        }
        const int64_t gkey = k0 + key;
        const int r = key_row((int)(gkey & (kPK - 1)));
        uint8_t *rec = kv + ((int64_t)h * kv_tiles + (gkey >> 5)) * kTileBytes;
        uint8_t *row = rec + r * 512;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int pos = (4 * b + j) ^ (r & 7);
            const uint4 x = make_uint4(out[4 * j], out[4 * j + 1], out[4 * j + 2], out[4 * j + 3]);
            *reinterpret_cast<uint4 *>(row + 16 * pos) = swap_halves(x, r & 8);
        }
        *reinterpret_cast<uint16_t *>(rec + kOffDk + (b * kPK + r) * 2) = src[0];
    }
    // V: thread t takes dword m of block beta's qs (dims 32 beta + 4m + i from the
    // low nibbles, 32 beta + 16 + 4m + i from the high ones, i < 4) for the 8 keys
    // 8 kg .. 8 kg + 7 and writes those keys' 16-byte chunk of each of its 8 Vc
    // rows (tile kg >> 2, chunk kg & 3); the first wavefront also writes the Dv
    // rows (below)
    {
        const int beta = (t >> 2) & 7, m = t & 3, kg = t >> 5;
        uint32_t w[8];
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) {
            uint32_t q1[1];
            qs_dwords<1>(sv + kHeadRowBytes * (8 * kg + kk), 18 * beta + 2 + 4 * m, q1);
            w[kk] = q1[0];
        }
        uint8_t *vrec = kv + ((int64_t)h * kv_tiles + ((k0 >> 5) + (kg >> 2))) * kTileBytes + kKHalf;
        const int c = kg & 3;  // keys 8c..8c+7 of the tile
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // byte i of keys 2j (bits 0-7) and 2j + 1 (bits 16-23)
            const uint32_t sel = (uint32_t)i | 0x0c00u | ((uint32_t)(4 + i) << 16) | 0x0c000000u;
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t x = __builtin_amdgcn_perm(w[2 * j + 1], w[2 * j], sel);
                lo[j] = codes_f16(x);
                hi[j] = codes_f16(x >> 4);
            }
            // chunk c of dim d at c ^ ((d >> 1) & 3), halves swapped when d & 8
            const int dl = 32 * beta + 4 * m + i, dh = dl + 16;
            *reinterpret_cast<uint4 *>(vrec + 64 * dl + 16 * (c ^ ((dl >> 1) & 3))) =
                swap_halves(make_uint4(lo[0], lo[1], lo[2], lo[3]), dl & 8);
            *reinterpret_cast<uint4 *>(vrec + 64 * dh + 16 * (c ^ ((dh >> 1) & 3))) =
                swap_halves(make_uint4(hi[0], hi[1], hi[2], hi[3]), dh & 8);
        }
        // Dv rows: thread t < 64 takes tile u, block b, keys 8q..8q+7 of the tile
        uint32_t dmax = 0;
        if (t < 64) {
            const int u = t >> 5, b = (t >> 2) & 7, q = t & 3;
            uint16_t dd[8];
#pragma unroll
            for (int kk = 0; kk < 8; ++kk) {
                dd[kk] = *reinterpret_cast<const uint16_t *>(sv + kHeadRowBytes * (32 * u + 8 * q + kk) + 18 * b);
                // a NaN/Inf scale (bytes that are not q4_0) reads as 0: such a key, if
                // masked, adds exactly 0 (P d_v is formed in fp16, where 0 * NaN = NaN)
                dd[kk] = (dd[kk] & 0x7C00u) == 0x7C00u ? (uint16_t)0 : dd[kk];
                const uint32_t mag = dd[kk] & 0x7fffu;
                dmax = mag > dmax ? mag : dmax;
            }
            uint8_t *vrec = kv + ((int64_t)h * kv_tiles + ((k0 >> 5) + u)) * kTileBytes + kKHalf;
            uint4 x;
            __builtin_memcpy(&x, dd, 16);
            *reinterpret_cast<uint4 *>(vrec + kOffDv + 64 * b + 16 * q) = x;
        }
        if (t < 64) {
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1) {
                const uint32_t other = (uint32_t)__shfl_xor((int)dmax, o);
                dmax = other > dmax ? other : dmax;
            }
            if (t == 0) p.dvmax[(int64_t)h * p.groups + group] = dmax;
        }
    }
}

// A quad of threads per 32-value block of one (query, head) row, 8 values each:
// q8_0 with ggml's x86 rounding (d = amax/127 over the block, codes =
// rint(x * 127/amax)), then Q' = code * qd with qd = fp16(d) * scale * log2(e) in
// fp32, written as fp16 hi = fp16(Q') and lo = fp16(Q' - hi).
// Exclusive key limit of query tile `tile` under an F16 mask: 1 + the last
// key any of its qb rows leaves visible (an entry other than -inf), 0 if none.
// Keys past it are masked in every row of the tile, so the main kernel stops
// there, as it does at the causal limit of the position form. Run by one
// 256-thread workgroup: each wavefront takes 4 rows at a time and reads them
// backwards 1024 keys per step (a lane takes two 8-key 16-byte loads per
// row, all 8 loads in flight at once) until a step holds a visible key, so a
// causal row costs its masked tail only: one step at pp512 (tails up to 511
// keys), two for a 2048-token ubatch. Rows are 16-byte aligned with len (a
// multiple of 8) readable keys. Every thread of the workgroup must call it.
__device__ __forceinline__ void mask_tile_limit(const char *__restrict__ mask, int64_t nb1, int64_t len, int n_q, int qb, int tile,
                                int32_t *__restrict__ lim) {
    __shared__ int32_t best[4];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int q0 = tile * qb;
    const int64_t c_top = (len - 1) / 1024 * 1024;
    const uint4 none = make_uint4(0xFC00FC00u, 0xFC00FC00u, 0xFC00FC00u, 0xFC00FC00u);
    auto last_of = [&](uint4 a, uint4 b, int64_t c0) {  // the wavefront's last visible key in one step, or -1
        int last = -1;
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int e = 0; e < 16; ++e)
            if (((w[e >> 1] >> (16 * (e & 1))) & 0xFFFFu) != 0xFC00u)
                last = (int)(c0 + 512 * (e >> 3) + 8 * lane + (e & 7));
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) last = max(last, __shfl_xor(last, o));
        return last;
    };
    auto load = [&](const uint16_t *row, int64_t k) {
        return k < len ? *reinterpret_cast<const uint4 *>(row + k) : none;
    };
    int32_t mine = -1;  // wave-uniform
    for (int r0 = 4 * wave; r0 < qb; r0 += 16) {
        uint4 a[4], b[4];
        const uint16_t *rows[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // the first step of four rows at once
            const bool ok = r0 + j < qb && q0 + r0 + j < n_q;
            rows[j] = ok ? reinterpret_cast<const uint16_t *>(mask + (int64_t)(q0 + r0 + j) * nb1) : nullptr;
            a[j] = ok ? load(rows[j], c_top + 8 * lane) : none;
            b[j] = ok ? load(rows[j], c_top + 512 + 8 * lane) : none;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            int last = last_of(a[j], b[j], c_top);
            for (int64_t c0 = c_top - 1024; last < 0 && rows[j] && c0 >= 0; c0 -= 1024)  // longer tails
                last = last_of(load(rows[j], c0 + 8 * lane), load(rows[j], c0 + 512 + 8 * lane), c0);
            mine = max(mine, last);
        }
    }
    if (lane == 0) best[wave] = mine;
    __syncthreads();
    if (threadIdx.x == 0) lim[tile] = max(max(best[0], best[1]), max(best[2], best[3])) + 1;
}

// The same as a kernel of its own, for a packed mask copy (written after the
// Q pre-pass): one workgroup per query tile.
__global__ __launch_bounds__(256) void mask_tile_limit_kernel(const char *__restrict__ mask, int64_t nb1, int64_t len,
                                                              int n_q, int qb, int32_t *__restrict__ lim) {
    mask_tile_limit(mask, nb1, len, n_q, qb, blockIdx.x, lim);
}

// The mask scan (mask_tile_limit) of every query tile, when the kernel reads the
// caller's mask in place.
struct MaskScan {
    const char *mask;  // null: no scan here
    int64_t nb1, len;
    int qb, tiles;
    int32_t *lim;
};

struct QPrep {
    const char *q;
    int64_t nb1, nb2;
    int n_q, H;
    float qscale;
    uint16_t *qh, *ql;
    bool aligned;
};

__device__ __forceinline__ void qprep(const QPrep &p, int64_t gid) {
    const char *q = p.q;
    const int64_t nb1 = p.nb1, nb2 = p.nb2;
    const int n_q = p.n_q, H = p.H;
    const float qscale = p.qscale;
    uint16_t *qh = p.qh, *ql = p.ql;
    const bool aligned = p.aligned;
    // one thread per 8 values: a quad of lanes owns a 32-value block
    if (gid >= (int64_t)n_q * H * kBlocksPerHead * 4) return;  // whole quads: the total is a multiple of 4
    const int qtr = (int)(gid & 3);
    const int64_t bid = gid >> 2;
    const int b = (int)(bid % kBlocksPerHead);
    const int64_t row = bid / kBlocksPerHead;  // t * H + h
    const int h = (int)(row % H);
    const int64_t t = row / H;
    const float *x = reinterpret_cast<const float *>(q + t * nb1 + h * nb2) + 32 * b + 8 * qtr;
    float v[8];
    if (aligned) {  // 16-byte aligned rows: vector loads
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float4 f = reinterpret_cast<const float4 *>(x)[j];
            v[4 * j] = f.x; v[4 * j + 1] = f.y; v[4 * j + 2] = f.z; v[4 * j + 3] = f.w;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = x[j];
    }
    float amax = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    // the block's amax over the quad (quad_perm [1,0,3,2], then [2,3,0,1])
    amax = fmaxf(amax, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(amax), 0xB1, 0xf, 0xf, false)));
    amax = fmaxf(amax, __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(amax), 0x4E, 0xf, 0xf, false)));
    const float d = amax / 127.f;
    const float id = amax != 0.0f ? 127.f / amax : 0.0f;
    const float qd = (float)(_Float16)d * qscale;
    uint16_t oh[8], ol[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        // x opaque: left visible, the compiler may round code * qd to fp16 twice
        // (once from the fp32 product for hi, once from the exact product for the
        // hi it subtracts), and a hi + lo off by one fp16 ulp of hi
        float xx = rintf(v[j] * id) * qd;
        asm volatile("" : "+v"(xx));
        const _Float16 hh = (_Float16)xx;
        const _Float16 ll = (_Float16)(xx - (float)hh);
        __builtin_memcpy(&oh[j], &hh, 2);
        __builtin_memcpy(&ol[j], &ll, 2);
    }
    uint4 a, c;
    __builtin_memcpy(&a, oh, 16);
    __builtin_memcpy(&c, ol, 16);
    *reinterpret_cast<uint4 *>(qh + row * kHeadDim + 32 * b + 8 * qtr) = a;
    *reinterpret_cast<uint4 *>(ql + row * kHeadDim + 32 * b + 8 * qtr) = c;
}

// The pre-passes in one launch: the K/V groups first (the longest workgroups),
// then the mask scans, then Q. As two launches, with the scans beside Q, they took
// 8.3 + 5.1 us for 512 queries on 512 keys (8.4 now), 6.5 + 17 on 16896 keys
// (16.8), 4.7 + 17.7 for 37 on 20048 (17.1), and the gap between them.
__global__ __launch_bounds__(256) void prep_kernel(KvPrep kv, QPrep q, MaskScan ms) {
    int id = (int)blockIdx.x;
    const int n_kv = kv.groups * kv.hkv;
    if (id < n_kv) {
        kvprep(kv, id % kv.groups, id / kv.groups);
        return;
    }
    id -= n_kv;
    if (ms.mask) {
        if (id < ms.tiles) {
            mask_tile_limit(ms.mask, ms.nb1, ms.len, q.n_q, ms.qb, id, ms.lim);
            return;
        }
        id -= ms.tiles;
    }
    qprep(q, (int64_t)id * 256 + threadIdx.x);
}

// Copies an F16 mask whose rows are unaligned or whose length is not a
// multiple of 8 into [n_q][len8] rows (len8 = n_kv rounded up to 8, -inf pad).
__global__ __launch_bounds__(256) void pf_mask_pack_kernel(const char *__restrict__ src, int64_t nb1, int64_t n_kv,
                                                           int n_q, int64_t len8, uint16_t *__restrict__ dst) {
    const int64_t total = len8 * n_q;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t t = i / len8, kk = i - t * len8;
        dst[i] = kk < n_kv ? reinterpret_cast<const uint16_t *>(src + t * nb1)[kk] : (uint16_t)0xFC00;
    }
}

// ------------------------------------------------------------ main kernel

// 16 bytes per lane from sbase + voff into LDS at m0 + 16 * lane (asynchronous;
// the caller waits with s_waitcnt vmcnt).
__device__ __forceinline__ void dma16(uint32_t voff, const void *sbase, uint32_t m0v) {
    // m0 as an operand: the compiler writes it and knows it holds the LDS base
    asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(m0v) : "memory");
}

// Two 8-byte LDS reads into one MFMA operand. volatile keeps them two single
// ds_read_b64 straight into the operand's registers: merged into ds_read2 pairs
// they would bring halves of different operands and need register moves.
__device__ __forceinline__ half8 lds_half8(const uint8_t *base, int off_lo, int off_hi) {
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    typedef const volatile __attribute__((address_space(3))) u32x2 lds_u32x2;
    const u32x2 a = *(lds_u32x2 *)(base + off_lo);
    const u32x2 b = *(lds_u32x2 *)(base + off_hi);
    const uint4 u = make_uint4(a.x, a.y, b.x, b.y);
    half8 h;
    __builtin_memcpy(&h, &u, 16);
    return h;
}


struct PrefillParams {
    const uint8_t *kv;        // [Hkv][kv_tiles] tile records
    const uint32_t *dvmax;    // [Hkv][kv_tiles / 2] fp16 magnitude bits
    const uint16_t *qh, *ql;  // [n_q*H][256] fp16 Q' hi and lo
    int64_t n_kv, kv_tiles;
    int n_q, H, G, Hkv;
    const char *mask;  // F16 rows 16-byte aligned, mask_len (a multiple of 8) keys each, or null
    int64_t mask_nb1, mask_len;
    int64_t q_pos0;    // >= 0: causal from positions (mask ignored)
    const int32_t *tile_lim;  // with a mask: [q_tiles] exclusive key limit of each query tile
    int n_splits;
    int q_tiles;        // workgroups per (KV head, split)
    bool skew;          // order of the workgroups, see the kernel
    int64_t split_len;  // keys per split, a multiple of kPK
    int qb;             // query positions per workgroup (64 or 128 rows / G)
    int mask_stage;     // LDS bytes per mask stage (qb x 64)
    float *part_acc, *part_ml;  // n_splits > 1
    float *dst;                 // n_splits == 1: [n_q][H][256]
    const char *gate;
    int64_t gate_nb1, gate_nb2;
};

// kRG = 2: 128 query rows; 1: 64 rows (see plan for where).
template <int kRG>
__global__ __launch_bounds__(kThreads, 1) void fa_prefill_kernel(PrefillParams p) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, g = lane >> 4, n = lane & 15;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

    // Workgroups are dealt round-robin to the 8 XCDs (each with its own L2).
    // Renumber so that each XCD gets a contiguous run of ids, i.e. the query
    // tiles of the same (KV head, split): they stream the same K/V range, which
    // that XCD's L2 then serves to all of them.
    // With p.skew (a causal chunk whose query tiles see ranges of very different
    // length) such runs would give whole XCDs the long tiles. The workgroups then
    // go out longest first: split by split (the early ones are seen whole), the
    // last query tile first, neighbours on different XCDs.
    const int nb = (int)gridDim.x;
    const int lin = (int)blockIdx.x;
    const int x = lin & 7, per = nb >> 3, rem = nb & 7;
    int q_tile, kvh, split;
    if (p.skew) {
        const int wgs = p.q_tiles * p.Hkv, r = lin % wgs;
        split = lin / wgs;
        q_tile = p.q_tiles - 1 - r / p.Hkv;
        kvh = r % p.Hkv;
    } else {
        const int id = x * per + (x < rem ? x : rem) + (lin >> 3), grp = id / p.q_tiles;
        q_tile = id % p.q_tiles;
        kvh = grp / p.n_splits;
        split = grp % p.n_splits;
    }
    const int q_base = q_tile * p.qb;

    // Key range: the split, cut at the last key any query of the workgroup sees.
    const int64_t k_begin = (int64_t)split * p.split_len;
    int64_t k_end = k_begin + p.split_len < p.n_kv ? k_begin + p.split_len : p.n_kv;
    if (p.q_pos0 >= 0) {
        const int64_t q_last = (q_base + p.qb < p.n_q ? q_base + p.qb : p.n_q) - 1;
        const int64_t lim = p.q_pos0 + q_last + 1;
        if (k_end > lim) k_end = lim;
    } else if (p.tile_lim) {  // the mask's last visible key over the tile's rows
        const int64_t lim = p.tile_lim[q_tile];
        if (k_end > lim) k_end = lim;
    }
    const int n_tiles = k_end > k_begin ? (int)((k_end - k_begin + kPK - 1) / kPK) : 0;
    if (n_tiles == 0 && p.n_splits > 1) {
        // a split past the tile's last visible key leaves its O unwritten: the
        // merge takes no partial whose m is -inf
        const int pos = q_base + tid / p.G;
        if (tid < rows_per_wg(kRG) && pos < p.n_q) {
            const int64_t row = (int64_t)split * p.n_q * p.H + (int64_t)pos * p.H + kvh * p.G + tid % p.G;
            store_through(p.part_ml + row * 2, -INFINITY);
            store_through(p.part_ml + row * 2 + 1, 0.0f);
        }
        return;
    }

    // ---------------- DMA: 1 KB per instruction, issued by the value waves --------
    // Iteration t: K half + mask of tile t + 1, V half of tile t (stage = tile & 1).
    // K and V instructions jj (0..16, the last one 512 bytes) go to value wave jj %
    // 4 and (jj + 2) % 4, mask instructions jm (< 8) to value waves (jm + 1) % 4: the
    // score waves' chain is the longer one, they issue none (us per call, all waves
    // issuing / this: 512 queries on 16896 keys 286 / 278.5, 2048 on 32048 1834 / 1807;
    // raising the value waves' priority made the first 10% slower).
    const int n_mask_inst = p.mask ? (p.qb + 15) / 16 : 0;
    const uint8_t *kv_h = p.kv + (int64_t)kvh * p.kv_tiles * kTileBytes;
    const int vw = wave & 3;
    const int jv0 = (vw + 2) & 3;
    static_assert(kKInst == 4 * kValueWaves + 1 && kVInst == 4 * kValueWaves + 1, "four full DMA instructions per value wave and half");
    const bool k_half = vw == 0, v_half = jv0 == 0;  // the wave that issues the 512-byte instruction
    // mask row of this lane's slot in instruction jm: position q_base + r (clamped
    // to n_q - 1), chunk c = (s & 3) ^ ((r >> 1) & 3) of the row's 32 keys
    const int jm0 = (vw + 3) & 3;
    uint32_t m_row[2];
    int m_c[2];
    bool m_lane[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int jm = jm0 + 4 * u, r = (64 * jm + lane) >> 2;
        m_c[u] = ((64 * jm + lane) & 3) ^ ((r >> 1) & 3);
        m_lane[u] = jm < n_mask_inst && r < p.qb;
        m_row[u] = m_lane[u] ? (uint32_t)((int64_t)(q_base + r < p.n_q ? q_base + r : p.n_q - 1) * p.mask_nb1) : 0u;
    }
    // record of the split's first tile (k_begin is a multiple of kPK); tile t's
    // record is t records further on
    const uint8_t *rec0 = kv_h + (k_begin / kPK) * kTileBytes;
    auto issue = [&](int t_k, int t_v) {  // tile indices or -1
        if (t_k >= 0) {
            const uint8_t *rec = rec0 + (int64_t)t_k * kTileBytes;
            const uint32_t st = lds0 + (uint32_t)((t_k & 1) * kKStage);
#pragma unroll
            for (int r = 0; r < 4; ++r) dma16(1024u * (vw + 4 * r) + 16u * lane, rec, st + 1024u * (vw + 4 * r));
            if (k_half && lane < 32) dma16(1024u * (kKInst - 1) + 16u * lane, rec, st + 1024u * (kKInst - 1));
            if (jm0 < n_mask_inst) {
                const int64_t kt = k_begin + (int64_t)t_k * kPK;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int64_t col = kt + 8 * m_c[u] < p.mask_len ? kt + 8 * m_c[u] : p.mask_len - 8;
                    const uint32_t sm = lds0 + (uint32_t)(kLdsMask + (t_k & 1) * p.mask_stage + 1024 * (jm0 + 4 * u));
                    if (m_lane[u]) dma16(m_row[u] + (uint32_t)(2 * col), p.mask, sm);
                }
            }
        }
        if (t_v >= 0) {
            const uint8_t *rec = rec0 + (int64_t)t_v * kTileBytes + kKHalf;
            const uint32_t st = lds0 + (uint32_t)(kLdsV + (t_v & 1) * kVStage);
#pragma unroll
            for (int r = 0; r < 4; ++r) dma16(1024u * (jv0 + 4 * r) + 16u * lane, rec, st + 1024u * (jv0 + 4 * r));
            if (v_half && lane < 32) dma16(1024u * (kVInst - 1) + 16u * lane, rec, st + 1024u * (kVInst - 1));
        }
    };
    if (n_tiles > 0 && wave >= kScoreWaves) issue(0, -1);

    // the head's largest |d_v| over its 64-key groups, by every wavefront for itself
    uint32_t dv = 0;
    {
        const int groups = (int)(p.kv_tiles >> 1);
        const uint32_t *m = p.dvmax + (int64_t)kvh * groups;
        for (int i = lane; i < groups; i += 256) {
            uint32_t a[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) a[j] = i + 64 * j < groups ? m[i + 64 * j] : 0u;
            dv = max(max(dv, max(a[0], a[1])), max(a[2], a[3]));
        }
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) dv = max(dv, (uint32_t)__shfl_xor((int)dv, o));
        dv = (uint32_t)__builtin_amdgcn_readfirstlane((int)dv);
    }
    // e2 with max |d_v| * 2^e2 in [1, 2) (at most 15)
    int e2 = 0;
    {
        const float dm = h2f(dv);
        if (dm > 0.0f) {
            int e;
            (void)frexpf(dm, &e);
            e2 = 1 - e < 15 ? 1 - e : 15;
        }
    }
    // 2^ep rides on P (the score waves' exp2 argument); O and l both carry it,
    // so it cancels in O / l. The lazy rescale keeps P 2^ep <= 2^(ks + ep), and
    // |d_v| < 2^(1 - e2), so A = P 2^ep d_v < 2^(ks + ep + 1 - e2):
    //   e2 >= 0: ep = e2 (at most 7), ks = 8: A < 2^9, P 2^ep <= 2^15;
    //   e2 < 0: ks + ep = 14 + e2 (A < 2^15), ep = 0 while ks can give way
    //     (down to 3), then ep < 0 (to -4 at fp16's largest d_v).
    // Lowering ep instead (ep = e2 for large V, max |d_v| >= 2) put the P of keys
    // a few binades below the row maximum into the fp16 subnormals, where its
    // lo half vanishes: outputs up to 3e-3 x RMS from the exact result. A smaller
    // slack only moves the reference maximum more often.
    int ep = e2 > 7 ? 7 : e2, ks = kSlack;
    if (e2 < 0) {
        const int top = 14 + e2;  // log2 of the largest P 2^ep that A's range admits
        ks = top >= kSlack ? kSlack : (top >= 3 ? top : 3);
        ep = top >= 3 ? 0 : top - 3;
    }
    const float lim_top = (float)(ks + ep);  // the lazy test's bound on s'
    const int nh = (n >> 3) & 1;

    // The two kinds of wave run separate code with the same barrier count:
    // n_tiles + 1 in the loop, then two for the hand-over of m and l.
    if (wave < kScoreWaves) {
        const int w = wave;
        float *ml = reinterpret_cast<float *>(smem + kLdsP) + w * (kRG * 32);  // [rg][row][m, l]
        // Q' hi and lo of rows r = 16 kRG w + 16rg + n (position q_base + r / G, head
        // kvh*G + r % G) as B operands, dims 32b + 8g..+7
        half8 bqh[kRG][8], bql[kRG][8];
        int my_pos[kRG], m_off[kRG];
        float m_run[kRG], l_part[kRG];
        // The logits are accumulated relative to the row's P reference mref =
        // (m_run, or 0 before the first visible key) - ep: s' = s - mref, so that
        // P = 2^s' needs no subtraction, and the lazy-maximum test s > m_run +
        // ks reads s' > lim_s (ks + ep, or -inf before the first visible key).
        // Both change only when the maximum moves.
        float mref[kRG], lim_s[kRG];
#pragma unroll
        for (int rg = 0; rg < kRG; ++rg) {
            const int r = 16 * kRG * w + 16 * rg + n;
            const int pos = q_base + r / p.G;
            my_pos[rg] = pos;
            const bool ok = pos < p.n_q;
            const uint32_t m = ok ? 0xffffffffu : 0u;
            const int64_t row = (int64_t)(ok ? pos : 0) * p.H + kvh * p.G + r % p.G;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                uint4 u = *reinterpret_cast<const uint4 *>(p.qh + row * kHeadDim + 32 * b + 8 * g);
                uint4 v = *reinterpret_cast<const uint4 *>(p.ql + row * kHeadDim + 32 * b + 8 * g);
                u = make_uint4(u.x & m, u.y & m, u.z & m, u.w & m);
                v = make_uint4(v.x & m, v.y & m, v.z & m, v.w & m);
                __builtin_memcpy(&bqh[rg][b], &u, 16);
                __builtin_memcpy(&bql[rg][b], &v, 16);
            }
            const int pl = r / p.G;  // mask row of the position, keys 8g..8g+7
            m_off[rg] = kLdsMask + 64 * pl + 16 * (g ^ ((pl >> 1) & 3));
            m_run[rg] = -INFINITY;
            l_part[rg] = 0.0f;
            mref[rg] = -(float)ep;
            lim_s[rg] = -INFINITY;
        }
        // K operand of key row 16kg + n, dims 32b + 8g..+7: chunk (4b + g) ^ (n & 7),
        // halves swapped when n & 8; the XOR touches bit 2 of 4b + g, so even and odd
        // b use two bases and b >> 1 adds 128 bytes.
        int k_off[2][2];  // [b & 1][half]
#pragma unroll
        for (int bp = 0; bp < 2; ++bp)
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) k_off[bp][hf] = n * 512 + 16 * ((4 * bp + g) ^ (n & 7)) + 8 * (hf ^ nh);
        const int p_off = w * (kRG * 2048) + 16 * lane;  // P slots [w][rg][half][lane]

        for (int t = 0; t <= n_tiles && n_tiles > 0; ++t) {
            // the value waves wait for their DMAs before this barrier, which makes them
            // visible and retires the buffers the new ones overwrite
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (t == n_tiles) break;
            const int64_t kt = k_begin + (int64_t)t * kPK;
            const int nvalid = (int)(k_end - kt < kPK ? k_end - kt : kPK);
            // this tile's four per-lane K bases, opaque to the compiler: every K read
            // is then one of them plus an immediate offset (hoisting all 64
            // base + offset sums out of the loop would need 64 more registers)
            int kb[2][2];
#pragma unroll
            for (int bp = 0; bp < 2; ++bp)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    kb[bp][hf] = (t & 1) * kKStage + k_off[bp][hf];
                    asm volatile("" : "+v"(kb[bp][hf]));
                }
            // mask rows of the tile, read now so that their latency hides behind QK
            uint4 mrow[kRG];
            if (p.mask) {
#pragma unroll
                for (int rg = 0; rg < kRG; ++rg)
                    mrow[rg] = *reinterpret_cast<const uint4 *>(smem + m_off[rg] + (t & 1) * p.mask_stage);
            }
            // ---- S^T: sa[rg][kg][i] = S[key kt + 8g + 4kg + i][row n of group rg] ----
            floatx4 sa[kRG][2];
#pragma unroll
            for (int rg = 0; rg < kRG; ++rg) sa[rg][0] = sa[rg][1] = -mref[rg];
            // d_k of the lane's four C rows 16kg + 4g + i, block b: 8 bytes at
            // Dk[b][16kg + 4g]
            const uint8_t *dkb = smem + (t & 1) * kKStage + kOffDk + 8 * g;
            // Software-pipelined by one step: step j = (block j >> 1, key group j & 1)
            // issues its MFMAs, then the d_k scaling of step j - 1 runs while they
            // execute. The scheduling barrier keeps the compiler from pulling the
            // scaling back next to the MFMAs it reads (it did, leaving 4-12
            // instructions between an MFMA and its consumer). The sum into sa keeps
            // the block order of the plain loop.
            floatx4 cp[kRG];
            uint2 dkp;
#pragma unroll
            for (int j = 0; j <= 16; ++j) {
                floatx4 cn[kRG];
                uint2 dkn;
                if (j < 16) {
                    const int b = j >> 1, kg = j & 1;
                    const int o = kg * 8192 + 128 * (b >> 1);
                    const half8 ak = lds_half8(smem, kb[b & 1][0] + o, kb[b & 1][1] + o);
                    dkn = *reinterpret_cast<const uint2 *>(dkb + 64 * b + 32 * kg);
#pragma unroll
                    for (int rg = 0; rg < kRG; ++rg) {
                        const floatx4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ak, bqh[rg][b],
                                                                                 floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                        cn[rg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ak, bql[rg][b], c, 0, 0, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
                if (j > 0) {
                    const int kg = (j - 1) & 1;
                    _Float16 dk[4];
                    __builtin_memcpy(dk, &dkp, 8);
#pragma unroll
                    for (int rg = 0; rg < kRG; ++rg)
#pragma unroll
                        for (int i = 0; i < 4; ++i) sa[rg][kg][i] = fmaf(cp[rg][i], (float)dk[i], sa[rg][kg][i]);
                }
                if (j < 16) {
                    dkp = dkn;
#pragma unroll
                    for (int rg = 0; rg < kRG; ++rg) cp[rg] = cn[rg];
                }
            }
            float s[kRG][8];  // keys 8g + jj, base-2 logits
#pragma unroll
            for (int rg = 0; rg < kRG; ++rg)
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) s[rg][jj] = sa[rg][jj >> 2][jj & 3];
            // ---- mask / causal / ragged tail ----------------------------------------
            // a block of the mask that is +0 for all of this wave's rows and keys (every
            // fully visible tile of a causal mask) changes no logit: skip it
            bool mask_live = false;
            if (p.mask) {
                uint32_t any = 0;
#pragma unroll
                for (int rg = 0; rg < kRG; ++rg) any |= mrow[rg].x | mrow[rg].y | mrow[rg].z | mrow[rg].w;
                mask_live = __any(any != 0u);
            }
            if (mask_live) {
#pragma unroll
                for (int rg = 0; rg < kRG; ++rg) {
                    const uint32_t mw[4] = {mrow[rg].x, mrow[rg].y, mrow[rg].z, mrow[rg].w};
#pragma unroll
                    for (int jj = 0; jj < 8; ++jj) {
                        // a -inf entry excludes the key whatever its logit (even NaN from
                        // a garbage scale): ggml's CPU loop skips such keys
                        const uint32_t mb = (mw[jj >> 1] >> (16 * (jj & 1))) & 0xffff;
                        s[rg][jj] = mb == 0xFC00u ? -INFINITY : fmaf(h2f(mb), kLog2e, s[rg][jj]);
                    }
                }
            }
            if (nvalid < kPK || (p.q_pos0 >= 0 && kt + kPK - 1 > p.q_pos0 + q_base)) {
#pragma unroll
                for (int rg = 0; rg < kRG; ++rg) {
                    int64_t lim = nvalid;  // keys at or past lim are dead for this row
                    if (p.q_pos0 >= 0 && p.q_pos0 + my_pos[rg] + 1 - kt < lim) lim = p.q_pos0 + my_pos[rg] + 1 - kt;
#pragma unroll
                    for (int jj = 0; jj < 8; ++jj) s[rg][jj] = 8 * g + jj < lim ? s[rg][jj] : -INFINITY;
                }
            }
            // ---- online softmax (base 2); P and the rescale factors to LDS -----------
            uint8_t *pb = smem + kLdsP + (t & 1) * kPBuf + p_off;
            float *ab = reinterpret_cast<float *>(smem + kLdsA + (t & 1) * kABuf) + w * (kRG * 16);
#pragma unroll
            for (int rg = 0; rg < kRG; ++rg) {
                // lazy maximum: the reference moves only when a logit passes it by more
                // than ks, so P <= 2^ks and most tiles need no rescale of O
                float alpha = 1.0f;
                bool over = false;
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) over |= s[rg][jj] > lim_s[rg];
                if (__any(over)) {
                    float mt = fmaxf(fmaxf(fmaxf(s[rg][0], s[rg][1]), fmaxf(s[rg][2], s[rg][3])),
                                     fmaxf(fmaxf(s[rg][4], s[rg][5]), fmaxf(s[rg][6], s[rg][7])));
                    mt = xmax16(mt);
                    mt = xmax32(mt);
                    const float m_new = fmaxf(m_run[rg], mt + mref[rg]);
                    alpha = m_run[rg] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run[rg] - m_new);
                    l_part[rg] *= alpha;
                    m_run[rg] = m_new;
                    // onto the new reference: s - mref_new = s' + (mref - mref_new)
                    const float mref_new = (m_new == -INFINITY ? 0.0f : m_new) - (float)ep;
                    const float d = mref[rg] - mref_new;
#pragma unroll
                    for (int jj = 0; jj < 8; ++jj) s[rg][jj] += d;
                    mref[rg] = mref_new;
                    lim_s[rg] = m_new == -INFINITY ? -INFINITY : lim_top;
                }
                float pf[8], psum = 0.0f;
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) {
                    pf[jj] = __builtin_amdgcn_exp2f(s[rg][jj]);
                    psum += pf[jj];
                }
                l_part[rg] += psum;
                // P as an fp16 hi + lo pair (22 bits): the value waves form P d_v from it
                half8 ph, pl;
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) ph[jj] = (_Float16)pf[jj];
                // the exact residual p - hi, with hi read from its packed fp16 half by
                // v_fma_mix (no conversion of hi back to fp32)
                uint32_t hw[4];
                __builtin_memcpy(hw, &ph, 16);
#pragma unroll
                for (int jj = 0; jj < 8; ++jj) {
                    float r;
                    if (jj & 1)
                        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r) : "v"(pf[jj]), "v"(hw[jj >> 1]));
                    else
                        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,0] op_sel_hi:[0,0,1]" : "=v"(r) : "v"(pf[jj]), "v"(hw[jj >> 1]));
                    pl[jj] = (_Float16)r;
                }
                *reinterpret_cast<half8 *>(pb + rg * 2048) = ph;
                *reinterpret_cast<half8 *>(pb + rg * 2048 + 1024) = pl;
                if (g == 0) ab[rg * 16 + n] = alpha;
            }
        }
        // ---- hand m and l of the rows to the value waves ----------------------------
        __syncthreads();
        if (n_tiles > 0) {
#pragma unroll
            for (int rg = 0; rg < kRG; ++rg) {
                float lp = l_part[rg];
                lp += __shfl_xor(lp, 16);
                lp += __shfl_xor(lp, 32);
                if (g == 0) {
                    ml[rg * 32 + 2 * n] = m_run[rg];
                    ml[rg * 32 + 2 * n + 1] = lp;
                }
            }
        }
        __syncthreads();
        return;
    }

    // ---- value waves: O[row 16 kRG w + 16rg + 4g + i][dim 16T + n] ----------------
    const int w = wave - kScoreWaves;
    const float *ml = reinterpret_cast<const float *>(smem + kLdsP) + w * (kRG * 32);  // [rg][row][m, l]
    // V operand of dim 16T + n, keys 8g..8g+7: chunk g ^ ((n >> 1) & 3), halves swapped when n & 8.
    const int v_off0 = 64 * n + 16 * (g ^ ((n >> 1) & 3)) + 8 * nh;
    const int v_off1 = v_off0 ^ 8;
    const int p_off = w * (kRG * 2048) + 16 * lane;
    floatx4 acc[kRG][16];
#pragma unroll
    for (int rg = 0; rg < kRG; ++rg)
#pragma unroll
        for (int T = 0; T < 16; ++T) acc[rg][T] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t <= n_tiles && n_tiles > 0; ++t) {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        issue(t + 1 < n_tiles ? t + 1 : -1, t < n_tiles ? t : -1);
        if (t == 0) continue;
        const int tp = t - 1;
        const uint8_t *vs = smem + kLdsV + (tp & 1) * kVStage;
        // this tile's two per-lane V bases, opaque to the compiler (see the K reads)
        int vb0 = kLdsV + (tp & 1) * kVStage + v_off0, vb1 = kLdsV + (tp & 1) * kVStage + v_off1;
        asm volatile("" : "+v"(vb0), "+v"(vb1));
        const uint8_t *pb = smem + kLdsP + (tp & 1) * kPBuf + p_off;
        const float *ab = reinterpret_cast<const float *>(smem + kLdsA + (tp & 1) * kABuf) + w * (kRG * 16);
        half8 ph[kRG], pl[kRG];
        bool resc = false;
#pragma unroll
        for (int rg = 0; rg < kRG; ++rg) {
            // rescale factors of rows 4g..4g+3: exactly 1 unless a maximum moved
            const floatx4 a4 = *reinterpret_cast<const floatx4 *>(ab + rg * 16 + 4 * g);
            resc |= (a4[0] != 1.0f) | (a4[1] != 1.0f) | (a4[2] != 1.0f) | (a4[3] != 1.0f);
            ph[rg] = *reinterpret_cast<const half8 *>(pb + rg * 2048);
            pl[rg] = *reinterpret_cast<const half8 *>(pb + rg * 2048 + 1024);
        }
        if (__any(resc)) {  // rare with the lazy maximum: O = alpha O
#pragma unroll
            for (int rg = 0; rg < kRG; ++rg) {
                const floatx4 a4 = *reinterpret_cast<const floatx4 *>(ab + rg * 16 + 4 * g);
#pragma unroll
                for (int T = 0; T < 16; ++T) acc[rg][T] *= a4;
            }
        }
        // d_v of the 8 blocks and V of block 0 first, then V of block b + 1 while
        // block b computes: the LDS latency stays off the MFMA chain
        uint4 dvr[8];
#pragma unroll
        for (int b = 0; b < 8; ++b) dvr[b] = *reinterpret_cast<const uint4 *>(vs + kOffDv + 64 * b + 16 * g);
        half8 bvn[2];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) bvn[hf] = lds_half8(smem, vb0 + 1024 * hf, vb1 + 1024 * hf);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const half8 bv[2] = {bvn[0], bvn[1]};
            if (b < 7) {
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
                    bvn[hf] = lds_half8(smem, vb0 + 1024 * (2 * b + 2 + hf), vb1 + 1024 * (2 * b + 2 + hf));
            }
            half8 dvb;
            __builtin_memcpy(&dvb, &dvr[b], 16);
            // A = P 2^ep d_v as an fp16 hi + lo pair (22 bits): the products with the
            // exact V codes are then exact in fp32, so a row that a few keys
            // dominate carries no fp16 rounding of P d_v into its output. Ph d_v has
            // at most 22 significant bits, so its residual after rounding to fp16
            // (at most 11 bits) is exact in one fma; Pl d_v is 2^-11 of it and
            // rounds once.
            half8 ah[kRG], al[kRG];
#pragma unroll
            for (int rg = 0; rg < kRG; ++rg) {
                ah[rg] = ph[rg] * dvb;
                const half8 r = __builtin_elementwise_fma(ph[rg], dvb, -ah[rg]);
                al[rg] = __builtin_elementwise_fma(pl[rg], dvb, r);
            }
#pragma unroll
            for (int rg = 0; rg < kRG; ++rg)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
                    acc[rg][2 * b + hf] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[rg], bv[hf], acc[rg][2 * b + hf], 0, 0, 0);
#pragma unroll
            for (int rg = 0; rg < kRG; ++rg)
#pragma unroll
                for (int hf = 0; hf < 2; ++hf)
                    acc[rg][2 * b + hf] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al[rg], bv[hf], acc[rg][2 * b + hf], 0, 0, 0);
        }
    }
    __syncthreads();  // m and l of the rows ...
    __syncthreads();  // ... are in LDS
    const int rows_total = p.n_q * p.H;
#pragma unroll
    for (int rg = 0; rg < kRG; ++rg) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 16 * kRG * w + 16 * rg + 4 * g + i;
            const int qrow = q_base + r / p.G, hrow = kvh * p.G + r % p.G;
            if (qrow >= p.n_q) continue;
            const float mrow = n_tiles > 0 ? ml[rg * 32 + 2 * (4 * g + i)] : -INFINITY;
            const float lrow = n_tiles > 0 ? ml[rg * 32 + 2 * (4 * g + i) + 1] : 0.0f;
            const int64_t ridx = (int64_t)qrow * p.H + hrow;
            if (p.n_splits == 1) {
                const float inv = lrow == 0.0f ? 0.0f : 1.0f / lrow;
#pragma unroll
                for (int T = 0; T < 16; ++T) {
                    float o = acc[rg][T][i] * inv;
                    if (p.gate) {
                        const float gv = reinterpret_cast<const float *>(p.gate + qrow * p.gate_nb2 +
                                                                         hrow * p.gate_nb1)[16 * T + n];
                        o = o * (1.0f / (1.0f + expf(-gv)));
                    }
                    store_through(p.dst + ridx * kHeadDim + 16 * T + n, o);
                }
            } else {
                float *pa_out = p.part_acc + ((int64_t)split * rows_total + ridx) * kHeadDim;
#pragma unroll
                for (int T = 0; T < 16; ++T) store_through(pa_out + 16 * T + n, acc[rg][T][i]);
                if (n == 0) {
                    // the combine works in base e: m * ln 2 (acc and l of every split
                    // carry the same 2^ep, which cancels in the merge)
                    store_through(p.part_ml + ((int64_t)split * rows_total + ridx) * 2,
                                  mrow == -INFINITY ? mrow : mrow * 0.6931471805599453f);
                    store_through(p.part_ml + ((int64_t)split * rows_total + ridx) * 2 + 1, lrow);
                }
            }
        }
    }
}

struct PrefillPlan {
    int64_t kv_tiles;
    int rg, qb, q_tiles, mask_stage;
    int64_t most, least;  // key splits: that the plan may choose; that a workspace has to hold
    size_t off_kv, off_dvmax, off_qh, off_ql, off_mask, off_lim, off_pa, total;
};

size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

// Bytes of the split partials of `rows` rows: O [n_splits][rows][256], then (m, l)
size_t partial_acc_bytes(int64_t n_splits, int64_t rows) { return al256((size_t)(n_splits * rows) * kHeadDim * 4); }
size_t partial_bytes(int64_t n_splits, int64_t rows) {
    return n_splits > 1 ? partial_acc_bytes(n_splits, rows) + al256((size_t)(n_splits * rows) * 8) : 0;
}

// Key splits that are worth a try. A workgroup fills a CU (LDS), so the workgroups
// of one split (wgs = q_tiles per KV head) run in rounds of one per CU. Up to an
// eighth of the CUs, whole splits fill a round to 8/9 or more. With more workgroups
// per split, the fewest splits that fill their rounds best, of up to kMaxRounds
// rounds: 160 workgroups run 2 rounds of 3 splits, where one or two splits leave
// 3/8 of each round idle; 64 run one round of 4, and no more fill it better (us per
// call with the count that 4 rounds would allow and the estimate then takes / with
// this one: 1233 queries on 5303 keys 315 / 248, 1345 on 8800 (4 KV heads) 474 / 438,
// 1555 on 9975 (8 heads on 1) 355 / 278). A skewed chunk, half of whose workgroups
// may see no key, is tried up to twice the splits that one round takes; its context is
// short, so the size that the longest one of them asks for is kept for all longer ones.
// Up to kOneSplitKeys keys a chunk stays whole: its output and gate leave in the
// attention kernel's epilogue, with no partials and no merge. The line is a bound on
// what a short context asks for, not where the forms cross: first chunks, us per call
// whole in 64-row workgroups / in 128-row ones with the best split count: 448 queries
// 30.0 / 33.2, 512 32.6 / 34.7, 544 34.0 / 36.5, 640 37.9 / 38.3, 768 42.8 / 42.9, 1024 52.1 /
// 53.8 (with 2 or 3 splits of 64-row workgroups 28.8 at 512, 33.8 at 640), so the first
// is taken up to the line and the second past it; and a few queries on a full 512 keys
// walk 16 tiles in a row (8 queries 29.9, 19.9 on 768 keys in 64-key splits).
constexpr int kMinSplitTiles = 2;  // 64 keys
constexpr int kMaxRounds = 4;
constexpr int kRoundTiles = 16;  // tiles of a split past the first round: the estimate hardly ever takes fewer
constexpr int kOneSplitKeys = 512;
bool skewed(int64_t n_q, int64_t n_kv) { return n_kv < 4 * n_q; }
int64_t max_splits(int64_t n_kv, int64_t wgs, bool skew) {
    if (n_kv <= kOneSplitKeys) return 1;
    const int64_t cus = device_cu_count();
    const int64_t by_len = ((n_kv + kPK - 1) / kPK + kMinSplitTiles - 1) / kMinSplitTiles;
    int64_t s = cus / wgs;
    if (8 * wgs > cus) {
        const int64_t rounds = kMaxRounds * cus / wgs;
        float best = 0.0f;
        s = 1;
        for (int64_t i = 1; i <= rounds; ++i) {
            const float fill = (float)(i * wgs) / (float)((i * wgs + cus - 1) / cus * cus);
            if (fill > 1.01f * best) best = fill, s = i;
        }
        const int64_t one = (cus + wgs - 1) / wgs, filled = (n_kv + kRoundTiles * kPK - 1) / (kRoundTiles * kPK);
        if (!skew && s > one && s > filled) s = one > filled ? one : filled;
        if (skew) s = 2 * one < rounds ? 2 * one : rounds;
    }
    if (s > by_len) s = by_len;
    if (s > kMaxSplits) s = kMaxSplits;
    return s < 1 ? 1 : s;
}

// Keys per split, a multiple of kPK: the candidate of least estimated time, in
// units of one tile of one workgroup. Measured: 2.2 us with the chip full, down to
// 0.75 of that with few CUs busy; a workgroup costs about kWgTiles tiles beside
// its own (start, Q rows, fill and drain, output), the merge kMergeTiles plus
// kMergeRow per row and split (1 KB written and read). The chunk is taken as
// causal and the last n_q keys as its own (a mask or a position may say
// otherwise: the estimate is then off, the result not). Workgroups that see no
// key leave at once; of the others, in dispatch order, round k starts with
// workgroup k * CUs and is taken to last as long as that one. Splitting at all
// must be worth kMargin: the estimate is no better than that. us per call (16
// heads on 2, pre-passes and merge included) with ceil(CUs / wgs) splits of 512
// keys or more, with this choice, and with the best split count of all tried:
//   37 queries on 20048 keys    75.0  65.1
//   300 on 3301                 94   65   64 (7 splits were 266 workgroups)
//   600 on 20600               610  432  426
//   405 on 171568             4390 2331
//   1280 on 6280               401  297  293
constexpr float kWgTiles = 2.0f, kMergeTiles = 2.0f, kMergeRow = 1.2e-4f, kMargin = 0.98f;
float tile_time(float busy) { return 0.75f + 0.25f * busy; }  // busy: share of the CUs
int64_t split_keys(int64_t n_q, int64_t n_kv, int64_t Hkv, int64_t qb, int64_t q_tiles, int64_t rows, int64_t most) {
    const int64_t cus = device_cu_count(), wgs = q_tiles * Hkv;
    const int64_t tiles = (n_kv + kPK - 1) / kPK;
    // key tiles that query tile i sees: first + i * step, at most all
    const float step = (float)qb / kPK;
    const float first = ((float)(n_kv > n_q ? n_kv - n_q : 0) + (float)qb) / kPK;
    int64_t best_len = tiles, last_len = 0;
    float best = INFINITY;
    for (int64_t s = 1; s <= most; ++s) {
        const int64_t len = (tiles + s - 1) / s;
        if (len == last_len) continue;
        last_len = len;
        const int64_t n_s = (tiles + len - 1) / len;
        float t = 0.0f, last = 0.0f;  // estimate, its last round
        int64_t next = 0;             // first workgroup of the next round
        auto round = [&](float n) {
            last = n + kWgTiles;
            t += last;
            next += cus;
        };
        // the splits that every query tile sees whole, then the others one by one
        int64_t j = (int64_t)(first / (float)len);
        if (j > n_s - 1) j = n_s - 1;
        int64_t live = j * wgs;  // workgroups with keys
        float work = (float)(live * len);
        while (next < live) round((float)len);
        for (; j < n_s; ++j) {
            const float at = (float)(j * len);
            // query tiles i0 .. q_tiles - 1 reach into it, the last one furthest
            const int64_t i0 = first > at ? 0 : (int64_t)((at - first) / step) + 1;
            if (i0 >= q_tiles) break;
            const float all = (float)(j == n_s - 1 ? tiles - j * len : len);
            const float lo = first + (float)i0 * step - at, hi = first + (float)(q_tiles - 1) * step - at;
            const int64_t here = (q_tiles - i0) * Hkv;
            while (next < live + here) round(fminf(all, hi - (float)((next - live) / Hkv) * step));
            live += here;
            work += (float)here * (lo >= all ? all : 0.5f * (lo + fminf(hi, all)));
        }
        const float part = live > cus ? (float)(live - (next - cus)) / (float)cus : work / ((float)cus * (last - kWgTiles));
        t += last * (tile_time(fminf(part, 1.0f)) - 1.0f);
        t = n_s > 1 ? t + kMergeTiles + kMergeRow * (float)(n_s * rows) : kMargin * t;
        if (t < best) best = t, best_len = len;
    }
    return best_len * kPK;
}

// The same for a chunk whose query tiles see ranges of very different length (its
// workgroups go out longest first, see the kernel), by walking through the dispatch:
// workgroups are dealt strictly in turn to the XCDs and, inside one, in order and in
// turn to its shader engines. One that finds its engine's CUs taken waits, and all
// behind it with it, while CUs of the other engines are free; the dead workgroups of
// a split take their turns. With that, 512 times of 64 causal chunks (300 to 2048
// queries on 300 to 7169 keys, 1 to 8 splits, 16 heads on 2 or 4, 8 on 1) are met to
// 2.3% RMS; with CUs taken as they come free inside an XCD to 4.4%. In tiles of 1.78
// us. us per call with the estimate above, which takes dead workgroups as gone, with
// this one, and with the best count of 1 to 12:
//   768 queries on 768 keys     55.5  43.2  43.2 (before either 51.7)
//   1500 on 1951               126.8 107.2 107.2
//   1500 on 3001               180.4 157.2 157.2
//   2000 on 2000, 4 KV heads   129.0 112.9 112.9
//   600 on 1201, 8 heads on 1   49.0  36.0  36.0
//   1300 on 1700, 4 on 4        54.9  41.7  41.7
//   800 on 800, 4 on 4          35.7  34.8  30.8 (9 splits; kSkewMany: 245 on 576,
//   8 on 2, 28.7 with 6 splits and 30.7 with 9)
// Over 142 random shapes (132 to 2048 queries, 1 to 8 KV heads, every count up to 16)
// its choice costs 0.4% more than the best count on average, 5% of the shapes lose
// more than 3%; with the estimate above it was 3.2% and 25%. Host time 1 to 5 us.
constexpr int kXcds = 8, kEngines = 4, kMaxEngineCus = 16;
constexpr float kSkewWg = 5.0f, kSkewDead = 0.5f, kSkewMerge = 3.3f, kSkewRow = 0.85e-4f, kSkewMany = 0.55f;
// a split chunk has to be clearly ahead of an unsplit one, and a second round of a
// first one (2000 queries on 4001 keys, 8 on 1: 135 us with 2 splits, 142 with 5)
constexpr float kSkewMargin = 0.96f, kSkewLate = 1.04f;
constexpr int64_t kSkewFew = 8;  // splits up to which a wavefront merges a row by itself
int64_t split_skewed(int64_t n_q, int64_t n_kv, int64_t Hkv, int64_t qb, int64_t q_tiles, int64_t rows, int64_t most) {
    // at most kMaxRounds * CUs workgroups where there is a choice, and n_kv < 4 n_q
    const int wgs = (int)(q_tiles * Hkv), tiles = (int)((n_kv + kPK - 1) / kPK), hkv = (int)Hkv;
    if (most <= 1) return (int64_t)tiles * kPK;
    // keys up to the end of the last query tile, were it whole
    const int ends = (int)((n_kv > n_q ? n_kv - n_q : 0) + q_tiles * qb), rows_qb = (int)qb;
    int cus = device_cu_count() / (kXcds * kEngines);  // of an engine
    cus = cus < 1 ? 1 : (cus > kMaxEngineCus ? kMaxEngineCus : cus);
    int best_len = tiles, last_len = 0;
    float best = INFINITY;
    for (int s = 1; s <= (int)most; ++s) {
        const int len = (tiles + s - 1) / s;
        if (len == last_len) continue;
        last_len = len;
        const int n_s = (tiles + len - 1) / len, total = n_s * wgs;
        const float first = (float)len + kSkewWg;
        const float merge = n_s == 1 ? (kSkewMargin - 1.0f) * first
                                     : kSkewMerge + kSkewRow * (float)(n_s * rows) + (n_s > kSkewFew ? kSkewMany : 0.0f);
        float end = first, late = 1.0f;  // of the last workgroup; that of the first one at least
        for (int x : {0, kXcds / 2}) {  // two XCDs stand for all (the same picks)
            if (end + merge >= best) break;
            float at[kEngines][kMaxEngineCus], now = 0.0f;  // a CU is busy up to here; the time of the dispatch
            int r = x, from = 0, e = 0, c = 0, live = 0;    // place in its split, the split's first tile; engine, CU
            for (int i = x; i < total; i += kXcds, r += kXcds) {
                for (; r >= wgs; r -= wgs) from += len;
                // tiles up to the last query of its query tile, inside the split
                const int keys = ends - r / hkv * rows_qb;
                const int sees = (keys < (int)n_kv ? (keys + kPK - 1) / kPK : tiles) - from;
                const float busy = sees > 0 ? (float)(sees < len ? sees : len) + kSkewWg : kSkewDead;
                live += sees > 0;
                float *cu = &at[e][c];
                if (c == cus) {  // all taken once: the one that is free first
                    cu = at[e];
                    for (int j = 1; j < cus; ++j) cu = at[e][j] < *cu ? &at[e][j] : cu;
                    now = *cu > now ? *cu : now;
                }
                *cu = now + busy;
                end = *cu > end ? *cu : end;
                if (++e == kEngines) e = 0, c += c < cus;
            }
            if (live > cus * kEngines) late = kSkewLate;
        }
        end *= late;
        if (end + merge < best) best = end + merge, best_len = len;
    }
    return (int64_t)best_len * kPK;
}

PrefillPlan plan(int64_t n_q, int64_t H, int64_t Hkv, int64_t n_kv) {
    PrefillPlan pl{};
    const int G = (int)(H / Hkv);
    // 64-row workgroups where 128 rows would leave most of their work to padding or
    // most of the chip idle: a query tile of all the rows, and an unsplit chunk (for
    // that line see max_splits) whose 64-row workgroups still run in one round. A tile
    // of keys costs them about 1.5 us where 128 rows take 2.2 to 2.4: us per call 128
    // rows / 64 rows 512 first queries 48.3 / 35.1, 200 first queries 32.3 / 21.5, 8 on
    // 3008 keys 34 / 24.
    const int64_t cus = device_cu_count();
    const int64_t wgs64 = (n_q + rows_per_wg(1) / G - 1) / (rows_per_wg(1) / G) * Hkv;
    pl.rg = n_q * G <= rows_per_wg(1) || (n_kv <= kOneSplitKeys && wgs64 <= cus) ? 1 : 2;
    pl.qb = rows_per_wg(pl.rg) / G;
    pl.mask_stage = pl.qb * kPK * 2;
    pl.kv_tiles = (n_kv + 63) / 64 * 2;  // the pre-pass writes 64-key groups
    pl.q_tiles = (int)((n_q + pl.qb - 1) / pl.qb);
    const int64_t wgs = pl.q_tiles * Hkv, rows = n_q * H;
    pl.most = max_splits(n_kv, wgs, skewed(n_q, n_kv));
    // one round of splits of 512 keys or more
    pl.least = (cus + wgs - 1) / wgs;
    if (pl.least > (n_kv + 511) / 512) pl.least = (n_kv + 511) / 512;
    if (pl.least > pl.most) pl.least = pl.most;
    size_t o = 0;
    pl.off_kv = o; o = al256(o + (size_t)Hkv * pl.kv_tiles * kTileBytes);
    pl.off_dvmax = o; o = al256(o + (size_t)Hkv * (size_t)(pl.kv_tiles / 2) * 4);
    pl.off_qh = o; o = al256(o + (size_t)n_q * H * kHeadDim * 2);
    pl.off_ql = o; o = al256(o + (size_t)n_q * H * kHeadDim * 2);
    pl.off_mask = o; o = al256(o + (size_t)n_q * ((n_kv + 7) / 8 * 8) * 2);
    pl.off_lim = o; o = al256(o + (size_t)pl.q_tiles * 4);
    pl.off_pa = o;
    pl.total = o + partial_bytes(pl.most, rows) + 256;
    return pl;
}

// A workspace sized for a longer cache serves every shorter one: the layout before
// the partials grows with n_kv, the splits of a chunk that is not skewed do, and
// those of skewed chunks are all asked for by the longest of them.
size_t plan_bytes(int64_t n_q, int64_t H, int64_t Hkv, int64_t n_kv) {
    const size_t here = plan(n_q, H, Hkv, n_kv).total;
    if (skewed(n_q, n_kv)) return here;
    const size_t skew = plan(n_q, H, Hkv, 4 * n_q - 1).total;
    return here > skew ? here : skew;
}

// Keys per split with partials of at most `most` splits
int64_t split_len(const PrefillPlan &pl, int64_t n_q, int64_t H, int64_t Hkv, int64_t n_kv, int64_t most) {
    return skewed(n_q, n_kv) ? split_skewed(n_q, n_kv, Hkv, pl.qb, pl.q_tiles, n_q * H, most)
                             : split_keys(n_q, n_kv, Hkv, pl.qb, pl.q_tiles, n_q * H, most);
}

}  // namespace

size_t fa_prefill_workspace(int64_t n_q, int64_t H, int64_t Hkv, int64_t n_kv) {
    return plan_bytes(n_q, H, Hkv, n_kv);
}

int launch_fa_prefill(const FaArgs &a, hipStream_t s) {
    const sqa_tensor &q = *a.q, &k = *a.k, &v = *a.v;
    const int64_t n_q = q.ne[1], H = q.ne[2], n_kv = k.ne[1], Hkv = k.ne[2];
    const int G = (int)(H / Hkv);
    if (16 % G != 0) return set_error(SQA_ERR_UNSUPPORTED, "prefill: n_head/n_head_kv must divide 16");
    const PrefillPlan pl = plan(n_q, H, Hkv, n_kv);
    // A workspace sized for another shape may hold fewer partials than the plan would
    // use (the size is not monotone in n_q): the chunk then takes fewer splits.
    const int64_t rows = n_q * H;
    const size_t need = pl.off_pa + partial_bytes(pl.least, rows) + 256;
    if (!a.ws || a.ws_bytes < need)
        return set_error(SQA_ERR_WORKSPACE, "flash_attn_ext: workspace %zu bytes < %zu needed", a.ws_bytes, need);
    int64_t most = pl.most;
    while (a.ws_bytes < pl.off_pa + partial_bytes(most, rows) + 256) --most;  // down to pl.least
    const int64_t len = split_len(pl, n_q, H, Hkv, n_kv, most);
    const int n_splits = (int)((n_kv + len - 1) / len);
    uint8_t *base = reinterpret_cast<uint8_t *>(((uintptr_t)a.ws + 255) & ~(uintptr_t)255);
    uint8_t *kv = base + pl.off_kv;
    uint32_t *dvmax = reinterpret_cast<uint32_t *>(base + pl.off_dvmax);
    uint16_t *qh = reinterpret_cast<uint16_t *>(base + pl.off_qh);
    uint16_t *ql = reinterpret_cast<uint16_t *>(base + pl.off_ql);

    PrefillParams p;
    p.mask = nullptr;
    p.mask_nb1 = 0;
    p.mask_len = 0;
    const char *mask_src = nullptr;
    int64_t mask_src_nb1 = 0;
    if (a.q_pos0 < 0 && a.mask) {
        mask_src = (const char *)a.mask->data;
        mask_src_nb1 = (int64_t)a.mask->nb[1];
        if ((uintptr_t)mask_src % 16 == 0 && mask_src_nb1 % 16 == 0 && n_kv % 8 == 0) {
            p.mask = mask_src;
            p.mask_nb1 = mask_src_nb1;
            p.mask_len = n_kv;
            mask_src = nullptr;
        } else {
            const int64_t len8 = (n_kv + 7) / 8 * 8;
            p.mask = (const char *)(base + pl.off_mask);
            p.mask_nb1 = len8 * 2;
            p.mask_len = len8;
        }
        // the mask DMA addresses rows with 32-bit offsets
        if ((n_q - 1) * p.mask_nb1 + p.mask_len * 2 > (int64_t)UINT32_MAX)
            return set_error(SQA_ERR_UNSUPPORTED, "prefill: mask of %lld rows x %lld bytes exceeds 4 GiB",
                             (long long)n_q, (long long)p.mask_nb1);
    }

    int prof = profile_start("fa_prefill_prep", s);
    {
        const int64_t nqb = n_q * H * kBlocksPerHead;
        const int qblocks = (int)((4 * nqb + 255) / 256);
        int32_t *lim = reinterpret_cast<int32_t *>(base + pl.off_lim);
        // an in-place mask is scanned by extra workgroups of the pre-pass, a packed
        // copy by a kernel of its own once it is written
        const MaskScan ms{p.mask && !mask_src ? p.mask : nullptr, p.mask_nb1, p.mask_len, pl.qb, pl.q_tiles, lim};
        const QPrep qp{(const char *)q.data, (int64_t)q.nb[1], (int64_t)q.nb[2], (int)n_q, (int)H, a.scale * kLog2e,
                       qh, ql, (uintptr_t)q.data % 16 == 0 && q.nb[1] % 16 == 0 && q.nb[2] % 16 == 0};
        const KvPrep kp{(const uint8_t *)k.data, (const uint8_t *)v.data, (int64_t)k.nb[1], (int64_t)k.nb[2],
                        (int64_t)v.nb[1], (int64_t)v.nb[2], n_kv, pl.kv_tiles, (int)Hkv, (int)(pl.kv_tiles / 2), kv,
                        dvmax};
        prep_kernel<<<dim3((unsigned)(kp.groups * kp.hkv + (ms.mask ? pl.q_tiles : 0) + qblocks)), dim3(256), 0, s>>>(
            kp, qp, ms);
        if (mask_src) {
            int64_t grid = (p.mask_len * n_q + 255) / 256;
            if (grid > 2048) grid = 2048;
            pf_mask_pack_kernel<<<dim3((unsigned)grid), dim3(256), 0, s>>>(
                mask_src, mask_src_nb1, n_kv, (int)n_q, p.mask_len, (uint16_t *)(base + pl.off_mask));
        }
        if (mask_src)  // the packed copy, just written
            mask_tile_limit_kernel<<<dim3((unsigned)pl.q_tiles), dim3(256), 0, s>>>(
                p.mask, p.mask_nb1, p.mask_len, (int)n_q, pl.qb, reinterpret_cast<int32_t *>(base + pl.off_lim));
    }
    profile_stop(prof, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_status(e, "prefill pre-pass launch");

    p.tile_lim = p.mask ? reinterpret_cast<const int32_t *>(base + pl.off_lim) : nullptr;
    p.kv = kv;
    p.dvmax = dvmax;
    p.qh = qh;
    p.ql = ql;
    p.n_kv = n_kv;
    p.kv_tiles = pl.kv_tiles;
    p.n_q = (int)n_q;
    p.H = (int)H;
    p.G = G;
    p.Hkv = (int)Hkv;
    p.q_pos0 = a.q_pos0;
    p.n_splits = n_splits;
    p.q_tiles = pl.q_tiles;
    p.split_len = len;
    p.skew = skewed(n_q, n_kv);
    p.qb = pl.qb;
    p.mask_stage = pl.mask_stage;
    p.part_acc = reinterpret_cast<float *>(base + pl.off_pa);
    p.part_ml = reinterpret_cast<float *>(base + pl.off_pa + partial_acc_bytes(n_splits, rows));
    p.dst = (float *)a.dst->data;
    p.gate = (n_splits == 1 && a.gate) ? (const char *)a.gate->data : nullptr;
    p.gate_nb1 = a.gate ? (int64_t)a.gate->nb[1] : 0;
    p.gate_nb2 = a.gate ? (int64_t)a.gate->nb[2] : 0;

    const int lds_bytes = kLdsMask + (p.mask ? 2 * pl.mask_stage : 0);
    // The function's LDS limit is raised once per process to the largest size
    // any launch uses, so concurrent first calls cannot leave a smaller one set.
    static std::once_flag lds_once;
    static hipError_t lds_err = hipSuccess;
    std::call_once(lds_once, [] {
        lds_err = hipFuncSetAttribute((const void *)fa_prefill_kernel<1>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      kLdsMaxBytes);
        if (lds_err == hipSuccess)
            lds_err = hipFuncSetAttribute((const void *)fa_prefill_kernel<2>,
                                          hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMaxBytes);
    });
    if (lds_err != hipSuccess) return hip_status(lds_err, "fa_prefill LDS attribute");
    prof = profile_start("fa_prefill", s);
    const dim3 grid((unsigned)(pl.q_tiles * Hkv * n_splits));
    if (pl.rg == 1)
        fa_prefill_kernel<1><<<grid, dim3(kThreads), lds_bytes, s>>>(p);
    else
        fa_prefill_kernel<2><<<grid, dim3(kThreads), lds_bytes, s>>>(p);
    profile_stop(prof, s);
    e = hipGetLastError();
    if (e != hipSuccess) return hip_status(e, "fa_prefill launch");
    if (n_splits > 1)
        return launch_fa_combine(p.part_acc, p.part_ml, n_splits, (int)rows, p.dst, a.gate, (int)H, s);
    return SQA_OK;
}

}  // namespace sqa
