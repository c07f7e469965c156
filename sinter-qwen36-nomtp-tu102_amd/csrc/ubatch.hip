// Batched GEMV over a ubatch of tokens: the trunk GEMM of a batched prefill
// (docs/PREFILL-SEMANTICS.md:286-313 in the reference: the fork's prefill
// multiplies quantised weights by quantised activations on int8 tensor
// cores, MMQ, instead of running the single-token GEMV once per token).
//
//   y[t][r] = (float) sum_i term(W[r] item i, X[t] item i),  t < n_tokens
//
// W: rows x K of ggml Q4_K or Q6_K super-blocks (the GGUF layout as-is);
// X: n_tokens Q8_K activations (ggml block_q8_K {f32 d; i8 qs[256];
// i16 bsums[16]}, K/256 blocks per token; the sums are taken from the codes).
// The item terms and their fold are the single-token GEMV's (gemv.h: one fp64
// term per 256-element super-block, summed in item order), so every output is
// bit-identical to the decode GEMV of the same token; only the integer dot
// products move to MFMA.
//
// Both kernels below work on 16 rows x 16 tokens x one item: A = the tokens'
// codes (lane l: token l%16), B = the rows' codes times their sub-block
// scales (lane l: row l%16), D (lane l: row l%16, tokens 4(l/16)+v) the item's
// exact integer sums.  An item takes four 64-deep v_mfma_i32_16x16x64_i8 per
// digit of code x scale.  Lane group g = l/16 holds 16 consecutive elements
// of each 64 (WItem::chunk), all of one sub-block: one scale per lane and MFMA.
//   Q4_K: the 6-bit scale is 8 hi + lo; code x digit (<= 15 * 7) is an int8.
//     The min term sum_s m_s (sum of sub-block s's codes) is a third MFMA per
//     chunk, against m_s in every byte.
//   Q6_K: (code - 32) x scale, at most 4096 in magnitude, is split into
//     256 h + l with l the signed low byte.
// Each lane then forms the fp64 terms of its four (token, row) pairs: per
// pair ((dw * isum) * dx) [- ((dmin * msum) * dx)], equal bit for bit to the
// decode's (dw * dx) * isum: dw (f16), dx (f32) and the integer leave either
// first product exact, so both round once, the same exact value.
#include <algorithm>
#include <cmath>

#include "batched.h"
#include "internal.h"
#include "dev_common.h"

namespace sinter {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));
typedef double v2d __attribute__((ext_vector_type(2)));
// 16 bytes at a 4-byte boundary (one global_load_dwordx4), 4 at a 2-byte one
typedef struct __attribute__((packed, aligned(4))) { uint32_t d[4]; } u128_a4;
typedef struct __attribute__((packed, aligned(2))) { uint32_t d; } u32_a2;

constexpr uint32_t UB_TOK = 16;      // tokens per tile: the MFMA's M
constexpr uint32_t UB_ROWS = 16;     // rows per wave: the MFMA's N
constexpr uint32_t UB_CONV_MAX = 8;    // conv taps
constexpr uint32_t Q8K_BYTES = 292;  // block_q8_K
constexpr uint32_t Q4K_BYTES = 144, Q6K_BYTES = 210;

__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}
// both 16-bit halves of x times s, modulo 2^16 (one v_pk_mul_lo_u16: four
// byte codes times a digit when no product leaves its byte; a 32-bit multiply
// would take four times the issue slots)
__device__ __forceinline__ uint32_t pk_mul(uint32_t x, uint32_t s) {
    const us2 r = __builtin_bit_cast(us2, x) * (us2)((unsigned short)s);
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t pk_mad(uint32_t x, uint32_t s, uint32_t c) {
    const us2 r = __builtin_bit_cast(us2, x) * (us2)((unsigned short)s) + (us2)((unsigned short)c);
    return __builtin_bit_cast(uint32_t, r);
}

// One item's MFMA operands of a wave: chunk m of four, the low and high
// digits of code x scale; the block scales.
struct BItem {
    v4i lo[4], hi[4];
    v4i mn[4];       // Q4_K: the chunk's min in every byte
    float dw, dmin;
};

template <int WT>
struct WItem;

// Q4_K.  Chunk m = 2P + n of lane group g: elements 128P + 64(g/2) + 32n +
// 16(g%2) .. +15 -- n is the nibble, so the lane's two 16-byte loads of qs
// (at 64P + 16g) serve two chunks each and no byte is loaded twice.
template <>
struct WItem<SINTER_Q4_K> {
    static constexpr uint32_t BYTES = Q4K_BYTES;
    static constexpr int HI_SHIFT = 3;   // value = lo + (hi << 3)
    uint32_t h[4];
    uint32_t q[8];
    // the 16-byte chunk (of the item's 16) that lane group g multiplies in MFMA m
    static __device__ __forceinline__ uint32_t chunk(uint32_t m, uint32_t g) {
        return 8u * (m >> 1) + 4u * (g >> 1) + 2u * (m & 1u) + (g & 1u);
    }
    __host__ __device__ __forceinline__ void load(const uint8_t *b, uint32_t g) {
        const uint4 hv = *(const uint4 *)b;
        h[0] = hv.x; h[1] = hv.y; h[2] = hv.z; h[3] = hv.w;
#pragma unroll
        for (uint32_t P = 0; P < 2; P++) {
            const uint4 v = *(const uint4 *)(b + 16u + 64u * P + 16u * g);
            q[4 * P] = v.x; q[4 * P + 1] = v.y; q[4 * P + 2] = v.z; q[4 * P + 3] = v.w;
        }
    }
    __device__ __forceinline__ void unpack(BItem &b, uint32_t g) const {
        // ggml get_scale_min_k4, four sub-blocks at a time; the lane's two
        // sub-blocks of each half are 2(g/2) and 2(g/2) + 1
        const uint32_t s0 = h[1], s1 = h[2], s2 = h[3], sh = 16u * (g >> 1);
        const uint32_t sd[2] = {(s0 & 0x3F3F3F3Fu) >> sh,
                                ((s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u)) >> sh};
        const uint32_t sm[2] = {(s1 & 0x3F3F3F3Fu) >> sh,
                                (((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u)) >> sh};
#pragma unroll
        for (uint32_t m = 0; m < 4; m++) {
            const uint32_t P = m >> 1, n = m & 1u;
            const uint32_t sc = (sd[P] >> (8u * n)) & 0xFFu, dl = sc & 7u, dh = sc >> 3;
            const int mb = (int)(((sm[P] >> (8u * n)) & 0xFFu) * 0x01010101u);
            b.mn[m] = v4i{mb, mb, mb, mb};
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const uint32_t c = (q[4 * P + j] >> (4u * n)) & 0x0F0F0F0Fu;
                b.lo[m][j] = (int)pk_mul(c, dl);
                b.hi[m][j] = (int)pk_mul(c, dh);
            }
        }
        b.dw = f16_bits_to_f32(h[0] & 0xFFFFu);
        b.dmin = f16_bits_to_f32(h[0] >> 16);
    }
};

// Q6_K.  Chunk m = 2n + k of lane group g: sub-block 8n + 4k + g, elements
// 128n + 64k + 16g .. +15: the low (k = 0) or high (k = 1) nibbles of the 16
// bytes ql[64n + 16g ..] and a 2-bit field of the 16 bytes qh[32n + 16(g%2) ..].
template <>
struct WItem<SINTER_Q6_K> {
    static constexpr uint32_t BYTES = Q6K_BYTES;
    static constexpr int HI_SHIFT = 8;
    uint32_t l[8], hq[8], sc[5], sh;
    static __device__ __forceinline__ uint32_t chunk(uint32_t m, uint32_t g) { return 4u * m + g; }
    // Blocks start on 2-byte boundaries and a 16-byte load that is not
    // 4-aligned takes four times as long (a wave's load from cache on a busy
    // CU: 586 cycles at 2 bytes past a boundary, 160 at 4 or 8): each field is
    // loaded from the 4-aligned address at or before it and shifted into place
    // with the dword that follows, which is another lane's first (a load of
    // its own would take as long as the 16 bytes).  The last dword is the
    // block's own last four bytes, off a 4-byte boundary where the block is on
    // one: a read on past the block's end would pass the end of a matrix of an
    // odd number of blocks (no slower: Q6_K 151936 x 5120, 1 token 153.3 ->
    // 152.2 us, 5120 x 17408, 256 tokens 117.9 -> 117.4).
    __host__ __device__ __forceinline__ void load(const uint8_t *b, uint32_t g) {
        sh = (uint32_t)((uintptr_t)b & 3u);
        b -= sh;
#pragma unroll
        for (uint32_t n = 0; n < 2; n++) {
            const uint8_t *p = b + 64u * n + 16u * g, *q = b + 128u + 32u * n + 16u * (g & 1u);
            const u128_a4 x = *(const u128_a4 *)p, y = *(const u128_a4 *)q;
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) { l[4 * n + j] = x.d[j]; hq[4 * n + j] = y.d[j]; }
        }
        const u128_a4 s = *(const u128_a4 *)(b + 192u);   // the scales
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) sc[j] = s.d[j];
        sc[4] = ((const u32_a2 *)(b + sh + 206u))->d;   // the last two scales, d
    }
    __device__ __forceinline__ void unpack(BItem &b, uint32_t g) const {
        const uint32_t f = 2u * (g >> 1);   // the lane's qh field of a nibble: bits f, f + 1 (low), f + 4, f + 5 (high)
        // the dword after the lane's 16 bytes: the first of lane group g + 1,
        // and after a field's last group the next field's first
        const int nl = (int)(4u * ((threadIdx.x + 16u) & 63u));
        uint32_t ln[2], hn[2];
#pragma unroll
        for (uint32_t n = 0; n < 2; n++) {
            ln[n] = (uint32_t)__builtin_amdgcn_ds_bpermute(nl, (int)(g == 0 ? (n ? hq[0] : l[4]) : l[4 * n]));
            hn[n] = (uint32_t)__builtin_amdgcn_ds_bpermute(nl, (int)((g & 1u) == 0 ? (n ? sc[0] : hq[4]) : hq[4 * n]));
        }
#pragma unroll
        for (uint32_t n = 0; n < 2; n++) {
            uint32_t s[2], bias[2];
#pragma unroll
            for (uint32_t k = 0; k < 2; k++) {
                // sub-block 4 (2n + k) + g's signed scale, 16 bits (mod 2^16 arithmetic)
                const uint32_t w = __builtin_amdgcn_alignbyte(sc[2 * n + k + 1], sc[2 * n + k], sh);
                s[k] = (uint32_t)(int)(int8_t)((w >> (8u * g)) & 0xFFu) & 0xFFFFu;
                bias[k] = 128u - 32u * s[k];
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const uint32_t lw = __builtin_amdgcn_alignbyte(j < 3 ? l[4 * n + j + 1] : ln[n], l[4 * n + j], sh);
                const uint32_t hw = __builtin_amdgcn_alignbyte(j < 3 ? hq[4 * n + j + 1] : hn[n], hq[4 * n + j], sh) >> f;
#pragma unroll
                for (uint32_t k = 0; k < 2; k++) {
                    const uint32_t m = 2 * n + k;
                    // code + 32, 0..63
                    const uint32_t u = ((lw >> (4u * k)) & 0x0F0F0F0Fu) | ((k ? hw : hw << 4) & 0x30303030u);
                    // p + 128 of the even and odd bytes, p = (u - 32) * scale:
                    // the high byte of p + 128 is h, its low byte l + 128
                    const uint32_t pe = pk_mad(u & 0x00FF00FFu, s[k], bias[k]);
                    const uint32_t po = pk_mad((u >> 8) & 0x00FF00FFu, s[k], bias[k]);
                    b.lo[m][j] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
                    b.hi[m][j] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
                }
            }
        }
        b.dw = f16_bits_to_f32(sc[4] >> 16);
        b.dmin = 0.0f;
    }
};

// The exact integer sums of one tile: lo / hi digits and (Q4_K) the min sums.
struct Sums {
    v4i lo, hi, mn;
};
template <int WT>
__device__ __forceinline__ Sums tile_sums(const v4i a[4], const BItem &b) {
    const v4i z = {0, 0, 0, 0};
    Sums s = {z, z, z};
#pragma unroll
    for (uint32_t m = 0; m < 4; m++) {
        s.lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m], b.lo[m], s.lo, 0, 0, 0);
        s.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m], b.hi[m], s.hi, 0, 0, 0);
        if constexpr (WT == SINTER_Q4_K) s.mn = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[m], b.mn[m], s.mn, 0, 0, 0);
    }
    return s;
}
// the fp64 terms of the lane's four pairs
template <int WT>
__device__ __forceinline__ void tile_terms(const Sums &s, double dw, double dmin, const double dx[4], double t[4]) {
    double p[4], q[4];
#pragma unroll
    for (uint32_t v = 0; v < 4; v++)
        p[v] = (double)(int)((uint32_t)s.lo[v] + ((uint32_t)s.hi[v] << WItem<WT>::HI_SHIFT));
    if constexpr (WT == SINTER_Q4_K) {
#pragma unroll
        for (uint32_t v = 0; v < 4; v++) q[v] = (double)s.mn[v];
    }
#pragma unroll
    for (uint32_t v = 0; v < 4; v++) p[v] = (dw * p[v]) * dx[v];
    if constexpr (WT == SINTER_Q4_K) {
#pragma unroll
        for (uint32_t v = 0; v < 4; v++) q[v] = (dmin * q[v]) * dx[v];
#pragma unroll
        for (uint32_t v = 0; v < 4; v++) p[v] = p[v] - q[v];
    }
#pragma unroll
    for (uint32_t v = 0; v < 4; v++) t[v] = p[v];
}

// One launch multiplies up to UB_SEGS matrices of one type by the same
// activations (a layer's projections): row tiles of all of them in one grid.
struct UbArgs {
    const uint8_t *xq;
    uint32_t nb, n_tok, n_tg, accumulate, n_seg;
    uint32_t rt0[UB_SEGS];     // first row tile of each matrix
    uint32_t rows[UB_SEGS];
    const uint8_t *w[UB_SEGS];
    float *y[UB_SEGS];
};
// workgroup -> (row tile, token group): workgroups are dealt to the 8 XCDs in
// turn, so XCD x takes the x-th eighth of the tiles and the token groups of
// one row tile (which read the same weights) share its L2
__device__ __forceinline__ void ub_tile(const UbArgs &a, uint32_t &rt, uint32_t &tg) {
    const uint32_t n = gridDim.x, x = blockIdx.x & 7u, q = n >> 3, r = n & 7u;
    const uint32_t id = x * q + min(x, r) + (blockIdx.x >> 3);
    rt = id / a.n_tg;
    tg = id % a.n_tg;
}

// ---------------------------------------------------------------- many tokens

// A workgroup of four waves owns 64 rows (16 per wave) and NT token tiles.
// Per item the tokens' codes arrive in LDS by LDS-DMA (double-buffered, one
// item ahead) and each wave unpacks its rows' weights (in registers, two items
// ahead) once for its NT tiles.  A token's 256 codes are 16 chunks of 16
// bytes; chunk c of token r lies in slot c ^ (r % 16), so the 16 tokens' reads
// of one chunk fall on distinct banks without padding, which the DMA's
// contiguous kilobyte per wave could not leave.
//
// SHORT: rows of at most UB_SHORT items.  Both buffers are filled and both
// items' weights loaded before the first is multiplied, and nothing is loaded
// ahead, so a workgroup reads each byte once and a CU holds twice the
// workgroups (the loop below loads past the row's end: its items again, never
// used).  us, the loop or the few-token kernel -> so: Q6_K 40000 x 512, 1 token
// 9.8 -> 6.4, 256 tokens 26.5 -> 25.0; Q4_K 40000 x 256, 64 tokens 8.3 -> 6.3.
constexpr uint32_t UB_THREADS = 256;
constexpr uint32_t UB_WG_ROWS = UB_ROWS * (UB_THREADS / 64u);
constexpr uint32_t UB_TILE_BYTES = UB_TOK * 256u;
// a buffer: codes | dx f64 [token]
template <uint32_t NT>
constexpr uint32_t ub_buf() { return NT * (UB_TILE_BYTES + UB_TOK * 8u); }
// the DMA's 32-bit lane offsets reach 128 tokens of items
constexpr uint32_t UB_MAX_NB = 50000;
constexpr uint32_t UB_SHORT = 2;

template <int WT, uint32_t NT, bool SHORT>
__global__ __launch_bounds__(UB_THREADS, SHORT ? 4 : 2) void ubatch_gemm_kernel(UbArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned char xs[2 * ub_buf<NT>()];
    LDS unsigned char *L = (LDS unsigned char *)xs;
    const uint32_t lbase = (uint32_t)(uintptr_t)L;
    const uint32_t lane = threadIdx.x & 63u, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t r = lane & 15u, g = lane >> 4;
    uint32_t rt, tg;
    ub_tile(a, rt, tg);
    uint32_t sg = 0;
    while (sg + 1u < a.n_seg && rt >= a.rt0[sg + 1u]) sg++;
    const uint32_t rows = a.rows[sg], nb = a.nb, n_tok = a.n_tok;
    const uint32_t row = (rt - a.rt0[sg]) * UB_WG_ROWS + wv * UB_ROWS + r;
    const uint32_t tok0 = tg * UB_TOK * NT, tl = n_tok - 1u - tok0;   // (tokens past the last repeat it, never stored)
    const uint8_t *wp = a.w[sg] + (size_t)min(row, rows - 1u) * nb * WItem<WT>::BYTES;
    const uint8_t *xp = a.xq + (size_t)tok0 * nb * Q8K_BYTES;   // (uniform)
    // DMA j of wave w fills tokens 16 j + 4 w .. + 3: lane l token l / 16 of
    // them, slot l % 16
    uint32_t xo[NT];
#pragma unroll
    for (uint32_t j = 0; j < NT; j++) {
        const uint32_t tk = 4u * wv + g;
        xo[j] = min(UB_TOK * j + tk, tl) * nb * Q8K_BYTES + 4u + 16u * (r ^ tk);
    }
    const uint32_t dxo = min(min(threadIdx.x, UB_TOK * NT - 1u), tl) * nb * Q8K_BYTES;
    uint32_t ao[4];   // the lane's four chunks of tile 0
#pragma unroll
    for (uint32_t m = 0; m < 4; m++) ao[m] = r * 256u + 16u * (WItem<WT>::chunk(m, g) ^ r);

    double acc[NT][4];
#pragma unroll
    for (uint32_t t = 0; t < NT; t++)
#pragma unroll
        for (uint32_t v = 0; v < 4; v++) acc[t][v] = 0.0;

    // item i's codes into buffer buf; its d of the thread's token
    auto stage = [&](uint32_t i, uint32_t buf) {
        const uint8_t *q = xp + (size_t)i * Q8K_BYTES;
        const uintptr_t p = (uintptr_t)q;
#pragma unroll
        for (uint32_t j = 0; j < NT; j++)
            lds_dma16<false>(p, xo[j], lbase + buf * ub_buf<NT>() + j * UB_TILE_BYTES + wv * 1024u);
        return *(const float *)(q + dxo);
    };
    auto park = [&](uint32_t buf, float dxn) {
        if (threadIdx.x < UB_TOK * NT)
            *reinterpret_cast<LDS double *>(L + buf * ub_buf<NT>() + NT * UB_TILE_BYTES + 8u * threadIdx.x) = (double)dxn;
    };
    struct AFrag { v4i x[4]; v2d d0, d1; };
    auto read = [&](uint32_t buf, uint32_t t) {   // tile t of buffer buf
        const LDS unsigned char *xb = L + buf * ub_buf<NT>(), *dxs = xb + NT * UB_TILE_BYTES + 32u * g;
        AFrag f;
#pragma unroll
        for (uint32_t m = 0; m < 4; m++) f.x[m] = *reinterpret_cast<const LDS v4i *>(xb + ao[m] + t * UB_TILE_BYTES);
        const LDS v2d *q = reinterpret_cast<const LDS v2d *>(dxs + t * UB_TOK * 8u);
        f.d0 = q[0];
        f.d1 = q[1];
        return f;
    };
    // item i: its codes in buffer `buf`, its weights in w
    auto item = [&](uint32_t i, uint32_t buf, WItem<WT> &w) {
        auto lda = [&](uint32_t t) { return read(buf, t); };
        // (the empty asm statements keep the compiler from sinking the
        // arithmetic past the loads that it is to run beside, or past the
        // barrier: the unpacking would wait for the loads behind it)
        BItem b;
        w.unpack(b, g);
#pragma unroll
        for (uint32_t m = 0; m < 4; m++) {
            asm volatile("" : "+v"(b.lo[m]), "+v"(b.hi[m]));
            if constexpr (WT == SINTER_Q4_K) asm volatile("" : "+v"(b.mn[m]));
        }
        sched_fence();
        // the next item's activations, then the weights of the one after it:
        // loads complete in order, so the wait below leaves the weights in
        // flight (past the end: the last item again, never used)
        float dxn = stage(min(i + 1u, nb - 1u), buf ^ 1u);
        sched_fence();
        w.load(wp + (size_t)min(i + 2u, nb - 1u) * WItem<WT>::BYTES, g);
        AFrag f = lda(0), fn;
        sched_fence();
        const double dw = (double)b.dw, dmin = (double)b.dmin;
        // tile t's MFMAs run beside tile t - 1's fp64 terms and tile t + 1's reads
        Sums s, sp;
        double dxp[4];
#pragma unroll
        for (uint32_t t = 0; t <= NT; t++) {
            if (t + 1 < NT) fn = lda(t + 1);
            sched_fence();
            if (t < NT) s = tile_sums<WT>(f.x, b);
            if (t > 0) {
                double tm[4];
                tile_terms<WT>(sp, dw, dmin, dxp, tm);
#pragma unroll
                for (uint32_t v = 0; v < 4; v++) acc[t - 1][v] += tm[v];
                asm volatile("" : "+v"(acc[t - 1][0]), "+v"(acc[t - 1][1]), "+v"(acc[t - 1][2]), "+v"(acc[t - 1][3]));
            }
            if (t < NT) asm volatile("" : "+v"(s.lo), "+v"(s.hi));
            sched_fence();
            if (t < NT) {
                sp = s;
                dxp[0] = f.d0[0]; dxp[1] = f.d0[1]; dxp[2] = f.d1[0]; dxp[3] = f.d1[1];
            }
            f = fn;
        }
        // every wave waits for dxn, which it loaded after its share of the
        // DMAs: loads complete in order, so they have landed (the weights
        // behind them may still fly)
        asm volatile("" : "+v"(dxn)::"memory");
        park(buf ^ 1u, dxn);
        __syncthreads();
    };
    // the same item with nothing loaded beside it
    auto item_only = [&](uint32_t buf, const WItem<WT> &w) {
        BItem b;
        w.unpack(b, g);
#pragma unroll
        for (uint32_t t = 0; t < NT; t++) {
            const AFrag f = read(buf, t);
            const double dx[4] = {f.d0[0], f.d0[1], f.d1[0], f.d1[1]};
            double tm[4];
            tile_terms<WT>(tile_sums<WT>(f.x, b), (double)b.dw, (double)b.dmin, dx, tm);
#pragma unroll
            for (uint32_t v = 0; v < 4; v++) acc[t][v] += tm[v];
        }
    };
    WItem<WT> w0, w1;
    if constexpr (SHORT) {
        w0.load(wp, g);
        const float d0 = stage(0, 0);
        if (nb > 1u) {
            w1.load(wp + WItem<WT>::BYTES, g);
            const float d1 = stage(1, 1);
            park(1, d1);
        }
        park(0, d0);
        dma_wait();
        __syncthreads();
        item_only(0, w0);
        if (nb > 1u) item_only(1, w1);
    } else {
        const float d0 = stage(0, 0);
        sched_fence();
        w0.load(wp, g);
        w1.load(wp + (size_t)min(1u, nb - 1u) * WItem<WT>::BYTES, g);
        park(0, d0);
        dma_wait();
        __syncthreads();
        for (uint32_t i = 0; i < nb; i += 2) {
            item(i, 0, w0);
            if (i + 1u < nb) item(i + 1u, 1, w1);
        }
        dma_wait();   // (the last item's staging must not outlive the workgroup's LDS)
    }

    if (row < rows) {
        float *y = a.y[sg] + row;
#pragma unroll
        for (uint32_t t = 0; t < NT; t++)
#pragma unroll
            for (uint32_t v = 0; v < 4; v++) {
                const uint32_t tok = tok0 + t * UB_TOK + 4u * g + v;
                if (tok < n_tok) {
                    // accumulate: the residual add of the single-token GEMV's
                    // RESID epilogue (y = y + result, one fp32 add)
                    float *yp = y + (size_t)tok * rows;
                    *yp = a.accumulate ? *yp + (float)acc[t][v] : (float)acc[t][v];
                }
            }
    }
}

// ---------------------------------------------------------------- few tokens

// With few tokens the weights bound the time: a workgroup owns 16 rows and NT
// token tiles, and its KW waves take the items in turn (wave w items w, w +
// KW, ...), each wave's weights and activations straight from memory, so the
// loads of a whole row are in flight at once.  The terms of a round of KW
// items meet in LDS (double-buffered), where each (row, token) is folded by
// one thread in item order.  One token tile is held to 128 registers, four
// workgroups on a CU instead of three: Q6_K 248320 x 5120, 1 token 262 -> 244 us,
// Q4_K 12416 x 5120 15.0 -> 13.5 (eight waves of a workgroup to the items: 15.4).
constexpr uint32_t UB_KW = 4;
template <int WT, uint32_t NT>
__global__ __launch_bounds__(64 * UB_KW, NT == 1 ? 4 : 2) void ubatch_gemv_kernel(UbArgs a) {
    constexpr uint32_t KW = UB_KW, OUT = NT * UB_TOK * UB_ROWS, THREADS = 64u * KW, PT = (OUT + THREADS - 1u) / THREADS;
    __shared__ double terms[2][KW][OUT];
    LDS double *T = (LDS double *)terms;
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6, r = lane & 15u, g = lane >> 4;
    uint32_t rt, tg;
    ub_tile(a, rt, tg);
    uint32_t sg = 0;
    while (sg + 1u < a.n_seg && rt >= a.rt0[sg + 1u]) sg++;
    const uint32_t rows = a.rows[sg], nb = a.nb, n_tok = a.n_tok;
    const uint32_t row0 = (rt - a.rt0[sg]) * UB_ROWS, tok0 = tg * UB_TOK * NT;
    const uint8_t *wrow = a.w[sg] + (size_t)min(row0 + r, rows - 1u) * nb * WItem<WT>::BYTES;
    const uint8_t *xrow[NT], *drow[NT][4];
#pragma unroll
    for (uint32_t t = 0; t < NT; t++) {   // (tokens past the last repeat it, never stored)
        xrow[t] = a.xq + (size_t)min(tok0 + UB_TOK * t + r, n_tok - 1u) * nb * Q8K_BYTES;
#pragma unroll
        for (uint32_t v = 0; v < 4; v++)
            drow[t][v] = a.xq + (size_t)min(tok0 + UB_TOK * t + 4u * g + v, n_tok - 1u) * nb * Q8K_BYTES;
    }
    double acc[PT];
#pragma unroll
    for (uint32_t p = 0; p < PT; p++) acc[p] = 0.0;
    const uint32_t rounds = (nb + KW - 1u) / KW;
    struct XItem { v4i x[NT][4]; float dx[NT][4]; };
    WItem<WT> w;
    auto load_x = [&](XItem &X, uint32_t i) {
#pragma unroll
        for (uint32_t t = 0; t < NT; t++) {
#pragma unroll
            for (uint32_t m = 0; m < 4; m++) {
                const u128_a4 c = *(const u128_a4 *)(xrow[t] + (size_t)i * Q8K_BYTES + 4u + 16u * WItem<WT>::chunk(m, g));
                X.x[t][m] = v4i{(int)c.d[0], (int)c.d[1], (int)c.d[2], (int)c.d[3]};
            }
#pragma unroll
            for (uint32_t v = 0; v < 4; v++) X.dx[t][v] = *(const float *)(drow[t][v] + (size_t)i * Q8K_BYTES);
        }
    };
    // round q: this wave's item from X, the next round's loads (into w and
    // Xn) in flight behind its arithmetic, the terms folded
    auto round = [&](uint32_t q, const XItem &X, XItem &Xn) {
        const uint32_t i = q * KW + wv;   // (items past the last repeat it, their terms never folded)
        BItem b;
        w.unpack(b, g);
        __builtin_amdgcn_sched_barrier(0);
        if (q + 1u < rounds) {
            const uint32_t in = min(i + KW, nb - 1u);
            w.load(wrow + (size_t)in * WItem<WT>::BYTES, g);
            load_x(Xn, in);
        }
        __builtin_amdgcn_sched_barrier(0);
        const double dw = (double)b.dw, dmin = (double)b.dmin;
        LDS double *Tb = T + (q & 1u) * KW * OUT;
#pragma unroll
        for (uint32_t t = 0; t < NT; t++) {
            const Sums u = tile_sums<WT>(X.x[t], b);
            const double dx[4] = {(double)X.dx[t][0], (double)X.dx[t][1], (double)X.dx[t][2], (double)X.dx[t][3]};
            double tm[4];
            tile_terms<WT>(u, dw, dmin, dx, tm);
#pragma unroll
            for (uint32_t v = 0; v < 4; v++) Tb[wv * OUT + (UB_TOK * t + 4u * g + v) * UB_ROWS + r] = tm[v];
        }
        __syncthreads();   // (the other buffer's readers are past it: they wrote their terms after reading)
        const uint32_t n = min(KW, nb - q * KW);
#pragma unroll
        for (uint32_t p = 0; p < PT; p++) {
            const uint32_t o = threadIdx.x + p * THREADS;
            if (OUT % THREADS == 0 || o < OUT) {
#pragma unroll
                for (uint32_t k = 0; k < KW; k++)
                    if (k < n) acc[p] += Tb[k * OUT + o];
            }
        }
    };
    XItem X0, X1;
    w.load(wrow + (size_t)min(wv, nb - 1u) * WItem<WT>::BYTES, g);
    load_x(X0, min(wv, nb - 1u));
    for (uint32_t q = 0; q < rounds; q += 2) {
        round(q, X0, X1);
        if (q + 1u < rounds) round(q + 1u, X1, X0);
    }
#pragma unroll
    for (uint32_t p = 0; p < PT; p++) {
        const uint32_t o = threadIdx.x + p * THREADS, tok = tok0 + o / UB_ROWS, row = row0 + o % UB_ROWS;
        if (o < OUT && tok < n_tok && row < rows) {
            float *yp = a.y[sg] + (size_t)tok * rows + row;
            *yp = a.accumulate ? *yp + (float)acc[p] : (float)acc[p];
        }
    }
}

// ggml quantize_row_q8_K_ref over a ubatch (the oracle's or_quant_q8_K):
// one wave per 256-element block, lane l holding elements 4l..4l+3.  The
// block's scale comes from its first element of largest |x| (sequentially:
// `if (|x| > amax)`, so a tie keeps the lower index: that of the
// first lane with the wave's maximum), iscale = -127 / that element, codes
// min(127, rint(iscale * x)) (ggml's nearest_int: round half to even), d =
// 1 / iscale, bsums the 16-element sums of the codes; an all-zero block is
// all zeros.  Inputs are finite.
__device__ __forceinline__ void quant_block_q8k(const float e[4], uint32_t lane, uint8_t *ob) {
    float amax = 0.0f, mx = 0.0f;
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
        const float ax = fabsf(e[j]);
        if (ax > amax) { amax = ax; mx = e[j]; }
    }
    // (by DPP, readlanes and a ballot: a chain of 18 LDS shuffles of (|x|, x,
    // index) took longer than the rest of the block)
    auto lane_f = [](float v, uint32_t l) {
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), (int)l));
    };
    const float rm = row16_max(amax);
    const float wm = fmaxf(fmaxf(lane_f(rm, 0), lane_f(rm, 16)), fmaxf(lane_f(rm, 32), lane_f(rm, 48)));
    mx = lane_f(mx, (uint32_t)__builtin_ctzll(__builtin_amdgcn_ballot_w64(amax == wm)));
    amax = wm;
    int q[4] = {0, 0, 0, 0};
    float d = 0.0f;
    if (amax != 0.0f) {
        const float iscale = -127.f / mx;
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            const int t = (int)rintf(iscale * e[j]);
            q[j] = t < 127 ? t : 127;
        }
        d = 1.0f / iscale;
    }
    *(uint32_t *)(ob + 4u + 4u * lane) =
        (uint32_t)(q[0] & 0xFF) | ((uint32_t)(q[1] & 0xFF) << 8) | ((uint32_t)(q[2] & 0xFF) << 16) | ((uint32_t)q[3] << 24);
    int bs = q[0] + q[1] + q[2] + q[3];
    bs += dpp_i<DPP_XOR1>(bs);
    bs += dpp_i<DPP_XOR2>(bs);
    if ((lane & 3u) == 0) *(int16_t *)(ob + 260u + 2u * (lane >> 2)) = (int16_t)bs;
    if (lane == 0) *(float *)ob = d;
}

__global__ __launch_bounds__(64) void quant_q8k_kernel(const float *__restrict__ x, uint8_t *__restrict__ xq) {
    const uint32_t lane = threadIdx.x;
    const size_t blk = blockIdx.x;   // token * (k / 256) + block: x and xq in the same order
    const float4 v = ((const float4 *)(x + blk * 256u))[lane];
    const float e[4] = {v.x, v.y, v.z, v.w};
    quant_block_q8k(e, lane, xq + blk * Q8K_BYTES);
}

// SwiGLU then the Q8_K quantiser over a ubatch: f = silu(gate) * up (the
// single-token GEMV's SWIGLU epilogue and the oracle's or_ffn: silu(x) =
// x / (1 + (float)exp(-(double)x))), quantised for the down projection.
__global__ __launch_bounds__(64) void swiglu_quant_q8k_kernel(const float *__restrict__ gate,
                                                             const float *__restrict__ up, uint8_t *__restrict__ xq) {
    const uint32_t lane = threadIdx.x;
    const size_t blk = blockIdx.x;
    const float4 g = ((const float4 *)(gate + blk * 256u))[lane];
    const float4 u = ((const float4 *)(up + blk * 256u))[lane];
    const float e[4] = {dev_silu(g.x) * u.x, dev_silu(g.y) * u.y, dev_silu(g.z) * u.z, dev_silu(g.w) * u.w};
    quant_block_q8k(e, lane, xq + blk * Q8K_BYTES);
}

// Gated RMSNorm per head then the Q8_K quantiser over a ubatch (the input of
// a gated-DeltaNet layer's ssm_out): for each head of d elements (d a power
// of two, 4..256), y = ((x * scale) * w[i]) * silu(z) with scale = 1 /
// sqrtf(mean + eps) from the head's fp32 squares summed in fp64 -- the
// single-token GEMV's GATED prologue and the oracle's or_gated_rmsnorm.  One
// wave per 256-element block: the d / 4 lanes of a head reduce its sum by xor
// shuffles (a fixed tree; the mean divides by a power of two, exactly).
__global__ __launch_bounds__(64) void gated_norm_quant_q8k_kernel(const float *__restrict__ x,
                                                                 const float *__restrict__ z,
                                                                 const float *__restrict__ w, uint32_t log2d,
                                                                 float eps, uint8_t *__restrict__ xq) {
    const uint32_t lane = threadIdx.x;
    const size_t blk = blockIdx.x;
    const float4 v = ((const float4 *)(x + blk * 256u))[lane];
    const float4 g = ((const float4 *)(z + blk * 256u))[lane];
    const uint32_t d = 1u << log2d, i0 = (4u * lane) & (d - 1u);   // element of the head
    double sq = (double)(v.x * v.x);
    sq += (double)(v.y * v.y);
    sq += (double)(v.z * v.z);
    sq += (double)(v.w * v.w);
    for (uint32_t o = 1; o < d / 4u; o <<= 1) sq += __shfl_xor(sq, o);
    const double inv_d = 1.0 / (double)d;   // a power of two: exact
    const float scale = 1.0f / sqrtf((float)(sq * inv_d) + eps);
    const float e[4] = {((v.x * scale) * w[i0]) * dev_silu(g.x), ((v.y * scale) * w[i0 + 1]) * dev_silu(g.y),
                        ((v.z * scale) * w[i0 + 2]) * dev_silu(g.z), ((v.w * scale) * w[i0 + 3]) * dev_silu(g.w)};
    quant_block_q8k(e, lane, xq + blk * Q8K_BYTES);
}

// The causal conv + silu of a gated-DeltaNet layer's qkv rows over a ubatch
// (the single-token GEMV's CONV epilogue and the oracle's or_conv_silu, token
// after token): with input(tau) = x[tau][c] for tau >= 0 and the conv state
// st[c][nh + tau] for -nh <= tau < 0 (nh = dconv - 1, oldest first),
// y[t][c] = silu(sum_j input(t - nh + j) * w[c][j]), the sum in fp64 in tap
// order rounded once.  Outputs do not depend on each other, so a thread
// takes channel c over UB_CONV_TOK consecutive tokens (blockIdx.y), all their
// inputs loaded before the first sum.  The state moves on to the last nh
// inputs (old entries when the ubatch is shorter than nh) in the threads of
// the first tokens, the only ones that read it: UB_CONV_TOK >= nh.  8192
// channels, 4 taps: with loads inside the token loop and a second launch for
// the state 6.9 + 4.7 us at 24 tokens, 11.7 + 4.7 at 256; 4.8 and 7.5 so (7.4
// and 11.9 with the tap count a variable, whose branches keep a token's taps
// and the exponentials of different tokens apart).
constexpr uint32_t UB_CONV_TOK = 8;
static_assert(UB_CONV_TOK >= UB_CONV_MAX - 1, "only a channel's first thread reads the conv state");
template <uint32_t DC>   // taps
__global__ __launch_bounds__(256) void conv_silu_kernel(const float *__restrict__ x, float *__restrict__ st,
                                                       const float *__restrict__ cw, float *__restrict__ y,
                                                       uint32_t channels, uint32_t n_tok) {
    constexpr uint32_t NH = DC - 1;
    const uint32_t c = blockIdx.x * 256u + threadIdx.x;
    if (c >= channels) return;
    const uint32_t t0 = blockIdx.y * UB_CONV_TOK;
    // input(tau), past the ubatch its last token's
    auto input = [&](int tau) {
        return tau >= 0 ? x[(size_t)min((uint32_t)tau, n_tok - 1u) * channels + c]
                        : st[(size_t)c * NH + (uint32_t)(tau + (int)NH)];
    };
    float in[NH + UB_CONV_TOK];   // inputs t0 - NH ..
    double wt[DC];
#pragma unroll
    for (uint32_t j = 0; j < NH + UB_CONV_TOK; j++) in[j] = input((int)(t0 + j) - (int)NH);
#pragma unroll
    for (uint32_t j = 0; j < DC; j++) wt[j] = (double)cw[(size_t)c * DC + j];
#pragma unroll
    for (uint32_t i = 0; i < UB_CONV_TOK; i++) {
        if (t0 + i >= n_tok) break;
        double acc = 0.0;
#pragma unroll
        for (uint32_t j = 0; j < DC; j++) acc += (double)in[i + j] * wt[j];
        y[(size_t)(t0 + i) * channels + c] = dev_silu((float)acc);
    }
    if (t0 == 0) {
        float nv[NH + 1];
#pragma unroll
        for (uint32_t j = 0; j < NH; j++) nv[j] = input((int)n_tok - (int)NH + (int)j);
#pragma unroll
        for (uint32_t j = 0; j < NH; j++) st[(size_t)c * NH + j] = nv[j];
    }
}

// RMSNorm then the Q8_K quantiser, one workgroup per token: the norm of the
// single-token GEMV's SINTER_PRO_RMSNORM prologue (gemv.h) and of the
// oracle's or_rmsnorm (ggml: fp32 squares summed in fp64, the mean rounded
// to fp32, scale = 1 / sqrtf(mean + eps), y = (x * scale) * w).  The fp64 sum
// is the prologue's tree exactly, so prefill and decode normalise a row to
// the same bits: row g = t / 16 (16 lanes) owns the 256-element chunks g,
// g + 16, ..., lane r = t % 16 elements 16r..16r+15 of each; the lane keeps
// four partial sums (element i into sum i / 4) over its chunks g + 32,
// g + 48, ... and then g and g + 16; the row adds them as
// (s0 + s1) + (s2 + s3) and by its DPP butterfly, the wave its four rows in
// order, the workgroup its four waves in order.  Those are the first four of NW
// waves; the normalised row is quantised by all, wave v blocks v, v + NW, ....
// PRE: everything the sum reads, and the wave's first two blocks, are loaded
// at once ahead of it (a row is one chain of latencies), for twice the
// registers and loads past a short row's end.
__device__ __forceinline__ void ub_add_sq(const float4 x[4], double s4[4]) {
#pragma unroll
    for (uint32_t q = 0; q < 4; q++) {
        s4[q] += (double)(x[q].x * x[q].x);
        s4[q] += (double)(x[q].y * x[q].y);
        s4[q] += (double)(x[q].z * x[q].z);
        s4[q] += (double)(x[q].w * x[q].w);
    }
}
template <uint32_t NW, bool PRE>
__global__ __launch_bounds__(64 * NW) void rmsnorm_quant_q8k_kernel(const float *__restrict__ x,
                                                                   const float *__restrict__ w, float eps, uint32_t k,
                                                                   uint8_t *__restrict__ xq) {
    __shared__ double red[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, r = tid & 15u, g = tid >> 4, nchunk = k / 256u;
    const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const float *xr = x + (size_t)blockIdx.x * k;
    auto chunk = [&](uint32_t c, float4 v[4]) {   // the lane's elements of chunk c (past the last: the last's)
#pragma unroll
        for (uint32_t q = 0; q < 4; q++) v[q] = ((const float4 *)(xr + 256u * min(c, nchunk - 1u) + 16u * r))[q];
    };
    float4 a[4], b[4], xv[2], gv[2];
    if constexpr (PRE) {
        if (wv < 4u) {
            chunk(g, a);
            chunk(g + 16u, b);
        }
#pragma unroll
        for (uint32_t j = 0; j < 2; j++) {
            const uint32_t bl = min(wv + NW * j, nchunk - 1u);
            xv[j] = ((const float4 *)(xr + 256u * bl))[lane];
            gv[j] = w ? ((const float4 *)(w + 256u * bl))[lane] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        }
    }
    if (wv < 4u) {
        double s4[4] = {0.0, 0.0, 0.0, 0.0};
        for (uint32_t c = g + 32u; c < nchunk; c += 16u) {
            float4 v[4];
            chunk(c, v);
            ub_add_sq(v, s4);
        }
        if (g < nchunk) {
            if constexpr (!PRE) chunk(g, a);
            ub_add_sq(a, s4);
        }
        if (g + 16u < nchunk) {
            if constexpr (!PRE) chunk(g + 16u, b);
            ub_add_sq(b, s4);
        }
        double s = row16_sum_f64((s4[0] + s4[1]) + (s4[2] + s4[3]));
        s = ((readlane_f64(s, 0) + readlane_f64(s, 16)) + readlane_f64(s, 32)) + readlane_f64(s, 48);
        if (lane == 0) red[wv] = s;
    }
    __syncthreads();
    const double s = ((red[0] + red[1]) + red[2]) + red[3];
    const float mean = (float)(s / (double)k);
    const float scale = 1.0f / sqrtf(mean + eps);
    uint8_t *orow = xq + (size_t)blockIdx.x * nchunk * Q8K_BYTES;
    auto quant = [&](uint32_t bl, const float4 &v, const float4 &gm) {
        float e[4] = {v.x * scale, v.y * scale, v.z * scale, v.w * scale};
        if (w) { e[0] = e[0] * gm.x; e[1] = e[1] * gm.y; e[2] = e[2] * gm.z; e[3] = e[3] * gm.w; }
        quant_block_q8k(e, lane, orow + (size_t)bl * Q8K_BYTES);
    };
    if constexpr (PRE) {
#pragma unroll
        for (uint32_t j = 0; j < 2; j++)
            if (wv + NW * j < nchunk) quant(wv + NW * j, xv[j], gv[j]);
    }
    for (uint32_t bl = wv + (PRE ? 2u * NW : 0u); bl < nchunk; bl += NW) {
        const float4 v = ((const float4 *)(xr + 256u * bl))[lane];
        quant(bl, v, w ? ((const float4 *)(w + 256u * bl))[lane] : v);
    }
}

}  // namespace
}  // namespace sinter

using namespace sinter;

namespace sinter {
namespace {

// The split of a launch: the kernel and its token tiles per workgroup.
struct UbSplit {
    enum Kernel { FEW, MANY, SHORT } kernel;
    uint32_t nt, wg_rows, n_tg;
    uint64_t wgs;
};
template <int WT>
UbSplit ub_split_of(const UbArgs &a, UbSplit::Kernel kernel, uint32_t nt) {
    UbSplit s = {kernel, nt, kernel == UbSplit::FEW ? UB_ROWS : UB_WG_ROWS, 0, 0};
    s.n_tg = ((a.n_tok + UB_TOK - 1) / UB_TOK + nt - 1) / nt;
    for (uint32_t i = 0; i < a.n_seg; i++) s.wgs += ((uint64_t)a.rows[i] + s.wg_rows - 1) / s.wg_rows;
    s.wgs *= s.n_tg;
    return s;
}

// The cheapest of the compiled splits by a cost per item, fitted to times of
// 11 matrices (32..34816 rows, K 4096..17408) x 10 token counts (8..512); ns:
//   many-token kernel: up to one workgroup per CU it runs at its latency
//   `lone`; with w > 1 per CU the CU's issue slots bound it, `thr` per
//   workgroup, and a started last round takes about two thirds of one;
//   few-token kernel: latency, or `thr` per workgroup of a CU over a start-up;
//   each further token's activations are another line of a load.
// E.g. Q6_K 5120 x 17408 at 256 tokens (us): nt 2 180, 3 131, 4 143, 6 118,
// 8 143; at 5 tokens few-token 37, many-token 90; 151936 x 5120 at 1, 5 and 16
// tokens: few-token 154, 162, 193, many-token 175, 186, 195 (its price leaves
// the tokens of a tile out: at 16 it is taken, 1 % over).  Q4_K 34816 x 5120 at 256:
// nt 2 205, 4 180, 6 181, 8 166; 8192 x 5120 at 24: few-token 15, nt 1 15.5.
// Short rows are mostly start-up, which these prices leave out: one item goes
// to SHORT, two do where the few-token kernel would take them with more than
// two workgroups per CU, or the many-token kernel with many or for one or two
// token tiles (us, the price's choice -> SHORT: Q6_K 160000 x 256, 1 token 30.1
// -> 8.5, 10000 x 256, 16 tokens 4.9 -> 3.4, 40000 x 512, 16 tokens 9.9 -> 6.9,
// 20 tokens 10.1 -> 7.8; but 1000 x 512, 64 tokens 3.7, SHORT 4.3, and 5000 x
// 512, 256 tokens 7.6, SHORT 8.0).  The more workgroups one token tile each
// would give, the more tiles one takes (us at nt 1, 2, 4: Q4_K 20000 x 256, 64
// tokens 4.8, 5.7, 5.4, 40000 x 256, 64 tokens 7.2, 6.3, 6.7, 160000 x 256, 40
// tokens 15.7, 15.6, 13.6; Q6_K 10000 x 256, 64 tokens 4.6, 4.5, 5.0, 40000 x
// 256, 64 tokens 9.7, 7.3, 7.1).
template <int WT>
UbSplit ub_split(const UbArgs &a) {
    constexpr bool Q4 = WT == SINTER_Q4_K;
    const uint32_t tiles = (a.n_tok + UB_TOK - 1) / UB_TOK;
    UbSplit best = {};
    double cost = 1e300;
    auto consider = [&](UbSplit::Kernel kernel, uint32_t nt, double lone, double thr, double start) {
        const UbSplit s = ub_split_of<WT>(a, kernel, nt);
        const double w = (double)s.wgs / 256.0;
        double c;
        if (kernel == UbSplit::FEW) c = std::max(lone, start + w * thr);
        else c = start + (w <= 1.0 ? lone : std::max(lone, std::floor(w) * thr) + (w > std::floor(w) ? 0.65 * thr : 0.0));
        // (a launch holds fewer than 2^32 threads; the few-token kernel's row
        // tiles are the smaller: Q6_K with 1-4 tokens past 2^28 rows)
        if (s.wgs > UINT32_MAX / UB_THREADS) c += 1e200;
        if (c < cost) { cost = c; best = s; }
    };
    // (not compiled, as never the cheapest: few-token nt 2 for Q4_K, whose
    // unpacking is cheap enough to repeat; many-token nt 1 for Q6_K, whose is not)
    const uint32_t tok = std::min(a.n_tok, UB_TOK);
    consider(UbSplit::FEW, 1, Q4 ? 370 : 560, Q4 ? 166 : 200 + 3 * tok, Q4 ? 200 : 150);
    if (!Q4 && tiles > 1) consider(UbSplit::FEW, 2, 700, 420, 150);
    if (a.nb > UB_MAX_NB) return best;
    for (uint32_t nt : {Q4 ? 1u : 2u, 2u, 3u, 4u, 6u, 8u})
        consider(UbSplit::MANY, nt, Q4 ? 477 + 168 * nt : 1030 + 108 * nt, Q4 ? 190 + 215 * nt : 550 + 150 * nt, 125);
    if (a.nb <= UB_SHORT) {
        const uint64_t w = ub_split_of<WT>(a, UbSplit::SHORT, 1).wgs, few = ub_split_of<WT>(a, UbSplit::FEW, 1).wgs;
        if (a.nb == 1 || (best.kernel == UbSplit::FEW ? few > 512 : w >= 1400 || tiles <= 2))
            return ub_split_of<WT>(a, UbSplit::SHORT, w >= (Q4 ? 4096 : 1024) && tiles > 2  ? 4
                                                      : w >= (Q4 ? 1400 : 512) && tiles > 1 ? 2
                                                                                            : 1);
    }
    return best;
}

template <int WT, uint32_t NT, bool SHORT = false>
void launch_gemm(const UbArgs &a, uint32_t grid, hipStream_t s) {
    hipLaunchKernelGGL((ubatch_gemm_kernel<WT, NT, SHORT>), dim3(grid), dim3(UB_THREADS), 0, s, a);
}
template <int WT, uint32_t NT>
void launch_gemv(const UbArgs &a, uint32_t grid, hipStream_t s) {
    hipLaunchKernelGGL((ubatch_gemv_kernel<WT, NT>), dim3(grid), dim3(64 * UB_KW), 0, s, a);
}

template <int WT>
hipError_t launch_ubatch(UbArgs &a, hipStream_t s) {
    const UbSplit p = ub_split<WT>(a);
    if (p.wgs > (uint64_t)INT32_MAX) return hipErrorInvalidValue;
    a.n_tg = p.n_tg;
    uint32_t n_rt = 0;
    for (uint32_t i = 0; i < a.n_seg; i++) {
        a.rt0[i] = n_rt;
        n_rt += (uint32_t)(((uint64_t)a.rows[i] + p.wg_rows - 1) / p.wg_rows);
    }
    const uint32_t grid = (uint32_t)p.wgs;
    if (p.kernel == UbSplit::SHORT) {
        if (p.nt == 1) launch_gemm<WT, 1, true>(a, grid, s);
        else if (p.nt == 2) launch_gemm<WT, 2, true>(a, grid, s);
        else launch_gemm<WT, 4, true>(a, grid, s);
    } else if (p.kernel == UbSplit::FEW) {
        if constexpr (WT == SINTER_Q6_K) {
            if (p.nt == 2) {
                launch_gemv<WT, 2>(a, grid, s);
                return hipGetLastError();
            }
        }
        launch_gemv<WT, 1>(a, grid, s);
    } else switch (p.nt) {
        case 1:
            if constexpr (WT == SINTER_Q4_K) launch_gemm<WT, 1>(a, grid, s);
            break;
        case 2: launch_gemm<WT, 2>(a, grid, s); break;
        case 3: launch_gemm<WT, 3>(a, grid, s); break;
        case 4: launch_gemm<WT, 4>(a, grid, s); break;
        case 6: launch_gemm<WT, 6>(a, grid, s); break;
        default: launch_gemm<WT, 8>(a, grid, s); break;
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_gemv_ubatch(int type, const UbMat *m, uint32_t n, uint32_t nb, const void *xq, uint32_t n_tok,
                              bool accumulate, hipStream_t s) {
    UbArgs a = {};
    a.xq = (const uint8_t *)xq;
    a.nb = nb;
    a.n_tok = n_tok;
    a.accumulate = accumulate;
    a.n_seg = n;
    for (uint32_t i = 0; i < n; i++) {
        a.rows[i] = m[i].rows;
        a.w[i] = (const uint8_t *)m[i].w;
        a.y[i] = m[i].y;
    }
    return type == SINTER_Q4_K ? launch_ubatch<SINTER_Q4_K>(a, s) : launch_ubatch<SINTER_Q6_K>(a, s);
}

}  // namespace sinter

extern "C" int sinter_op_gemv_ubatch(int type, const void *w, int64_t rows, int64_t k, const void *xq,
                                     uint32_t n_tokens, float *y, int accumulate, void *stream) {
    if (type != SINTER_Q4_K && type != SINTER_Q6_K)
        return set_error(SINTER_ERR_ARG, "gemv_ubatch: weight type %d (Q4_K or Q6_K)", type);
    if (rows <= 0 || rows > (int64_t)UINT32_MAX - UB_ROWS || k <= 0 || k % 256 != 0 || k / 256 > (int64_t)UINT32_MAX)
        return set_error(SINTER_ERR_ARG, "gemv_ubatch: rows %lld / k %lld (k a positive multiple of 256)",
                         (long long)rows, (long long)k);
    if (n_tokens == 0) return SINTER_OK;
    if (!w || !xq || !y) return set_error(SINTER_ERR_ARG, "gemv_ubatch: null pointer");
    const uintptr_t wa = type == SINTER_Q4_K ? 16u : 4u;
    if ((uintptr_t)w % wa || (uintptr_t)xq % 4u || (uintptr_t)y % 4u)
        return set_error(SINTER_ERR_ARG, "gemv_ubatch: alignment (weights %u B, activations and output 4 B)",
                         (unsigned)wa);
    const UbMat m = {w, y, (uint32_t)rows};
    const hipError_t e = launch_gemv_ubatch(type, &m, 1, (uint32_t)(k / 256), xq, n_tokens, accumulate != 0,
                                            (hipStream_t)stream);
    if (e == hipErrorInvalidValue) return set_error(SINTER_ERR_ARG, "gemv_ubatch: grid too large");
    return hip_ok(e, "gemv_ubatch: launch") ? SINTER_OK : SINTER_ERR_HIP;
}

extern "C" int sinter_quant_q8k_ubatch(const float *x, int64_t k, uint32_t n_tokens, void *xq, void *stream) {
    if (k <= 0 || k % 256 != 0) return set_error(SINTER_ERR_ARG, "quant_q8k_ubatch: k %lld (a positive multiple of 256)",
                                                 (long long)k);
    if (n_tokens == 0) return SINTER_OK;
    if (!x || !xq) return set_error(SINTER_ERR_ARG, "quant_q8k_ubatch: null pointer");
    if ((uintptr_t)x % 16u || (uintptr_t)xq % 4u)
        return set_error(SINTER_ERR_ARG, "quant_q8k_ubatch: alignment (x 16 bytes, xq 4 bytes)");
    const uint64_t n_blk = (uint64_t)n_tokens * (uint64_t)(k / 256);
    if (n_blk > (uint64_t)INT32_MAX) return set_error(SINTER_ERR_ARG, "quant_q8k_ubatch: too many blocks");
    hipLaunchKernelGGL(quant_q8k_kernel, dim3((uint32_t)n_blk), dim3(64), 0, (hipStream_t)stream, x, (uint8_t *)xq);
    return hip_ok(hipGetLastError(), "quant_q8k_ubatch: launch") ? SINTER_OK : SINTER_ERR_HIP;
}

extern "C" int sinter_rmsnorm_quant_q8k_ubatch(const float *x, const float *w, float eps, int64_t k, uint32_t n_tokens,
                                               void *xq, void *stream) {
    if (k <= 0 || k % 256 != 0 || k > (int64_t)UINT32_MAX)
        return set_error(SINTER_ERR_ARG, "rmsnorm_quant_q8k_ubatch: k %lld (a positive multiple of 256)", (long long)k);
    if (n_tokens == 0) return SINTER_OK;
    if (!x || !xq) return set_error(SINTER_ERR_ARG, "rmsnorm_quant_q8k_ubatch: null pointer");
    if ((uintptr_t)x % 16u || (uintptr_t)w % 16u || (uintptr_t)xq % 4u)
        return set_error(SINTER_ERR_ARG, "rmsnorm_quant_q8k_ubatch: alignment (x, w 16 bytes, xq 4 bytes)");
    if (!(eps >= 0.0f)) return set_error(SINTER_ERR_ARG, "rmsnorm_quant_q8k_ubatch: eps must be >= 0");
    auto launch = [&](auto kernel, uint32_t waves) {
        hipLaunchKernelGGL(kernel, dim3(n_tokens), dim3(64 * waves), 0, (hipStream_t)stream, x, w, eps, (uint32_t)k,
                           (uint8_t *)xq);
    };
    // Up to one row per CU a row's latency is the time: 16 waves (us, four
    // waves with their loads behind the sum -> so: K 5120, 24 rows 7.3 -> 3.5,
    // 17408 20.0 -> 7.2).  Then 8, while a CU's rows are few for their length
    // (5120, 512 rows 8.0, 16 waves 6.3, 8 waves 5.1).  Past that the waves
    // that start and the registers they hold are the time: 4 without PRE
    // (1024, 65536 rows: 16 waves 512, 4 with PRE 169, without 106; 5120, 8192
    // rows: 84, 55, 49; 2048, 768 rows: 8 waves 4.7, 1024 rows: 5.7, 4 without
    // PRE 4.7).
    const uint32_t nchunk = (uint32_t)(k / 256);
    if (n_tokens <= 256) launch(rmsnorm_quant_q8k_kernel<16, true>, 16);
    else if (nchunk >= 8 && n_tokens <= 96ull * nchunk) launch(rmsnorm_quant_q8k_kernel<8, true>, 8);
    else launch(rmsnorm_quant_q8k_kernel<4, false>, 4);
    return hip_ok(hipGetLastError(), "rmsnorm_quant_q8k_ubatch: launch") ? SINTER_OK : SINTER_ERR_HIP;
}

extern "C" int sinter_swiglu_quant_q8k_ubatch(const float *gate, const float *up, int64_t k, uint32_t n_tokens, void *xq,
                                              void *stream) {
    if (k <= 0 || k % 256 != 0)
        return set_error(SINTER_ERR_ARG, "swiglu_quant_q8k_ubatch: k %lld (a positive multiple of 256)", (long long)k);
    if (n_tokens == 0) return SINTER_OK;
    if (!gate || !up || !xq) return set_error(SINTER_ERR_ARG, "swiglu_quant_q8k_ubatch: null pointer");
    if ((uintptr_t)gate % 16u || (uintptr_t)up % 16u || (uintptr_t)xq % 4u)
        return set_error(SINTER_ERR_ARG, "swiglu_quant_q8k_ubatch: alignment (gate, up 16 bytes, xq 4 bytes)");
    const uint64_t n_blk = (uint64_t)n_tokens * (uint64_t)(k / 256);
    if (n_blk > (uint64_t)INT32_MAX) return set_error(SINTER_ERR_ARG, "swiglu_quant_q8k_ubatch: too many blocks");
    hipLaunchKernelGGL(swiglu_quant_q8k_kernel, dim3((uint32_t)n_blk), dim3(64), 0, (hipStream_t)stream, gate, up,
                       (uint8_t *)xq);
    return hip_ok(hipGetLastError(), "swiglu_quant_q8k_ubatch: launch") ? SINTER_OK : SINTER_ERR_HIP;
}

extern "C" int sinter_gated_rmsnorm_quant_q8k_ubatch(const float *x, const float *z, const float *w, uint32_t head_dim,
                                                     float eps, int64_t k, uint32_t n_tokens, void *xq, void *stream) {
    if (k <= 0 || k % 256 != 0)
        return set_error(SINTER_ERR_ARG, "gated_rmsnorm_quant_q8k_ubatch: k %lld (a positive multiple of 256)",
                         (long long)k);
    if (head_dim < 4 || head_dim > 256 || (head_dim & (head_dim - 1)))
        return set_error(SINTER_ERR_ARG, "gated_rmsnorm_quant_q8k_ubatch: head_dim %u (a power of two, 4..256)",
                         head_dim);
    if (n_tokens == 0) return SINTER_OK;
    if (!x || !z || !w || !xq) return set_error(SINTER_ERR_ARG, "gated_rmsnorm_quant_q8k_ubatch: null pointer");
    if ((uintptr_t)x % 16u || (uintptr_t)z % 16u || (uintptr_t)w % 4u || (uintptr_t)xq % 4u)
        return set_error(SINTER_ERR_ARG, "gated_rmsnorm_quant_q8k_ubatch: alignment (x, z 16 bytes, w, xq 4 bytes)");
    if (!(eps >= 0.0f)) return set_error(SINTER_ERR_ARG, "gated_rmsnorm_quant_q8k_ubatch: eps must be >= 0");
    const uint64_t n_blk = (uint64_t)n_tokens * (uint64_t)(k / 256);
    if (n_blk > (uint64_t)INT32_MAX) return set_error(SINTER_ERR_ARG, "gated_rmsnorm_quant_q8k_ubatch: too many blocks");
    hipLaunchKernelGGL(gated_norm_quant_q8k_kernel, dim3((uint32_t)n_blk), dim3(64), 0, (hipStream_t)stream, x, z, w,
                       (uint32_t)__builtin_ctz(head_dim), eps, (uint8_t *)xq);
    return hip_ok(hipGetLastError(), "gated_rmsnorm_quant_q8k_ubatch: launch") ? SINTER_OK : SINTER_ERR_HIP;
}

extern "C" int sinter_conv_silu_ubatch(const float *x, float *state, const float *conv_w, float *y, int64_t channels,
                                       uint32_t dconv, uint32_t n_tokens, void *stream) {
    if (channels <= 0 || channels > (int64_t)INT32_MAX || dconv < 1 || dconv > UB_CONV_MAX)
        return set_error(SINTER_ERR_ARG, "conv_silu_ubatch: channels %lld / dconv %u (1..%u)", (long long)channels,
                         dconv, UB_CONV_MAX);
    if (n_tokens == 0) return SINTER_OK;
    if (!x || !conv_w || !y || (dconv > 1 && !state)) return set_error(SINTER_ERR_ARG, "conv_silu_ubatch: null pointer");
    if ((uintptr_t)x % 4u || (uintptr_t)state % 4u || (uintptr_t)conv_w % 4u || (uintptr_t)y % 4u)
        return set_error(SINTER_ERR_ARG, "conv_silu_ubatch: alignment (4 bytes)");
    const uint32_t nblk = (uint32_t)((channels + 255) / 256);
    const dim3 grid(nblk, (n_tokens + UB_CONV_TOK - 1) / UB_CONV_TOK);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, x, state, conv_w, y, (uint32_t)channels,
                           n_tokens);
    };
    switch (dconv) {
        case 1: launch(conv_silu_kernel<1>); break;
        case 2: launch(conv_silu_kernel<2>); break;
        case 3: launch(conv_silu_kernel<3>); break;
        case 4: launch(conv_silu_kernel<4>); break;
        case 5: launch(conv_silu_kernel<5>); break;
        case 6: launch(conv_silu_kernel<6>); break;
        case 7: launch(conv_silu_kernel<7>); break;
        default: launch(conv_silu_kernel<8>); break;
    }
    return hip_ok(hipGetLastError(), "conv_silu_ubatch: launch") ? SINTER_OK : SINTER_ERR_HIP;
}
