// The batched prefill's own kernels (sinter_model_prefill runs a prompt layer
// by layer over ubatches of tokens; docs/PREFILL-SEMANTICS.md:379-426 of the
// reference calls this the "(b)" stage: each layer once per ubatch, the
// recurrence looping over the ubatch's tokens inside one launch).  The trunk
// GEMMs, norms, quantisers, SwiGLU and the conv come from ubatch.hip; here:
//   embed_ubatch_kernel      token rows of the embedding, dequantised
//   gdn_prep_ubatch_kernel   the l2 norms of q and k and the gates of every
//                            token of the ubatch
//   gdn_scan_ubatch_kernel   the delta rule over the ubatch, token after
//                            token, the state slice in registers
//   attn_prep_ubatch_kernel  q/k RMSNorm + NEOX RoPE per token and head, the
//                            ubatch's K/V rows appended to the cache
//   attn_prefill_split_kernel, attn_prefill_merge_kernel
//                            causal attention of the ubatch's queries over
//                            the cache, split over chunks and merged as the
//                            decode does, gated by sigmoid(gate)
// All compute what the decode ops compute, expression for expression (same
// helpers, same fp64 folds, same chunks), so a prefilled state, KV cache and
// logits are bit-identical to the decode program's.
#include <algorithm>

#include "batched.h"
#include "internal.h"
#include "gemv.h"
#include "attn.h"

namespace sinter {
namespace {

// ------------------------------------------------------------------ embedding

// x[t] = dequant(embd[tokens[t]]) (the decode's SINTER_PRO_EMBED rows, ggml's
// dequantize_row_*); blockIdx.y is the token
__global__ __launch_bounds__(256) void embed_ubatch_kernel(const char *__restrict__ embd, int type, uint32_t E,
                                                          uint64_t row_bytes, const int32_t *__restrict__ tokens,
                                                          float *__restrict__ x) {
    const uint32_t t = blockIdx.y;
    const char *row = embd + (size_t)tokens[t] * row_bytes;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < E / 4u; i += gridDim.x * 256u) {
        float v[4];
        dequant4(row, type, 4u * i, v);
        reinterpret_cast<float4 *>(x + (size_t)t * E)[i] = make_float4(v[0], v[1], v[2], v[3]);
    }
}

// ------------------------------------------------------------------ GDN step over a ubatch

struct GdnUb {
    const float *qkv;     // [T][C] conv outputs: q[HK*D] | k[HK*D] | v[HV*D]
    const float *alpha;   // [T][HV]
    const float *beta;    // [T][HV]
    const float *dt_bias, *ssm_a;
    float *qn, *kn;       // [T][HK][D] l2-normalised q and k
    float *gate, *bgate;  // [T][HV] decay g and beta
    float *state;         // [HV][D][D] (column-major per head), updated in place
    float *o;             // [T][HV*D]
    uint32_t hk, hv, d, n_tok, c_stride;
    float eps, scale;
};

// The per-token inputs of the recurrence, for every token at once: the l2
// norms of q and k head hk (blockIdx.y) of token blockIdx.x -- the decode
// op_gdn_step's block_sum2_f64 over the same 256-thread layout, scale
// 1/fmaxf(sqrtf(sum), eps) -- and, in the hk = 0 workgroup, the token's gates
// g = exp(softplus(alpha + dt_bias) * a) and beta = sigmoid(beta_raw).
__global__ __launch_bounds__(256) void gdn_prep_ubatch_kernel(GdnUb a) {
    __shared__ double red[16];
    const uint32_t t = blockIdx.x, hk = blockIdx.y, D = a.d, HK = a.hk;
    const float *qkv = a.qkv + (size_t)t * a.c_stride;
    const uint32_t tq = threadIdx.x & (D - 1);
    const float qv = qkv[(size_t)hk * D + tq], kv = qkv[(size_t)HK * D + (size_t)hk * D + tq];
    const bool mine = threadIdx.x < D;
    double sq = mine ? (double)(qv * qv) : 0.0, sk = mine ? (double)(kv * kv) : 0.0;
    block_sum2_f64(sq, sk, red);
    if (mine) {
        const size_t o = ((size_t)t * HK + hk) * D + threadIdx.x;
        a.qn[o] = qv * (1.0f / fmaxf(sqrtf((float)sq), a.eps));
        a.kn[o] = kv * (1.0f / fmaxf(sqrtf((float)sk), a.eps));
    }
    if (hk == 0) {
        for (uint32_t h = threadIdx.x; h < a.hv; h += 256u) {
            const float alpha = a.alpha[(size_t)t * a.hv + h], braw = a.beta[(size_t)t * a.hv + h];
            const float sp = dev_softplus(alpha + a.dt_bias[h]);
            a.gate[(size_t)t * a.hv + h] = (float)exp((double)(sp * a.ssm_a[h]));
            a.bgate[(size_t)t * a.hv + h] = dev_sigmoid(braw);
        }
    }
}

// The delta rule over the ubatch: one wave per (v-head, 64 / TPC state
// columns), the decode op_gdn_step's column layout and folds (gdn.h): TPC
// threads of RPT rows per column, kv and o as sequential fp32 sums over the
// thread's rows then lanes_sum_f32 over the column's threads, delta and the
// update in the same fp32 expressions.  The state stays in registers from the
// first token to the last.
//
// A token is 7 RPT instructions of one wave's own issue (per row the decay, the
// update's product and sum, two products and two running sums), and the next
// token's update waits for this one's sums: what else a token waits for decides
// the time.  k and q come by LDS-DMA, GDN_STAGE tokens at a time and one stage
// ahead, in the order the lanes read them -- position j TPC + p holds rows
// RPT p + 4j .. + 3, so the TPC threads of a column read consecutive 16-byte
// units (row order put them 64 bytes apart, four to a bank) -- and are read
// into registers a token ahead; a stage belongs to one wave, so there is no
// barrier.  27B shapes, 256 tokens: 139 us with four-wave workgroups, row
// order and a barrier per stage, 80 us so; with the prep kernel and 32 heads,
// head size 64 99 -> 53, 128 147 -> 90, 256 229 -> 163 (one wave per SIMD).
constexpr uint32_t GDN_STAGE = 8;
static_assert(GDN_STAGE <= 8, "a stage's outputs fit the threads of a column");
template <uint32_t RPT, uint32_t TPC>
__global__ __launch_bounds__(64) void gdn_scan_ubatch_kernel(GdnUb a) {
    constexpr uint32_t D = RPT * TPC, COLS = 64u / TPC, VEC = D * 4u, BUF = GDN_STAGE * 2u * VEC;
    __shared__ __attribute__((aligned(16))) unsigned char sm[2 * BUF];
    LDS unsigned char *L = (LDS unsigned char *)sm;
    const uint32_t lbase = (uint32_t)(uintptr_t)L;
    const uint32_t HK = a.hk, HV = a.hv, lane = threadIdx.x, p = lane % TPC;
    const uint32_t h = blockIdx.x / (D / COLS), col = (blockIdx.x % (D / COLS)) * COLS + lane / TPC, hk = h % HK;
    const uint32_t n = a.n_tok, last = n - 1u;
    float *srow = a.state + ((size_t)h * D + col) * D + p * RPT;
    float s[RPT];
    auto load = [&](const LDS unsigned char *v, float (&d)[RPT]) {
#pragma unroll
        for (uint32_t j = 0; j < RPT / 4; j++) {
            const f32x4 t = *reinterpret_cast<const LDS f32x4 *>(v + 16u * (j * TPC + p));
            d[4 * j] = t.x; d[4 * j + 1] = t.y; d[4 * j + 2] = t.z; d[4 * j + 3] = t.w;
        }
    };
#pragma unroll
    for (uint32_t r = 0; r < RPT; r += 4) {
        const f32x4 t = *reinterpret_cast<const f32x4 *>(srow + r);
        s[r] = t.x; s[r + 1] = t.y; s[r + 2] = t.z; s[r + 3] = t.w;
    }
    // stage st's inputs: k | q of its tokens into buffer `buf`, v of the
    // lane's column, g and beta of token lane % GDN_STAGE in registers
    // (tokens past the last repeat it, never used)
    struct Small { float v[GDN_STAGE], g, b; };
    auto issue = [&](uint32_t st, uint32_t buf, Small &w) {
        const uint32_t tb = st * GDN_STAGE;
#pragma unroll
        for (uint32_t i = 0; i < BUF / 1024u; i++) {
            const uint32_t u = 64u * i + lane, tk = u / (D / 2), half = (u / (D / 4)) & 1u, pos = u % (D / 4);
            const uint32_t t = min(tb + tk, last), c = (pos % TPC) * (RPT / 4) + pos / TPC;
            // (byte offset from the first token: kn follows qn in one buffer)
            const uint32_t voff = (((half ? 0u : n) + t) * HK + hk) * VEC + 16u * c;
            lds_dma16<false>((uintptr_t)a.qn, voff, lbase + buf * BUF + 1024u * i);
        }
        const uint32_t tg = min(tb + lane % GDN_STAGE, last);
        w.g = a.gate[(size_t)tg * HV + h];
        w.b = a.bgate[(size_t)tg * HV + h];
#pragma unroll
        for (uint32_t i = 0; i < GDN_STAGE; i++)
            w.v[i] = a.qkv[(size_t)min(tb + i, last) * a.c_stride + (size_t)2 * HK * D + (size_t)h * D + col];
    };
    // the stage has landed: its last load has, and loads complete in order
    auto landed = [&](Small &w) { asm volatile("" : "+v"(w.v[GDN_STAGE - 1])::"memory"); };
    auto kvec = [&](uint32_t st, uint32_t i) { return L + (st & 1u) * BUF + i * 2u * VEC; };
    auto qvec = [&](uint32_t st, uint32_t i) { return L + (st & 1u) * BUF + i * 2u * VEC + VEC; };
    const uint32_t nst = (n + GDN_STAGE - 1) / GDN_STAGE;
    Small cur, nxt;
    issue(0, 0, cur);
    landed(cur);
    float kc[RPT], qc[RPT], kn[RPT];
    load(kvec(0, 0), kc);
    load(qvec(0, 0), qc);
    float dkv = 0.0f;
#pragma unroll
    for (uint32_t r = 0; r < RPT; r++) {
        const float pr = s[r] * kc[r];
        dkv = dkv + pr;
    }
    dkv = lanes_sum_f32(dkv, TPC);
    load(kvec(0, 1), kn);
    // one token: its update and o sum beside the next token's kv sum (two
    // independent chains on the same updated state)
    auto token = [&](float vcol, float g, float beta) -> float {
        float u1[RPT];
#pragma unroll
        for (uint32_t r = 0; r < RPT; r++) u1[r] = g * s[r];
        const float t1 = g * dkv;
        const float t2 = vcol - t1;
        const float delta = t2 * beta;
        float dout = 0.0f, dkn = 0.0f;
#pragma unroll
        for (uint32_t r = 0; r < RPT; r++) {
            const float u2 = kc[r] * delta;
            s[r] = u1[r] + u2;
            const float po = s[r] * qc[r], pn = s[r] * kn[r];
            dout = dout + po;
            dkn = dkn + pn;
        }
        dkv = lanes_sum_f32(dkn, TPC);
        return lanes_sum_f32(dout, TPC) * a.scale;
    };
    float *orow = a.o + (size_t)h * D + col;
    auto lane_f = [](float v, uint32_t i) {
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), (int)i));
    };
    uint32_t st = 0;
    // whole stages (kc, qc of the stage's first token and kn of the one after
    // it are loaded, dkv is the first token's)
    for (; (st + 1) * GDN_STAGE <= n; st++) {
        // every LDS read so far has landed, the last ones of the buffer that
        // is filled next among them, in whatever order they were issued (the
        // last stage fills it too, with its own tokens, which nothing uses: a
        // branch here cost 6 % at 1024 tokens, 27 % at head size 256)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        issue(min(st + 1, nst - 1), (st + 1) & 1u, nxt);
        const uint32_t tb = st * GDN_STAGE;
        float ov = 0.0f;   // token tb + p's output (every thread of a column has it: one store per stage)
#pragma unroll
        for (uint32_t i = 0; i < GDN_STAGE; i++) {
            float qx[RPT], kx[RPT];   // the next token's q, the k after that
            if (i == GDN_STAGE - 2) landed(nxt);
            load(i + 1 < GDN_STAGE ? qvec(st, i + 1) : qvec(st + 1, 0), qx);
            load(i + 2 < GDN_STAGE ? kvec(st, i + 2) : kvec(st + 1, i + 2 - GDN_STAGE), kx);
            const float o = token(cur.v[i], lane_f(cur.g, i), lane_f(cur.b, i));
            ov = p == i ? o : ov;
#pragma unroll
            for (uint32_t r = 0; r < RPT; r++) { kc[r] = kn[r]; qc[r] = qx[r]; kn[r] = kx[r]; }
        }
        if (TPC == GDN_STAGE || p < GDN_STAGE) orow[(size_t)(tb + p) * HV * D] = ov;
        cur = nxt;
    }
    // the last, partial stage (already staged; sums for tokens past the end are dropped)
    for (uint32_t i = 0; i < n - st * GDN_STAGE; i++) {
        const uint32_t i1 = min(i + 1, GDN_STAGE - 1), i2 = min(i + 2, GDN_STAGE - 1);
        float qx[RPT], kx[RPT];
        load(qvec(st, i1), qx);
        load(kvec(st, i2), kx);
        float v = cur.v[0];
#pragma unroll
        for (uint32_t j = 1; j < GDN_STAGE; j++) v = i == j ? cur.v[j] : v;
        const float o = token(v, lane_f(cur.g, i), lane_f(cur.b, i));
        if (p == 0) orow[(size_t)(st * GDN_STAGE + i) * HV * D] = o;
#pragma unroll
        for (uint32_t r = 0; r < RPT; r++) { kc[r] = kn[r]; qc[r] = qx[r]; kn[r] = kx[r]; }
    }
#pragma unroll
    for (uint32_t r = 0; r < RPT; r += 4) {
        const f32x4 v = {s[r], s[r + 1], s[r + 2], s[r + 3]};
        *reinterpret_cast<f32x4 *>(srow + r) = v;
    }
}

// ------------------------------------------------------------------ attention prep

struct AttnPrepUb {
    const float *qg;      // [T][NQ][2*HD]: q | gate
    const float *k, *v;   // [T][NKV*HD]
    const float *q_norm, *k_norm;
    void *kc, *vc;        // the cache: rows [n_ctx][NKV heads], f16 or Q8_0
    float *qr;            // [T][NQ][HD] normalised, rotated q
    int32_t pos0;
    uint32_t n_tok, nq, nkv, hd, rope_dims, kv_type;
    float theta_scale, eps;
};

// One wave per (token, head): heads j < NQ are the token's q heads (into qr),
// heads NQ + g its k head g, appended (with v head g, raw) at row pos0 + t.
// The decode's att_prep arithmetic: lane l holds elements 4l..4l+3; the sum
// of squares is the lane's four fp32 squares added in fp64 in order, then
// wave_sum_f64; y = (x * (1/sqrtf(mean + eps))) * w; rope pair (i, i + half)
// turns by theta_i = pos * theta_scale^i (repeated fp32 products), cos and
// sin evaluated in fp64 and rounded; the cache gets f16 (round to nearest
// even) or ggml's reference Q8_0 blocks (amax / 127, codes roundf(x * 1/d)).
__global__ __launch_bounds__(256) void attn_prep_ubatch_kernel(AttnPrepUb a) {
    const uint32_t t = blockIdx.x, lane = threadIdx.x & 63u;
    const uint32_t j = blockIdx.y * 4u + (threadIdx.x >> 6);
    if (j >= a.nq + a.nkv) return;   // (wave-uniform)
    const int pos = a.pos0 + (int)t;
    const uint32_t HD = a.hd, RW = a.nkv * HD, e0 = 4 * lane;
    const bool isq = j < a.nq;
    const uint32_t g = isq ? 0u : j - a.nq;
    const float *src = isq ? a.qg + ((size_t)t * a.nq + j) * 2 * HD : a.k + (size_t)t * RW + (size_t)g * HD;
    const float4 x = reinterpret_cast<const float4 *>(src)[lane];
    const float4 wt = reinterpret_cast<const float4 *>(isq ? a.q_norm : a.k_norm)[lane];
    double ss = (double)(x.x * x.x);
    ss += (double)(x.y * x.y);
    ss += (double)(x.z * x.z);
    ss += (double)(x.w * x.w);
    ss = wave_sum_f64(ss);
    const float hs = 1.0f / sqrtf((float)(ss / 256.0) + a.eps);
    const float xv[4] = {x.x, x.y, x.z, x.w}, wv[4] = {wt.x, wt.y, wt.z, wt.w};
    float y[4], o[4];
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
        const float nrm = xv[c] * hs;
        y[c] = nrm * wv[c];
    }
    const uint32_t half = a.rope_dims / 2, pl = half / 4, partner = lane < pl ? lane + pl : lane - pl;
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) o[c] = __shfl(y[c], (int)partner, 64);
#pragma unroll
    for (uint32_t c = 0; c < 4; c++) {
        const uint32_t i = e0 + c;
        if (i < 2 * half) {
            const uint32_t ri = i < half ? i : i - half;
            float th = (float)pos;
            for (uint32_t k = 0; k < ri; k++) th *= a.theta_scale;
            const float cs = (float)cos((double)th), sn = (float)sin((double)th);
            if (i < half) {
                const float a0 = y[c] * cs, a1 = o[c] * sn;
                y[c] = a0 - a1;
            } else {
                const float b0 = o[c] * sn, b1 = y[c] * cs;
                y[c] = b0 + b1;
            }
        }
    }
    if (isq) {
        reinterpret_cast<float4 *>(a.qr + ((size_t)t * a.nq + j) * HD)[lane] = make_float4(y[0], y[1], y[2], y[3]);
        return;
    }
    const float4 vr4 = reinterpret_cast<const float4 *>(a.v + (size_t)t * RW + (size_t)g * HD)[lane];
    const float vv[4] = {vr4.x, vr4.y, vr4.z, vr4.w};
    if (a.kv_type != SINTER_Q8_0) {
        uint16_t *kr = static_cast<uint16_t *>(a.kc) + (size_t)pos * RW + (size_t)g * HD + e0;
        uint16_t *vrow = static_cast<uint16_t *>(a.vc) + (size_t)pos * RW + (size_t)g * HD + e0;
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) {
            kr[c] = f2h(y[c]);
            vrow[c] = f2h(vv[c]);
        }
        return;
    }
    // Q8_0: block b = lane / 8 of the head row holds the lane's 4 elements
    const size_t row_bytes = (size_t)a.nkv * ATT_Q8_HEAD;
    auto q8 = [&](const float val[4], unsigned char *row) {
        float am = fmaxf(fmaxf(fabsf(val[0]), fabsf(val[1])), fmaxf(fabsf(val[2]), fabsf(val[3])));
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) am = fmaxf(am, __shfl_xor(am, off, 64));
        const float d = am / 127.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        unsigned char *blk = row + (lane >> 3) * 34u;
#pragma unroll
        for (uint32_t c = 0; c < 4; c++) blk[2 + 4 * (lane & 7u) + c] = (unsigned char)(int8_t)roundf(val[c] * id);
        if ((lane & 7u) == 0) {
            const uint16_t dh = f2h(d);
            blk[0] = (unsigned char)(dh & 0xff);
            blk[1] = (unsigned char)(dh >> 8);
        }
    };
    q8(y, static_cast<unsigned char *>(a.kc) + (size_t)pos * row_bytes + (size_t)g * ATT_Q8_HEAD);
    q8(vv, static_cast<unsigned char *>(a.vc) + (size_t)pos * row_bytes + (size_t)g * ATT_Q8_HEAD);
}

// ------------------------------------------------------------------ causal attention of the ubatch

struct AttnPrefill {
    const float *qr;      // [T][NQ][HD]
    const float *qg;      // [T][NQ][2*HD] (the gate halves)
    const void *kc, *vc;
    float *part;          // [T][NQ][C][att_rec(HD)] chunk partials: O[HD], M, L
    float *out;           // [T][NQ*HD] gated attention output
    int32_t pos0;
    uint32_t n_tok, nq, nkv, hd, kv_type, n_chunks, chunk_min;
    float scale;
};

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr uint32_t PF_SLOTS = 16;   // queries per work item: the MFMA's 16
// K/V tile buffers (tile j + 1 loads while tile j is computed): two, so that
// the workgroup's LDS fits two workgroups per CU
constexpr uint32_t PF_NBUF = 2;
constexpr uint32_t PF_Q8_KC = 2 * PF_NBUF * ATT_Q8_RAWB, PF_Q8_VC = PF_Q8_KC + 32 * 256;
constexpr uint32_t PF_Q8_KS = PF_Q8_VC + 32 * 256, PF_Q8_VS = PF_Q8_KS + 32 * 8 * 4;
constexpr uint32_t PF_COMB = 8u * 8u * 256u * 4u;   // the row groups' V sums of 8 queries
constexpr uint32_t PF_TILES = PF_NBUF * ATT_F16_BUF > PF_COMB ? PF_NBUF * ATT_F16_BUF : PF_COMB;
static_assert(PF_Q8_VS + 32 * 8 * 4 <= PF_TILES, "Q8_0 tiles fit the tile region");

// Work item = (kv head g, split chunk c, q head hh of g's group, block of 16
// consecutive queries), the block index running over the query blocks
// first, so the items that read one chunk of one kv head run side by side.
// Query i of the ubatch (position pos0 + i) is split exactly as the decode
// splits it at that position: att_geom(pos0 + i + 1, C, chunk_min) chunks of
// tpc tiles, chunk c holding rows [c tpc 32, min((c + 1) tpc 32, pos0 + i +
// 1)).  The item runs the union of its queries' chunk-c rows in the decode
// attention's tiles; a row outside a query's own range is masked out of its
// scores and enters its V sums as fmaf(0, v, acc) (no change but the sign of a
// zero sum, which the Q8_K quantisation of the attention output erases), or
// not at all where v is not finite.  Per query the chunk partial -- the 8 row
// groups merged, O, M, L -- is the decode's, bit for bit.
//
// The decode's fmaf chains run on v_mfma_f32_16x16x1_4b_f32: four 16 x 16
// blocks, one product each, every output a single fmaf (checked bit for bit,
// subnormals included), at twice the VALU's rate and without the lanes'
// exchanges:
//   scores  wave w takes the dims of the decode's lanes p in {w, 15 - w,
//           7 - w, 8 + w} (a block each) and p + 16: blocks of 16 rows (A) x
//           16 queries (B) over the 8 dims of each p, ascending.  The first
//           three levels of the decode's sum over the lanes (masks 16, 15, 7)
//           are then adds between registers of a lane, the last two (2, 1)
//           adds of the four waves' results, exchanged through LDS.
//   V sums  wave w holds row groups 2w and 2w + 1: 16 queries (A, their
//           weights of one row) x 64 dims (B) per MFMA, lane l's B being dim
//           4l + jj of the row; the groups' 4 rows of a tile ascending.
// The softmax state of row groups 2w and 2w + 1 lives in wave w (a thread per
// two rows and query), so only the scores cross waves: one barrier beside the
// tile's.  K rows lie in LDS as 16-byte chunks, chunk p at slot p ^ (row %
// 16), so 16 rows' reads of one chunk hit distinct banks.  256 queries behind
// 8192 positions, 27B shapes: 1.60 ms with VALU chains (8 queries per item),
// 0.99 ms so.  An item costs the same for fewer queries, where the chains took
// half the slots: 8 queries behind 8192 positions 75 and 73 us, behind 131,008
// 630 and 715.
template <bool Q8>
__global__ __launch_bounds__(256, 2) void attn_prefill_split_kernel(AttnPrefill a, uint32_t cmax) {
    __shared__ __attribute__((aligned(16))) unsigned char tiles[PF_TILES];
    __shared__ __attribute__((aligned(16))) float sx[4 * 32 * PF_SLOTS];         // scores: [wave][row][query]
    __shared__ __attribute__((aligned(16))) float wl[32 * PF_SLOTS + 8 * PF_SLOTS];   // weights [row][query], corrections [group][query]
    __shared__ __attribute__((aligned(16))) float gm[2 * 8 * PF_SLOTS];           // m, l [group][query]
    const uint32_t t = threadIdx.x, HD = a.hd, NQ = a.nq, NKV = a.nkv, gqa = NQ / NKV, C = a.n_chunks;
    const uint32_t n_qb = (a.n_tok + PF_SLOTS - 1) / PF_SLOTS;
    uint32_t it = blockIdx.x;
    const uint32_t qb = it % n_qb; it /= n_qb;
    const uint32_t hh = it % gqa; it /= gqa;
    const uint32_t c = it % cmax, g = it / cmax;
    const uint32_t head = g * gqa + hh, q0 = qb * PF_SLOTS, nqs = min(PF_SLOTS, a.n_tok - q0);
    const uint32_t lane = t & 63u, w = __builtin_amdgcn_readfirstlane(t >> 6), l16 = lane & 15u, lb = lane >> 4;
    // the chunk-c rows [k0, k1) of query `lane % 16` (empty when its split has
    // fewer chunks), and their union U0, U1 over the item's queries
    uint32_t k0 = 0, k1 = 0;
    if (l16 < nqs) {
        const uint32_t n_kv = (uint32_t)a.pos0 + q0 + l16 + 1u;
        const AttGeom geo = att_geom(n_kv, C, a.chunk_min);
        if (c < geo.n) {
            k0 = c * geo.tpc * ATT_TILE;
            k1 = min(k0 + geo.tpc * ATT_TILE, n_kv);
        }
    }
    uint32_t U0 = k1 > k0 ? k0 : 0xffffffffu, U1 = k1;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
        U0 = min(U0, (uint32_t)__shfl_xor((int)U0, o, 64));
        U1 = max(U1, (uint32_t)__shfl_xor((int)U1, o, 64));
    }
    U0 = __builtin_amdgcn_readfirstlane(U0);
    U1 = __builtin_amdgcn_readfirstlane(U1);
    if (U1 == 0) return;   // (uniform) no query of the block has a chunk c
    const uint32_t ntile = (U1 - U0 + ATT_TILE - 1) / ATT_TILE;
    const uint32_t HB = Q8 ? ATT_Q8_HEAD : HD * 2u, RWB = NKV * HB;
    LDS unsigned char *Lu = (LDS unsigned char *)tiles;
    const uint32_t kbase = (uint32_t)(uintptr_t)Lu;
    // tile j (rows U0 + 32 j ..) into buffer j % PF_NBUF; rows past U1 re-read
    // row U1 - 1
    auto issue_tile = [&](uint32_t j) {
        const uint32_t t0 = U0 + j * ATT_TILE;
        if constexpr (!Q8) {
            const uint32_t bo = (j % PF_NBUF) * ATT_F16_BUF;
#pragma unroll
            for (uint32_t kk = 0; kk < 4; kk++) {
                const uint32_t k = w + 4 * kk, r = 2 * k + (lane >> 5), row = min(t0 + r, U1 - 1);
                const uint32_t off = row * RWB + g * HB, slot = lane & 31;
                lds_dma16<false>((uintptr_t)a.kc, off + (slot ^ (r & 15u)) * 16, kbase + bo + k * 1024);
                lds_dma16<false>((uintptr_t)a.vc, off + slot * 16, kbase + bo + ATT_TILE * 512 + k * 1024);
            }
        } else {
            const uint32_t rb = (j % PF_NBUF) * 2 * ATT_Q8_RAWB;
#pragma unroll
            for (uint32_t kk = 0; kk < 3; kk++) {
                const uint32_t c0 = 136u * w + 64u * kk, ci = c0 + lane;
                const uint32_t row = min(t0 + ci / 17u, U1 - 1), voff = row * RWB + g * HB + (ci % 17u) * 16u;
                lds_dma16<false>((uintptr_t)a.kc, voff, kbase + rb + c0 * 16u);
                lds_dma16<false>((uintptr_t)a.vc, voff, kbase + rb + ATT_Q8_RAWB + c0 * 16u);
            }
        }
    };
    issue_tile(0);
    // score operands: block lb of the MFMAs holds lane group p = xp (+ 16)
    const uint32_t xp = lb == 0 ? w : lb == 1 ? 15u - w : lb == 2 ? 7u - w : 8u + w;
    float qv[2][8];
#pragma unroll
    for (uint32_t j = 0; j < 2; j++) {
        const bool ok = l16 < nqs;
        const float *src = a.qr + ((size_t)(q0 + (ok ? l16 : 0u)) * NQ + head) * HD + 8 * (xp + 16 * j);
        const float4 v0 = reinterpret_cast<const float4 *>(src)[0], v1 = reinterpret_cast<const float4 *>(src)[1];
        const float q8v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (uint32_t d = 0; d < 8; d++) qv[j][d] = ok ? q8v[d] : 0.0f;
        // (waited for here: the loop's waits would be for the next tile's DMA too)
#pragma unroll
        for (uint32_t d = 0; d < 8; d++) asm volatile("" : "+v"(qv[j][d]));
    }
    const f32x16 z16 = {0.0f};
    f32x16 acc[2][4];   // V sums: [row group 2w + gi][jj]: query 4 lb + v, dim 64 b + 4 l16 + jj at element 4 b + v
#pragma unroll
    for (uint32_t gi = 0; gi < 2; gi++)
#pragma unroll
        for (uint32_t jj = 0; jj < 4; jj++) acc[gi][jj] = z16;
    // softmax: this thread's row group, query, and pair of the group's rows of a tile
    const uint32_t rr = t >> 5, sq = (t >> 1) & 15u, hf = t & 1u;
    const uint32_t my0 = (uint32_t)__shfl((int)k0, (int)sq, 64), my1 = (uint32_t)__shfl((int)k1, (int)sq, 64);
    float mrun = -INFINITY, lrun = 0.0f;
    LDS float *S = (LDS float *)sx, *W = (LDS float *)wl, *CF = W + 32 * PF_SLOTS, *gml = (LDS float *)gm;

    for (uint32_t j = 0; j < ntile; j++) {
        const uint32_t t0 = U0 + j * ATT_TILE, b = j % PF_NBUF;
        dma_wait();
        __syncthreads();   // tile j landed for every wave; every wave is past tile j - 1
        if (j + 1 < ntile) issue_tile(j + 1);   // into the buffer tile j - 1 used
        const LDS unsigned char *kt = Lu + b * ATT_F16_BUF, *vt = kt + ATT_TILE * 512;
        if constexpr (Q8) {
            // thread t: block bb of row rq; K codes as 16-byte chunks, chunk i
            // at slot i ^ (row % 16)
            const uint32_t rq = t >> 3, bb = t & 7u, rb = b * 2 * ATT_Q8_RAWB;
            const LDS unsigned char *raw = Lu + rb + rq * ATT_Q8_HEAD + 34u * bb;
            const LDS uint16_t *hw = reinterpret_cast<const LDS uint16_t *>(raw);
            uint32_t cw[8];
#pragma unroll
            for (int i = 0; i < 8; i++) cw[i] = (uint32_t)hw[1 + 2 * i] | ((uint32_t)hw[2 + 2 * i] << 16);
            LDS unsigned char *krow = Lu + PF_Q8_KC + rq * 256;
            const u32x4 c0 = {cw[0], cw[1], cw[2], cw[3]}, c1 = {cw[4], cw[5], cw[6], cw[7]};
            *reinterpret_cast<LDS u32x4 *>(krow + 16u * ((2u * bb) ^ (rq & 15u))) = c0;
            *reinterpret_cast<LDS u32x4 *>(krow + 16u * ((2u * bb + 1u) ^ (rq & 15u))) = c1;
            reinterpret_cast<LDS float *>(Lu + PF_Q8_KS)[t] = h2f(hw[0]);
            sched_fence();
            att_q8_split(raw + ATT_Q8_RAWB, Lu + PF_Q8_VC + rq * 256 + 32u * bb,
                         reinterpret_cast<LDS float *>(Lu + PF_Q8_VS) + t);
            __syncthreads();
            kt = Lu + PF_Q8_KC;
            vt = Lu + PF_Q8_VC;
        }
        // scores: rows 16 rb + l16 (A), queries (B); all of the tile's reads first
        u32x4 kraw[2][2];
        float ks[2][2];
#pragma unroll
        for (uint32_t rb = 0; rb < 2; rb++)
#pragma unroll
            for (uint32_t jj = 0; jj < 2; jj++) {
                const uint32_t row = 16 * rb + l16, p = xp + 16 * jj;
                if constexpr (!Q8) {
                    kraw[rb][jj] = *reinterpret_cast<const LDS u32x4 *>(kt + row * 512u + 16u * (p ^ l16));
                } else {
                    // (8 codes: half p % 2 of 16-byte chunk p / 2, in its slot)
                    const u32x2 u = *reinterpret_cast<const LDS u32x2 *>(kt + row * 256u + 16u * ((p >> 1) ^ l16) + 8u * (p & 1u));
                    kraw[rb][jj] = u32x4{u.x, u.y, 0u, 0u};
                    ks[rb][jj] = reinterpret_cast<const LDS float *>(Lu + PF_Q8_KS)[row * 8 + (p >> 2)];
                }
            }
        sched_fence();
#pragma unroll
        for (uint32_t rb = 0; rb < 2; rb++) {
            f32x16 d[2];
#pragma unroll
            for (uint32_t jj = 0; jj < 2; jj++) {
                float kd[8];
#pragma unroll
                for (uint32_t k = 0; k < 8; k++) {
                    const uint32_t u = kraw[rb][jj][Q8 ? k >> 2 : k >> 1];
                    if constexpr (!Q8) kd[k] = h2f((uint16_t)(u >> (16 * (k & 1u))));
                    else kd[k] = (float)(int)(int8_t)((u >> (8 * (k & 3u))) & 0xffu) * ks[rb][jj];
                }
                d[jj] = z16;
#pragma unroll
                for (uint32_t dd = 0; dd < 8; dd++)
                    d[jj] = __builtin_amdgcn_mfma_f32_16x16x1f32(kd[dd], qv[jj][dd], d[jj], 0, 0, 0);
            }
            // lane masks 16, 15, 7: elements 4 b + v of both, blocks (0, 1) and (2, 3), the two pairs
#pragma unroll
            for (uint32_t v = 0; v < 4; v++) {
                const float b0 = d[0][v] + d[1][v], b1 = d[0][4 + v] + d[1][4 + v];
                const float b2 = d[0][8 + v] + d[1][8 + v], b3 = d[0][12 + v] + d[1][12 + v];
                const float c0 = b0 + b1, c1 = b2 + b3;
                S[(w * 32 + 16 * rb + 4 * lb + v) * PF_SLOTS + l16] = c0 + c1;
            }
        }
        // the V rows of row groups 2w and 2w + 1, read while the scores cross
        // (f16; the Q8_0 codes and scales where they are used, for registers)
        u32x2 vraw[4][2];
        if constexpr (!Q8) {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++)
#pragma unroll
                for (uint32_t gi = 0; gi < 2; gi++)
                    vraw[i][gi] = *reinterpret_cast<const LDS u32x2 *>(vt + (2 * w + gi + 8 * i) * 512u + 8u * lane);
        }
        __syncthreads();
        bool changed;
        const bool partial = my1 > my0 && (t0 < my0 || t0 + ATT_TILE > my1);
        {
            float sv[2], wg[2];
            bool ok[2];
#pragma unroll
            for (uint32_t i = 0; i < 2; i++) {
                const uint32_t r = rr + 8 * (2 * hf + i), o = r * PF_SLOTS + sq;
                // lane masks 2, 1
                const float e0 = S[o] + S[2 * 32 * PF_SLOTS + o], e1 = S[32 * PF_SLOTS + o] + S[3 * 32 * PF_SLOTS + o];
                ok[i] = t0 + r >= my0 && t0 + r < my1;
                sv[i] = ok[i] ? (e0 + e1) * a.scale : -INFINITY;
            }
            float mt = fmaxf(sv[0], sv[1]);
            mt = fmaxf(mt, dpp_f<DPP_XOR1>(mt));
            const float mn = fmaxf(mrun, mt);
#pragma unroll
            for (uint32_t i = 0; i < 2; i++) {
                wg[i] = ok[i] ? att_exp(sv[i] - mn) : 0.0f;
                W[(rr + 8 * (2 * hf + i)) * PF_SLOTS + sq] = wg[i];
            }
            float ws = wg[0] + wg[1];
            ws = ws + dpp_f<DPP_XOR1>(ws);
            // the correction is 1 unless the maximum moved, in few tiles
            float cf = mrun == -INFINITY ? 0.0f : 1.0f;
            const bool moved = mrun != -INFINITY && mrun != mn;
            if (__builtin_amdgcn_ballot_w64(moved) != 0) {
                const float ce = att_exp(mrun - mn);
                cf = moved ? ce : cf;
            }
            const float lc = lrun * cf;
            lrun = lc + ws;
            mrun = mn;
            if (hf == 0) CF[rr * PF_SLOTS + sq] = cf;
            changed = cf != 1.0f;
        }
        // (weights and corrections are read back by this wave only: LDS
        // accesses of a wave complete in order)
        if (__builtin_amdgcn_ballot_w64(changed || partial) != 0) {
            if (__builtin_amdgcn_ballot_w64(changed) != 0) {
#pragma unroll
                for (uint32_t gi = 0; gi < 2; gi++) {
                    const f32x4 cv = *reinterpret_cast<const LDS f32x4 *>(CF + (2 * w + gi) * PF_SLOTS + 4 * lb);
#pragma unroll
                    for (uint32_t jj = 0; jj < 4; jj++)
#pragma unroll
                        for (uint32_t e = 0; e < 16; e++) acc[gi][jj][e] = acc[gi][jj][e] * cv[e & 3u];
                }
            }
            // a tile with rows that some query does not hold: a V value in it
            // that is not finite is added here, to the queries that hold its
            // row, and is 0 below, where a zero weight would not keep it out of
            // the others.  (Selects and no branches inside, and out of the
            // loop's way: 256 queries behind 8192 positions 968 us without,
            // 985 so, 989 with a branch per value; behind 131,008 10.76, 10.90
            // and 11.21 ms.)
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(partial) != 0, 0)) {
                // (the lane is opaque: addresses made of it would be kept in
                // registers through the loop, and spill)
                uint32_t ln = lane;
                asm volatile("" : "+v"(ln));
                const uint32_t n16 = ln & 15u, nb4 = ln >> 4;
                LDS float *vs = reinterpret_cast<LDS float *>(Lu + PF_Q8_VS);
                const uint32_t vo = (2 * w + ((ln >> 3) & 1u) + 8 * nb4) * 8 + (ln & 7u);   // the wave's 64 scales
                bool bad = false;
                if constexpr (Q8) {
                    bad = !(fabsf(vs[vo]) < INFINITY);
                } else {
#pragma unroll
                    for (uint32_t i = 0; i < 4; i++)
#pragma unroll
                        for (uint32_t gi = 0; gi < 2; gi++) {
                            const uint32_t x = ~vraw[i][gi].x & 0x7c007c00u, y = ~vraw[i][gi].y & 0x7c007c00u;
                            bad |= !(x & 0xffffu) || !(x >> 16) || !(y & 0xffffu) || !(y >> 16);
                        }
                }
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(bad) != 0, 0)) {
#pragma unroll 1
                    for (uint32_t i = 0; i < 4; i++)
#pragma unroll
                        for (uint32_t gi = 0; gi < 2; gi++) {
                            const uint32_t r = 2 * w + gi + 8 * i;
                            // (query q's bounds: lane 2 q)
                            const uint64_t holds = __builtin_amdgcn_ballot_w64(t0 + r >= my0 && t0 + r < my1) >> (8 * nb4);
                            const f32x4 wq = *reinterpret_cast<const LDS f32x4 *>(W + r * PF_SLOTS + 4 * nb4);
#pragma unroll
                            for (uint32_t b4 = 0; b4 < 4; b4++) {
                                sched_fence();
                                float vd[4];
                                if constexpr (!Q8) {
                                    const u32x2 u = *reinterpret_cast<const LDS u32x2 *>(vt + r * 512u + 8u * (16 * b4 + n16));
#pragma unroll
                                    for (uint32_t k = 0; k < 4; k++) vd[k] = h2f((uint16_t)((k < 2 ? u.x : u.y) >> (16 * (k & 1u))));
                                } else {
                                    const uint32_t u = *reinterpret_cast<const LDS uint32_t *>(vt + r * 256u + 4u * (16 * b4 + n16));
#pragma unroll
                                    for (uint32_t k = 0; k < 4; k++)
                                        vd[k] = (float)(int)(int8_t)((u >> (8 * k)) & 0xffu) * vs[r * 8 + ((16 * b4 + n16) >> 3)];
                                }
#pragma unroll
                                for (uint32_t jj = 0; jj < 4; jj++)
#pragma unroll
                                    for (uint32_t v = 0; v < 4; v++) {
                                        const float o = acc[gi][jj][4 * b4 + v], n = fmaf(wq[v], vd[jj], o);
                                        acc[gi][jj][4 * b4 + v] = !(fabsf(vd[jj]) < INFINITY) && ((holds >> (2 * v)) & 1u) ? n : o;
                                    }
                            }
                        }
                    if constexpr (Q8) {
                        if (bad) vs[vo] = 0.0f;
                    } else {
#pragma unroll
                        for (uint32_t i = 0; i < 4; i++)
#pragma unroll
                            for (uint32_t gi = 0; gi < 2; gi++)
#pragma unroll
                                for (uint32_t k = 0; k < 2; k++) {
                                    uint32_t &u = reinterpret_cast<uint32_t *>(&vraw[i][gi])[k];
                                    if (!(~u & 0x7c00u)) u &= 0xffff0000u;
                                    if (!(~u & 0x7c000000u)) u &= 0xffffu;
                                }
                    }
                }
            }
        }
        float wt[4][2];
#pragma unroll
        for (uint32_t i = 0; i < 4; i++)
#pragma unroll
            for (uint32_t gi = 0; gi < 2; gi++) wt[i][gi] = W[(2 * w + gi + 8 * i) * PF_SLOTS + l16];
#pragma unroll
        for (uint32_t i = 0; i < 4; i++)
#pragma unroll
            for (uint32_t gi = 0; gi < 2; gi++) {
                float vd[4];
                if constexpr (!Q8) {
                    const u32x2 u = vraw[i][gi];
#pragma unroll
                    for (uint32_t k = 0; k < 4; k++) vd[k] = h2f((uint16_t)((k < 2 ? u.x : u.y) >> (16 * (k & 1u))));
                } else {
                    const uint32_t r = 2 * w + gi + 8 * i, u = *reinterpret_cast<const LDS uint32_t *>(vt + r * 256u + 4u * lane);
                    const float vs = reinterpret_cast<const LDS float *>(Lu + PF_Q8_VS)[r * 8 + (lane >> 3)];
#pragma unroll
                    for (uint32_t k = 0; k < 4; k++) vd[k] = (float)(int)(int8_t)((u >> (8 * k)) & 0xffu) * vs;
                }
#pragma unroll
                for (uint32_t jj = 0; jj < 4; jj++)
                    acc[gi][jj] = __builtin_amdgcn_mfma_f32_16x16x1f32(wt[i][gi], vd[jj], acc[gi][jj], 0, 0, 0);
            }
    }
    // the chunk's partial per query: the eight row groups merged (through
    // LDS, in the tile region, 8 queries at a time) as the decode merges them
    LDS float *comb = reinterpret_cast<LDS float *>(Lu);   // [8 groups][8 queries][256]
    if (hf == 0) {
        gml[rr * PF_SLOTS + sq] = mrun;
        gml[(8 + rr) * PF_SLOTS + sq] = lrun;
    }
    __syncthreads();
    // each group's weight once (threads 0-127: group t / 16, query t % 16)
    LDS float *ge = W, *gM = W + 8 * PF_SLOTS;
    if (t < 8 * PF_SLOTS) {
        float M = -INFINITY;
#pragma unroll
        for (uint32_t g2 = 0; g2 < 8; g2++) M = fmaxf(M, gml[g2 * PF_SLOTS + l16]);
        const float mg = gml[t];
        ge[t] = mg != -INFINITY ? att_exp(mg - M) : 0.0f;
        if (t < PF_SLOTS) gM[t] = M;
    }
#pragma unroll
    for (uint32_t qh = 0; qh < 2; qh++) {
        if (qh) __syncthreads();
        if (lb >> 1 == qh) {
#pragma unroll
            for (uint32_t gi = 0; gi < 2; gi++)
#pragma unroll
                for (uint32_t v = 0; v < 4; v++)
#pragma unroll
                    for (uint32_t b = 0; b < 4; b++) {
                        const f32x4 o = {acc[gi][0][4 * b + v], acc[gi][1][4 * b + v], acc[gi][2][4 * b + v],
                                         acc[gi][3][4 * b + v]};
                        *reinterpret_cast<LDS f32x4 *>(comb + ((2 * w + gi) * 8 + 4 * (lb & 1u) + v) * 256 + 64 * b +
                                                       4 * l16) = o;
                    }
        }
        __syncthreads();
        const uint32_t s = t >> 5, po = t & 31, q = 8 * qh + s;
        const float M = gM[q];
        float Lc = 0.0f, o[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (uint32_t g2 = 0; g2 < 8; g2++) {
            const float e = ge[g2 * PF_SLOTS + q];
            Lc = fmaf(e, gml[(8 + g2) * PF_SLOTS + q], Lc);
            const f32x4 c0 = *reinterpret_cast<const LDS f32x4 *>(comb + (g2 * 8 + s) * 256 + 8 * po);
            const f32x4 c1 = *reinterpret_cast<const LDS f32x4 *>(comb + (g2 * 8 + s) * 256 + 8 * po + 4);
            const float cv[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
            for (uint32_t dd = 0; dd < 8; dd++) o[dd] = fmaf(e, cv[dd], o[dd]);
        }
        const uint32_t m0 = (uint32_t)__shfl((int)my0, (int)(2 * q), 64), m1 = (uint32_t)__shfl((int)my1, (int)(2 * q), 64);
        if (m1 > m0) {
            const uint32_t PS = att_rec(HD);
            float *d = a.part + (((size_t)(q0 + q) * NQ + head) * C + c) * PS;
            reinterpret_cast<float4 *>(d + 8 * po)[0] = make_float4(o[0], o[1], o[2], o[3]);
            reinterpret_cast<float4 *>(d + 8 * po)[1] = make_float4(o[4], o[5], o[6], o[7]);
            if (po == 0) {
                d[HD] = M;
                d[HD + 1] = Lc;
            }
        }
    }
}

// The decode attention's merge per (query, q head) -- one workgroup each,
// thread d the output element d: M = max over the query's chunks of m_c,
// e_c = exp(m_c - M), L = sum e_c l_c and O = sum e_c O_c as fmaf chains
// over the chunks ascending; out = O / L * sigmoid(gate).
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(AttnPrefill a) {
    __shared__ float e[64];
    __shared__ float Ls;
    const uint32_t q = blockIdx.x / a.nq, head = blockIdx.x % a.nq, HD = a.hd, C = a.n_chunks, PS = att_rec(HD);
    const uint32_t NC = att_geom((uint32_t)a.pos0 + q + 1u, C, a.chunk_min).n;
    const float *pb = a.part + ((size_t)q * a.nq + head) * C * PS;
    const uint32_t t = threadIdx.x;
    if (t < 64) {
        const uint32_t ci = min(t, NC - 1);
        const float m = pb[(size_t)ci * PS + HD], l = pb[(size_t)ci * PS + HD + 1];
        float M = t < NC ? m : -INFINITY;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
        const float ev = t < NC ? att_exp(m - M) : 0.0f;
        float L = 0.0f;
        for (uint32_t k = 0; k < NC; k++) {
            const float ek = __shfl(ev, (int)k, 64), lk = __shfl(l, (int)k, 64);
            L = fmaf(ek, lk, L);
        }
        e[t] = ev;
        if (t == 0) Ls = L;
    }
    __syncthreads();
    if (t < HD) {
        // eight chunks' values in flight (past the last: re-read, weight and
        // add skipped)
        float O = 0.0f;
        for (uint32_t k = 0; k < NC; k += 8) {
            float v[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) v[i] = pb[(size_t)min(k + i, NC - 1) * PS + t];
#pragma unroll
            for (uint32_t i = 0; i < 8; i++)
                if (k + i < NC) O = fmaf(e[k + i], v[i], O);
        }
        const float gate = a.qg[((size_t)q * a.nq + head) * 2 * HD + HD + t];
        a.out[((size_t)q * a.nq + head) * HD + t] = (O / Ls) * dev_sigmoid(gate);
    }
}

}  // namespace

hipError_t launch_embed_ubatch(const void *embd, int type, uint32_t E, const int32_t *tokens, uint32_t n_tok, float *x,
                               hipStream_t s) {
    const dim3 grid((E / 4 + 255) / 256, n_tok);
    hipLaunchKernelGGL(embed_ubatch_kernel, grid, dim3(256), 0, s, static_cast<const char *>(embd), type, E,
                       (uint64_t)sinter_row_bytes_dev(type, E), tokens, x);
    return hipGetLastError();
}

hipError_t launch_gdn_ubatch(const float *qkv, const float *alpha, const float *beta, const float *dt_bias,
                             const float *ssm_a, float *state, float *o, float *work, uint32_t hk, uint32_t hv,
                             uint32_t d, uint32_t n_tok, float eps, float scale, hipStream_t s) {
    GdnUb a;
    a.qkv = qkv; a.alpha = alpha; a.beta = beta; a.dt_bias = dt_bias; a.ssm_a = ssm_a; a.state = state; a.o = o;
    a.qn = work;
    a.kn = a.qn + (size_t)n_tok * hk * d;
    a.gate = a.kn + (size_t)n_tok * hk * d;
    a.bgate = a.gate + (size_t)n_tok * hv;
    a.hk = hk; a.hv = hv; a.d = d; a.n_tok = n_tok;
    a.c_stride = (2 * hk + hv) * d;
    a.eps = eps; a.scale = scale;
    if (n_tok == 0) return hipSuccess;
    hipLaunchKernelGGL(gdn_prep_ubatch_kernel, dim3(n_tok, hk), dim3(256), 0, s, a);
    // the decode op's threads per column: 256 / cols, cols 32 (16 at d = 64)
    switch (d) {
    case 64: hipLaunchKernelGGL((gdn_scan_ubatch_kernel<4, 16>), dim3(hv * 16), dim3(64), 0, s, a); break;
    case 128: hipLaunchKernelGGL((gdn_scan_ubatch_kernel<16, 8>), dim3(hv * 16), dim3(64), 0, s, a); break;
    case 256: hipLaunchKernelGGL((gdn_scan_ubatch_kernel<32, 8>), dim3(hv * 32), dim3(64), 0, s, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// floats of launch_gdn_ubatch's work buffer
size_t gdn_ubatch_work(uint32_t hk, uint32_t hv, uint32_t d, uint32_t n_tok) {
    return (size_t)n_tok * (2 * (size_t)hk * d + 2 * (size_t)hv);
}

hipError_t launch_attn_prep_ubatch(const float *qg, const float *k, const float *v, const float *q_norm,
                                   const float *k_norm, void *kc, void *vc, uint32_t kv_type, int32_t pos0,
                                   uint32_t n_tok, uint32_t nq, uint32_t nkv, uint32_t hd, uint32_t rope_dims,
                                   float theta_scale, float eps, float *qr, hipStream_t s) {
    AttnPrepUb a;
    a.qg = qg; a.k = k; a.v = v; a.q_norm = q_norm; a.k_norm = k_norm; a.kc = kc; a.vc = vc; a.qr = qr;
    a.pos0 = pos0; a.n_tok = n_tok; a.nq = nq; a.nkv = nkv; a.hd = hd; a.rope_dims = rope_dims; a.kv_type = kv_type;
    a.theta_scale = theta_scale; a.eps = eps;
    hipLaunchKernelGGL(attn_prep_ubatch_kernel, dim3(n_tok, (nq + nkv + 3) / 4), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_attn_prefill(const float *qr, const float *qg, const void *kc, const void *vc, uint32_t kv_type,
                               int32_t pos0, uint32_t n_tok, uint32_t nq, uint32_t nkv, uint32_t hd,
                               uint32_t n_chunks, uint32_t chunk_min, float scale, float *part, float *out,
                               hipStream_t s) {
    AttnPrefill a;
    a.qr = qr; a.qg = qg; a.kc = kc; a.vc = vc; a.part = part; a.out = out; a.pos0 = pos0; a.n_tok = n_tok;
    a.nq = nq; a.nkv = nkv; a.hd = hd; a.kv_type = kv_type; a.n_chunks = n_chunks; a.chunk_min = chunk_min;
    a.scale = scale;
    if (n_tok == 0) return hipSuccess;
    // the most chunks any of the queries is split into: not the deepest one's,
    // whose tiles per chunk may just have grown (64 chunks of 4 tiles up to
    // 8192 positions, 52 of 5 at 8193)
    uint32_t cmax = 0;
    for (uint32_t n_kv = (uint32_t)pos0 + 1; n_kv <= (uint32_t)pos0 + n_tok; n_kv = (n_kv + 31u) / 32u * 32u + 1u)
        cmax = std::max(cmax, att_geom(n_kv, n_chunks, chunk_min).n);
    const uint32_t items = nkv * cmax * (nq / nkv) * ((n_tok + PF_SLOTS - 1) / PF_SLOTS);
    if (kv_type == SINTER_Q8_0)
        hipLaunchKernelGGL(attn_prefill_split_kernel<true>, dim3(items), dim3(256), 0, s, a, cmax);
    else
        hipLaunchKernelGGL(attn_prefill_split_kernel<false>, dim3(items), dim3(256), 0, s, a, cmax);
    hipLaunchKernelGGL(attn_prefill_merge_kernel, dim3(n_tok * nq), dim3(256), 0, s, a);
    return hipGetLastError();
}

// floats of launch_attn_prefill's partials buffer
size_t attn_prefill_part(uint32_t n_tok, uint32_t nq, uint32_t hd, uint32_t n_chunks) {
    return (size_t)n_tok * nq * n_chunks * att_rec(hd);
}

}  // namespace sinter
