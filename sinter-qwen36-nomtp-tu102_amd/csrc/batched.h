// Launchers of the batched prefill's kernels (ubatch.hip, prefill.hip) that
// the model (model.cpp) calls; the interpreter's units do not include this.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sinter {

// the batched GEMV (ubatch.hip): n <= UB_SEGS matrices of one type (Q4_K or
// Q6_K, nb 256-element items per row) by the same n_tok >= 1 Q8_K activations,
// one launch; pointers aligned as sinter_op_gemv_ubatch asks
constexpr uint32_t UB_SEGS = 4;
struct UbMat {
    const void *w;
    float *y;
    uint32_t rows;
};
hipError_t launch_gemv_ubatch(int type, const UbMat *m, uint32_t n, uint32_t nb, const void *xq, uint32_t n_tok,
                              bool accumulate, hipStream_t s);

// the batched prefill's own kernels (prefill.hip), launched on s
hipError_t launch_embed_ubatch(const void *embd, int type, uint32_t E, const int32_t *tokens, uint32_t n_tok, float *x,
                               hipStream_t s);
// the GDN step over n_tok tokens; work: gdn_ubatch_work(...) floats
hipError_t launch_gdn_ubatch(const float *qkv, const float *alpha, const float *beta, const float *dt_bias,
                             const float *ssm_a, float *state, float *o, float *work, uint32_t hk, uint32_t hv,
                             uint32_t d, uint32_t n_tok, float eps, float scale, hipStream_t s);
size_t gdn_ubatch_work(uint32_t hk, uint32_t hv, uint32_t d, uint32_t n_tok);
hipError_t launch_attn_prep_ubatch(const float *qg, const float *k, const float *v, const float *q_norm,
                                   const float *k_norm, void *kc, void *vc, uint32_t kv_type, int32_t pos0,
                                   uint32_t n_tok, uint32_t nq, uint32_t nkv, uint32_t hd, uint32_t rope_dims,
                                   float theta_scale, float eps, float *qr, hipStream_t s);
// causal attention of n_tok queries at positions pos0.. over the cache, split
// per query as the decode splits it; part: attn_prefill_part(...) floats
hipError_t launch_attn_prefill(const float *qr, const float *qg, const void *kc, const void *vc, uint32_t kv_type,
                               int32_t pos0, uint32_t n_tok, uint32_t nq, uint32_t nkv, uint32_t hd,
                               uint32_t n_chunks, uint32_t chunk_min, float scale, float *part, float *out,
                               hipStream_t s);
size_t attn_prefill_part(uint32_t n_tok, uint32_t nq, uint32_t hd, uint32_t n_chunks);

}  // namespace sinter
