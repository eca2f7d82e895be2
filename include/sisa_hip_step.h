/*
 * sisa_hip_step.h -- generation entry points of libsisa_hip.so: a decoder layer's step for one new token, and the
 * filling of its cache after a prefill. Conventions (views, status codes, streams, caller-owned buffers) are those of
 * sisa_hip.h.
 */
#ifndef SISA_HIP_STEP_H
#define SISA_HIP_STEP_H

#include "sisa_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

/* One new token of each of B rows through a decoder layer with a filled cache (src/sisa/modeling.py:171-199, 224-238,
 * 288-291 at L = 1), all tensors in one 16-bit dtype:
 *   x' = x + res; n = RMSNorm(x'); q, k, v, b, c, theta, alpha = projections of n; z = forget logits of n (fp32)
 *   Phi, g, F advanced by theta, -softplus(alpha), logsigmoid(z); b~, c~ rotated by Phi; the position appended to the
 *   cache at `pos`; y = attention of the new row over positions 0 .. pos;
 *   h = x' + W_O y;  ffn = w_down(silu(w_gate m) * (w_up m)), m = RMSNorm(h).  The layer's output is h + ffn. */
#define SISA_STEP_MAX_ROWS 64
#define SISA_STEP_MAX_D 1024
typedef struct {
    int32_t B, H, D, FF;       /* rows 1..SISA_STEP_MAX_ROWS, heads, width (64 H), hidden width of the FFN */
    int32_t dtype;             /* SISA_BF16 or SISA_F16 */
    int32_t pos;               /* cached positions before this one (>= 1): where the new one goes */
    float eps_attn, eps_ffn;
    const void* x; int64_t sx;         /* (B, D), row stride sx */
    const void* res;                   /* (B, D) contiguous, added to x first, or NULL */
    const void *attn_norm, *w_q, *w_k, *w_v, *w_b, *w_c, *w_theta, *w_alpha, *b_alpha, *w_forget, *b_forget, *w_o;
    const void *ffn_norm, *w_gate, *w_up, *w_down;     /* all contiguous, (outputs, inputs) */
    const float* lambda_raw;           /* (H) */
    sisa_view k, v, b, g, f;           /* cache slabs (B,H,capacity,64|64|32) in dtype, (B,H,capacity) fp32 */
    const float* phi_in;               /* (B,H,16) contiguous: phase at position pos - 1 */
    float* phi_out;                    /* (B,H,16) contiguous: phase at position pos */
    void *h, *ffn;                     /* (B, D) contiguous outputs */
    void* workspace;                   /* sisa_step_workspace_bytes(B,H,D,FF,pos + 1), 256-byte aligned */
} sisa_step_args;

int64_t sisa_step_workspace_bytes(int32_t B, int32_t H, int32_t D, int32_t FF, int32_t N);
int sisa_step(const sisa_step_args* a, void* stream);

/* Positions 0 .. L-1 of a layer's cache from a prefill's fused projection and preparation: k and v from the columns
 * col_k, col_v of proj (B, L, .), b~, g, F and, from the chunk totals of sisa_prep_fwd, the phase at position L-1
 * (the cache fill of src/sisa/modeling.py:224-238 after the prompt). */
typedef struct {
    int32_t B, H, L;
    int32_t dtype;             /* SISA_BF16 or SISA_F16 */
    const void* proj; int64_t s_b, s_l;
    int32_t col_k, col_v;
    const void* br;            /* (B,L,H,32) contiguous */
    const float *gs, *fs;      /* (B,H,L) contiguous */
    const float* totals;       /* (B*H, ceil(L/64), 18) contiguous */
    sisa_view k, v, b, g, f;   /* cache slabs */
    float* phi;                /* (B,H,16) contiguous */
} sisa_cache_fill_args;

int sisa_cache_fill(const sisa_cache_fill_args* a, void* stream);

/* A prompt of B rows of L positions through a decoder layer with an empty cache, all tensors in one 16-bit dtype: the
 * layer as above for every position (attention among the prompt's own), its cache filled. Outputs: h, the residual
 * stream after the attention; act, silu(w_gate m) * (w_up m), zero in columns FF .. act_ld - 1; and, unless ffn is
 * NULL, ffn = w_down act. rise_ok (or NULL): one byte, whether the cumulative log-decay g nowhere rises by more than
 * rise_tol between neighbours (left alone for L = 1). */
#define SISA_PREFILL_MAX_ROWS 8192
typedef struct {
    int32_t B, L, H, FF;
    int32_t dtype;             /* SISA_BF16 or SISA_F16 */
    float eps_attn, eps_ffn, rise_tol;
    const void *x, *res;               /* (B*L, D) contiguous; res added to x first, or NULL */
    const void *attn_norm, *w_q, *w_k, *w_v, *w_b, *w_c, *w_theta, *w_alpha, *b_alpha, *w_forget, *b_forget, *w_o;
    const void *ffn_norm, *w_gate, *w_up, *w_down;     /* all contiguous, (outputs, inputs) */
    const float* lambda_raw;           /* (H) */
    sisa_view k, v, b, g, f;           /* cache slabs (B,H,capacity,64|64|32) in dtype, (B,H,capacity) fp32 */
    float* phi;                        /* (B,H,16) contiguous: phase at position L - 1 */
    void *h, *act, *ffn;               /* (B*L, D), (B*L, act_ld), (B*L, D) */
    int64_t act_ld;                    /* FF rounded up to a multiple of 64; act, like each weight, spans less than 2 GiB */
    unsigned char* rise_ok;
    void* workspace;                   /* sisa_prefill_workspace_bytes(B,L,H), 256-byte aligned */
} sisa_prefill_args;

int64_t sisa_prefill_workspace_bytes(int32_t B, int32_t L, int32_t H);
int sisa_prefill(const sisa_prefill_args* a, void* stream);

#ifdef __cplusplus
}
#endif

#endif
