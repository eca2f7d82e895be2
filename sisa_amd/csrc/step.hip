// One generated token through a decoder layer for gfx950: the cached route of a block (norm, projections, cache append,
// attention over the cache, W_O, residual, norm, SwiGLU) for B rows of one new position each, as seven launches; and
// the filling of a layer's cache after a prefill, as one.
//
// Reference: the block and its cached attention (src/sisa/modeling.py:171-199, 224-238, 288-291) at L = 1, computed
// there by about seventy torch kernels per layer. With B rows the weights are read once and nothing else is large, so
// what such a step costs is launches and memory latency, not arithmetic: 11 ms of host time per token for 2.9 ms of
// kernels in the 152M model, against about 0.06 ms for its bytes; here 0.73 ms of host time for 0.48 ms of kernels. Rounding points are those of the modules: every
// projection is an fp32 sum rounded once to the weights' dtype (biases added before it), the norm's rows, the
// residual sums and the activation are rounded once, the forget logits stay fp32, the gates and the rotation are fp32.
//
// Skinny products y = W x (B <= 64 rows of x as the columns of 16x16x32 MFMA blocks, 16 rows of W as the rows): a
// workgroup owns 16 rows of W and splits K over its waves, 32 elements a step, wave w taking steps w, w + NWV, ...;
// each lane reads 16 consecutive bytes of one row of W per step, up to eight steps ahead, straight into the operand
// registers (W is used once: LDS would only add a trip); the waves' partial blocks are added in wave order in LDS.
// That gives (rows / 16) workgroups, 206 for the projections of a 768-wide layer. The norm in front of a product is
// recomputed by every workgroup (B short rows, served by L2) while its first weights are on their way: one launch and
// one dependent round trip less than a norm of its own.
#include "common.h"
#include "host.h"
#include "sisa_hip_step.h"

namespace sisa {
namespace detail {
__attribute__((visibility("hidden"))) int decode_attn_out16(const sisa_decode_args* a, void* out, hipStream_t st);   // decode.hip
}
}  // namespace sisa

namespace {

constexpr int DH = 64, DS = 32;
constexpr int AHEAD = 8;               // weight fragments in flight per wave
constexpr int NORM_NWV = 8;            // waves of the products behind a norm and of W_O
constexpr int DOWN_NWV = 16;           // waves of the down projection (K = d_ff)
constexpr int ROW_PAD = 8;             // padding of the staged rows: 16 rows of a fragment read fall on distinct banks

template <class T> SISA_DEV float rnd(float x) { return (float)cvt<T>(x); }

// 8 consecutive elements at any 2-byte alignment (global memory takes unaligned vector loads on this chip)
template <class T> struct __attribute__((packed, aligned(2))) Unaligned8 { frag8<T> v; };

// Fragment of W: row `row`, elements k .. k + 7, zero past K or for row < 0.
template <class T, bool ALIGNED>
SISA_DEV frag8<T> weight_frag(const T* w, int64_t row, int64_t ld, int k, int K) {
    if (row < 0 || k >= K) return zero8<T>();
    const T* p = w + row * ld + k;
    if (ALIGNED || k + 8 <= K)
        return ALIGNED ? load8<T>(p) : reinterpret_cast<const Unaligned8<T>*>(p)->v;
    frag8<T> r = zero8<T>();
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if (k + j < K) r[j] = p[j];
    return r;
}

// The partial blocks of the waves added in wave order; afterwards wave j < JB holds column group j's block.
template <int NWV, int JB>
SISA_DEV f32x4 combine_waves(f32x4* red, const f32x4 (&acc)[JB], int w, int lane) {
#pragma unroll
    for (int j = 0; j < JB; ++j) red[(w * JB + j) * 64 + lane] = acc[j];
    __syncthreads();
    f32x4 s = zero4();
    if (w < JB) {
        s = red[w * 64 + lane];
        for (int k = 1; k < NWV; ++k) s += red[(k * JB + w) * 64 + lane];
    }
    return s;
}

// ------------------------------------------------------------------------------------------------ norm in front
struct NormRows {
    const void* x;                     // (B, D), row stride sx
    int64_t sx;
    const void* res;                   // (B, D) contiguous to add first, or null
    const void* weight;                // (D)
    void* sum;                         // (B, D) contiguous: x + res, written by workgroup 0 (null: not wanted)
    float eps;
    int B, D;
};

// Rows of RMSNorm(x + res) * weight in LDS, (16 JB) x (D + ROW_PAD), rows past B zero.
template <class T, int NWV, int JB>
SISA_DEV void stage_norm(const NormRows& a, T* n, int w, int lane) {
    const int ld = a.D + ROW_PAD, nv = a.D / 8;
    for (int m = w; m < 16 * JB; m += NWV) {
        T* row = n + m * ld;
        if (m >= a.B) {
            for (int c = lane; c < nv; c += 64) *reinterpret_cast<frag8<T>*>(row + 8 * c) = zero8<T>();
            continue;
        }
        float ss = 0.f;
        for (int c = lane; c < nv; c += 64) {
            f32x8 v = load_f32x8<T>((const T*)a.x + m * a.sx + 8 * c);
            if (a.res) {
                const f32x8 r = load_f32x8<T>((const T*)a.res + (int64_t)m * a.D + 8 * c);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = rnd<T>(v[e] + r[e]);
            }
            store_f32x8<T>(row + 8 * c, v);
            if (a.sum && blockIdx.x == 0) store_f32x8<T>((T*)a.sum + (int64_t)m * a.D + 8 * c, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
        const float rstd = 1.f / sqrtf(ss / (float)a.D + a.eps);
        for (int c = lane; c < nv; c += 64) {      // the lane's own chunks again
            const f32x8 v = load_f32x8<T>(row + 8 * c), g = load_f32x8<T>((const T*)a.weight + 8 * c);
            f32x8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (v[e] * rstd) * g[e];
            store_f32x8<T>(row + 8 * c, o);
        }
    }
}

// acc[s] += W_s[rows] . n over the wave's steps, for NS weights of K = D (row < 0: no such row)
template <class T, int NWV, int JB, int NS>
SISA_DEV void norm_product(const NormRows& a, T* n, const T* const (&wt)[NS], int64_t row, int w, int lane,
                           f32x4 (&acc)[NS][JB]) {
    const int grp = lane >> 4, lc = lane & 15, D = a.D, steps = D / 32;
    constexpr int LOOK = AHEAD / NS;
    frag8<T> wf[NS][LOOK];
    auto fetch = [&](int s0) {
#pragma unroll
        for (int i = 0; i < LOOK; ++i)
#pragma unroll
            for (int s = 0; s < NS; ++s)
                wf[s][i] = weight_frag<T, true>(wt[s], row, D, 32 * (s0 + NWV * i) + 8 * grp, D);
    };
    fetch(w);
    stage_norm<T, NWV, JB>(a, n, w, lane);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int j = 0; j < JB; ++j) acc[s][j] = zero4();
    for (int s0 = w; s0 < steps; s0 += NWV * LOOK) {
        if (s0 != w) fetch(s0);
#pragma unroll
        for (int i = 0; i < LOOK; ++i) {
            const int st = s0 + NWV * i;
            if (st < steps) {
#pragma unroll
                for (int j = 0; j < JB; ++j) {
                    const frag8<T> xf = load8<T>(n + (16 * j + lc) * (D + ROW_PAD) + 32 * st + 8 * grp);
#pragma unroll
                    for (int s = 0; s < NS; ++s) acc[s][j] = mma(wf[s][i], xf, acc[s][j]);
                }
            }
        }
    }
    __syncthreads();                   // every wave is done with the rows: their LDS becomes the waves' partials
}

// ------------------------------------------------------------------------------------------------ projections
// The weights of the projections in the order q, k, v, b, c, theta (rows of a multiple of 16, written side by side in
// that order), alpha and forget (H rows each).
struct ProjArgs {
    NormRows nr;
    const void* w[8];
    const void* bias[2];               // of alpha and forget
    void* out;                         // (B, 272 H) q | k | v | b | c | theta
    float* alpha;                      // (B, H): rounded to T as the module's output
    float* z;                          // (B, H) fp32
    int H;
};

template <class T, int JB>
__global__ __launch_bounds__(64 * NORM_NWV) void step_proj_kernel(ProjArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, grp = lane >> 4, lc = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int H = a.H, main = 17 * H;  // 16-row groups of the six wide weights: 272 H rows
    const int g = blockIdx.x;
    int seg, r0;                       // weight and first row of the group
    if (g < main) {
        const int h4 = 4 * H;
        if (g < 3 * h4) seg = g / h4, r0 = 16 * (g % h4);
        else if (g < 16 * H) seg = 3 + (g - 3 * h4) / (2 * H), r0 = 16 * ((g - 3 * h4) % (2 * H));
        else seg = 5, r0 = 16 * (g - 16 * H);
    } else {
        const int gh = (H + 15) / 16;
        seg = 6 + (g - main) / gh, r0 = 16 * ((g - main) % gh);
    }
    const int rows = seg < 6 ? 1 << 30 : H;
    const T* const wt[1] = {(const T*)a.w[seg]};
    f32x4 acc[1][JB];
    norm_product<T, NORM_NWV, JB, 1>(a.nr, (T*)lds, wt, r0 + lc < rows ? r0 + lc : -1, w, lane, acc);
    const f32x4 s = combine_waves<NORM_NWV, JB>((f32x4*)lds, acc[0], w, lane);
    const int m = 16 * w + lc;         // lane: outputs 4 grp .. + 3 of the group for row m
    if (w >= JB || m >= a.nr.B) return;
    if (seg < 6) {
        store4<T>((T*)a.out + (int64_t)m * 272 * H + 16 * g + 4 * grp, to_vec4<T>(s));
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int h = r0 + 4 * grp + i;
        if (h >= H) continue;
        const float v = s[i] + (float)((const T*)a.bias[seg - 6])[h];
        if (seg == 6) a.alpha[m * H + h] = rnd<T>(v);
        else a.z[m * H + h] = v;
    }
}

// ------------------------------------------------------------------------------------------------ cache append
struct AppendArgs {
    const void* proj;                  // (B, 272 H)
    const float *alpha, *z;            // (B, H)
    const float *phi_in, *lambda_raw;  // (B, H, 16), (H)
    sisa_view k, v, b, g, f;           // cache slabs (B, H, capacity, .)
    float *phi_out, *gq, *fq, *lam;    // (B, H, 16), (B, H), (B, H), (H)
    void* c;                           // (B, H, 32) rotated c
    int H, pos;
};

// One wave per (batch row, head): the recurrences advanced by the new position, c and b rotated by the new phase, the
// position's k, v, b~, g and F written to the cache.
template <class T>
__global__ __launch_bounds__(64) void step_append_kernel(AppendArgs a) {
    const int lane = threadIdx.x, H = a.H, bh = blockIdx.x, b = bh / H, h = bh % H;
    const T* P = (const T*)a.proj + (int64_t)b * 272 * H;
    const int64_t pos = a.pos;
    ((T*)a.k.ptr)[b * a.k.sb + h * a.k.sh + pos * a.k.sl + lane] = P[(H + h) * DH + lane];
    ((T*)a.v.ptr)[b * a.v.sb + h * a.v.sh + pos * a.v.sl + lane] = P[(2 * H + h) * DH + lane];
    if (lane < DS / 2) {
        const int64_t p = (int64_t)bh * (DS / 2) + lane;
        const float phi = a.phi_in[p] + (float)P[256 * H + h * (DS / 2) + lane];
        a.phi_out[p] = phi;
        const float cs = cosf(phi), sn = sinf(phi);
        const T* bp = P + 192 * H + h * DS + 2 * lane;
        const T* cp = P + 224 * H + h * DS + 2 * lane;
        const float b0 = (float)bp[0], b1 = (float)bp[1], c0 = (float)cp[0], c1 = (float)cp[1];
        T* bo = (T*)a.b.ptr + b * a.b.sb + h * a.b.sh + pos * a.b.sl + 2 * lane;
        T* co = (T*)a.c + (int64_t)bh * DS + 2 * lane;
        bo[0] = cvt<T>(b0 * cs - b1 * sn);
        bo[1] = cvt<T>(b1 * cs + b0 * sn);
        co[0] = cvt<T>(c0 * cs - c1 * sn);
        co[1] = cvt<T>(c1 * cs + c0 * sn);
    } else if (lane == 32) {           // g = g_prev - softplus(alpha), as torch's softplus (threshold 20)
        float* g = (float*)a.g.ptr + b * a.g.sb + h * a.g.sh + pos * a.g.sl;
        const float al = a.alpha[bh];
        const float v = g[-a.g.sl] - (al > 20.f ? al : log1pf(expf(al)));
        g[0] = v;
        a.gq[bh] = v;
    } else if (lane == 33) {           // F = F_prev + logsigmoid(z)
        float* f = (float*)a.f.ptr + b * a.f.sb + h * a.f.sh + pos * a.f.sl;
        const float z = a.z[bh];
        const float v = f[-a.f.sl] + ((z < 0.f ? z : (z != z ? z : 0.f)) - log1pf(expf(-fabsf(z))));
        f[0] = v;
        a.fq[bh] = v;
    } else if (lane == 34 && b == 0) {
        const float r = a.lambda_raw[h];
        a.lam[h] = r > 20.f ? r : log1pf(expf(r));
    }
}

// ------------------------------------------------------------------------------------------------ W_O, down
// y = x W^T for W (rows, K), row stride K; OUT = add + y when `add` is given (both rounded to T in turn).
struct LinArgs {
    const void *x, *w, *add;           // x (B, ldx) zero past K, up to a multiple of 32; add (B, rows) contiguous
    void* out;                         // (B, rows) contiguous
    int64_t ldx;
    int B, K, rows;
};

template <class T, int NWV, int JB, bool ALIGNED>
__global__ __launch_bounds__(64 * NWV) void step_linear_kernel(LinArgs a) {
    __shared__ f32x4 red[NWV * JB * 64];
    const int lane = threadIdx.x & 63, grp = lane >> 4, lc = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = 16 * blockIdx.x, K = a.K, steps = (K + 31) / 32;
    constexpr int LOOK = JB == 1 ? AHEAD : AHEAD / JB;
    f32x4 acc[JB];
#pragma unroll
    for (int j = 0; j < JB; ++j) acc[j] = zero4();
    for (int s0 = w; s0 < steps; s0 += NWV * LOOK) {
        frag8<T> wf[LOOK], xf[LOOK][JB];
#pragma unroll
        for (int i = 0; i < LOOK; ++i) {
            const int k = 32 * (s0 + NWV * i) + 8 * grp;
            wf[i] = weight_frag<T, ALIGNED>((const T*)a.w, r0 + lc < a.rows ? r0 + lc : -1, K, k, K);
#pragma unroll
            for (int j = 0; j < JB; ++j)
                xf[i][j] = (16 * j + lc < a.B && s0 + NWV * i < steps)
                               ? load8<T>((const T*)a.x + (16 * j + lc) * a.ldx + k) : zero8<T>();
        }
#pragma unroll
        for (int i = 0; i < LOOK; ++i)
#pragma unroll
            for (int j = 0; j < JB; ++j) acc[j] = mma(wf[i], xf[i][j], acc[j]);
    }
    const f32x4 s = combine_waves<NWV, JB>(red, acc, w, lane);
    const int m = 16 * w + lc, r = r0 + 4 * grp;
    if (w >= JB || m >= a.B || r >= a.rows) return;
    vec4<T> y = to_vec4<T>(s);         // rows is a multiple of 4
    if (a.add) {
        const vec4<T> x = load4<T>((const T*)a.add + (int64_t)m * a.rows + r);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = cvt<T>((float)x[i] + (float)y[i]);
    }
    store4<T>((T*)a.out + (int64_t)m * a.rows + r, y);
}

// ------------------------------------------------------------------------------------------------ gate, up, SwiGLU
struct GateArgs {
    NormRows nr;
    const void *w_gate, *w_up;         // (FF, D)
    void* act;                         // (B, FP): silu(gate) * up, zero for columns FF .. FP - 1
    int FF, FP;                        // FP: FF rounded up to a multiple of 32
};

template <class T, int JB>
__global__ __launch_bounds__(64 * NORM_NWV) void step_gate_kernel(GateArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int lane = threadIdx.x & 63, grp = lane >> 4, lc = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = 16 * blockIdx.x;
    const T* const wt[2] = {(const T*)a.w_gate, (const T*)a.w_up};
    f32x4 acc[2][JB];
    norm_product<T, NORM_NWV, JB, 2>(a.nr, (T*)lds, wt, r0 + lc < a.FF ? r0 + lc : -1, w, lane, acc);
    const f32x4 gate = combine_waves<NORM_NWV, JB>((f32x4*)lds, acc[0], w, lane);
    const f32x4 up = combine_waves<NORM_NWV, JB>((f32x4*)lds + NORM_NWV * JB * 64, acc[1], w, lane);
    const int m = 16 * w + lc;
    if (w >= JB || m >= a.nr.B) return;
    vec4<T> h;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = rnd<T>(gate[i]), y = rnd<T>(up[i]);
        h[i] = cvt<T>((x * (1.f / (1.f + expf(-x)))) * y);
    }
    store4<T>((T*)a.act + (int64_t)m * a.FP + r0 + 4 * grp, h);
}

// ------------------------------------------------------------------------------------------------ workspace, launches
struct Ws {
    char *proj, *act, *c, *y, *h0;
    float *alpha, *z, *gq, *fq, *lam, *attn;
    int64_t bytes;
};

int64_t pad256(int64_t b) { return (b + 255) / 256 * 256; }

Ws workspace(char* base, int64_t B, int64_t H, int64_t D, int64_t FF, int64_t N) {
    Ws w{};
    int64_t at = 0;
    auto take = [&](int64_t bytes) {
        char* p = base + at;
        at += pad256(bytes);
        return p;
    };
    w.proj = take(B * 272 * H * 2);
    w.act = take(B * ((FF + 31) / 32 * 32) * 2);
    w.c = take(B * H * DS * 2);
    w.y = take(B * H * DH * 2);
    w.h0 = take(B * D * 2);
    w.alpha = (float*)take(B * H * 4);
    w.z = (float*)take(B * H * 4);
    w.gq = (float*)take(B * H * 4);
    w.fq = (float*)take(B * H * 4);
    w.lam = (float*)take(H * 4);
    w.attn = (float*)take(sisa_decode_workspace_bytes((int32_t)B, (int32_t)H, 1, (int32_t)N));
    w.bytes = at;
    return w;
}

// Dynamic LDS of a product behind a norm: the staged rows, later NS sets of the waves' partial blocks.
int64_t norm_lds(int JB, int D, int NS) {
    const int64_t rows = (int64_t)16 * JB * (D + ROW_PAD) * 2, part = (int64_t)NS * NORM_NWV * JB * 64 * 16;
    return rows > part ? rows : part;
}

template <class T, int JB>
int launch_step(const sisa_step_args* a, hipStream_t st) {
    const int B = a->B, H = a->H, D = a->D, FF = a->FF, FP = (FF + 31) / 32 * 32;
    const Ws ws = workspace((char*)a->workspace, B, H, D, FF, a->pos + 1);
    ProjArgs p{};
    p.nr = NormRows{a->x, a->sx, a->res, a->attn_norm, ws.h0, a->eps_attn, B, D};
    const void* w[8] = {a->w_q, a->w_k, a->w_v, a->w_b, a->w_c, a->w_theta, a->w_alpha, a->w_forget};
    for (int i = 0; i < 8; ++i) p.w[i] = w[i];
    p.bias[0] = a->b_alpha;
    p.bias[1] = a->b_forget;
    p.out = ws.proj;
    p.alpha = ws.alpha;
    p.z = ws.z;
    p.H = H;
    const unsigned groups = (unsigned)(17 * H + 2 * ((H + 15) / 16));
    step_proj_kernel<T, JB><<<groups, 64 * NORM_NWV, norm_lds(JB, D, 1), st>>>(p);
    int rc = sisa::launch_status("sisa_step (projections)");
    if (rc) return rc;
    step_append_kernel<T><<<(unsigned)(B * H), 64, 0, st>>>(AppendArgs{ws.proj, ws.alpha, ws.z, a->phi_in, a->lambda_raw,
                                                                       a->k, a->v, a->b, a->g, a->f, a->phi_out, ws.gq,
                                                                       ws.fq, ws.lam, ws.c, H, a->pos});
    rc = sisa::launch_status("sisa_step (append)");
    if (rc) return rc;
    sisa_decode_args d{};
    d.B = B;
    d.H = H;
    d.M = 1;
    d.N = a->pos + 1;
    d.dtype = a->dtype;
    d.q_start = a->pos;
    d.q = sisa_view{ws.proj, (int64_t)272 * H, DH, DH};
    d.c = sisa_view{ws.c, (int64_t)H * DS, DS, DS};
    d.gq = sisa_view{ws.gq, H, 1, 1};
    d.fq = sisa_view{ws.fq, H, 1, 1};
    d.k = a->k;
    d.v = a->v;
    d.b = a->b;
    d.gk = a->g;
    d.fk = a->f;
    d.lam = ws.lam;
    d.s_lam = 1;
    d.workspace = ws.attn;
    rc = sisa::detail::decode_attn_out16(&d, ws.y, st);
    if (rc) return rc;
    // h = (x + res) + W_O y, then the FFN of its norm
    step_linear_kernel<T, NORM_NWV, JB, true><<<(unsigned)(D / 16), 64 * NORM_NWV, 0, st>>>(
        LinArgs{ws.y, a->w_o, ws.h0, a->h, (int64_t)H * DH, B, H * DH, D});
    rc = sisa::launch_status("sisa_step (W_O)");
    if (rc) return rc;
    GateArgs g{};
    g.nr = NormRows{a->h, D, nullptr, a->ffn_norm, nullptr, a->eps_ffn, B, D};
    g.w_gate = a->w_gate;
    g.w_up = a->w_up;
    g.act = ws.act;
    g.FF = FF;
    g.FP = FP;
    step_gate_kernel<T, JB><<<(unsigned)(FP / 16), 64 * NORM_NWV, norm_lds(JB, D, 2), st>>>(g);
    rc = sisa::launch_status("sisa_step (gate, up)");
    if (rc) return rc;
    const LinArgs dn{ws.act, a->w_down, nullptr, a->ffn, FP, B, FF, D};
    if (FF % 8 == 0) step_linear_kernel<T, DOWN_NWV, JB, true><<<(unsigned)(D / 16), 64 * DOWN_NWV, 0, st>>>(dn);
    else step_linear_kernel<T, DOWN_NWV, JB, false><<<(unsigned)(D / 16), 64 * DOWN_NWV, 0, st>>>(dn);
    return sisa::launch_status("sisa_step (down)");
}

template <class T>
int launch_step_rows(const sisa_step_args* a, hipStream_t st) {
    if (a->B <= 16) return launch_step<T, 1>(a, st);
    if (a->B <= 32) return launch_step<T, 2>(a, st);
    return launch_step<T, 4>(a, st);
}

// ------------------------------------------------------------------------------------------------ cache fill
// 32 threads per (batch row, position, head): 16-byte pieces of k (8), v (8) and b~ (4) and the two gates; the head's
// last phase, the sum of the chunk totals in order, by the threads of the last position.
template <class T>
__global__ __launch_bounds__(256) void cache_fill_kernel(sisa_cache_fill_args a) {
    const int64_t id = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 5);
    const int t = threadIdx.x & 31;
    if (id >= (int64_t)a.B * a.L * a.H) return;
    const int h = (int)(id % a.H);
    const int64_t l = (id / a.H) % a.L, b = id / a.H / a.L;
    if (t < 16) {
        const T* src = (const T*)a.proj + b * a.s_b + l * a.s_l + (t < 8 ? a.col_k : a.col_v) + h * DH + 8 * (t & 7);
        const sisa_view& d = t < 8 ? a.k : a.v;
        *reinterpret_cast<frag8<T>*>((T*)d.ptr + b * d.sb + h * d.sh + l * d.sl + 8 * (t & 7)) = load8<T>(src);
    } else if (t < 20) {
        const T* src = (const T*)a.br + ((b * a.L + l) * a.H + h) * DS + 8 * (t - 16);
        *reinterpret_cast<frag8<T>*>((T*)a.b.ptr + b * a.b.sb + h * a.b.sh + l * a.b.sl + 8 * (t - 16)) = load8<T>(src);
    } else if (t < 22) {
        const sisa_view& d = t == 20 ? a.g : a.f;
        ((float*)d.ptr)[b * d.sb + h * d.sh + l * d.sl] = (t == 20 ? a.gs : a.fs)[(b * a.H + h) * a.L + l];
    }
    if (l == a.L - 1 && t < DS / 2) {
        const int64_t bh = b * a.H + h, nc = (a.L + 63) / 64;
        float s = 0.f;
        for (int64_t c = 0; c < nc; ++c) s += a.totals[(bh * nc + c) * (2 + DS / 2) + 2 + t];
        a.phi[bh * (DS / 2) + t] = s;
    }
}

bool slab_ok(const sisa_view& v, int dtype) { return sisa::view_ok(v, dtype); }

}  // namespace

extern "C" int64_t sisa_step_workspace_bytes(int32_t B, int32_t H, int32_t D, int32_t FF, int32_t N) {
    if (B < 1 || H < 1 || D < 1 || FF < 1 || N < 1) return 0;
    return workspace(nullptr, B, H, D, FF, N).bytes;
}

extern "C" int sisa_step(const sisa_step_args* a, void* stream) {
    SISA_REQUIRE(a != nullptr, "sisa_step: null args");
    SISA_REQUIRE(a->B >= 1 && a->B <= SISA_STEP_MAX_ROWS && a->H >= 1 && a->D == DH * a->H && a->D <= SISA_STEP_MAX_D &&
                     a->FF >= 1,
                 "sisa_step: B=%d (1..%d), H=%d, D=%d (64 H, at most %d), FF=%d", a->B, SISA_STEP_MAX_ROWS, a->H, a->D,
                 SISA_STEP_MAX_D, a->FF);
    SISA_REQUIRE(a->pos >= 1, "sisa_step: position %d (the cache must hold a previous one)", a->pos);
    SISA_REQUIRE(a->dtype == SISA_BF16 || a->dtype == SISA_F16, "sisa_step: dtype %d (bf16 or fp16)", a->dtype);
    const void* given[] = {a->x, a->attn_norm, a->w_q, a->w_k, a->w_v, a->w_b, a->w_c, a->w_theta, a->w_alpha, a->w_forget,
                           a->w_o, a->ffn_norm, a->w_gate, a->w_up, a->h, a->ffn};
    for (const void* p : given)
        SISA_REQUIRE(p && sisa::aligned16(p), "sisa_step: tensors must be given and 16-byte aligned");
    SISA_REQUIRE(a->w_down && (a->FF % 8 != 0 || sisa::aligned16(a->w_down)), "sisa_step: w_down not aligned");
    SISA_REQUIRE((a->res == nullptr || sisa::aligned16(a->res)) && a->sx >= a->D && a->sx % 8 == 0,
                 "sisa_step: x rows and res must be 16-byte aligned");
    SISA_REQUIRE(a->b_alpha && a->b_forget && a->lambda_raw && a->phi_in && a->phi_out && a->g.ptr && a->f.ptr &&
                     a->workspace && ((uintptr_t)a->workspace & 255) == 0,
                 "sisa_step: null pointer, or workspace not 256-byte aligned");
    SISA_REQUIRE(slab_ok(a->k, a->dtype) && slab_ok(a->v, a->dtype) && slab_ok(a->b, a->dtype),
                 "sisa_step: cache rows must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    return a->dtype == SISA_BF16 ? launch_step_rows<__bf16>(a, st) : launch_step_rows<_Float16>(a, st);
}

extern "C" int sisa_cache_fill(const sisa_cache_fill_args* a, void* stream) {
    SISA_REQUIRE(a != nullptr, "sisa_cache_fill: null args");
    SISA_REQUIRE(a->B >= 1 && a->H >= 1 && a->L >= 1, "sisa_cache_fill: bad shape B=%d H=%d L=%d", a->B, a->H, a->L);
    SISA_REQUIRE(a->dtype == SISA_BF16 || a->dtype == SISA_F16, "sisa_cache_fill: dtype %d (bf16 or fp16)", a->dtype);
    SISA_REQUIRE(a->proj && sisa::aligned16(a->proj) && a->s_b % 8 == 0 && a->s_l % 8 == 0 && a->col_k % 8 == 0 &&
                     a->col_v % 8 == 0 && a->br && sisa::aligned16(a->br) && a->gs && a->fs && a->totals && a->phi &&
                     a->g.ptr && a->f.ptr,
                 "sisa_cache_fill: null or unaligned pointer");
    SISA_REQUIRE(slab_ok(a->k, a->dtype) && slab_ok(a->v, a->dtype) && slab_ok(a->b, a->dtype),
                 "sisa_cache_fill: cache rows must be 16-byte aligned");
    const int64_t rows = (int64_t)a->B * a->L * a->H;
    SISA_REQUIRE(rows < ((int64_t)1 << 33), "sisa_cache_fill: B*L*H too large for one launch");
    const unsigned grid = (unsigned)sisa::cdiv(rows, 8);
    hipStream_t st = (hipStream_t)stream;
    if (a->dtype == SISA_BF16) cache_fill_kernel<__bf16><<<grid, 256, 0, st>>>(*a);
    else cache_fill_kernel<_Float16><<<grid, 256, 0, st>>>(*a);
    return sisa::launch_status("sisa_cache_fill");
}
