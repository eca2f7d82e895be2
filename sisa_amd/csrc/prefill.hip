// A prompt through a decoder layer for gfx950, filling the layer's cache: every kernel of the layer behind one call, for
// prompts so short that launching them one by one from the host costs more than running them.
//
// Reference: the block on a prompt with an empty cache (src/sisa/modeling.py:171-199, 224-238, 288-291). The same layer
// through torch and this library's separate entry points is about 24 launches and 430 us of host time (four of them
// library GEMMs at 27 us of host time each) for 110 us of kernels at 800 rows of 768; here it is 13 launches and 165 us
// in all (twelve layers, 800 tokens: 5.1 -> 2.0 ms; 8,192 tokens: 5.5 -> 4.6).
// Rounding points are those of the modules (see step.hip).
//
// The products y = x W^T (both operands contiguous along K) run on rows_gemm_kernel: 128 rows x 128 outputs a workgroup,
// 2 x 2 waves of 4 x 4 MFMA blocks, K in 64-wide stages staged by buffer loads straight into LDS, double-buffered. 128
// wide rather than the 256 of the linear CE's kernels: at 800 rows the projections are 189 tiles of this size, 52 of
// that. Several weights side by side are one launch (the projections without a concatenated weight), and gate and up
// are staged together so that a lane holds both of an output and writes the activation.
#include "common.h"
#include "host.h"
#include "sisa_hip_step.h"

namespace {

constexpr int DH = 64, DS = 32;
constexpr int TM = 128, TN = 128, TK = 64;   // rows, outputs and K per stage of a workgroup
constexpr int GW = 4;                        // waves: 2 along the outputs x 2 along the rows
constexpr int PER = TM * TK / 8 / 64 / GW;   // wave instructions per wave, operand and stage

template <class T> SISA_DEV float rnd(float x) { return (float)cvt<T>(x); }

struct Seg {
    const void *w, *bias;                    // (rows, K) contiguous; (rows) or null
    int rows, tile0, col;                    // outputs, first tile, first output column
};
struct GemmArgs {
    const void* x;                           // (M, ldx), zero or absent past K
    void* out;                               // (M, ldo)
    int64_t ldx, ldo;
    int M, K, ntile, nseg;                   // K a multiple of 8; ntile: tiles along the outputs
    Seg seg[7];                              // GLU: gate and up, seg[0].rows outputs, columns up to ldo written
};

template <class T>
struct __attribute__((aligned(16))) GemmLds {
    T x[2][TM * TK];
    T w[2][TN * TK];
};

template <class T, bool GLU>
__global__ __launch_bounds__(64 * GW) void rows_gemm_kernel(GemmArgs a) {
    __shared__ GemmLds<T> sm;
    const int lane = threadIdx.x & 63, grp = lane >> 4, lc = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tile = blockIdx.x % a.ntile, m0 = (int)(blockIdx.x / a.ntile) * TM;
    const int K = a.K, stages = (K + TK - 1) / TK;
    int s = 0;
    if constexpr (!GLU)
        while (s + 1 < a.nseg && tile >= a.seg[s + 1].tile0) ++s;
    const Seg sg = a.seg[s];
    const int r0 = GLU ? tile * (TN / 2) : (tile - sg.tile0) * TN;
    const int wo = w & 1, wm = w >> 1;

    // staging: wave instruction k of an operand fills rows 8 k .. 8 k + 7 (GLU: gate rows in 0 .. 63, up rows in 64 .. 127);
    // rows past the data and elements past K read as zero through the buffers' range
    int row[PER], col[PER];
#pragma unroll
    for (int p = 0; p < PER; ++p) {
        const int ci = 64 * (w + GW * p) + lane;
        row[p] = ci / 8;
        col[p] = 8 * ((ci % 8) ^ swz<T, TK>(row[p]));
    }
    const int64_t xbytes = ((int64_t)(a.M - 1) * a.ldx + K) * 2, wbytes = (int64_t)sg.rows * K * 2;
    const __amdgpu_buffer_rsrc_t xr = make_rsrc(a.x, xbytes), wr = make_rsrc(sg.w, wbytes);
    const __amdgpu_buffer_rsrc_t ur = make_rsrc(GLU ? a.seg[1].w : sg.w, wbytes);
    auto issue = [&](int g, int buf) {
        const int k0 = g * TK;
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            const bool ok = k0 + col[p] < K;
            const int xo = ok ? (int)(((m0 + row[p]) * a.ldx + k0 + col[p]) * 2) : 0x7ffffff0;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                xr, (__attribute__((address_space(3))) void*)(sm.x[buf] + (w + GW * p) * 512), 16, xo, 0, 0, 0);
            const bool up = GLU && 2 * p >= PER;
            const int wrow = r0 + (up ? row[p] - TN / 2 : row[p]);
            const int woff = ok ? (int)(((int64_t)wrow * K + k0 + col[p]) * 2) : 0x7ffffff0;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                up ? ur : wr, (__attribute__((address_space(3))) void*)(sm.w[buf] + (w + GW * p) * 512), 16, woff, 0, 0, 0);
        }
    };

    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = zero4();
    issue(0, 0);
    __syncthreads();
    for (int g = 0; g < stages; ++g) {
        const int buf = g & 1;
        if (g + 1 < stages) issue(g + 1, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int st = 0; st < TK / 32; ++st) {
            frag8<T> xf[4], wf[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) xf[j] = frag_rows<T, TK>(sm.x[buf], 64 * wm + 16 * j, st, lane);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int o = GLU ? 64 * (i >> 1) + 32 * wo + 16 * (i & 1) : 64 * wo + 16 * i;
                wf[i] = frag_rows<T, TK>(sm.w[buf], o, st, lane);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = mma(wf[i], xf[j], acc[i][j]);
        }
        __syncthreads();
    }
    // lane: outputs 4 grp .. + 3 of block i for row 16 j + lc
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = m0 + 64 * wm + 16 * j + lc;
        if (n >= a.M) continue;
        T* orow = (T*)a.out + (int64_t)n * a.ldo;
        if constexpr (GLU) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int o = r0 + 32 * wo + 16 * i + 4 * grp;     // columns past FF: products with zero rows, 0
                if (o >= a.ldo) continue;
                vec4<T> h;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float x = rnd<T>(acc[i][j][r]), y = rnd<T>(acc[i + 2][j][r]);
                    h[r] = cvt<T>((x * (1.f / (1.f + expf(-x)))) * y);
                }
                store4<T>(orow + o, h);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int o = r0 + 64 * wo + 16 * i + 4 * grp;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (sg.bias && o + r < sg.rows) acc[i][j][r] += (float)((const T*)sg.bias)[o + r];
                if (o + 3 < sg.rows) {
                    store4<T>(orow + sg.col + o, to_vec4<T>(acc[i][j]));
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (o + r < sg.rows) orow[sg.col + o + r] = cvt<T>(acc[i][j][r]);
                }
            }
        }
    }
}

// The fp32 copies of the small parameters that the norm and attention kernels read: both norm gains, W_f, b_f, and
// lam = softplus(lambda_raw).
struct SmallArgs {
    const void *g1, *g2, *wf, *bf;
    const float* lambda_raw;
    float *g1f, *g2f, *wff, *bff, *lam;
    int D, H;
};
template <class T>
__global__ __launch_bounds__(256) void small_params_kernel(SmallArgs a) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < a.D) {
        a.g1f[i] = (float)((const T*)a.g1)[i];
        a.g2f[i] = (float)((const T*)a.g2)[i];
    }
    if (i < a.H) {
        a.bff[i] = (float)((const T*)a.bf)[i];
        const float r = a.lambda_raw[i];
        a.lam[i] = r > 20.f ? r : log1pf(expf(r));
    }
    if (i < a.H * a.D) a.wff[i] = (float)((const T*)a.wf)[i];
}

// *ok = every rise of g within the tolerance (false for NaN)
__global__ __launch_bounds__(256) void rise_ok_kernel(const float* rise, int n, float tol, unsigned char* ok) {
    __shared__ int bad;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    bool b = false;
    for (int i = threadIdx.x; i < n; i += 256) b |= !(rise[i] <= tol);
    if (b) bad = 1;
    __syncthreads();
    if (threadIdx.x == 0) *ok = bad ? 0 : 1;
}

struct Ws {
    char *n, *proj, *cr, *br, *y, *a, *m, *h0;
    float *z, *g, *f, *rowf, *colf, *rowf2, *colf2, *rise, *tot, *lse, *g1, *g2, *wf, *bf, *lam;
    int64_t bytes;
};

int npad(int H) { return (273 * H + 15) / 16 * 16; }

Ws workspace(char* base, int64_t B, int64_t L, int64_t H) {
    Ws w{};
    int64_t at = 0;
    auto take = [&](int64_t bytes) {
        char* p = base + at;
        at += (bytes + 255) / 256 * 256;
        return p;
    };
    const int64_t N = B * L, D = DH * H, BHL = N * H, nc = (L + 63) / 64;
    w.n = take(N * D * 2);
    w.proj = take(N * npad((int)H) * 2);
    w.cr = take(BHL * DS * 2);
    w.br = take(BHL * DS * 2);
    w.y = take(N * D * 2);
    w.a = take(N * D * 2);
    w.m = take(N * D * 2);
    w.h0 = take(N * D * 2);
    w.z = (float*)take(BHL * 4);
    w.g = (float*)take(BHL * 4);
    w.f = (float*)take(BHL * 4);
    w.rowf = (float*)take(BHL * 4);
    w.colf = (float*)take(BHL * 4);
    w.rowf2 = (float*)take(BHL * 4);
    w.colf2 = (float*)take(BHL * 4);
    w.lse = (float*)take(BHL * 4);
    w.rise = (float*)take(B * H * nc * 4);
    w.tot = (float*)take(B * H * nc * 18 * 4);
    w.g1 = (float*)take(D * 4);
    w.g2 = (float*)take(D * 4);
    w.wf = (float*)take(H * D * 4);
    w.bf = (float*)take(H * 4);
    w.lam = (float*)take(H * 4);
    w.bytes = at;
    return w;
}

template <class T, bool GLU>
int gemm(GemmArgs g, hipStream_t st, const char* what) {
    int t = 0;
    if (GLU) {
        t = (int)sisa::cdiv(g.ldo, TN / 2);
    } else {
        for (int s = 0; s < g.nseg; ++s) {
            g.seg[s].tile0 = t;
            t += (int)sisa::cdiv(g.seg[s].rows, TN);
        }
    }
    g.ntile = t;
    rows_gemm_kernel<T, GLU><<<(unsigned)(t * sisa::cdiv(g.M, TM)), 64 * GW, 0, st>>>(g);
    return sisa::launch_status(what);
}

#define SISA_TRY(expr)      \
    do {                    \
        const int rc_ = (expr); \
        if (rc_) return rc_;    \
    } while (0)

template <class T>
int run_layer(const sisa_prefill_args* a, hipStream_t st) {
    const int B = a->B, L = a->L, H = a->H, D = DH * H, N = B * L, P = npad(H), FF = a->FF;
    const Ws ws = workspace((char*)a->workspace, B, L, H);
    small_params_kernel<T><<<(unsigned)sisa::cdiv(H * D > D ? H * D : D, 256), 256, 0, st>>>(
        SmallArgs{a->attn_norm, a->ffn_norm, a->w_forget, a->b_forget, a->lambda_raw, ws.g1, ws.g2, ws.wf, ws.bf, ws.lam, D,
                  H});
    SISA_TRY(sisa::launch_status("sisa_prefill (parameters)"));
    sisa_norm_args n{};
    n.N = N;
    n.D = D;
    n.H = H;
    n.xdtype = n.ydtype = a->dtype;
    n.eps = a->eps_attn;
    n.x = a->x;
    n.sx = D;
    n.w = ws.g1;
    n.wf = ws.wf;
    n.bf = ws.bf;
    n.y = ws.n;
    n.sy = D;
    n.z = ws.z;
    const void* h0 = a->x;
    if (a->res) {
        n.res = a->res;
        n.sres = D;
        n.h = ws.h0;
        n.sh = D;
        h0 = ws.h0;
    }
    SISA_TRY(sisa_norm_fwd(&n, st));
    GemmArgs g{};
    g.x = ws.n;
    g.ldx = D;
    g.out = ws.proj;
    g.ldo = P;
    g.M = N;
    g.K = D;
    g.nseg = 7;
    const void* w[7] = {a->w_q, a->w_k, a->w_v, a->w_b, a->w_c, a->w_theta, a->w_alpha};
    const int rows[7] = {D, D, D, DS * H, DS * H, DS / 2 * H, H};
    for (int s = 0, col = 0; s < 7; ++s) {
        g.seg[s] = Seg{w[s], s == 6 ? a->b_alpha : nullptr, rows[s], 0, col};
        col += rows[s];
    }
    SISA_TRY((gemm<T, false>(g, st, "sisa_prefill (projections)")));
    const sisa_prep_fwd_args p{B, L, H, a->dtype, ws.proj, (int64_t)L * P, P, ws.z, (int64_t)L * H, H, ws.cr, ws.br, ws.g,
                               ws.f, ws.rowf, ws.colf, ws.tot};
    SISA_TRY(sisa_prep_fwd(&p, st));
    const int64_t hl = (int64_t)H * L;
    const sisa_view gv{ws.g, hl, L, 1}, fv{ws.f, hl, L, 1};
    if (a->rise_ok && L > 1) {               // the unfused route's check of g
        const sisa_factors_args fa{B, H, L, gv, ws.rowf2, ws.colf2, ws.rise};
        SISA_TRY(sisa_factors(&fa, st));
        rise_ok_kernel<<<1, 256, 0, st>>>(ws.rise, (int)(B * H * sisa::cdiv(L, 64)), a->rise_tol, a->rise_ok);
        SISA_TRY(sisa::launch_status("sisa_prefill (check)"));
    }
    const int es = 2;
    auto heads = [&](char* base, int col) { return sisa_view{base + (int64_t)col * es, (int64_t)L * P, DH, P}; };
    auto state = [&](char* base) { return sisa_view{base, (int64_t)L * H * DS, DS, (int64_t)H * DS}; };
    sisa_attn_fwd_args at{};
    at.B = B;
    at.H = H;
    at.L = L;
    at.dtype = a->dtype;
    at.q = heads(ws.proj, 0);
    at.k = heads(ws.proj, D);
    at.v = heads(ws.proj, 2 * D);
    at.c = state(ws.cr);
    at.b = state(ws.br);
    at.g = gv;
    at.f = fv;
    at.lam = ws.lam;
    at.s_lam = 1;
    at.rowf = ws.rowf;
    at.colf = ws.colf;
    at.o = sisa_view{ws.y, (int64_t)L * D, DH, D};
    at.lse = ws.lse;
    SISA_TRY(sisa_attn_fwd(&at, st));
    const sisa_cache_fill_args cf{B, H, L, a->dtype, ws.proj, (int64_t)L * P, P, D, 2 * D, ws.br, ws.g, ws.f, ws.tot,
                                  a->k, a->v, a->b, a->g, a->f, a->phi};
    SISA_TRY(sisa_cache_fill(&cf, st));
    g = GemmArgs{};
    g.x = ws.y;
    g.ldx = D;
    g.out = ws.a;
    g.ldo = D;
    g.M = N;
    g.K = D;
    g.nseg = 1;
    g.seg[0] = Seg{a->w_o, nullptr, D, 0, 0};
    SISA_TRY((gemm<T, false>(g, st, "sisa_prefill (W_O)")));
    n = sisa_norm_args{};
    n.N = N;
    n.D = D;
    n.xdtype = n.ydtype = a->dtype;
    n.eps = a->eps_ffn;
    n.x = h0;
    n.sx = D;
    n.w = ws.g2;
    n.y = ws.m;
    n.sy = D;
    n.res = ws.a;
    n.sres = D;
    n.h = a->h;
    n.sh = D;
    SISA_TRY(sisa_norm_fwd(&n, st));
    g.x = ws.m;
    g.out = a->act;
    g.ldo = a->act_ld;
    g.seg[0] = Seg{a->w_gate, nullptr, FF, 0, 0};
    g.seg[1] = Seg{a->w_up, nullptr, FF, 0, 0};
    SISA_TRY((gemm<T, true>(g, st, "sisa_prefill (gate, up)")));
    if (!a->ffn) return SISA_OK;
    g.x = a->act;
    g.ldx = a->act_ld;
    g.K = FF;
    g.out = a->ffn;
    g.ldo = D;
    g.seg[0] = Seg{a->w_down, nullptr, D, 0, 0};
    return gemm<T, false>(g, st, "sisa_prefill (down)");
}

}  // namespace

extern "C" int64_t sisa_prefill_workspace_bytes(int32_t B, int32_t L, int32_t H) {
    if (B < 1 || L < 1 || H < 1) return 0;
    return workspace(nullptr, B, L, H).bytes;
}

extern "C" int sisa_prefill(const sisa_prefill_args* a, void* stream) {
    SISA_REQUIRE(a != nullptr, "sisa_prefill: null args");
    SISA_REQUIRE(a->B >= 1 && a->L >= 1 && a->H >= 1 && a->H <= 64 && a->FF >= 1 &&
                     (int64_t)a->B * a->L <= SISA_PREFILL_MAX_ROWS,
                 "sisa_prefill: B=%d L=%d (at most %d rows), H=%d (1..64), FF=%d", a->B, a->L, SISA_PREFILL_MAX_ROWS, a->H,
                 a->FF);
    SISA_REQUIRE(a->dtype == SISA_BF16 || a->dtype == SISA_F16, "sisa_prefill: dtype %d (bf16 or fp16)", a->dtype);
    const void* given[] = {a->x, a->attn_norm, a->w_q, a->w_k, a->w_v, a->w_b, a->w_c, a->w_theta, a->w_alpha, a->w_forget,
                           a->w_o, a->ffn_norm, a->w_gate, a->w_up, a->h, a->act};
    for (const void* p : given)
        SISA_REQUIRE(p && sisa::aligned16(p), "sisa_prefill: tensors must be given and 16-byte aligned");
    SISA_REQUIRE(a->res == nullptr || sisa::aligned16(a->res), "sisa_prefill: res not aligned");
    SISA_REQUIRE(a->act_ld >= a->FF && a->act_ld % 64 == 0 && a->act_ld < a->FF + 64,
                 "sisa_prefill: act_ld %lld must be FF = %d rounded up to a multiple of 64", (long long)a->act_ld, a->FF);
    SISA_REQUIRE(a->ffn == nullptr || (sisa::aligned16(a->ffn) && a->w_down && sisa::aligned16(a->w_down) && a->FF % 8 == 0),
                 "sisa_prefill: the down projection needs FF %% 8 == 0 and aligned w_down, ffn");
    SISA_REQUIRE((int64_t)a->FF * a->H * DH * 2 < ((int64_t)1 << 31) &&
                     (int64_t)a->B * a->L * a->act_ld * 2 < ((int64_t)1 << 31),
                 "sisa_prefill: a weight or the activation spans 2 GiB or more");
    SISA_REQUIRE(a->b_alpha && a->b_forget && a->lambda_raw && a->phi && a->workspace &&
                     ((uintptr_t)a->workspace & 255) == 0,
                 "sisa_prefill: null pointer, or workspace not 256-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    return a->dtype == SISA_BF16 ? run_layer<__bf16>(a, st) : run_layer<_Float16>(a, st);
}
