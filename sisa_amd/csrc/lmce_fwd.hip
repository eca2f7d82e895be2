// Fused forward of the linear cross-entropy for gfx950: logits = x W_pad^T computed tile by tile on bf16/fp16 MFMA
// and reduced on the fly to each row's log-sum-exp and label logit. The (N x Vp) logits never exist in memory.
//
// Reference: the forward of `_LinearCrossEntropyFn` (src/sisa/kernels/linear_ce.py:138-191: logits chunk GEMM, then
// `_lmce_row_kernel`'s online max / sum-exp and the label pick, linear_ce.py:60-96). The reference materialises a
// (chunk, Vp) logits buffer; here the GEMM's output tiles never leave registers. As there, each logit (an fp32 MFMA
// accumulation) is rounded once to the compute dtype before the reduction, so lse and the loss are those of the
// reference's stored logits.
//
// Decomposition: a workgroup of 2 x 4 waves owns 256 rows of x and walks a range of 256-column vocabulary tiles (one
// of S vocabulary splits). Per tile, K = D is streamed through LDS in 64-wide stages (buffer loads straight into
// LDS, double-buffered, XOR-swizzled 16-byte chunks); a wave computes a 128 (vocabulary) x 64 (rows) block as 8 x 4
// v_mfma_f32_16x16x32 blocks with W as the A operand, so that a lane holds 32 logits of one row per block column
// (12 operand fragments per 32 MFMAs, to keep the LDS reads below the matrix rate). After a tile's last stage each
// wave takes every row's maximum over its 128 columns of the tile (log2 units, shared by the row's four lane groups),
// sums the row's exponentials relative to it and folds that sum into the row's running (max, sum of exponentials);
// when the tile holds a row's label it keeps that logit. At the end the lane groups and the two waves sharing rows
// combine their partials; a second launch combines the S splits of each row in a fixed order.
//
// bf16 takes the exponentials against one reference per row, its label's logit (REF; lmce_ref_kernel), and goes over the
// 256-row blocks with a row that reference does not suit again, against the maxima described above; see launch_logits. At
// 4,094 rows of 1,024 (V 50,277, weights of standard deviation 0.02) the launch takes about 350 us with REF and 372 against
// the maxima (the difference of two whole passes without and with every block marked, less its small launches).
//
// The training pass (sisa_lmce_train, lmce_train.hip) runs the same kernel with STORE: each exponential is also stored in
// the compute dtype into a (N, Vp) buffer, and without REF the maxima m_t it is relative to into a (2 * tiles, N) table.
// Both passes give bitwise the same loss rows.
// Deterministic: no atomics. Workgroup i runs on XCD i % 8; each XCD takes an equal, contiguous range of (row block,
// split) items, whole row blocks with all their splits where there are enough, so that its L2 keeps those rows of x for
// every vocabulary tile and fewer than eight row blocks still fill all XCDs.
#include "common.h"
#include "host.h"

namespace {

constexpr int NWC = 8;            // waves per workgroup: 2 along the vocabulary x 4 along the rows
constexpr int TR = 256;           // rows of x per workgroup
constexpr int TV = 256;           // vocabulary columns per tile
constexpr int RGRP = 4;           // row blocks that walk the same vocabulary tiles side by side
constexpr int WV = 128;           // vocabulary columns of a wave (8 MFMA blocks)
constexpr int WR = 64;            // rows of a wave (4 MFMA blocks)
constexpr int IB = WV / 16, JB = WR / 16;
constexpr int TK = 64;            // hidden elements per LDS stage
constexpr float M_FLOOR_CE = -1e30f;
constexpr float LN2 = 0.69314718055994531f;

template <class T>
struct __attribute__((aligned(16))) CeLds {
    T x[2][TR * TK];
    T w[2][TV * TK];
    float red_m[TR], red_s[TR];   // the second wave of each row pair hands over its row partials
};

// What a launch stores and against what it takes its exponentials.
//   STORE: the exponentials go to probs. REF: they are relative to one given reference per row (ref, log2 units)
//   instead of the row's maxima over the tile halves, which go to mtab.
//   MARKED: only the row blocks that marks marks. (A kernel of its own: with the choice made in the kernel of all blocks its
//   main loop, short of scalar registers, took 1.5 % longer.)
template <class T>
struct CeStore {
    T* probs;                     // (N, Vp) in the compute dtype, row stride Vp; columns >= V hold 0
    float* mtab;                  // (2 * tiles, N): m_t of (tile t, half h) at row (2 t + h) * N + n, log2 units
    const float* ref;             // (N,)
    float* zlab;                  // (N,) the label's logit, natural units; left alone without a label that counts
    const int* marks;
};

// The vocabulary splits of `nrb` row blocks: S splits of `per` consecutive tiles (the last ones may be shorter or empty).
constexpr int CE_WGS = 512;                      // about as many workgroups: two rounds of one per CU
struct Split {
    int S, per;
};
__host__ __device__ inline Split ce_split(int nrb, int tiles) {
    int S = (CE_WGS + nrb - 1) / nrb;
    S = S > tiles ? tiles : S;
    return {S, (tiles + S - 1) / S};
}
// The most (row block, split) items that some of `nrb` row blocks make.
inline int64_t ce_items(int64_t nrb, int64_t tiles) {
    return tiles * nrb < CE_WGS - 1 + nrb ? tiles * nrb : CE_WGS - 1 + nrb;
}

// Marks over the row blocks: word 0 tells whether there are any, word 1 + rb marks block rb. The slot of a marked block is
// the number of marked ones before it; the marked blocks are split as a problem of that many. (Whole waves call these.)
SISA_DEV int marks_before(const int* marks, int rb, int lane) {
    int c = 0;
    for (int b = 0; b < rb; b += 64) c += __popcll(__builtin_amdgcn_ballot_w64(b + lane < rb && marks[1 + b + lane] != 0));
    return c;
}
SISA_DEV int marked_block(const int* marks, int nrb, int slot, int lane) {
    for (int b = 0; b < nrb; b += 64) {
        uint64_t m = __builtin_amdgcn_ballot_w64(b + lane < nrb && marks[1 + b + lane] != 0);
        const int c = __popcll(m);
        if (slot < c) {
            for (; slot > 0; --slot) m &= m - 1;
            return b + __builtin_ctzll(m);
        }
        slot -= c;
    }
    return 0;                                    // not reached for a slot below their number
}

template <class T, bool STORE, bool REF, bool MARKED>
__global__ __launch_bounds__(64 * NWC) void lmce_fwd_kernel(sisa_lmce_fwd_args a, int S, int per, CeStore<T> out) {
    __shared__ CeLds<T> sm;
    if (MARKED && out.marks[0] == 0) return;
    const int tid = threadIdx.x, lane = tid & 63, grp = lane >> 4, lc = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t N = a.N, V = a.V;
    const int blocks = (int)((N + TR - 1) / TR), tiles = (int)((a.Vp + TV - 1) / TV);
    int nrb = blocks;
    if constexpr (MARKED) {
        nrb = marks_before(out.marks, blocks, lane);
        const Split sp = ce_split(nrb, tiles);
        S = sp.S;
        per = sp.per;
    }
    const int item = xcd_item(blockIdx.x, nrb * S);
    if (item < 0) return;
    // Items (row block, split) in groups of RGRP row blocks, row blocks fastest: the 32 workgroups an XCD runs at a time
    // are then 4 row blocks x 8 splits, which read 12 tiles of x and W per tile time through its L2; one row block with 32
    // splits reads 33.
    const int grp_items = RGRP * S, g0 = item / grp_items * RGRP, in_grp = item % grp_items;
    const int rg = nrb - g0 < RGRP ? nrb - g0 : RGRP;
    const int split = in_grp / rg, slot = g0 + in_grp % rg;
    const int rb = MARKED ? marked_block(out.marks, blocks, slot, lane) : slot;
    const int t_begin = split * per;
    const int t_end = t_begin + per < tiles ? t_begin + per : tiles;
    const int ntiles = t_end > t_begin ? t_end - t_begin : 0;
    const int nks = a.D / TK;
    const int64_t row0 = (int64_t)rb * TR;
    const int wv = WV * (w & 1), wn = WR * (w >> 1);   // the wave's vocabulary and row offsets in the tile

    // staging: a 256-row tile is four 64-row DMA groups; rows past the data read as zero
    DmaStage<T, TK, NWC> sx, sw;
    sx.init(a.ldx, w, lane);
    sw.init(a.ldw, w, lane);
    const int64_t xbytes = ((N - 1) * a.ldx + a.D) * (int64_t)sizeof(T);
    const int64_t wbytes = ((a.Vp - 1) * a.ldw + a.D) * (int64_t)sizeof(T);
    const T* X = (const T*)a.x;
    const T* W = (const T*)a.w;
    constexpr int DMA = (STORE ? 8 : 4) + (REF ? 16 : 0) + (MARKED ? 32 : 0);   // one per kernel (dma_issue)
    auto issue = [&](int g, int buf) {   // stage g of the workgroup: vocabulary tile g / nks, K block g % nks
        const int64_t v0 = (int64_t)(t_begin + g / nks) * TV;
        const int k0 = (g % nks) * TK;
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            dma_issue<DMA>(sx, X, xbytes, (int)(((row0 + 64 * h) * a.ldx + k0) * (int64_t)sizeof(T)),
                           sm.x[buf] + 64 * h * TK, w);
            dma_issue<DMA + 1>(sw, W, wbytes, (int)(((v0 + 64 * h) * a.ldw + k0) * (int64_t)sizeof(T)),
                               sm.w[buf] + 64 * h * TK, w);
        }
    };

    // the label of each of the lane's 4 rows: which tile, and whether this lane holds it (and where)
    int lab_tile[JB], lab_idx[JB];
#pragma unroll
    for (int j = 0; j < JB; ++j) {
        const int64_t n = row0 + wn + 16 * j + lc;
        lab_tile[j] = -1;
        lab_idx[j] = 0;
        if (n < N) {
            const int64_t y = a.labels[n];
            if (y != a.ignore_index && y >= 0 && y < V) {
                const int pos = (int)(y % TV);
                const bool mine = (pos / WV) * WV == wv && ((pos % 16) >> 2) == grp;
                lab_tile[j] = mine ? (int)(y / TV) : -1;
                lab_idx[j] = ((pos % WV) >> 4) * 4 + (pos & 3);   // block i, register r
            }
        }
    }
    float m[JB], s[JB], zlab[JB];   // REF: m is the rows' reference
#pragma unroll
    for (int j = 0; j < JB; ++j) {
        const int64_t n = row0 + wn + 16 * j + lc;
        m[j] = REF ? (n < N ? out.ref[n] : 0.f) : M_FLOOR_CE;
        s[j] = 0.f;
        zlab[j] = 0.f;
    }
    bool got[JB] = {false, false, false, false};

    f32x4 acc[IB][JB];
#pragma unroll
    for (int i = 0; i < IB; ++i)
#pragma unroll
        for (int j = 0; j < JB; ++j) acc[i][j] = zero4();

    // STORE: the exponentials go out through one buffer resource over (N, Vp) (at most 0x7fffff00 bytes, checked by
    // sisa_lmce_train)
    const __amdgpu_buffer_rsrc_t prs =
        make_rsrc(STORE ? (const void*)out.probs : (const void*)a.x, STORE ? N * a.Vp * (int64_t)sizeof(T) : 0);
    const int total = ntiles * nks;
    if (total > 0) issue(0, 0);
    __syncthreads();
    for (int g = 0; g < total; ++g) {
        const int buf = g & 1;
        if (g + 1 < total) issue(g + 1, buf ^ 1);
        __builtin_amdgcn_sched_barrier(0);   // the next stage's DMA stays ahead of this stage's stores
        // all 12 operand fragments of a 32-deep step are read before its 32 MFMAs (two waves per SIMD leave room
        // for them), so one LDS wait per step instead of one per 4 MFMAs
#pragma unroll
        for (int step = 0; step < TK / 32; ++step) {
            frag8<T> xf[JB], wf[IB];
#pragma unroll
            for (int j = 0; j < JB; ++j) xf[j] = frag_rows<T, TK>(sm.x[buf], wn + 16 * j, step, lane);
#pragma unroll
            for (int i = 0; i < IB; ++i) wf[i] = frag_rows<T, TK>(sm.w[buf], wv + 16 * i, step, lane);
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int j = 0; j < JB; ++j) acc[i][j] = mma(wf[i], xf[j], acc[i][j]);
        }
        if (g % nks == nks - 1) {
            // the tile is complete: lane holds logits of rows wn + 16 j + lc at columns v0 + wv + 16 i + 4 grp + r,
            // rounded once to the compute dtype (the logits the reference's row kernel reads)
            const int vt = t_begin + g / nks;
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int j = 0; j < JB; ++j) acc[i][j] = __builtin_convertvector(to_vec4<T>(acc[i][j]), f32x4);
            if ((int64_t)(vt + 1) * TV > V) {   // the last tile: padding columns do not enter the sums
                const int lim = (int)(V - (int64_t)vt * TV) - wv - 4 * grp;
#pragma unroll
                for (int i = 0; i < IB; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int j = 0; j < JB; ++j)
                            acc[i][j][r] = 16 * i + r < lim ? acc[i][j][r] : -__builtin_inff();
            }
#pragma unroll
            for (int j = 0; j < JB; ++j) {
                float mt = -__builtin_inff();   // the row's maximum over the wave's 128 columns, in log2 units
                if constexpr (!REF) {
#pragma unroll
                    for (int i = 0; i < IB; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) mt = fmaxf(mt, acc[i][j][r]);
                    mt = group_max(mt) * LOG2E;
                }
                // a half made only of padding columns (-inf) takes the reference 0: its exponentials are 0
                const float mref = REF ? m[j] : (mt == -__builtin_inff() ? 0.f : mt);
                const int64_t n = row0 + wn + 16 * j + lc;
                float ls = 0.f;
                u32x2 prev = {0u, 0u};
#pragma unroll
                for (int i = 0; i < IB; ++i) {
                    f32x4 e;
#pragma unroll
                    for (int r = 0; r < 4; ++r) e[r] = fast_exp2(fmaf(acc[i][j][r], LOG2E, -mref));
                    ls += (e[0] + e[1]) + (e[2] + e[3]);
                    if constexpr (STORE) {
                        // Blocks i - 1 and i trade places between neighbouring lane groups: a lane then holds 8
                        // consecutive columns, 8 (grp / 2) .. + 7 of block i - 1 + grp % 2, and a store covers 64
                        // consecutive bytes of each of its 16 rows (32 without the trade, for twice the stores).
                        // Stores are unconditional: positions past the data go past the resource.
                        const u32x2 cur = __builtin_bit_cast(u32x2, to_vec4<T>(e));
                        if (i & 1) {
                            const auto lo = __builtin_amdgcn_permlane16_swap(prev[0], cur[0], false, false);
                            const auto hi = __builtin_amdgcn_permlane16_swap(prev[1], cur[1], false, false);
                            const u32x4 q = {lo[0], hi[0], lo[1], hi[1]};
                            const int64_t v = (int64_t)vt * TV + wv + 16 * (i - 1 + (grp & 1)) + 8 * (grp >> 1);
                            const int off = (n < N && v < a.Vp) ? (int)((n * a.Vp + v) * (int64_t)sizeof(T)) : 0x7ffffff0;
                            __builtin_amdgcn_raw_buffer_store_b128(q, prs, off, 0, 0);
                        }
                        prev = cur;
                    }
                }
                if constexpr (STORE && !REF) {
                    if (grp == 0 && n < N) out.mtab[(int64_t)(2 * vt + (w & 1)) * N + n] = mref;
                }
                if constexpr (REF) {
                    s[j] += ls;
                } else if (mt > m[j]) {
                    s[j] = fmaf(s[j], fast_exp2(m[j] - mt), ls);
                    m[j] = mt;
                } else {
                    s[j] = fmaf(ls, fast_exp2(mt - m[j]), s[j]);
                }
                if (lab_tile[j] == vt) {   // rare: pick the label's logit (natural units)
                    float z = 0.f;
#pragma unroll
                    for (int i = 0; i < IB; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) z = (lab_idx[j] == 4 * i + r) ? acc[i][j][r] : z;
                    zlab[j] = z;
                    got[j] = true;
                }
            }
#pragma unroll
            for (int i = 0; i < IB; ++i)
#pragma unroll
                for (int j = 0; j < JB; ++j) acc[i][j] = zero4();
            if constexpr (STORE) {
                // The barrier after a tile's stores waits only until the next stage's DMA (issued before them) has
                // landed: vector memory operations complete in issue order, and at least the 16 exponential stores
                // (unconditional instructions) follow it, so vmcnt <= 16 implies the DMA is done; the stores
                // themselves complete under the next stage (its barrier waits for everything).
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(0x4070);   // vmcnt(16) expcnt(7) lgkmcnt(0)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                continue;
            }
        }
        __syncthreads();
    }

    // combine the four lane groups of each row, then the two waves sharing the rows (w and w ^ 1)
    const int64_t np = MARKED ? (int64_t)nrb * TR : (N + TR - 1) / TR * TR;
    float* part = a.workspace + (MARKED ? (int64_t)slot * TR : row0);
    float rm[JB], rsum[JB];
#pragma unroll
    for (int j = 0; j < JB; ++j) {
        rm[j] = REF ? m[j] : group_max(m[j]);
        rsum[j] = group_sum(REF ? s[j] : s[j] * fast_exp2(m[j] - rm[j]));
        if (got[j]) out.zlab[row0 + wn + 16 * j + lc] = zlab[j];
    }
    if ((w & 1) && grp == 0) {
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            sm.red_m[wn + 16 * j + lc] = rm[j];
            sm.red_s[wn + 16 * j + lc] = rsum[j];
        }
    }
    __syncthreads();
    if ((w & 1) == 0 && grp == 0) {
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            const int r = wn + 16 * j + lc;
            if (row0 + r >= N) continue;
            const float m2 = sm.red_m[r], s2 = sm.red_s[r];
            if constexpr (REF) {
                part[(S + split) * np + r] = rsum[j] + s2;
                continue;
            }
            const float mm = fmaxf(rm[j], m2);
            part[split * np + r] = mm;
            part[(S + split) * np + r] = rsum[j] * fast_exp2(rm[j] - mm) + s2 * fast_exp2(m2 - mm);
        }
    }
}

// Per row: the S split partials combined in split order; lse (natural log) and the loss row, and what the training pass
// keeps of them. The partials of a row lie at its block's slot (256 rows each) plus its place in the block.
//   LABEL: of exponentials against the rows' references, all rows; marks the row blocks that must be gone over again.
//   TOP: of exponentials against maxima: fp16's only pass, or bf16's marked row blocks.
//   AGAIN: of exponentials stored again against the log-sum-exp, bf16's marked row blocks; the loss stays.
enum CombineMode { LABEL, TOP, AGAIN };
struct CeTrainRows {
    float* lse2;                  // fp16: (N,) lse in log2 units, or nullptr (the no-gradient pass)
    float2* rinfo;                // (N,): s_n (bf16: s_n (1 - p_label), what G holds at the label, negated), and the
                                  // label as the bit pattern of an int (-1 outside [0, V) or ignored)
    const float* inv_n;           // device scalar 1 / N_valid
    float gscale;
    float* ref;                   // bf16: (N,) the reference of the row's exponentials, log2 units
    float* cn;                    // bf16: (N,) s_n / Z_n, or nullptr (the no-gradient pass)
    __bf16* probs;                // bf16 with cn: the stored exponentials (N, Vp); the label's is zeroed here
    int* marks;                   // LABEL: marks a block with a row that its reference did not suit; else: the blocks to run
                                  // on (null: all)
};

// 16 rows per workgroup, 16 threads per row: each folds every sixteenth split, and the row's first thread the sixteen
// partial results in order. (One thread per row walks S splits in dependent loads: with the 128 splits of 1,023 rows
// that took 66 us.)
constexpr int CRW = 16, CSP = 16;
// Sums of exponentials that a reference is good for: an actual logit's term is 1, and products of up to 2^90 with weights
// stay far inside fp32, as s_n / 2^90 does.
constexpr float Z_MIN = 0x1p-20f, Z_MAX = 0x1p90f;

// An ignored row adds nothing: unless its log-sum-exp is asked for it takes a reference above any logit, so that its
// exponentials are 0 and products with them finite, and marks no row block. (No column's logit represents such a row, and
// one prompt token that the loss masks would have a block gone over again.)
constexpr float REF_IGNORED = 0x1p126f;
SISA_DEV bool left_out(const sisa_lmce_fwd_args& a, int64_t y) { return y == a.ignore_index && !a.lse; }

template <CombineMode MODE>
__global__ __launch_bounds__(CRW * CSP) void lmce_combine_kernel(sisa_lmce_fwd_args a, int S, const float* zlab,
                                                                 CeTrainRows tr) {
    constexpr bool REF = MODE != TOP;
    __shared__ float pm[CSP][CRW], ps[CSP][CRW];
    const int lane = threadIdx.x & 63;
    const int64_t N = a.N;
    const int rb = (int)((int64_t)blockIdx.x * CRW / TR), blocks = (int)((N + TR - 1) / TR);
    int nrb = blocks, slot = rb;
    if (MODE != LABEL && tr.marks) {
        if (tr.marks[0] == 0 || tr.marks[1 + rb] == 0) return;
        nrb = marks_before(tr.marks, blocks, lane);
        slot = marks_before(tr.marks, rb, lane);
        S = ce_split(nrb, (int)((a.Vp + TV - 1) / TV)).S;
    }
    const int lr = threadIdx.x % CRW, part = threadIdx.x / CRW;
    const int64_t n = (int64_t)blockIdx.x * CRW + lr, np = (int64_t)nrb * TR;
    const float* in = a.workspace + (int64_t)slot * TR + (n - (int64_t)rb * TR);
    float mm = M_FLOOR_CE, ss = 0.f;
    if (n < N) {
        for (int sp = part; sp < S; sp += CSP) {
            const float s = in[(S + sp) * np];
            if constexpr (REF) {
                ss += s;
            } else {
                const float m = in[sp * np];
                const float mn = fmaxf(mm, m);
                ss = fmaf(ss, fast_exp2(mm - mn), s * fast_exp2(m - mn));
                mm = mn;
            }
        }
    }
    pm[part][lr] = mm;
    ps[part][lr] = ss;
    __syncthreads();
    if (part != 0 || n >= N) return;
    const int64_t y = a.labels[n];
    const bool out = left_out(a, y);
    if constexpr (REF) {
        mm = tr.ref[n];
        ss = 0.f;
#pragma unroll
        for (int p = 0; p < CSP; ++p) ss += ps[p][lr];
    } else {
#pragma unroll
        for (int p = 1; p < CSP; ++p) mm = fmaxf(mm, pm[p][lr]);
        ss = 0.f;
#pragma unroll
        for (int p = 0; p < CSP; ++p) ss = fmaf(ps[p][lr], fast_exp2(pm[p][lr] - mm), ss);
    }
    if constexpr (MODE == LABEL)         // NaN too; all who mark store the same value
        if (!out && !(ss >= Z_MIN && ss <= Z_MAX)) tr.marks[0] = tr.marks[1 + rb] = 1;
    const float l2 = mm + __builtin_amdgcn_logf(ss);
    if constexpr (MODE != AGAIN) {
        const float lse = l2 * LN2;
        float loss;
        if (y == a.ignore_index) loss = 0.f;
        else if (y < 0 || y >= a.V) loss = __builtin_nanf("");
        else loss = lse - zlab[n];
        a.loss_rows[n] = loss;
        if (a.lse) a.lse[n] = lse;
        if (MODE == TOP && tr.cn && !out) tr.ref[n] = l2;
    }
    const int lab = (y != a.ignore_index && y >= 0 && y < a.V) ? (int)y : -1;   // its logit exists only then
    const float sn = y == a.ignore_index || !tr.inv_n ? 0.f : tr.inv_n[0] * tr.gscale;
    if constexpr (REF) {
        if (!tr.cn) return;
        float gl = sn;
        tr.cn[n] = out ? 0.f : sn / ss;
        if (lab >= 0) {   // p - 1 is formed here in fp32: taken apart, the two roundings of p would outweigh it near p = 1
            gl = sn * (1.f - fast_exp2(fmaf(zlab[n], LOG2E, -mm)) / ss);
            tr.probs[n * a.Vp + lab] = (__bf16)0.f;
        }
        tr.rinfo[n] = float2{gl, __int_as_float(lab)};
    } else if (tr.lse2) {
        tr.lse2[n] = l2;
        tr.rinfo[n] = float2{sn, __int_as_float(lab)};
    }
}

// The reference of a row's exponentials: the logit of its label (of column 0 without a valid one), in log2 units. Any
// column's logit bounds the row's sum below by 1; the label's is near the largest wherever the loss is small. Rows left
// out: REF_IGNORED. LPR lanes a row, 8 elements each at a time (a whole wave for a row of 64
// elements keeps 8 lanes busy: 140,000 such rows took 30 us). Also clears the marks.
template <class T, int LPR>
__global__ __launch_bounds__(256) void lmce_ref_kernel(sisa_lmce_fwd_args a, float* ref, int* marks) {
    constexpr int RPB = 256 / LPR;                        // rows of a workgroup; 256 = TR is a multiple of it
    const int64_t n = (int64_t)blockIdx.x * RPB + threadIdx.x / LPR;
    const int lane = threadIdx.x % LPR;
    if (threadIdx.x == 0 && blockIdx.x % (TR / RPB) == 0) {
        const int rb = blockIdx.x / (TR / RPB);
        marks[1 + rb] = 0;
        if (rb == 0) marks[0] = 0;
    }
    if (n >= a.N) return;
    const int64_t y = a.labels[n];
    if (left_out(a, y)) {
        if (lane == 0) ref[n] = REF_IGNORED;
        return;
    }
    const T* x = (const T*)a.x + n * a.ldx;
    const T* w = (const T*)a.w + (y >= 0 && y < a.V ? y : 0) * a.ldw;
    float d = 0.f;
    for (int c = 8 * lane; c < a.D; c += 8 * LPR) {
        const f32x8 xv = load_f32x8<T>(x + c), wv = load_f32x8<T>(w + c);
#pragma unroll
        for (int e = 0; e < 8; ++e) d = fmaf(xv[e], wv[e], d);
    }
#pragma unroll
    for (int o = LPR / 2; o > 0; o >>= 1) d += __shfl_xor(d, o);
    if (lane == 0) ref[n] = d * LOG2E;
}

template <class T>
void launch_ref(const sisa_lmce_fwd_args* a, float* ref, int* marks, hipStream_t st) {
    if (a->D <= 64) lmce_ref_kernel<T, 8><<<(unsigned)sisa::cdiv(a->N, 32), 256, 0, st>>>(*a, ref, marks);
    else if (a->D <= 256) lmce_ref_kernel<T, 32><<<(unsigned)sisa::cdiv(a->N, 8), 256, 0, st>>>(*a, ref, marks);
    else lmce_ref_kernel<T, 64><<<(unsigned)sisa::cdiv(a->N, 4), 256, 0, st>>>(*a, ref, marks);
}

// The workspace of the logits pass: the split partials (max and sum rows), label logits, the rows' references, the marks.
struct CeWs {
    float *zlab, *ref;
    int* marks;
    int64_t bytes;
};
CeWs ce_ws(float* base, int64_t N, int64_t Vp) {
    const int64_t nrb = sisa::cdiv(N, TR);
    CeWs w;
    w.zlab = base + 2 * TR * ce_items(nrb, sisa::cdiv(Vp, TV));
    w.ref = w.zlab + N;
    w.marks = (int*)(w.ref + N);
    w.bytes = (char*)(w.marks + 1 + nrb) - (char*)base;
    return w;
}

// Logits GEMM and combine. bf16: against the label logits (REF). That spares each logit the running maximum, and lets the
// gradient products of the training pass take the stored exponentials as they are. A row that counts may have a sum its
// reference was not good for: its label's logit more than 62 below its largest, or non-finite values. Its block of 256
// rows is then gone over again, for the loss against the maxima, and in the training pass once more, storing exponentials
// against the log-sum-exp. Those launches split the marked blocks over the whole chip and end at once without any. (16,384
// rows of 768: 4,340 us, 4,400 with one such row, 6,830 with one in every block; taking the whole chunk through maxima
// and forming G for dx as fp16 does took 6,090 with any.) fp16 has too little exponent range for a reference per row and
// always takes the maxima.
template <class T, bool STORE>
int launch_logits(const sisa_lmce_fwd_args* a, T* probs, float* mtab, CeTrainRows r, hipStream_t st) {
    const int64_t nrb = sisa::cdiv(a->N, TR), tiles = sisa::cdiv(a->Vp, TV);
    const Split sp = ce_split((int)nrb, (int)tiles);
    const CeWs ws = ce_ws(a->workspace, a->N, a->Vp);
    const unsigned grid = (unsigned)(8 * sisa::cdiv(nrb * sp.S, 8));
    const unsigned again = (unsigned)(8 * sisa::cdiv(ce_items(nrb, tiles), 8));
    const unsigned cgrid = (unsigned)sisa::cdiv(a->N, CRW);
    CeStore<T> out{probs, mtab, nullptr, ws.zlab, nullptr};
    if constexpr (__is_same(T, __bf16)) {
        out.ref = r.ref = ws.ref;
        r.marks = ws.marks;
        launch_ref<T>(a, ws.ref, ws.marks, st);
        int rc = sisa::launch_status("linear CE (reference)");
        if (rc) return rc;
        lmce_fwd_kernel<T, STORE, true, false><<<grid, 64 * NWC, 0, st>>>(*a, sp.S, sp.per, out);
        rc = sisa::launch_status("linear CE (logits)");
        if (rc) return rc;
        lmce_combine_kernel<LABEL><<<cgrid, CRW * CSP, 0, st>>>(*a, sp.S, ws.zlab, r);
        rc = sisa::launch_status("linear CE (combine)");
        if (rc) return rc;
        out.marks = ws.marks;
        lmce_fwd_kernel<T, false, false, true><<<again, 64 * NWC, 0, st>>>(*a, 0, 0, out);
        rc = sisa::launch_status("linear CE (logits again)");
        if (rc) return rc;
        lmce_combine_kernel<TOP><<<cgrid, CRW * CSP, 0, st>>>(*a, 0, ws.zlab, r);
        rc = sisa::launch_status("linear CE (combine again)");
        if (rc || !STORE) return rc;
        lmce_fwd_kernel<T, true, true, true><<<again, 64 * NWC, 0, st>>>(*a, 0, 0, out);
        rc = sisa::launch_status("linear CE (exponentials again)");
        if (rc) return rc;
        lmce_combine_kernel<AGAIN><<<cgrid, CRW * CSP, 0, st>>>(*a, 0, ws.zlab, r);
        return sisa::launch_status("linear CE (scales again)");
    } else {
        lmce_fwd_kernel<T, STORE, false, false><<<grid, 64 * NWC, 0, st>>>(*a, sp.S, sp.per, out);
        const int rc = sisa::launch_status("linear CE (logits)");
        if (rc) return rc;
        lmce_combine_kernel<TOP><<<cgrid, CRW * CSP, 0, st>>>(*a, sp.S, ws.zlab, r);
        return sisa::launch_status("linear CE (combine)");
    }
}

template <class T>
int launch_lmce_fwd(const sisa_lmce_fwd_args* a, hipStream_t st) {
    return launch_logits<T, false>(a, nullptr, nullptr, CeTrainRows{}, st);
}

}  // namespace

namespace sisa {
namespace detail {

int64_t lmce_fwd_ws_bytes(int64_t N, int64_t Vp) { return ce_ws(nullptr, N, Vp).bytes; }

// The training pass's forward: the logits GEMM storing the exponentials (probs: (N, Vp) in the compute dtype), then the
// split combine writing the loss rows and each row's gradient scale. bf16: exponentials against one reference per row,
// G = probs * cn off the label, whose entry of probs is zero, and -rinfo.x at it. fp16: exponentials against the tile-half
// maxima in mtab ((2 * ceil(Vp / 256), N) fp32), lse in log2 units, rinfo.x = s_n. a->workspace: lmce_fwd_ws_bytes.
int lmce_train_forward(const sisa_lmce_fwd_args* a, void* probs, float* mtab, float* lse2, float2* rinfo, float* cn,
                       const float* inv_n, float gscale, hipStream_t st) {
    CeTrainRows r{};
    r.rinfo = rinfo;
    r.inv_n = inv_n;
    r.gscale = gscale;
    if (a->dtype == SISA_BF16) {
        r.cn = cn;
        r.probs = (__bf16*)probs;
        return launch_logits<__bf16, true>(a, (__bf16*)probs, nullptr, r, st);
    }
    r.lse2 = lse2;
    return launch_logits<_Float16, true>(a, (_Float16*)probs, mtab, r, st);
}

}  // namespace detail
}  // namespace sisa

extern "C" int64_t sisa_lmce_fwd_workspace_bytes(int64_t N, int64_t Vp) {
    if (N < 1 || Vp < 1) return 0;
    return sisa::detail::lmce_fwd_ws_bytes(N, Vp);
}

extern "C" int sisa_lmce_fwd(const sisa_lmce_fwd_args* a, void* stream) {
    SISA_REQUIRE(a != nullptr, "sisa_lmce_fwd: null args");
    if (a->N == 0) return SISA_OK;
    SISA_REQUIRE(a->N >= 1 && a->V >= 1 && a->Vp >= a->V, "sisa_lmce_fwd: bad shape N=%lld V=%lld Vp=%lld",
                 (long long)a->N, (long long)a->V, (long long)a->Vp);
    SISA_REQUIRE(a->D >= TK && a->D % TK == 0, "sisa_lmce_fwd: hidden size %d must be a positive multiple of %d", a->D,
                 TK);
    SISA_REQUIRE(a->dtype == SISA_BF16 || a->dtype == SISA_F16, "sisa_lmce_fwd: dtype %d (bf16 or fp16)", a->dtype);
    SISA_REQUIRE(a->x && a->w && a->labels && a->loss_rows && a->workspace && sisa::aligned16(a->x) &&
                     sisa::aligned16(a->w) && a->ldx >= a->D && a->ldw >= a->D && a->ldx % 8 == 0 && a->ldw % 8 == 0,
                 "sisa_lmce_fwd: x, w must be 16-byte aligned with row strides >= D (multiples of 8); labels, "
                 "loss_rows, workspace given");
    // one buffer resource per operand: both extents below 2 GiB
    SISA_REQUIRE(((sisa::cdiv(a->N, TR) * TR - 1) * a->ldx + a->D) * 2 < ((int64_t)1 << 31) &&
                     ((sisa::cdiv(a->Vp, TV) * TV - 1) * a->ldw + a->D) * 2 < ((int64_t)1 << 31),
                 "sisa_lmce_fwd: x or w spans 2 GiB or more");
    hipStream_t st = (hipStream_t)stream;
    return a->dtype == SISA_BF16 ? launch_lmce_fwd<__bf16>(a, st) : launch_lmce_fwd<_Float16>(a, st);
}
