/*
 * k_gemm.hip — weight repacking, activation quantization and the matrix products of
 * the verify step on gfx950.
 *
 * Reference semantics: NUMERICS §2-3 (engine/src/quant.c:325-427). Every (token, row)
 * output is one lane's fold acc = acc + (float)isum_g * (dw_g * dx_g) over the blocks
 * g of its row in ascending order; isum_g is the exact int32 block sum from one
 * v_mfma_i32_16x16x64_i8 (K = one 64-block). Which other tokens share the MFMA tile
 * cannot change any output, so a batch equals T single-token calls bit for bit
 * (reference INV-DET-2, governance/INVARIANTS.md:12).
 */
#include "hx_device.h"
#include "hx_launch.h"
#include <hip/hip_ext.h>
#include <type_traits>

using namespace hxd;

namespace {

constexpr uint32_t LO4 = 0x0F0F0F0Fu;

/* ------------------------------------------------------------ repacking */

/* FORMAT.md §6 Q8 rows (66-byte blocks) -> tiles + transposed scales. src holds rows
 * [r0, r0 + count) (pad rows beyond `rows` are not read); one thread per (row, block);
 * pad rows and the pad block get zeros. */
__global__ void k_repack_q8(const uint8_t *__restrict__ src, int r0, int count, int rows, int nb, QMat m, uint8_t *w,
                            uint16_t *d) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)count * m.nbp) return;
    const int r = r0 + (int)(idx / m.nbp), g = (int)(idx % m.nbp);
    const bool real = r < rows && g < nb;
    const uint8_t *blk = src + ((size_t)(r - r0) * nb + g) * 66;
    d[(size_t)g * m.rows_pad + r] = real ? (uint16_t)(blk[0] | (blk[1] << 8)) : (uint16_t)0;
    uint8_t *tile = w + ((size_t)(r >> 4) * m.nbp + g) * 1024;
    for (int kg = 0; kg < 4; kg++)
        for (int b = 0; b < 16; b++) {
            const int e = b < 8 ? 8 * kg + b : 32 + 8 * kg + (b - 8);
            tile[(size_t)((r & 15) + 16 * kg) * 16 + b] = real ? blk[2 + e] : (uint8_t)0;
        }
}

/* FORMAT.md §6 Q4 rows (34-byte blocks) -> tiles of block pairs + transposed scales. */
__global__ void k_repack_q4(const uint8_t *__restrict__ src, int r0, int count, int rows, int nb, QMat m, uint8_t *w,
                            uint16_t *d) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)count * m.nbp) return;
    const int r = r0 + (int)(idx / m.nbp), g = (int)(idx % m.nbp);
    const bool real = r < rows && g < nb;
    const uint8_t *blk = src + ((size_t)(r - r0) * nb + g) * 34;
    d[(size_t)g * m.rows_pad + r] = real ? (uint16_t)(blk[0] | (blk[1] << 8)) : (uint16_t)0;
    uint8_t *tile = w + ((size_t)(r >> 4) * (m.nbp / 2) + (g >> 1)) * 1024;
    for (int kg = 0; kg < 4; kg++)
        for (int b = 0; b < 8; b++)
            tile[(size_t)((r & 15) + 16 * kg) * 16 + (g & 1) * 8 + b] = real ? blk[2 + 8 * kg + b] : (uint8_t)0;
}

/* ------------------------------------------------------------ activation quantization */

/* NUMERICS §2 on rows of x (f32 [T][n], row stride ldx): one wave per (row, block). */
__global__ void k_quant_rows(const float *__restrict__ x, int64_t ldx, int T, int nb, Act a) {
    const int wave = (int)((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6);
    if (wave >= T * a.nbp) return;   /* uniform per wave */
    const int t = wave / a.nbp, g = wave % a.nbp, lane = threadIdx.x & 63;
    const float v = g < nb ? x[(size_t)t * ldx + (size_t)g * 64 + lane] : 0.0f;
    quant_block_wave(v, a, t, g);
}

/* ------------------------------------------------------------ the MFMA fold */

__device__ __forceinline__ v4i load16(const uint8_t *p) { return *(const v4i *)p; }

__device__ __forceinline__ void unpack_q4(v4i raw, v4i &a0, v4i &a1) {
    a0.x = raw.x & LO4; a0.y = raw.y & LO4; a0.z = (raw.x >> 4) & LO4; a0.w = (raw.y >> 4) & LO4;
    a1.x = raw.z & LO4; a1.y = raw.w & LO4; a1.z = (raw.z >> 4) & LO4; a1.w = (raw.w >> 4) & LO4;
}

/* ------------------------------------------------------------ split-K products (few tokens) */

/* With few tokens a product is bound by how many weight bytes are in flight, not by the
 * MFMA rate. The split-K kernels give each wave of a workgroup a contiguous range of
 * block pairs of one 16-row tile and issue all its loads at once; each wave writes the
 * NUMERICS §3 terms (float)isum_g * (dw_g * dx_g) of its blocks to LDS, and after one
 * barrier one thread per (row, token) folds the terms of blocks 0, 1, ... in order, so
 * the result is the one-lane fold bit for bit. */
constexpr int SK_MAXP = 4;      /* block pairs per wave */
constexpr int TK_WAVES_GATEUP = 8;   /* waves per workgroup of k_expert_tk: gate/up (token blocks staged once for 8 waves) */
constexpr int TK_WAVES_DOWN = 4;     /* and down (more, smaller workgroups over the shorter rows) */
constexpr size_t TK_LDS_MAX = 65536;
constexpr int TK_MIXED_T = 4;        /* k_expert_tk for experts of both dtypes: tokens at most */
constexpr int TK_CHUNK_ROWS = 128;   /* rows of a slot kept on one XCD (two 128-byte scale lines) */
constexpr int SK_LDS = 65536;   /* bytes of terms per workgroup */
constexpr int SK_DUMMY = 1024;  /* LDS after the terms: stores of padding token columns */
/* the split-K kernels of the experts: tokens at most, and the workgroups of the chunked
 * kernels from which those are the faster ones (few_workgroups) */
constexpr int SK_T = 4, SK_WGS_GATEUP = 96, SK_WGS_DOWN = 256;

/* Terms of pairs [p0, p1) of row tile rt of the NM matrices ms (same dtype DT and
 * blocks, one shared activation) for tokens t0 .. t0 + 15 (token t's activation row
 * is row_of(t); tokens >= n repeat row_of(n - 1)). Term (matrix mi, block g, token c,
 * row r) goes to P[mi * pstride + (g * ntok + c) * 16 + r] for c < ntok. */
template <int DT, int NM>
__device__ __forceinline__ void tile_terms_chunk(const QMat *ms, int rt, const Act &a, int arow, int ntok, int p0,
                                                 int p1, float *P, int pstride) {
    const int lane = threadIdx.x & 63, kg = lane >> 4, lr = lane & 15;
    const int npair = ms[0].nbp >> 1, nb = ms[0].nb;
    v4i raw[NM][SK_MAXP][DT == 4 ? 1 : 2];
    uint2 sc[NM][SK_MAXP][2];
    v4i xq[SK_MAXP][2];
    float dx[SK_MAXP][2];
    int sx[SK_MAXP][2];
#pragma unroll
    for (int k = 0; k < SK_MAXP; k++) {
        const int gp = p0 + k < p1 ? p0 + k : p1 - 1;
#pragma unroll
        for (int mi = 0; mi < NM; mi++) {
            const QMat &m = ms[mi];
            if (DT == 4) {
                raw[mi][k][0] = load16(m.w + ((size_t)rt * npair + gp) * 1024 + lane * 16);
            } else {
                const uint8_t *base = m.w + ((size_t)rt * m.nbp + 2 * gp) * 1024 + lane * 16;
                raw[mi][k][0] = load16(base);
                raw[mi][k][DT == 4 ? 0 : 1] = load16(base + 1024);
            }
            const uint16_t *dcol = m.d + rt * 16 + 4 * kg;
            sc[mi][k][0] = *(const uint2 *)(dcol + (size_t)(2 * gp) * m.rows_pad);
            sc[mi][k][1] = *(const uint2 *)(dcol + (size_t)(2 * gp + 1) * m.rows_pad);
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const size_t ab = (size_t)arow * a.nbp + 2 * gp + j;
            xq[k][j] = load16((const uint8_t *)(a.q + ab * 64 + kg * 16));
            dx[k][j] = a.d[ab];
            sx[k][j] = DT == 4 ? a.s[ab] : 0;
        }
    }
    /* all MFMAs first (each into its own registers), then the f32 terms: no term waits on
     * the MFMA just issued. Lanes of token columns >= ntok store to the dummy area. */
    const v4i zero = {0, 0, 0, 0};
    v4i cc[NM][SK_MAXP][2];
#pragma unroll
    for (int k = 0; k < SK_MAXP; k++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int mi = 0; mi < NM; mi++) {
                v4i wa;
                if (DT == 4) {
                    v4i w0, w1;
                    unpack_q4(raw[mi][k][0], w0, w1);
                    wa = j ? w1 : w0;
                } else {
                    wa = raw[mi][k][DT == 4 ? 0 : j];
                }
                cc[mi][k][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa, xq[k][j], zero, 0, 0, 0);
            }
    float *dmy = P + (size_t)NM * nb * ntok * 16 + lane * 4;   /* after the NM matrices' terms */
#pragma unroll
    for (int k = 0; k < SK_MAXP; k++) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int g = 2 * (p0 + k) + j;
            if (p0 + k >= p1 || g >= nb) continue;   /* uniform */
#pragma unroll
            for (int mi = 0; mi < NM; mi++) {
                v4i c = cc[mi][k][j];
                if (DT == 4) {
                    const int off = 8 * sx[k][j];   /* sum(nib * q) - 8 sum(q) = sum((nib - 8) q) */
                    c.x -= off; c.y -= off; c.z -= off; c.w -= off;
                }
                const uint2 sw = sc[mi][k][j];
                const float d = dx[k][j];
                float4 v;
                v.x = fmul((float)c.x, fmul(h2f((uint16_t)(sw.x & 0xffff)), d));
                v.y = fmul((float)c.y, fmul(h2f((uint16_t)(sw.x >> 16)), d));
                v.z = fmul((float)c.z, fmul(h2f((uint16_t)(sw.y & 0xffff)), d));
                v.w = fmul((float)c.w, fmul(h2f((uint16_t)(sw.y >> 16)), d));
                float *dst = lr < ntok ? P + (size_t)mi * pstride + ((size_t)g * ntok + lr) * 16 + 4 * kg : dmy;
                *(float4 *)dst = v;
            }
        }
    }
}

template <int DT, int NM, typename RowOf>
__device__ __forceinline__ void tile_terms(const QMat *ms, int rt, const Act &a, int t0, int n, int ntok,
                                           RowOf row_of, int p0, int p1, float *P, int pstride) {
    int t = t0 + (threadIdx.x & 15);
    t = t < n ? t : n - 1;
    const int arow = row_of(t);
    for (int pc = p0; pc < p1; pc += SK_MAXP)   /* uniform */
        tile_terms_chunk<DT, NM>(ms, rt, a, arow, ntok, pc, pc + SK_MAXP < p1 ? pc + SK_MAXP : p1, P, pstride);
}

/* sum of the terms P[(g * ntok) * 16 + tid] over blocks g = 0 .. nb-1, in order */
__device__ __forceinline__ float fold_terms(const float *P, int nb, int ntok, int tid) {
    float acc = 0.0f;
    const int st = ntok * 16;
    int g = 0;
    for (; g + 8 <= nb; g += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = P[(g + u) * st + tid];
#pragma unroll
        for (int u = 0; u < 8; u++) acc = fadd(acc, v[u]);
    }
    for (; g < nb; g++) acc = fadd(acc, P[g * st + tid]);
    return acc;
}

/* pair range of wave w of W over npair pairs */
__device__ __forceinline__ void wave_pairs(int npair, int W, int w, int &p0, int &p1) {
    const int ppw = (npair + W - 1) / W;
    p0 = w * ppw;
    p1 = p0 + ppw < npair ? p0 + ppw : npair;
}

/* dense product of few tokens: one workgroup per 16-row tile of a segment. */
template <int DT>
__global__ __launch_bounds__(512) void k_gemm_sk(GemmArgs args, int ntok) {
    extern __shared__ float P[];
    int s = 0;
    while (s + 1 < args.nseg && (int)blockIdx.x >= args.seg[s + 1].wg0) s++;
    const GemmSeg &sg = args.seg[s];
    const int rt = (int)blockIdx.x - sg.wg0;
    const int W = blockDim.x >> 6, wave = threadIdx.x >> 6, tid = threadIdx.x;
    int p0, p1;
    wave_pairs(sg.m.nbp >> 1, W, wave, p0, p1);
    /* padding tokens (t >= *live): no columns of their own (their activation loads repeat
     * the last live row's), no folds, no rows written. Bounding the columns only after
     * the loads (every padding row's activations loaded) cost 0.96 us a launch in a loop
     * with short drafts. */
    const int lv = args.live ? *args.live : args.T;
    const int T = lv < args.T ? lv : args.T;
    for (int t0 = 0; t0 < T; t0 += ntok) {
        tile_terms<DT, 1>(&sg.m, rt, args.a, t0, T, ntok, [](int t) { return t; }, p0, p1, P, 0);
        __syncthreads();
        const int nc = T - t0 < ntok ? T - t0 : ntok;
        for (int f = tid; f < nc * 16; f += blockDim.x) {
            const int c = f >> 4, row = rt * 16 + (f & 15), t = t0 + c;
            const float acc = fold_terms(P, sg.m.nb, ntok, f);
            if (row < sg.m.rows) {
                float y = canon(acc);
                if (sg.scale_on) y = canon(fmul(sg.scale, y));
                sg.Y[(size_t)t * sg.ldy + row] = y;
            }
        }
        __syncthreads();
    }
}

/* Expert products for experts of at most 16 tokens, K split over S waves per row tile:
 * gate and up with the SwiGLU epilogue (MODE TK_GATEUP), or the down projection of
 * quantized rows (TK_DOWN: the SwiGLU rows, MLA's W_UV).
 *
 * Workgroup = (token group g, active slot, rpw row tiles of 16 rows); S waves per row
 * tile. Wave (row tile r, part p) streams block pairs [p TK_NP, (p + 1) TK_NP) of the
 * tile's matrices into registers, every load issued at once. The slot's activation
 * blocks are staged once per workgroup in LDS by LDS-direct loads, [block][token][64 B]
 * (the Act block of each token, k-group kg at 16 kg).
 *
 * Tokens go in groups of four: for group g the B operand of column c is read from token
 * 4 g + c % 4, so the MFMA result holds each (row, token) pair four times and lane
 * (kg = l / 16, lr = l % 16) keeps register lr / 4: row 4 kg + lr / 4, token
 * 4 g + lr % 4 -- one useful term per lane, matrix and block, where the 16 token
 * columns of the plain layout would leave most lanes working on padding.
 *
 * Sums: part 0 folds its blocks from 0.0; part p > 0 keeps its terms in registers,
 * takes the running sums of part p - 1 through LDS after barrier p and adds its terms
 * in block order, so each sum is the sequential fold acc = acc + isum (dw dx) over
 * blocks 0 .. nb-1. The last part writes the result. */
template <int DT>
struct TkCfg {
    static constexpr int NP = DT == 4 ? 8 : 4;   /* block pairs per wave (registers) */
    static constexpr int NV = DT == 4 ? 1 : 2;   /* 16-byte loads per pair, matrix and lane */
};

/* register q of c */
__device__ __forceinline__ int pick4(const v4i &c, int q) {
    const int lo = (q & 1) ? c.y : c.x, hi = (q & 1) ? c.w : c.z;
    return (q & 2) ? hi : lo;
}

/* tile sets per XCD chunk: a workgroup of fewer than 64 rows shares the 128-byte scale
 * lines with its neighbours, so TK_CHUNK_ROWS rows stay on one XCD; from 64 rows on the
 * workgroups go round the XCDs one by one */
__host__ __device__ inline int tk_chunk(int rpw) {
    return 16 * rpw >= 64 ? 1 : TK_CHUNK_ROWS / (16 * rpw);
}

/* LDS bytes of one workgroup (qf: plus the SwiGLU rows [4 tokens][16 rpw] it quantizes) */
__host__ __device__ inline size_t tk_lds_bytes(int nbp, int nm, int np, int rpw, int S, bool qf = false) {
    const int nbp4 = (nbp + 3) & ~3;
    return (size_t)nbp * 1024 + (size_t)nbp4 * 128 + (size_t)rpw * S * nm * 2 * np * 32 + (size_t)rpw * nm * 64 * 4 +
           (qf ? (size_t)4 * 16 * rpw * 4 : 0);
}

/* TK_GATEUP_Q: gate/up whose workgroups cover whole 64-row blocks of the SwiGLU rows
 * (4 or 8 row tiles) and quantize them (NUMERICS §2) in the epilogue */
enum { TK_GATEUP = 0, TK_DOWN = 1, TK_GATEUP_Q = 2 };

/* s_waitcnt vmcnt(n) for an n known once loops are unrolled (0 <= n <= 31) */
__device__ __forceinline__ void wait_vmcnt_le(int n) {
    switch (n) {
#define HX_W(k) case k: HX_WAIT_VMCNT(k); break;
    HX_W(0) HX_W(1) HX_W(2) HX_W(3) HX_W(4) HX_W(5) HX_W(6) HX_W(7) HX_W(8) HX_W(9) HX_W(10) HX_W(11)
    HX_W(12) HX_W(13) HX_W(14) HX_W(15) HX_W(16) HX_W(17) HX_W(18) HX_W(19) HX_W(20) HX_W(21) HX_W(22)
    HX_W(23) HX_W(24) HX_W(25) HX_W(26) HX_W(27) HX_W(28) HX_W(29) HX_W(30) HX_W(31)
#undef HX_W
    default: HX_WAIT_VMCNT(0);
    }
}

template <int DT, int MODE>
__global__ __launch_bounds__(512) void k_expert_tk(MoeArgs a, int rpw, int S, int gmax, int n_slots) {
    constexpr bool DOWN = MODE == TK_DOWN, QF = MODE == TK_GATEUP_Q;
    extern __shared__ __attribute__((aligned(16))) uint8_t tk_lds[];
    /* the exp table of the SwiGLU epilogue, one entry per lane, loaded with the weights */
    const unsigned long long ev = DOWN ? 0ull : exp_table_lane();
    constexpr int NP = TkCfg<DT>::NP, NV = TkCfg<DT>::NV, NBK = 2 * NP, NM = DOWN ? 1 : 2;
    const int rows_out = DOWN ? a.D : a.F;
    const int ntile = (rows_out + 15) / 16, tpw = (ntile + rpw - 1) / rpw;
    /* workgroup i runs on XCD i % 8. Chunks of TK_CHUNK_ROWS rows of one slot are dealt
     * to the XCDs in turn and a chunk's workgroups follow each other on its XCD, so the
     * row tiles that share 128-byte lines of the scale rows meet in one L2 while every
     * XCD gets the same share of the bytes */
    const int ch = tk_chunk(rpw);   /* tile sets per chunk */
    const int cps = (tpw + ch - 1) / ch, per_chunk = ch * gmax;
    const int xcd = (int)blockIdx.x & 7, k = (int)blockIdx.x >> 3;
    const int c = xcd + 8 * (k / per_chunk), within = k % per_chunk;
    const int u = c / cps, tile = (c % cps) * ch + within / gmax, g = within % gmax;
    if (u >= n_slots || tile >= tpw) return;   /* uniform */
    int n, p0;
    QMat mat[NM];
    if (DOWN && a.head_slots) {
        n = a.T;
        p0 = u * a.T;
        mat[0] = a.table[u].down;
    } else {
        if (u >= *a.n_active) return;   /* uniform */
        const SlotDesc &sd = a.desc[u];
        n = sd.n;
        p0 = sd.p0;
        if (DOWN) {
            mat[0] = sd.w.down;
        } else {
            mat[0] = sd.w.gate;
            mat[NM - 1] = sd.w.up;
        }
    }
    if (mat[0].dtype != DT || 4 * g >= n) return;   /* uniform */
    const Act &x = DOWN ? a.mid : a.x;
    const int W = rpw * S;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rtl = wave / S, part = wave % S;
    const int lane = threadIdx.x & 63, kg = lane >> 4, lr = lane & 15;
    const int rt0 = tile * rpw + rtl;
    const bool live = rt0 < ntile;   /* uniform per wave */
    const int rt = live ? rt0 : ntile - 1;   /* a dead wave loads a live tile and discards it */
    const int nb = mat[0].nb, nbp = mat[0].nbp, npair = nbp >> 1, nbp4 = (nbp + 3) & ~3;
    const int g0 = part * NP, kb0 = 2 * g0;   /* first pair / block of this part */
    uint8_t *xs = tk_lds;                                   /* [nbp][16 tokens][64 B] */
    float *dxs = (float *)(xs + (size_t)nbp * 1024);        /* [nbp4][16 tokens] */
    int *sxs = (int *)(dxs + nbp4 * 16);                    /* [nbp4][16 tokens] */
    uint8_t *scl = (uint8_t *)(sxs + nbp4 * 16) + wave * NM * NBK * 32;   /* [NM][NBK][16 halves] */
    float *const relay0 = (float *)((uint8_t *)(sxs + nbp4 * 16) + W * NM * NBK * 32);   /* [rpw][NM][64] */
    float *relay = relay0 + rtl * NM * 64;
    /* issue order: the token rows, the weights (straight-line loads), then the
     * LDS-direct loads that need the token rows. The q loads cover token lane / 4,
     * k-group lane % 4 of a block; the d and s loads token lane % 16 of four blocks. */
    const int tq = (lane >> 2) < n ? (lane >> 2) : n - 1, tds = lr < n ? lr : n - 1;
    const int arow_q = !DOWN ? a.pair_tok[p0 + tq] : p0 + tq;
    const int arow_d = !DOWN ? a.pair_tok[p0 + tds] : p0 + tds;
    v4i w[NM][NP][NV];
    /* pairs [0, NA) go before the token rows, pairs [NA, NP) after them: the wait for the
     * token rows then leaves the later weights in flight, and each pair's MFMAs start as
     * soon as its own bytes are in (the compiler waits for each register as it is used) */
    constexpr int NA = NP / 4 > 0 ? NP / 4 : 1;
    auto load_pair = [&](int k, int dep) {
        const int gp = g0 + k < npair ? g0 + k : npair - 1;
#pragma unroll
        for (int mi = 0; mi < NM; mi++) {
            const QMat &m = mat[mi];
            if (DT == 4) {
                w[mi][k][0] = gload<v4i>(m.w + ((size_t)rt * npair + gp) * 1024 + lane * 16 + dep);
            } else {
                const uint8_t *base = m.w + ((size_t)rt * nbp + 2 * gp) * 1024 + lane * 16 + dep;
                w[mi][k][0] = gload<v4i>(base);
                w[mi][k][NV - 1] = gload<v4i>(base + 1024);
            }
        }
    };
#pragma unroll
    for (int k = 0; k < NA; k++) load_pair(k, 0);
    /* one loop for every LDS-direct load */
    {
        const int nxq = (nbp - wave + W - 1) / W, nit = nxq > NBK / 8 ? nxq : NBK / 8;
        int it = 0;
        do {   /* nit >= 1 */
            const int b = wave + it * W;
            if (b < nbp) lds_direct<16>(x.q + ((size_t)arow_q * x.nbp + b) * 64 + (lane & 3) * 16, xs + (size_t)b * 1024);
            if (4 * b < nbp4) {
                const int bb = 4 * b + kg < nbp ? 4 * b + kg : nbp - 1;
                lds_direct<4>(x.d + (size_t)arow_d * x.nbp + bb, dxs + 4 * b * 16);
                if (DT == 4) lds_direct<4>(x.s + (size_t)arow_d * x.nbp + bb, sxs + 4 * b * 16);
            }
            const int b0 = it * 8;
            if (b0 < NBK) {
                const int bg = kb0 + b0 + (lane >> 3), bs = bg < nbp ? bg : nbp - 1, h2 = (lane & 7) * 2;
#pragma unroll
                for (int mi = 0; mi < NM; mi++)
                    lds_direct<4>(mat[mi].d + (size_t)bs * mat[mi].rows_pad + rt * 16 + h2, scl + (mi * NBK + b0) * 32);
            }
        } while (++it < nit);
    }
    /* the later weights: their addresses depend on an empty volatile asm after the
     * LDS-direct loads, so no load of them can be issued before those */
    int dep = 0;
    asm volatile("" : "+v"(dep));
#pragma unroll
    for (int k = NA; k < NP; k++) load_pair(k, dep);
    HX_WAIT_VMCNT(NM * (NP - NA) * NV);   /* the token rows, scales and pairs [0, NA) */
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);    /* no weight use moves above the barrier */
    const int q = lr >> 2;                /* register of this lane's pair: row 4 kg + q */
    /* one group of 4 tokens: the MFMAs, the fold over the parts and the epilogue */
    auto group = [&](int g) {
        const int col = 4 * g + (lr & 3);     /* token of this lane's pair */
        const int colc = col < n ? col : n - 1;   /* its staged row (columns past n are discarded) */
        const v4i zero = {0, 0, 0, 0};
        const bool full = kb0 + NBK <= nb;    /* uniform */
        /* terms of local block kb (global kb0 + kb); the MFMA gives sum q x with q the
         * stored nibble (Q4), so isum = sum q x - 8 sx */
        auto terms = [&](const v4i (&wa)[NM], int kb, float (&t)[NM]) {
            const int blk = kb0 + kb;
            const v4i xq = *(const v4i *)(xs + ((size_t)blk * 16 + colc) * 64 + kg * 16);
            const float d = dxs[blk * 16 + colc];
            const int off = DT == 4 ? 8 * sxs[blk * 16 + colc] : 0;
#pragma unroll
            for (int mi = 0; mi < NM; mi++) {
                const v4i cc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[mi], xq, zero, 0, 0, 0);
                const float dw = h2f(*((const uint16_t *)(scl + (size_t)(mi * NBK + kb) * 32) + 4 * kg + q));
                t[mi] = fmul((float)(pick4(cc, q) - off), fmul(dw, d));
            }
        };
        float acc[NM];
        float tm[NBK][NM];
        auto run_part = [&](bool fold) {
#pragma unroll
            for (int k = 0; k < NP; k++) {
                /* pair k's loads are in when at most the later pairs' are outstanding */
                if (k >= NA) wait_vmcnt_le(NM * NV * (NP - 1 - k));
                v4i wv[2][NM];
#pragma unroll
                for (int mi = 0; mi < NM; mi++) {
                    if (DT == 4) {
                        unpack_q4(w[mi][k][0], wv[0][mi], wv[1][mi]);
                    } else {
                        wv[0][mi] = w[mi][k][0];
                        wv[1][mi] = w[mi][k][NV - 1];
                    }
                }
#pragma unroll
                for (int j2 = 0; j2 < 2; j2++) {
                    const int kb = 2 * k + j2;
                    if (!full && kb0 + kb >= nb) break;   /* uniform */
                    float t[NM];
                    terms(wv[j2], kb, t);
#pragma unroll
                    for (int mi = 0; mi < NM; mi++) {
                        if (fold) acc[mi] = fadd(acc[mi], t[mi]);
                        else tm[kb][mi] = t[mi];
                    }
                }
            }
        };
        if (part == 0) {
#pragma unroll
            for (int mi = 0; mi < NM; mi++) acc[mi] = 0.0f;
            run_part(true);
        } else {
            run_part(false);
        }
        for (int stage = 1; stage < S; stage++) {
            if (part == stage - 1) {
#pragma unroll
                for (int mi = 0; mi < NM; mi++) relay[mi * 64 + lane] = acc[mi];
            }
            __syncthreads();
            if (part == stage) {
#pragma unroll
                for (int mi = 0; mi < NM; mi++) acc[mi] = relay[mi * 64 + lane];
#pragma unroll
                for (int kb = 0; kb < NBK; kb++) {
                    if (!full && kb0 + kb >= nb) break;   /* uniform */
#pragma unroll
                    for (int mi = 0; mi < NM; mi++) acc[mi] = fadd(acc[mi], tm[kb][mi]);
                }
            }
            __syncthreads();   /* the relay slot is read before the next stage writes it */
        }
        const int row = rt * 16 + 4 * kg + q;
        const bool out = part == S - 1 && live && col < n;
        if (DOWN) {
            if (out && row < mat[0].rows) a.Y[(size_t)(p0 + col) * a.D + row] = canon(acc[0]);
            return;
        }
        float mv = 0.0f;
        {
            /* every lane takes the exp (the table is read across the wave); the outputs keep it */
            const float gv = canon(acc[0]), uv = canon(acc[NM - 1]);
            const float sg = fdiv(gv, fadd(1.0f, exp_glibc_f_wave(-gv, ev)));
            if (out) {
                mv = fmul(sg, uv);
                if (!QF) a.midf[(size_t)(p0 + col) * a.F + row] = mv;
            }
        }
        if constexpr (QF) {
            /* the workgroup's rows [16 rpw tile, +16 rpw) are whole blocks of F: the last
             * parts put them in LDS by (token, row), then wave j quantizes block j / 4 of
             * token 4 g + j % 4 -- the values k_quant_rows would read from midf */
            const int nr = 16 * rpw;
            float *qb = relay0 + rpw * NM * 64;   /* [4 tokens][16 rpw], after the relay slots */
            if (part == S - 1) qb[(lr & 3) * nr + rtl * 16 + 4 * kg + q] = mv;
            __syncthreads();
            if (wave < rpw) {
                const int tt = wave & 3, bb = wave >> 2, tcol = 4 * g + tt;
                if (tcol < n) quant_block_wave(qb[tt * nr + bb * 64 + lane], a.mid, p0 + tcol, (tile * nr) / 64 + bb);
            }
        }
    };
    if (DOWN) {
        /* down runs every group of the slot from the same weight registers (the
         * stage loop's last barrier orders the relay slots between groups) */
        const int ng = (n + 3) >> 2;
        for (int gi = 0; gi < ng; gi++) group(gi);
    } else {
        group(g);
    }
}

/* k_expert_tk of one dtype: workgroup shape, or W = 0 when it does not fit */
struct TkPlan {
    int rpw, S, W;
    size_t lds;
    bool qf;   /* gate/up: its workgroups can quantize the SwiGLU rows */
};

TkPlan tk_plan(const MoeArgs &a, bool down, int dt) {
    const int K = down ? a.F : a.D;
    const int nb = (K + 63) / 64, nbp = (nb + 1) & ~1, npair = nbp / 2;
    const int NP = dt == 4 ? TkCfg<4>::NP : TkCfg<3>::NP, NM = down ? 1 : 2;
    const int waves = down ? TK_WAVES_DOWN : TK_WAVES_GATEUP;
    TkPlan p;
    p.S = (npair + NP - 1) / NP;
    p.rpw = p.S < waves ? waves / p.S : 1;
    p.W = p.rpw * p.S;
    /* gate/up workgroups of 4 or 8 row tiles cover whole blocks of the SwiGLU rows: they
     * quantize them too (F a multiple of 128, so the blocks need no padding block) */
    p.qf = !down && a.mid.q && a.F % 128 == 0 && (p.rpw == 4 || p.rpw == 8) && a.mid.nbp == a.F / 64;
    p.lds = tk_lds_bytes(nbp, NM, NP, p.rpw, p.S, p.qf);
    if (p.W > 8 || p.lds > TK_LDS_MAX) p.W = 0;
    return p;
}

/* launches k_expert_tk for experts of at most 16 tokens; 0 when the shape does not fit (the
 * caller uses another kernel), 2 when the launch also quantized the SwiGLU rows. Experts of
 * both dtypes: a launch each, whose workgroups leave the other's slots alone, and for few
 * tokens only. Both products of 8 of 128 such experts a token (2048 x 768), these and the
 * chunked kernels, us: one token 32.5 / 39.6, four 43.1 / 45.5, six 52.4 / 49.6, 16 116 / 60. */
int launch_tk(const MoeArgs &a, int mode, int n_slots, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    const bool down = mode == TK_DOWN;
    const bool q4 = a.dtype_mask & (1 << 4), q8 = a.dtype_mask & (1 << 3);
    if (a.T > (q4 && q8 ? TK_MIXED_T : 16)) return 0;
    const TkPlan p4 = tk_plan(a, down, 4), p8 = tk_plan(a, down, 3);
    if ((q4 && !p4.W) || (q8 && !p8.W)) return 0;
    const bool qf = mode == TK_GATEUP && (!q4 || p4.qf) && (!q8 || p8.qf);
    const int rows = down ? a.D : a.F;
    /* gate/up: a workgroup per group of 4 tokens; down: one runs all of its slot's groups */
    const int gmax = down ? 1 : (a.T + 3) / 4;   /* tokens per slot <= T */
    auto run = [&](auto dt, const TkPlan &p, hipEvent_t e0, hipEvent_t e1) {
        constexpr int DT = decltype(dt)::value;
        const int tpw = ((rows + 15) / 16 + p.rpw - 1) / p.rpw;
        const int ch = tk_chunk(p.rpw);
        const int chunks = n_slots * ((tpw + ch - 1) / ch);
        const dim3 grid(8 * ((chunks + 7) / 8) * ch * gmax), block(64 * p.W);
#define TK_LAUNCH(MODE_) \
    hipExtLaunchKernelGGL(k_expert_tk<DT, MODE_>, grid, block, (uint32_t)p.lds, st, e0, e1, 0u, a, p.rpw, p.S, gmax, n_slots)
        if (down) TK_LAUNCH(TK_DOWN);
        else if (qf) TK_LAUNCH(TK_GATEUP_Q);
        else TK_LAUNCH(TK_GATEUP);
#undef TK_LAUNCH
    };
    if (q4) run(std::integral_constant<int, 4>{}, p4, ev0, q8 ? nullptr : ev1);
    if (q8) run(std::integral_constant<int, 3>{}, p8, q4 ? nullptr : ev0, ev1);
    return qf ? 2 : 1;
}

/* Split-K products of experts whose K does not fit k_expert_tk, for the few tokens at which
 * the chunked kernels (k_mm.hip) have too few workgroups: those walk K in order, so that a
 * launch takes the latency of its K however little work it has, while here each wave loads
 * its part of K at once. Bound by the weight bytes in flight. Measured, these / the chunked
 * ones, us a launch (in brackets the chunked workgroups of a dtype): down of K = 6144 to 2048
 * rows, two Q4 experts a token, 1 token (64) 10.3 / 18.2, 3 (192) 15.4 / 19.2, 4 (256) 22.0 /
 * 19.3, Q8 1 token 11.2 / 20.1; gate/up and the quantization of its rows, 768 rows of K =
 * 8192, 1 token (48) 21.8 / 39.9, 2 (96) 35.8 / 40.6, of K = 6144, 1 token (96) 32.8 / 32.4. */
template <int DT>
__global__ __launch_bounds__(512) void k_expert_gateup_sk(MoeArgs a, int ntok) {
    extern __shared__ float P[];
    const int ntile = a.F / 16;
    const int u = (int)blockIdx.x / ntile, rt = (int)blockIdx.x % ntile;
    if (u >= *a.n_active) return;   /* uniform */
    const SlotDesc &sd = a.desc[u];
    const int n = sd.n, p0 = sd.p0;
    const QMat ms[2] = {sd.w.gate, sd.w.up};
    if (ms[0].dtype != DT) return;   /* the launcher runs one instantiation per dtype */
    const int W = blockDim.x >> 6, wave = threadIdx.x >> 6, tid = threadIdx.x;
    int q0, q1;
    wave_pairs(ms[0].nbp >> 1, W, wave, q0, q1);
    const int pstride = ms[0].nb * ntok * 16;
    const int *ptok = a.pair_tok + p0;
    for (int t0 = 0; t0 < n; t0 += ntok) {
        tile_terms<DT, 2>(ms, rt, a.x, t0, n, ntok, [ptok](int t) { return ptok[t]; }, q0, q1, P, pstride);
        __syncthreads();
        const int nc = n - t0 < ntok ? n - t0 : ntok;
        for (int f = tid; f < nc * 16; f += blockDim.x) {
            const float gv = canon(fold_terms(P, ms[0].nb, ntok, f));
            const float uv = canon(fold_terms(P + pstride, ms[0].nb, ntok, f));
            const float sg = fdiv(gv, fadd(1.0f, exp_glibc_f(-gv)));
            a.midf[(size_t)(p0 + t0 + (f >> 4)) * a.F + rt * 16 + (f & 15)] = fmul(sg, uv);
        }
        __syncthreads();
    }
}

template <int DT>
__global__ __launch_bounds__(512) void k_expert_down_sk(MoeArgs a, int ntok) {
    extern __shared__ float P[];
    const int ntile = (a.D + 15) / 16;
    const int u = (int)blockIdx.x / ntile, rt = (int)blockIdx.x % ntile;
    if (u >= *a.n_active) return;   /* uniform */
    const SlotDesc &sd = a.desc[u];
    const int n = sd.n, p0 = sd.p0;
    const QMat m = sd.w.down;
    if (m.dtype != DT) return;
    const int W = blockDim.x >> 6, wave = threadIdx.x >> 6, tid = threadIdx.x;
    int q0, q1;
    wave_pairs(m.nbp >> 1, W, wave, q0, q1);
    for (int t0 = 0; t0 < n; t0 += ntok) {
        tile_terms<DT, 1>(&m, rt, a.mid, t0, n, ntok, [p0](int t) { return p0 + t; }, q0, q1, P, 0);
        __syncthreads();
        const int nc = n - t0 < ntok ? n - t0 : ntok;
        for (int f = tid; f < nc * 16; f += blockDim.x) {
            const int row = rt * 16 + (f & 15);
            if (row < m.rows) a.Y[(size_t)(p0 + t0 + (f >> 4)) * a.D + row] = canon(fold_terms(P, m.nb, ntok, f));
        }
        __syncthreads();
    }
}

/* ------------------------------------------------------------ float matrices (dot16) */

/* y = dot16(w_r, x_t) (NUMERICS §1/§3; quant.c:352-376): 16 lanes per (row, token),
 * lane j sums elements j, j+16, ... in order, then the 8/4/2/1 tree. Any shape. */
template <int WDT>
__global__ __launch_bounds__(256) void k_fgemv_any(const void *__restrict__ W, int rows, int cols,
                                                  const float *__restrict__ X, int ldx, int T, float *__restrict__ Y,
                                                  int ldy) {
    const int64_t pair = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 4;
    const int j = threadIdx.x & 15;
    const bool live = pair < (int64_t)rows * T;
    const int r = live ? (int)(pair % rows) : 0, t = live ? (int)(pair / rows) : 0;
    float L = 0.0f;
    if (live) {
        const float *x = X + (size_t)t * ldx;
        for (int i = j; i < cols; i += 16) {
            float w;
            if (WDT == 0) w = ((const float *)W)[(size_t)r * cols + i];
            else if (WDT == 1) w = h2f(((const uint16_t *)W)[(size_t)r * cols + i]);
            else w = __uint_as_float((uint32_t)((const uint16_t *)W)[(size_t)r * cols + i] << 16);
            L = fadd(L, fmul(w, x[i]));
        }
    }
#pragma unroll
    for (int s = 8; s >= 1; s >>= 1) L = fadd(L, __shfl_down(L, s, 16));
    if (live && j == 0) Y[(size_t)t * ldy + r] = canon(L);
}

/* The same products for cols % 4 == 0 and ldx % 4 == 0: a workgroup computes 4 rows x 4
 * tokens; the rows of W and X go to LDS in chunks of 2048 columns, each thread issuing
 * all its loads of a chunk at once, and the 16 lanes of each (row, token) then run their
 * sums from LDS (chunk boundaries are multiples of 16, so lane j keeps its elements). */
constexpr int FG_R = 4, FG_T = 4, FG_CH = 2048;
constexpr int FG_PER = (FG_R + FG_T) * FG_CH / 4 / 256;   /* float4 loads per thread per chunk */

template <int WDT>
__device__ __forceinline__ float4 fg_w4(const void *W, size_t idx) {
    if (WDT == 0) return *(const float4 *)((const float *)W + idx);
    const uint2 u = *(const uint2 *)((const uint16_t *)W + idx);
    float4 v;
    if (WDT == 1) {
        v.x = h2f((uint16_t)(u.x & 0xffff)); v.y = h2f((uint16_t)(u.x >> 16));
        v.z = h2f((uint16_t)(u.y & 0xffff)); v.w = h2f((uint16_t)(u.y >> 16));
    } else {
        v.x = __uint_as_float(u.x << 16); v.y = __uint_as_float(u.x & 0xffff0000u);
        v.z = __uint_as_float(u.y << 16); v.w = __uint_as_float(u.y & 0xffff0000u);
    }
    return v;
}

template <int WDT>
__global__ __launch_bounds__(256) void k_fgemv(const void *__restrict__ W, int rows, int cols,
                                              const float *__restrict__ X, int ldx, int T, float *__restrict__ Y,
                                              int ldy) {
    __shared__ float buf[FG_R + FG_T][FG_CH];
    const int nrb = (rows + FG_R - 1) / FG_R;
    const int rb = (int)blockIdx.x % nrb, tb = (int)blockIdx.x / nrb;
    const int tid = threadIdx.x, pr = tid >> 4, j = tid & 15;
    const int rr = pr % FG_R, tt = pr / FG_R;
    const int r = rb * FG_R + rr, t = tb * FG_T + tt;
    float L = 0.0f;
    for (int c0 = 0; c0 < cols; c0 += FG_CH) {
        const int n = cols - c0 < FG_CH ? cols - c0 : FG_CH;
        if (c0) __syncthreads();
        float4 v[FG_PER];
        /* load u: row q = u / 2 of the stage (rows of W first, then rows of X), float4
         * column tid + 256 (u % 2); columns past the chunk read column 0 and are unused */
#pragma unroll
        for (int u = 0; u < FG_PER; u++) {
            const int q = u >> 1;
            int c4 = (tid + 256 * (u & 1)) * 4;
            c4 = c4 < n ? c4 : 0;
            if (q < FG_R) {
                const int rq = rb * FG_R + q < rows ? rb * FG_R + q : rows - 1;
                v[u] = fg_w4<WDT>(W, (size_t)rq * cols + c0 + c4);
            } else {
                const int tq = tb * FG_T + (q - FG_R) < T ? tb * FG_T + (q - FG_R) : T - 1;
                v[u] = *(const float4 *)(X + (size_t)tq * ldx + c0 + c4);
            }
        }
#pragma unroll
        for (int u = 0; u < FG_PER; u++)
            *(float4 *)&buf[u >> 1][(tid + 256 * (u & 1)) * 4] = v[u];
        __syncthreads();
        const float *wr = buf[rr], *xr = buf[FG_R + tt];
        int i = j;
        for (; i + 112 < n; i += 128) {
            float a[8], b[8];
#pragma unroll
            for (int u = 0; u < 8; u++) { a[u] = wr[i + 16 * u]; b[u] = xr[i + 16 * u]; }
#pragma unroll
            for (int u = 0; u < 8; u++) L = fadd(L, fmul(a[u], b[u]));
        }
        for (; i < n; i += 16) L = fadd(L, fmul(wr[i], xr[i]));
    }
#pragma unroll
    for (int s = 8; s >= 1; s >>= 1) L = fadd(L, __shfl_down(L, s, 16));
    if (r < rows && t < T && j == 0) Y[(size_t)t * ldy + r] = canon(L);
}

} // namespace

/* ------------------------------------------------------------ launchers */

namespace hxl {

void repack(const uint8_t *src_dev, int r0, int count, const QMat &m, hipStream_t st) {
    const int64_t n = (int64_t)count * m.nbp;
    if (!n) return;
    const int blocks = (int)((n + 255) / 256);
    if (m.dtype == 3) k_repack_q8<<<blocks, 256, 0, st>>>(src_dev, r0, count, m.rows, m.nb, m, (uint8_t *)m.w, (uint16_t *)m.d);
    else k_repack_q4<<<blocks, 256, 0, st>>>(src_dev, r0, count, m.rows, m.nb, m, (uint8_t *)m.w, (uint16_t *)m.d);
}

void quant_rows(const float *x, int64_t ldx, int T, int nb, const Act &a, hipStream_t st) {
    const int64_t waves = (int64_t)T * a.nbp;
    if (!waves) return;
    k_quant_rows<<<(int)((waves + 3) / 4), 256, 0, st>>>(x, ldx, T, nb, a);
}

/* waves per split-K workgroup for npair block pairs */
static int sk_waves(int npair) {
    const int w = (npair + SK_MAXP - 1) / SK_MAXP;
    return w < 1 ? 1 : (w > 8 ? 8 : w);
}

/* tokens per split-K token tile: the terms of NM matrices of nb blocks fit SK_LDS */
static int sk_ntok(int T, int NM, int nb) {
    int n = T < 16 ? T : 16;
    const int fit = (SK_LDS - SK_DUMMY) / (NM * nb * 64);
    n = n < fit ? n : fit;
    return n < 1 ? 1 : n;
}

/* dense product through the split-K kernel: one launch per run of consecutive segments of
 * one dtype */
static void gemm_sk(const GemmArgs &in, hipStream_t st) {
    for (int s0 = 0; s0 < in.nseg;) {
        int s1 = s0 + 1;
        while (s1 < in.nseg && in.seg[s1].m.dtype == in.seg[s0].m.dtype && in.seg[s1].m.nb == in.seg[s0].m.nb) s1++;
        GemmArgs g = in;
        g.nseg = s1 - s0;
        int wg = 0;
        for (int s = 0; s < g.nseg; s++) {
            g.seg[s] = in.seg[s0 + s];
            g.seg[s].wg0 = wg;
            wg += g.seg[s].m.rows_pad / 16;
        }
        const QMat &m = g.seg[0].m;
        const int ntok = sk_ntok(in.T, 1, m.nb);
        const int threads = 64 * sk_waves(m.nbp / 2);
        const size_t lds = (size_t)m.nb * ntok * 64 + SK_DUMMY;
        if (wg) {
            if (m.dtype == 4) k_gemm_sk<4><<<wg, threads, lds, st>>>(g, ntok);
            else k_gemm_sk<3><<<wg, threads, lds, st>>>(g, ntok);
        }
        s0 = s1;
    }
}

void gemm(const GemmArgs &in, hipStream_t st) {
    bool few = in.T <= 16;   /* k_gemm_sk's terms of at least one token fit its LDS */
    for (int s = 0; s < in.nseg; s++) few = few && (size_t)in.seg[s].m.nb * 64 <= (size_t)(SK_LDS - SK_DUMMY);
    if (few) gemm_sk(in, st);
    else mm_dense(in, st);
}

/* few tokens whose chunked product (k_mm.hip) would be fewer than `least` workgroups of each
 * dtype: the split-K kernels of the experts */
static bool few_workgroups(const MoeArgs &a, int n_slots, int row_groups, int least) {
    const bool both = (a.dtype_mask & (1 << 4)) && (a.dtype_mask & (1 << 3));
    return a.T <= SK_T && n_slots * row_groups < (both ? 2 : 1) * least;
}

/* gate/up; true when the launch also quantized the SwiGLU rows into a.mid. ev0 / ev1
 * (optional) are recorded by the dispatch itself: ev0 at the start of the first launch, ev1
 * at the end of the last. */
bool expert_gateup(const MoeArgs &a, int n_slots, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    if (n_slots <= 0) return false;
    if (const int r = launch_tk(a, TK_GATEUP, n_slots, st, ev0, ev1)) return r == 2;
    if (!few_workgroups(a, n_slots, a.F / 64, SK_WGS_GATEUP)) {
        mm_gateup(a, n_slots, st, ev0, ev1);
        return true;
    }
    const int nb = (a.D + 63) / 64, ntok = sk_ntok(a.T, 2, nb), threads = 64 * sk_waves((nb + 1) / 2);
    const uint32_t lds = (uint32_t)2 * nb * ntok * 64 + SK_DUMMY;
    const dim3 grid(n_slots * (a.F / 16));
    const bool q4 = a.dtype_mask & (1 << 4), q8 = a.dtype_mask & (1 << 3);
    if (q4) hipExtLaunchKernelGGL(k_expert_gateup_sk<4>, grid, dim3(threads), lds, st, ev0, q8 ? nullptr : ev1, 0u, a, ntok);
    if (q8) hipExtLaunchKernelGGL(k_expert_gateup_sk<3>, grid, dim3(threads), lds, st, q4 ? nullptr : ev0, ev1, 0u, a, ntok);
    return false;
}

/* NUMERICS §2 of the SwiGLU rows of all T * top_k pairs (unless the gate/up launch did
 * it: mid_done), then the down projections */
void expert_down(const MoeArgs &a, int n_slots, hipStream_t st, bool mid_done) {
    if (n_slots <= 0) return;
    if (!mid_done) quant_rows(a.midf, a.F, a.P, a.F / 64, a.mid, st);
    expert_down_q(a, n_slots, st);
}

void expert_down_q(const MoeArgs &a, int n_slots, hipStream_t st) {
    if (n_slots <= 0) return;
    if (launch_tk(a, TK_DOWN, n_slots, st, nullptr, nullptr)) return;
    if (a.head_slots || !few_workgroups(a, n_slots, (a.D + 63) / 64, SK_WGS_DOWN)) {
        mm_down(a, n_slots, st);
        return;
    }
    const int nb = a.F / 64, ntok = sk_ntok(a.T, 1, nb), threads = 64 * sk_waves((nb + 1) / 2);
    const uint32_t lds = (uint32_t)nb * ntok * 64 + SK_DUMMY;
    const dim3 grid(n_slots * ((a.D + 15) / 16));
    if (a.dtype_mask & (1 << 4)) k_expert_down_sk<4><<<grid, threads, lds, st>>>(a, ntok);
    if (a.dtype_mask & (1 << 3)) k_expert_down_sk<3><<<grid, threads, lds, st>>>(a, ntok);
}

void fgemv(int dtype, const void *W, int rows, int cols, const float *X, int ldx, int T, float *Y, int ldy, hipStream_t st) {
    if (rows <= 0 || T <= 0) return;
    if (cols % 4 == 0 && ldx % 4 == 0) {
        const int grid = ((rows + FG_R - 1) / FG_R) * ((T + FG_T - 1) / FG_T);
        if (dtype == 0) k_fgemv<0><<<grid, 256, 0, st>>>(W, rows, cols, X, ldx, T, Y, ldy);
        else if (dtype == 1) k_fgemv<1><<<grid, 256, 0, st>>>(W, rows, cols, X, ldx, T, Y, ldy);
        else k_fgemv<2><<<grid, 256, 0, st>>>(W, rows, cols, X, ldx, T, Y, ldy);
        return;
    }
    const int64_t threads = (int64_t)rows * T * 16;
    const int blocks = (int)((threads + 255) / 256);
    if (dtype == 0) k_fgemv_any<0><<<blocks, 256, 0, st>>>(W, rows, cols, X, ldx, T, Y, ldy);
    else if (dtype == 1) k_fgemv_any<1><<<blocks, 256, 0, st>>>(W, rows, cols, X, ldx, T, Y, ldy);
    else k_fgemv_any<2><<<blocks, 256, 0, st>>>(W, rows, cols, X, ldx, T, Y, ldy);
}

} // namespace hxl
