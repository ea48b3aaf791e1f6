/*
 * k_mm.hip — int8 products of more tokens than the few-token kernels of k_gemm.hip take:
 * dense matrices (prefill chunks, trees), the routed experts' gate/up and down, MLA's
 * per-head W_UV, on gfx950.
 *
 * Reference semantics: NUMERICS §2-3 (engine/src/quant.c:325-427). Every (token, row)
 * output is one lane's fold acc = acc + (float)isum_g * (dw_g * dx_g) over the blocks g of
 * its row in ascending order; isum_g is the exact int32 block sum from
 * v_mfma_i32_16x16x64_i8. Which other tokens share a tile cannot change any output.
 */
#include "hx_device.h"
#include "hx_launch.h"
#include <hip/hip_ext.h>

using namespace hxd;

namespace {

/* One workgroup of four waves: wave w takes the 16-row tile 4 rg + w of one matrix (gate/up:
 * of both), all waves the same NT tiles of 16 tokens; K is walked in chunks of MM_CB blocks,
 * double-buffered. Of chunk c + 1 the tokens' blocks, their scales and the weights' scales go
 * to LDS by LDS-direct loads and the weights to registers while chunk c is folded: one
 * barrier a chunk, 8 blocks of every wave's rows in flight.
 *
 * What bounds it: the weight bytes for the experts (a slot's tokens share one pass over
 * them), the fold's four f32 operations per term and the first chunk's latency for the dense
 * products. Before, a wave kept 4 block pairs and its terms went through LDS to one thread
 * per output (dense, gate/up), or a wave walked all of K one pair ahead (wide K). Measured,
 * before -> now, us a launch: 2048-wide model at T = 512 gate/up 210 (+ 12 for the
 * quantization of its rows, now here) -> 82, down 152 -> 49, QKV and o-projection 80 -> 25
 * each; at T = 85 72 + 5 -> 40, 45 -> 22, 19.5 -> 11.5; 7168-wide model at T = 301
 * gate/up 4252 -> 483, down 792 -> 272, dense 82 a launch
 * on average against 190; at T = 9 (too wide for the few-token kernel) gate/up 366 -> 143. */
constexpr int MM_RT = 4;       /* row tiles (waves) per workgroup: 64 rows, one block of a product's K */
constexpr int MM_CB = 8;       /* blocks per chunk */
constexpr float MAGIC = 12582912.0f;     /* 1.5 * 2^23 */
constexpr int MAGIC_BITS = 0x4B400000;

/* LDS of one stage: blocks [MM_CB][NT][16 tokens as the MFMA reads them: 1 KiB], token
 * scales [16 NT][MM_CB], weight scales [NM][MM_CB][64 rows] */
template <int NM, int NT> struct MmStage {
    uint8_t q[MM_CB][NT][1024];
    float d[16 * NT][MM_CB];
    uint16_t w[NM][MM_CB][64];
};

enum { MM_DENSE = 0, MM_GATEUP = 1, MM_DOWN = 2 };

template <int DT, int NM>
struct MmTile {
    static constexpr int NW = DT == 4 ? MM_CB / 2 : MM_CB;   /* 16-byte weight loads per chunk */
    v4i w[NM][NW];

    __device__ __forceinline__ void load_w(const QMat *m, int rt, int c) {
        const unsigned lo = (threadIdx.x & 63) * 16;
#pragma unroll
        for (int mi = 0; mi < NM; mi++)
#pragma unroll
            for (int k = 0; k < NW; k++) {
                const int per = DT == 4 ? m[mi].nbp >> 1 : m[mi].nbp;   /* tiles of a row tile */
                int i = c * NW + k;
                i = i < per ? i : per - 1;
                w[mi][k] = gload<v4i>(m[mi].w + ((size_t)rt * per + i) * 1024 + lo);
            }
    }
};

/* what a lane stages: byte offsets of its tokens' blocks and scales and of its weight
 * scales, so that a chunk's addresses are scalar bases plus these */
template <int NT> struct MmLane {
    unsigned q, d[(NT + 1) / 2], w;
};

template <int NM, int NT>
__device__ __forceinline__ void mm_stage(MmStage<NM, NT> &__restrict__ s, const QMat *m, const Act &x, const MmLane<NT> &ln,
                                         int c) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nb = m[0].nb, b0 = c * MM_CB, left = nb - b0;   /* blocks from the chunk's first on */
    constexpr int PER = MM_CB * NT / MM_RT;    /* block loads of one wave */
    const int tt = wave % NT, j0 = (wave / NT) * PER;
    const uint8_t *xq = (const uint8_t *)x.q + (size_t)b0 * 64;
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int j = j0 + k, jc = j < left ? j : left - 1;
        lds_direct<16>(xq + jc * 64 + ln.q, s.q[j][tt]);
    }
    {
        const int j = lane & 7, jc = j < left ? j : left - 1;
        const uint8_t *xd = (const uint8_t *)(x.d + b0);
#pragma unroll
        for (int k = 0; k < (NT + 1) / 2; k++) {
            const int i = wave + MM_RT * k;
            if (i < 2 * NT) lds_direct<4>(xd + (ln.d[k] + 4u * jc), s.d[8 * i]);
        }
    }
    /* two blocks of 64 rows a load */
    const unsigned rb = 2u * m[0].rows_pad;
#pragma unroll
    for (int k = 0; k < NM; k++) {
        const int i = wave + MM_RT * k, mi = i / (MM_CB / 2), j = 2 * (i % (MM_CB / 2));
        const uint8_t *wd = (const uint8_t *)(NM == 2 && mi ? m[NM - 1].d : m[0].d) + (size_t)b0 * rb;
        const int jl = j + (lane >> 5), jc = jl < left ? jl : left - 1;
        lds_direct<4>(wd + (ln.w + (unsigned)jc * rb), s.w[mi][j]);
    }
}

/* folds the chunk's blocks [0, nblk) into acc (nblk <= MM_CB; CHECK: fewer are possible) */
template <int DT, int NM, int NT, bool CHECK>
__device__ __forceinline__ void mm_fold(const MmStage<NM, NT> &__restrict__ s, const MmTile<DT, NM> &t, int nblk,
                                        float (&acc)[NM][NT][4]) {
    const int lane = threadIdx.x & 63, kg = lane >> 4, lr = lane & 15, wave = threadIdx.x >> 6;
    const v4i magic = {MAGIC_BITS, MAGIC_BITS, MAGIC_BITS, MAGIC_BITS};
    const v4i m8 = {(int)0xF8F8F8F8, (int)0xF8F8F8F8, (int)0xF8F8F8F8, (int)0xF8F8F8F8};
    float4 dx[NT];
#pragma unroll
    for (int j = 0; j < MM_CB; j++) {
        if (CHECK && j >= nblk) break;   /* uniform */
        v4i c[NM][NT];
#pragma unroll
        for (int tt = 0; tt < NT; tt++) {
            if (j % 4 == 0) dx[tt] = *(const float4 *)&s.d[tt * 16 + lr][j];
            const v4i x = *(const v4i *)&s.q[j][tt][lane * 16];
            /* the block sum comes out as the float MAGIC + isum (|isum| < 2^21, so exact):
             * the accumulator starts from MAGIC's bits. Q4 stores nibbles q + 8: a product
             * with -8 everywhere takes 8 sum(x) off first. */
            const v4i z = DT == 4 ? __builtin_amdgcn_mfma_i32_16x16x64_i8(m8, x, magic, 0, 0, 0) : magic;
#pragma unroll
            for (int mi = 0; mi < NM; mi++) {
                v4i wa;
                if (DT == 4) {
                    const v4i raw = t.w[mi][j >> 1];
                    const int lo = j & 1 ? raw.z : raw.x, hi = j & 1 ? raw.w : raw.y;
                    wa.x = lo & 0x0F0F0F0F; wa.y = hi & 0x0F0F0F0F; wa.z = (lo >> 4) & 0x0F0F0F0F; wa.w = (hi >> 4) & 0x0F0F0F0F;
                } else {
                    wa = t.w[mi][DT == 4 ? 0 : j];
                }
                c[mi][tt] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa, x, z, 0, 0, 0);
            }
        }
#pragma unroll
        for (int mi = 0; mi < NM; mi++) {
            const uint2 sw = *(const uint2 *)&s.w[mi][j][wave * 16 + 4 * kg];
            const float dw[4] = {h2f((uint16_t)(sw.x & 0xffff)), h2f((uint16_t)(sw.x >> 16)),
                                 h2f((uint16_t)(sw.y & 0xffff)), h2f((uint16_t)(sw.y >> 16))};
#pragma unroll
            for (int tt = 0; tt < NT; tt++) {
                const float d = j % 4 == 0 ? dx[tt].x : j % 4 == 1 ? dx[tt].y : j % 4 == 2 ? dx[tt].z : dx[tt].w;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    acc[mi][tt][i] = fadd(acc[mi][tt][i], fmul(fsub(__int_as_float(c[mi][tt][i]), MAGIC), fmul(dw[i], d)));
            }
        }
    }
}

/* stages chunk c + 1 into nxt and folds chunk c from cur. The two never alias (restrict): the
 * compiler otherwise waits for the LDS-direct loads in flight before every LDS read. */
template <int DT, int NM, int NT>
__device__ __forceinline__ void mm_step(MmStage<NM, NT> *__restrict__ nxt, const MmStage<NM, NT> *__restrict__ cur,
                                        MmTile<DT, NM> (&t)[2], const QMat *m, const Act &x, const MmLane<NT> &ln,
                                        int rt, int c, float (&acc)[NM][NT][4]) {
    mm_stage<NM, NT>(*nxt, m, x, ln, c + 1);
    t[1].load_w(m, rt, c + 1);
    mm_fold<DT, NM, NT, false>(*cur, t[0], MM_CB, acc);
    t[0] = t[1];
}

/* the products of one workgroup for tokens t0 .. t0 + 16 NT - 1 of n (row_of(t): token t's
 * activation row; tokens past n repeat the last one and are discarded by the caller). On
 * return every wave is past its last read of the stages. */
template <int DT, int NM, int NT, typename RowOf>
__device__ __forceinline__ void mm_run(MmStage<NM, NT> (&st)[2], const QMat *m, const Act &x, int rg, int t0, int n,
                                       RowOf row_of, float (&acc)[NM][NT][4]) {
    const int lane = threadIdx.x & 63, lr = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int ntile = m[0].rows_pad >> 4, nb = m[0].nb;
    int rt = rg * MM_RT + wave;
    rt = rt < ntile ? rt : ntile - 1;       /* a dead wave repeats the last tile */
    auto clampt = [&](int t) { return t < n ? t : n - 1; };
    MmLane<NT> ln;
    ln.q = (unsigned)row_of(clampt(t0 + (wave % NT) * 16 + lr)) * (unsigned)x.nbp * 64u + (lane >> 4) * 16;
#pragma unroll
    for (int k = 0; k < (NT + 1) / 2; k++)
        ln.d[k] = (unsigned)row_of(clampt(t0 + (wave + MM_RT * k) * 8 + (lane >> 3))) * (unsigned)x.nbp * 4u;
    {
        const int r = rg * MM_RT * 16 + 2 * (lane & 31);
        ln.w = 2u * (r < m[0].rows_pad ? r : m[0].rows_pad - 2);
    }
#pragma unroll
    for (int mi = 0; mi < NM; mi++)
#pragma unroll
        for (int tt = 0; tt < NT; tt++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[mi][tt][i] = 0.0f;
    const int nc = (nb + MM_CB - 1) / MM_CB;
    MmTile<DT, NM> t[2];
    mm_stage<NM, NT>(st[0], m, x, ln, 0);
    t[0].load_w(m, rt, 0);
    HX_WAIT_VMCNT(0);
    __syncthreads();
    int c = 0;
    for (; c + 1 < nc; c++) {
        /* every chunk but the last is whole */
        mm_step<DT, NM, NT>(&st[(c + 1) & 1], &st[c & 1], t, m, x, ln, rt, c, acc);
        HX_WAIT_VMCNT(0);   /* this wave's share of the next stage is in */
        __syncthreads();
    }
    mm_fold<DT, NM, NT, true>(st[c & 1], t[0], nb - c * MM_CB, acc);
    __syncthreads();
}

template <int DT, int NT>
__global__ __launch_bounds__(256, 2) void k_mm_dense(GemmArgs a, int wgr) {
    __shared__ __attribute__((aligned(16))) MmStage<1, NT> st[2];
    /* workgroup b: row group b % wgr, token group b / wgr; wgr is a multiple of 8, so the
     * token groups of a row group run on one XCD and read its weights from that L2 */
    const int rw = (int)blockIdx.x % wgr, t0 = ((int)blockIdx.x / wgr) * 16 * NT;
    int s = 0;
    while (s + 1 < a.nseg && rw >= a.seg[s + 1].wg0) s++;
    const GemmSeg &sg = a.seg[s];
    const QMat m = sg.m;
    const int rg = rw - sg.wg0;
    if (rg * MM_RT * 16 >= m.rows_pad || t0 >= a.T) return;   /* uniform */
    Act x = a.a;   /* from token t0 on, so that a lane's 32-bit offsets hold for any T */
    x.q += (size_t)t0 * x.nbp * 64;
    x.d += (size_t)t0 * x.nbp;
    float acc[1][NT][4];
    mm_run<DT, 1, NT>(st, &m, x, rg, 0, a.T - t0, [](int t) { return t; }, acc);
    const int lane = threadIdx.x & 63, kg = lane >> 4, lr = lane & 15, wave = threadIdx.x >> 6;
    const int row = (rg * MM_RT + wave) * 16 + 4 * kg;
    const bool vec = ((sg.ldy & 3) | (int)((uintptr_t)sg.Y & 15)) == 0;
#pragma unroll
    for (int tt = 0; tt < NT; tt++) {
        const int t = t0 + tt * 16 + lr;
        if (t >= a.T || row >= m.rows) continue;
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            y[i] = canon(acc[0][tt][i]);
            if (sg.scale_on) y[i] = canon(fmul(sg.scale, y[i]));
        }
        float *dst = sg.Y + (size_t)t * sg.ldy + row;
        if (vec && row + 4 <= m.rows) {
            *(float4 *)dst = make_float4(y[0], y[1], y[2], y[3]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (row + i < m.rows) dst[i] = y[i];
        }
    }
}

/* Item `item` of the routed products: the items are the active slots' passes of G tokens, slot
 * after slot, so that a slot with many tokens is as many workgroups as it has passes. Returns
 * false past the last item; uniform over the wave. */
__device__ __forceinline__ bool mm_item(const MoeArgs &a, int item, int G, int &u, int &t0) {
    const int lane = threadIdx.x & 63, na = *a.n_active;
    for (int u0 = 0; u0 < na; u0 += 64) {
        const int cnt = u0 + lane < na ? (a.u_n[u0 + lane] + G - 1) / G : 0;
        const int inc = wave_scan_incl(cnt), total = __builtin_amdgcn_readlane(inc, 63);
        if (item < total) {
            const int l = __ffsll((unsigned long long)__ballot(inc > item)) - 1;
            u = u0 + l;
            t0 = (item - __builtin_amdgcn_readlane(inc - cnt, l)) * G;
            return true;
        }
        item -= total;
    }
    return false;
}

/* gate/up of 64 rows of one active expert (one block of the down product's K) for its n
 * tokens t0 .. t0 + 15 (an item): mid = silu(g) * u (NUMERICS §4, quant.c:644-649), then
 * NUMERICS §2 of the block, straight into the down product's activations. */
template <int DT>
__global__ __launch_bounds__(256, 2) void k_mm_gateup(MoeArgs a) {
    constexpr int NT = 1;
    __shared__ __attribute__((aligned(16))) MmStage<2, NT> st[2];
    __shared__ unsigned long long tab[32];
    const int nrg = a.F / 64;
    const int rg = (int)blockIdx.x % nrg;
    int u, t0;
    if (!mm_item(a, (int)blockIdx.x / nrg, 16 * NT, u, t0)) return;   /* uniform */
    const SlotDesc &sd = a.desc[u];
    const int n = sd.n, p0 = sd.p0;
    if (sd.w.gate.dtype != DT) return;   /* the launcher runs one instantiation per dtype */
    const QMat m[2] = {sd.w.gate, sd.w.up};
    exp_table_to_lds(tab);
    const int lane = threadIdx.x & 63, kg = lane >> 4, lr = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int *ptok = a.pair_tok + p0;
    float *v = (float *)&st[0];           /* [16 NT tokens][64 rows + 1] */
    static_assert(sizeof(MmStage<2, NT>) >= sizeof(float) * 16 * NT * 65, "SwiGLU rows fit a stage");
    float acc[2][NT][4];
    mm_run<DT, 2, NT>(st, m, a.x, rg, t0, n, [ptok](int t) { return ptok[t]; }, acc);
#pragma unroll
    for (int tt = 0; tt < NT; tt++) {
        if (t0 + tt * 16 >= n) break;   /* uniform */
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float gv = canon(acc[0][tt][i]), uv = canon(acc[1][tt][i]);
            const float sg = fdiv(gv, fadd(1.0f, exp_glibc_f(-gv, tab)));
            v[(tt * 16 + lr) * 65 + wave * 16 + 4 * kg + i] = fmul(sg, uv);
        }
    }
    __syncthreads();
    for (int t = wave; t < 16 * NT && t0 + t < n; t += MM_RT)   /* uniform per wave */
        quant_block_wave(v[t * 65 + lane], a.mid, p0 + t0 + t, rg);
}

/* down projection of 64 rows of one active expert (or one head's W_UV) for its n pairs */
template <int DT, int NT>
__global__ __launch_bounds__(256, 2) void k_mm_down(MoeArgs a) {
    __shared__ __attribute__((aligned(16))) MmStage<1, NT> st[2];
    const int nrg = (a.D + 63) / 64;
    const int rg = (int)blockIdx.x % nrg;
    int u, t0, n, p0;
    QMat m;
    if (a.head_slots) {
        const int ng = (a.T + 16 * NT - 1) / (16 * NT), item = (int)blockIdx.x / nrg;
        u = item / ng;
        t0 = (item % ng) * 16 * NT;
        n = a.T;
        p0 = u * a.T;
        m = a.table[u].down;
    } else {
        if (!mm_item(a, (int)blockIdx.x / nrg, 16 * NT, u, t0)) return;   /* uniform */
        const SlotDesc &sd = a.desc[u];
        n = sd.n;
        p0 = sd.p0;
        m = sd.w.down;
    }
    if (m.dtype != DT || rg * 64 >= m.rows_pad) return;   /* uniform */
    const int lane = threadIdx.x & 63, kg = lane >> 4, lr = lane & 15, wave = threadIdx.x >> 6;
    const int row = (rg * MM_RT + wave) * 16 + 4 * kg;
    const bool vec = ((a.D & 3) | (int)((uintptr_t)a.Y & 15)) == 0;
    float acc[1][NT][4];
    mm_run<DT, 1, NT>(st, &m, a.mid, rg, t0, n, [p0](int t) { return p0 + t; }, acc);
#pragma unroll
    for (int tt = 0; tt < NT; tt++) {
        const int t = t0 + tt * 16 + lr;
        if (t >= n || row >= m.rows) continue;
        float *dst = a.Y + (size_t)(p0 + t) * a.D + row;
        if (vec && row + 4 <= m.rows) {
            *(float4 *)dst = make_float4(canon(acc[0][tt][0]), canon(acc[0][tt][1]), canon(acc[0][tt][2]), canon(acc[0][tt][3]));
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (row + i < m.rows) dst[i] = canon(acc[0][tt][i]);
        }
    }
}

} // namespace

namespace hxl {

void mm_dense(const GemmArgs &in, hipStream_t st) {
    if (in.T <= 0) return;
    for (int s0 = 0; s0 < in.nseg;) {   /* one launch per run of segments of one dtype */
        int s1 = s0 + 1;
        while (s1 < in.nseg && in.seg[s1].m.dtype == in.seg[s0].m.dtype) s1++;
        GemmArgs g = in;
        g.nseg = s1 - s0;
        int wg = 0;
        for (int s = 0; s < g.nseg; s++) {
            g.seg[s] = in.seg[s0 + s];
            g.seg[s].wg0 = wg;
            wg += (g.seg[s].m.rows_pad + 63) / 64;
        }
        const int wgr = (wg + 7) & ~7;
        /* two token tiles a workgroup read a weight half as often, and pay while that still
         * leaves two workgroups a CU: a 2048-wide layer's products at T = 512 25.0 us against
         * 27.5 (four tiles: 29.5), a 7168-wide one's at T = 301 84 against 109 (89); below, at
         * T = 85 (240 workgroups), one tile 11.5 us against 13.2 */
        const int nt = wg * ((in.T + 31) / 32) >= 512 ? 2 : 1;
        const dim3 grid(wgr * ((in.T + 16 * nt - 1) / (16 * nt)));
#define MM_L(DT_) \
    if (nt == 2) k_mm_dense<DT_, 2><<<grid, 256, 0, st>>>(g, wgr); \
    else k_mm_dense<DT_, 1><<<grid, 256, 0, st>>>(g, wgr);
        if (wg && g.seg[0].m.dtype == 4) { MM_L(4) }
        else if (wg) { MM_L(3) }
#undef MM_L
        s0 = s1;
    }
}

/* items of the routed products at most: every slot's last pass may be short */
static int mm_items(const MoeArgs &a, int n_slots, int nt) { return n_slots + a.P / (16 * nt); }

void mm_gateup(const MoeArgs &a, int n_slots, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    const bool q4 = a.dtype_mask & (1 << 4), q8 = a.dtype_mask & (1 << 3);
    const dim3 grid(mm_items(a, n_slots, 1) * (a.F / 64));
#define MM_L(DT_, E0, E1) \
    hipExtLaunchKernelGGL(k_mm_gateup<DT_>, grid, dim3(256), 0, st, E0, E1, 0u, a);
    if (q4) { MM_L(4, ev0, q8 ? nullptr : ev1) }
    if (q8) { MM_L(3, q4 ? nullptr : ev0, ev1) }
#undef MM_L
}

void mm_down(const MoeArgs &a, int n_slots, hipStream_t st) {
    /* token tiles per pass by the pairs a slot has on average: at 32 (T = 512, 128 experts)
     * two tiles 49.5 us against 54, at 5 (T = 85) one tile 22.0 against 25.6; at 9 level */
    const int nt = a.head_slots ? (a.T > 16 ? 2 : 1) : a.P >= 12 * n_slots ? 2 : 1;
    const int items = a.head_slots ? n_slots * ((a.T + 16 * nt - 1) / (16 * nt)) : mm_items(a, n_slots, nt);
    const dim3 grid(items * ((a.D + 63) / 64));
#define MM_L(DT_) \
    if (nt == 2) k_mm_down<DT_, 2><<<grid, 256, 0, st>>>(a); \
    else k_mm_down<DT_, 1><<<grid, 256, 0, st>>>(a);
    if (a.dtype_mask & (1 << 4)) { MM_L(4) }
    if (a.dtype_mask & (1 << 3)) { MM_L(3) }
#undef MM_L
}

} // namespace hxl
