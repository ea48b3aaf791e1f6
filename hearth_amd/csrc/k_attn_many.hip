/*
 * k_attn_many.hip — the canonical attention's scores and value sums for many (token, head)
 * rows (prefill chunks, trees, the heads of latent attention), on gfx950.
 *
 * Reference semantics: docs/NUMERICS.md §5.1 (engine/src/model.c:519-589), and for the
 * latent attention's RoPE term model.c:690-703: every score is a dot16 (16 partials over
 * ascending elements, then the 8/4/2/1 tree), every output one sequential f32 sum over
 * the token's rows. The order of each sum is fixed and each product is rounded before it
 * is added, so the sums stay on the vector units. The products come from
 * v_mfma_f32_16x16x1_4b_f32 with a zero accumulator: one multiplication per output, rounded
 * once, subnormals kept: fmul (the sign of a zero product is not relied on: every sum here
 * starts at +0, which neither zero changes). What that buys is the operands: an instruction
 * takes one register of rows and one of columns for 1024 products, where the vector units
 * would need one operand of each product broadcast over the lanes -- by DPP 6 cycles an
 * instruction against 2 (32 terms a clock and CU), from LDS 4 bytes a lane. The MFMA and
 * the add together sustain 51 terms a clock and CU, multiply and add with both operands
 * already in place 57.
 */
#include <algorithm>
#include <type_traits>

#include "hx_device.h"
#include "hx_launch.h"

using namespace hxd;

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

/* p[4 b + r] = fmul(a of row 4 (lane / 16) + r, b of column lane % 16) for the operands that
 * lanes 16 b .. 16 b + 15 hold (lane 16 b + i: row i, column i), b = 0 .. 3 */
__device__ __forceinline__ v16f products(float a, float b) {
    const v16f zero = {};
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 0, 0, 0);
}

/* ---- scores ----------------------------------------------------------------------
 * A workgroup holds 64 (token, head) rows of one KV group in LDS (rows padded by 16 bytes,
 * so that 16 lanes' 16-byte reads of 16 rows hit all banks); wave w takes the 16 rows 16
 * (w % 4) .. and walks tiles of 16 cache slots of its share, whose K rows it loads straight
 * from the cache, half a 64-element chunk ahead (the four waves of a slot tile meet in L1).
 * Lane (b = lane / 16, i) holds elements 16 k + 4 b + e of row i and slot i, so the product
 * of register e gives partials j = 4 b + e, b = 0 .. 3: acc[e][4 b + r] is partial 4 b + e
 * of row 4 (lane / 16) + r and slot lane % 16, and the tree stays in the lane.
 * A slot past the context is node n = slot - pos0 of this step: a row of token t exactly
 * if it is the ancestor at its own depth, which is also its place in the row order (for a
 * chain: n <= t).
 * PE: the latent attention's RoPE term is a second dot16 over 64 more columns (its queries
 * lie behind the latent ones in LDS), added before the scale.
 *
 * Bound by the products and adds. Before (16 lanes a row, queries read from LDS for every
 * row, the tree across lanes; the RoPE term a pass over S of its own), now, us a launch
 * (32 heads of 128 in 4 groups; MLA: 128 heads of 512 + 64): 512 tokens at 2048 to 3536
 * 461 -> 278, 512 from empty 60 -> 43, a tree of 85 at 2047 60 -> 49; MLA 301 tokens
 * 306 + 85 -> 197, 9 tokens at 4095 153 + 64 -> 143. */
/* waves: rows of 128 elements leave room for two workgroups of 8 a CU, longer ones for one */
constexpr int sm_waves(int hd) { return hd <= 128 ? 8 : 16; }

template <int HD, bool PE>
__global__ __launch_bounds__(64 * sm_waves(HD), 4) void k_scores_many(AttnArgs a, int nsplit) {
    constexpr int NW = sm_waves(HD), KW = NW / 4;
    constexpr int W = HD + (PE ? 64 : 0), LD = W + 4, NS = W / 32;
    __shared__ __attribute__((aligned(16))) float qs[64 * LD];   /* [64 rows][LD] */
    const int Hkv = a.Hkv, grp = a.H / Hkv;
    int b = (int)blockIdx.x;
    const int g = b % Hkv;
    b /= Hkv;
    const int split = b % nsplit;
    const int pos0 = *a.g.pos;
    const int T = a.g.live && *a.g.live < a.T ? *a.g.live : a.T;
    const int nrows = T * grp;
    /* the last tokens of a chain, which have the most slots, go first */
    const int nblk = (a.T * grp + 63) / 64, row0 = (nblk - 1 - b / nsplit) * 64;
    if (row0 >= nrows) return;   /* uniform */
    const int t_hi = min(row0 + 63, nrows - 1) / grp;
    const int nslots = pos0 + t_hi + 1;   /* slots any of the rows can have */
    const int ntile = (nslots + 15) / 16, per = (ntile + nsplit - 1) / nsplit;
    const int k1 = min(ntile, (split + 1) * per);
    if (split * per >= k1) return;   /* uniform */
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int kg = lane >> 4, lr = lane & 15, tid = threadIdx.x;
    const float *kb = a.kc + (size_t)g * a.cap * HD;
    /* elements 32 u + 16 i + 4 kg .. + 3 (i = 0, 1) of slot 16 kt + lr */
    auto load_k = [&](v4f (&k)[2], int kt, int u) {
        const int slot = min(16 * kt + lr, nslots - 1);
        const float *p = PE && u >= HD / 32 ? a.kpe + (size_t)slot * 64 + 32 * u - HD : kb + (size_t)slot * HD + 32 * u;
#pragma unroll
        for (int i = 0; i < 2; i++) k[i] = gload<v4f>(p + 16 * i + 4 * kg);
    };
    int kt = split * per + (wave >> 2);
    v4f k[2], kn[2];
    load_k(k, min(kt, ntile - 1), 0);
    {
        constexpr int N = 64 * HD / 4 / (64 * NW);
        v4f v[N < 8 ? N : 8];
#pragma unroll
        for (int j0 = 0; j0 < N; j0 += 8) {
#pragma unroll
            for (int i = j0; i < N && i < j0 + 8; i++) {
                const int f = tid + 64 * NW * i, ri = min(row0 + f / (HD / 4), nrows - 1), c4 = f % (HD / 4);
                v[i - j0] = gload<v4f>(a.q + ((size_t)(ri / grp) * a.H + g * grp + ri % grp) * HD + 4 * c4);
            }
#pragma unroll
            for (int i = j0; i < N && i < j0 + 8; i++) {
                const int f = tid + 64 * NW * i, row = f / (HD / 4), c4 = f % (HD / 4);
                *(v4f *)&qs[row * LD + 4 * c4] = v[i - j0];
            }
        }
        if (PE) {
            static_assert(!PE || NW == 16, "one 16-byte load a thread covers the RoPE columns");
            const int row = tid / 16, c4 = tid % 16, ri = min(row0 + row, nrows - 1);
            *(v4f *)&qs[row * LD + HD + 4 * c4] =
                gload<v4f>(a.qpe + ((size_t)(ri / grp) * a.H + g * grp + ri % grp) * a.qpe_ld + 4 * c4);
        }
    }
    __syncthreads();
    const float *qrow = &qs[(16 * (wave & 3) + lr) * LD + 4 * kg];
    const int r0 = row0 + 16 * (wave & 3) + 4 * kg;   /* this lane's score rows r0 .. r0 + 3 */
    const int t0 = row0 / grp;
    float *Sb = a.S + ((size_t)t0 * a.H + g * grp) * a.ldS;   /* rows at 32-bit offsets from here (checked by the launcher) */
    unsigned So[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int ri = min(r0 + r, nrows - 1);
        So[r] = (unsigned)((ri / grp - t0) * a.H + ri % grp) * (unsigned)a.ldS;
    }
    for (; kt < k1; kt += KW) {
        const int slot = 16 * kt + lr;
        int v = slot;           /* the slot's place in the row order */
        unsigned in = 0;        /* bit r: row r0 + r has the slot */
        if (16 * kt + 16 <= pos0) {   /* uniform */
#pragma unroll
            for (int r = 0; r < 4; r++) in |= r0 + r < nrows ? 1u << r : 0u;
        } else if (slot < nslots) {
            const int node = slot - pos0;
            const int dn = node < 0 ? 0 : a.g.chain ? node : a.g.depth[node];
            if (node >= 0) v = pos0 + dn;
            int r0 = row0 + 16 * (wave & 3) + 4 * kg;
            asm volatile("" : "+v"(r0));   /* few tiles come here: no registers held for them */
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int t = min(r0 + r, nrows - 1) / grp;
                bool has = node <= t;
                if (!a.g.chain && node >= 0 && has)
                    has = dn <= a.g.depth[t] && a.g.anc[(size_t)t * a.g.anc_ld + dn] == node;
                in |= r0 + r < nrows && has ? 1u << r : 0u;
            }
        }
        v16f acc[4];
        float lat[4] = {};
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[e][i] = 0.0f;
        /* the 8/4/2/1 tree over the partials j = 4 b + e of row r */
        auto tree = [&](int r) {
            float L[16];
#pragma unroll
            for (int j = 0; j < 16; j++) L[j] = acc[j & 3][4 * (j >> 2) + r];
#pragma unroll
            for (int s = 8; s >= 1; s >>= 1)
#pragma unroll
                for (int j = 0; j < s; j++) L[j] = fadd(L[j], L[j + s]);
            return L[0];
        };
        const int nx = min(kt + KW, ntile - 1);
        int ns = NS;   /* opaque: one copy of the chunk's code */
        asm volatile("" : "+s"(ns));
#pragma unroll 1
        for (int u = 0; u < ns; u++) {
            if (u + 1 < ns) load_k(kn, kt, u + 1);
            else load_k(kn, nx, 0);
            if (PE && u == HD / 32) {
#pragma unroll
                for (int r = 0; r < 4; r++) lat[r] = canon(tree(r));
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[e][i] = 0.0f;
            }
            v4f q[2];
#pragma unroll
            for (int i = 0; i < 2; i++) q[i] = *(const v4f *)(qrow + 32 * u + 16 * i);
            /* each instruction's products are added while the next one runs */
            v16f p[2];
            p[0] = products(q[0][0], k[0][0]);
#pragma unroll
            for (int f = 0; f < 8; f++) {
                if (f < 7) p[(f + 1) & 1] = products(q[(f + 1) >> 2][(f + 1) & 3], k[(f + 1) >> 2][(f + 1) & 3]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int x = 0; x < 16; x++) acc[f & 3][x] = fadd(acc[f & 3][x], p[f & 1][x]);
            }
#pragma unroll
            for (int i = 0; i < 2; i++) k[i] = kn[i];
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float d = tree(r);
            const float s = PE ? fmul(a.pe_scale, fadd(lat[r], d)) : fmul(a.scale, canon(d));
            if (in >> r & 1) Sb[So[r] + (unsigned)v] = s;
        }
    }
}

/* ---- value sums --------------------------------------------------------------------
 * A wave sums 16 (token, head) rows of one KV group over 16 CT columns; a workgroup's four
 * waves are CT such row tiles of one 64-column chunk. Slots go by in order, 4 to an MFMA
 * (products of slot 4 s + b in p[4 b + r]), from tiles of 32 slots that LDS-direct loads
 * bring in NST - 1 tiles ahead: V as it lies in the cache, the rows' probabilities in the
 * order the MFMA reads them. A tile's sums are short (8 steps of 50 to 260 clocks) against
 * the latency of S, which the L2s do not hold.
 * A chain's token has the slots up to its own; a tree's token the context and, of this
 * step's nodes, its ancestors, whose slots ascend along the path, so that walking all slots
 * in order and leaving out the others is the sum in the row order. Steps that hold such
 * slots select per row; all others add.
 *
 * Bound by the products and adds. Before (loader waves and 8 summing waves of one head each,
 * V read from LDS once a head), now, us a launch: 512
 * tokens of 32 heads of 128 at 2048 to 3536 388 -> 258, 512 from empty 63 -> 45; 301
 * tokens of 128 latent heads of 512 425 -> 214. */
constexpr int VM_ROWS = 32;
constexpr int VM_TREE = 1024;   /* nodes of a tree */

template <int CT> struct VmCfg {
    static constexpr int NST = 4;                            /* tiles in LDS */
    static constexpr int PW = CT == 4 ? 2 : 1;               /* a wave's p loads: 16 rows x 16 slots each */
    static constexpr int TILE = VM_ROWS * 64 + 4 * PW * 256; /* floats of a tile: V, then p [row tile][16 slots][16 rows][16] */
    static constexpr int LOADS = 2 + PW;                     /* LDS-direct loads of a wave for a tile (a tree's path: more) */
};

template <int CT>
__global__ __launch_bounds__(256, 2) void k_values_many(AttnArgs a) {
    typedef VmCfg<CT> C;
    constexpr int CW = 4 / CT, LDO = 65, NST = C::NST;
    __shared__ __attribute__((aligned(16))) float vt[NST][C::TILE];
    __shared__ unsigned long long path_s[16 * CT][VM_TREE / 64 + 1];   /* a tree: the nodes on the path of token t_lo + i */
    __shared__ uint16_t depth_s[VM_TREE];
    static_assert(NST * C::TILE >= 16 * CT * LDO, "the output rows fit the tiles");
    const int Hkv = a.Hkv, grp = a.H / Hkv, hd = a.hd, nd = hd >> 6;
    int b = (int)blockIdx.x;
    const int dc = b % nd;
    b /= nd;
    const int g = b % Hkv;
    b /= Hkv;
    const int T = a.g.live && *a.g.live < a.T ? *a.g.live : a.T;
    const int nrows = T * grp;
    /* the last tokens of a chain, which have the most slots, go first */
    const int nblk = (a.T * grp + 16 * CT - 1) / (16 * CT), row0 = (nblk - 1 - b) * 16 * CT;
    if (row0 >= nrows) return;   /* uniform */
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int kg = lane >> 4, lr = lane & 15, cw = wave % CW, rw = wave / CW;
    const int pos0 = *a.g.pos;
    const bool chain = a.g.chain != 0;
    auto row_at = [&](int i) { return min(row0 + i, nrows - 1); };
    const int t_lo = row0 / grp, t_hi = row_at(16 * CT - 1) / grp;
    const int nslots = pos0 + t_hi + 1;                   /* slots any row of the workgroup can have */
    if (!chain) {
        for (int n = threadIdx.x; n <= t_hi; n += 256) depth_s[n] = (uint16_t)a.g.depth[n];
        const int nw = t_hi / 64 + 1;
        for (int i = wave; i < (t_hi - t_lo + 1) * nw; i += 4) {
            const int t = t_lo + i / nw, n = (i % nw) * 64 + lane;
            const int dn = a.g.depth[min(n, t)];
            /* n's place on a path is its depth */
            const bool on = n <= t && dn <= a.g.depth[t] && a.g.anc[(size_t)t * a.g.anc_ld + dn] == n;
            const unsigned long long m = __ballot(on);
            if (lane == 0) path_s[i / nw][i % nw] = m;
        }
        __syncthreads();
    }
    const int ntiles = (nslots + VM_ROWS - 1) / VM_ROWS;
    const int all = chain ? pos0 + row_at(16 * rw) / grp + 1 : pos0;   /* slots that each of the wave's rows has */
    const int hd4 = hd * 4;
    const __amdgpu_buffer_rsrc_t vrs =
        __builtin_amdgcn_make_buffer_rsrc((void *)(a.vc + (size_t)g * a.cap * hd), 0, a.cap * hd4, 0x00020000);
    const int voff = kg * hd4 + (dc * 64 + 4 * lr) * 4;
    /* p load f = [row tile][half of the tile's slots] (past the last row tile: a copy) */
    auto srow = [&](int i) {
        const int ri = row_at(i);
        return a.S + ((size_t)(ri / grp) * a.H + g * grp + ri % grp) * a.ldS;
    };
    const int pf0 = wave * C::PW, prt = pf0 / 2 % CT;     /* a wave's p loads are of one row tile */
    const float *prow = srow(16 * prt + (lane >> 2));
    auto load = [&](float *dst, int i) {
#pragma unroll
        for (int k = 0; k < VM_ROWS / 16; k++) {
            const int f = k * 4 + wave;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(vrs, (__attribute__((address_space(3))) void *)(dst + f * 256), 16,
                                                     voff + (i * VM_ROWS + 4 * f) * hd4, 0, 0, 0);
        }
        const bool path = !chain && (i + 1) * VM_ROWS > pos0;   /* uniform */
#pragma unroll
        for (int k = 0; k < C::PW; k++) {
            float *pd = dst + VM_ROWS * 64 + (pf0 + k) * 256;
            const int v0 = i * VM_ROWS + 16 * ((pf0 + k) & 1);
            if (!path) {
                /* 4 slots of a row a lane; past the rows' slots a copy (S rows hold whole 64s) */
                lds_direct<16>(prow + min(v0, (nslots - 1) & ~15) + 4 * (lane & 3), pd);
            } else {
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    int at = min(v0 + lr, nslots - 1);
                    if (at >= pos0) at = pos0 + depth_s[at - pos0];
                    lds_direct<4>(srow(16 * prt + 4 * q + kg) + at, pd + 64 * q);
                }
            }
        }
    };
    int lim[4], ti[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int t = row_at(16 * rw + 4 * kg + r) / grp;
        ti[r] = t - t_lo;
        lim[r] = pos0 + t + 1;
    }
    /* bit b: row 4 (lane / 16) + r has slot v + b */
    auto has4 = [&](int r, int v) {
        const unsigned below = (1u << min(max(lim[r] - v, 0), 4)) - 1u;
        if (chain) return below;
        const int n = v - pos0, c = max(-n, 0), m = max(n, 0);   /* the first c of the slots are context */
        const uint8_t *pb = (const uint8_t *)path_s[ti[r]] + (m >> 3);
        const unsigned w = (pb[0] | (unsigned)pb[1] << 8) >> (m & 7);
        return (w << c | ((1u << c) - 1u)) & below;
    };
    float acc[CT][4];
#pragma unroll
    for (int x = 0; x < CT; x++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[x][r] = 0.0f;
    /* step s's operands, and its products */
    struct Ops {
        float p, v[CT];
    };
    auto fetch = [&](const float *cur, int s) {
        Ops o;
        o.p = cur[VM_ROWS * 64 + (rw * 2 + (s >> 2)) * 256 + lr * 16 + 4 * (s & 3) + kg];
        const float *src = cur + (4 * s + kg) * 64 + cw * 16 * CT + lr * CT;
        typedef float vct __attribute__((ext_vector_type(CT)));
        const vct t = *(const vct *)src;
#pragma unroll
        for (int x = 0; x < CT; x++) o.v[x] = t[x];
        return o;
    };
    auto mul = [&](const Ops &o, v16f (&pr)[CT]) {
#pragma unroll
        for (int x = 0; x < CT; x++) pr[x] = products(o.p, o.v[x]);
    };
    auto add = [&](const v16f (&pr)[CT]) {
#pragma unroll
        for (int bb = 0; bb < 4; bb++)
#pragma unroll
            for (int x = 0; x < CT; x++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[x][r] = fadd(acc[x][r], pr[x][4 * bb + r]);
    };
    /* the two never alias (restrict): the compiler otherwise waits for the LDS-direct loads
     * in flight before every LDS read */
    auto tile = [&](float *__restrict__ nxt, const float *__restrict__ cur, int i) {
        load(nxt, i + NST - 1);
        const int v0 = i * VM_ROWS;
        if (v0 + VM_ROWS <= all) {   /* uniform */
            /* a step's products are added while the next one's are formed and the operands
             * of the one after that are read */
            constexpr int N = VM_ROWS / 4;
            v16f pr[2][CT];
            Ops o[3];
            o[0] = fetch(cur, 0);
            o[1] = fetch(cur, 1);
            mul(o[0], pr[0]);
#pragma unroll
            for (int s = 0; s < N; s++) {
                if (s + 2 < N) o[(s + 2) % 3] = fetch(cur, s + 2);
                __builtin_amdgcn_sched_barrier(0);
                if (s + 1 < N) mul(o[(s + 1) % 3], pr[(s + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
                add(pr[s & 1]);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            for (int s = 0; s < VM_ROWS / 4 && v0 + 4 * s < nslots; s++) {   /* uniform */
                v16f pr[CT];
                mul(fetch(cur, s), pr);
                if (v0 + 4 * s + 4 <= all) {
                    add(pr);
                    continue;
                }
                unsigned keep[4];
#pragma unroll
                for (int r = 0; r < 4; r++) keep[r] = has4(r, v0 + 4 * s);
#pragma unroll
                for (int bb = 0; bb < 4; bb++)
#pragma unroll
                    for (int x = 0; x < CT; x++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const float y = fadd(acc[x][r], pr[x][4 * bb + r]);
                            acc[x][r] = keep[r] >> bb & 1 ? y : acc[x][r];
                        }
            }
        }
    };
#pragma unroll
    for (int i = 0; i < NST - 1; i++) load(vt[i], i);
    int at = 0;   /* i % NST */
    for (int i = 0; i < ntiles; i++) {
        /* the loads of tiles i + 1 .. i + NST - 2 may still be in flight; tile i's are done,
         * here and, after the barrier, in every wave */
        asm volatile("" ::: "memory");
        HX_WAIT_VMCNT((NST - 2) * C::LOADS);
        __builtin_amdgcn_s_waitcnt(0xC07F);   /* lgkmcnt(0): this wave is done reading tile i - 1 */
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        tile(vt[at ? at - 1 : NST - 1], vt[at], i);
        at = at + 1 < NST ? at + 1 : 0;
    }
    /* the rows as whole 64-column blocks: stored, and quantized by a wave each */
    asm volatile("" ::: "memory");
    HX_WAIT_VMCNT(0);   /* no tile may land on the rows */
    __syncthreads();
    float *o = &vt[0][0];
#pragma unroll
    for (int x = 0; x < CT; x++)
#pragma unroll
        for (int r = 0; r < 4; r++) o[(16 * rw + 4 * kg + r) * LDO + cw * 16 * CT + lr * CT + x] = acc[x][r];
    __syncthreads();
    for (int i = wave; i < 16 * CT && row0 + i < nrows; i += 4) {   /* uniform per wave */
        const int t = (row0 + i) / grp, h = g * grp + (row0 + i) % grp;
        const float y = o[i * LDO + lane];
        a.out[((size_t)t * a.H + h) * hd + dc * 64 + lane] = y;
        if (a.qo_on) quant_block_wave(y, a.qo, a.qo_hm ? h * a.T + t : t, a.qo_hm ? dc : h * nd + dc);
    }
}

} // namespace

namespace hxl {

bool scores_many(const AttnArgs &a, hipStream_t st) {
    const int grp = a.H / a.Hkv;
    if (a.post || (a.hd != 64 && a.hd != 128 && a.hd != 256 && a.hd != 512)) return false;
    /* A workgroup takes the latency of its slot tiles however few its rows are; the others read
     * the rows of K once a token. Measured, these / the others, us a launch: latent rows (with
     * the RoPE term) of 16 heads, one token at 0 15 / 33, at 1000 30 / 39, at 4000 31 / 41, of 4
     * heads, one token at 4000 30 / 23, 9 tokens 32 / 37; single heads of 128, 32 tokens at 0
     * 6.4 / 7.2, at 1000 15 / 40 (17 at 0 level, but the whole call 1% slower); groups of 2 of
     * 256, 32 tokens at 0 9.4 / 6.5, at 1000 16 / 40; groups of 8 of 128, 17 tokens at 0 7.9 /
     * 6.8, at 4000 29.5 / 26.5, 24 at 4000 30 / 36 */
    const bool few = a.T * grp < 64 && !(a.hd == 512 && grp >= 16) && !(a.hd <= 128 && a.T >= 32);
    if (few) return false;
    const bool pe = a.qpe != nullptr;
    if (pe && (a.hd != 512 || a.qpe_ld % 4 || ((uintptr_t)a.qpe & 15))) return false;
    if ((64LL / grp + 2) * a.H * a.ldS >= 1LL << 32) return false;
    const long long base = ((long long)a.T * grp + 63) / 64 * a.Hkv;
    /* shares of the slots by rounds of the workgroups that fit the chip at once, times a
     * share's slot tiles a wave and one for its prologue. A prefill of mostly its own tokens
     * has shares of very different lengths: at least three rounds even out */
    const int kw = sm_waves(a.hd) / 4, nkt = (a.g.nr_max + 15) / 16, fit = a.hd <= 128 ? 512 : 256;
    const bool ragged = a.g.chain && 2 * a.T > a.g.nr_max;
    int ns = 1;
    long long best = 0;
    for (int n = 1; n <= (nkt + kw - 1) / kw && (n == 1 || base * n <= 6 * fit); n++) {
        const long long rounds = std::max((base * n + fit - 1) / fit, ragged ? 3LL : 1LL);
        const long long cost = rounds * (((nkt + n - 1) / n + kw - 1) / kw + 1);
        if (!best || cost < best) { ns = n; best = cost; }
    }
#define HX_SM(HD_, PE_) { k_scores_many<HD_, PE_><<<(int)(base * ns), 64 * sm_waves(HD_), 0, st>>>(a, ns); return true; }
    if (pe) HX_SM(512, true)
    if (a.hd == 64) HX_SM(64, false)
    if (a.hd == 128) HX_SM(128, false)
    if (a.hd == 256) HX_SM(256, false)
    HX_SM(512, false)
#undef HX_SM
}

/* ns of k_values_many<CT>: rounds of the workgroups that fit the chip at once (two a compute
 * unit), the longest rows first. A row is 64 / 42 ns (CT = 4 / 2) while a unit has one of them
 * and 79 / 49 with two; a tree's steps over its own nodes select per row. */
static double values_many_ns(const AttnArgs &a, int ct, long long wgs) {
    const bool four = ct == 4;
    double ns = four ? 12000 : 7000;
    for (long long w0 = 0; w0 < wgs; w0 += 512) {
        const double rows = a.g.nr_max - (a.g.chain ? (double)a.T * w0 / wgs : 0.0);
        ns += (wgs - w0 <= 256 ? (four ? 64 : 42) : (four ? 79 : 49)) * rows + (w0 ? 2000 : 0);
        if (!a.g.chain) ns += (four ? 120 : 75) * a.T;
    }
    return ns;
}

bool values_many(const AttnArgs &a, double other_ns, hipStream_t st) {
    if (a.hd % 64 || (!a.g.chain && a.T > VM_TREE)) return false;
    const int grp = a.H / a.Hkv, nd = a.hd / 64;
    auto wgs = [&](int ct) { return ((long long)a.T * grp + 16 * ct - 1) / (16 * ct) * a.Hkv * nd; };
    /* The line lies where the times cross: a workgroup here takes the latency of its rows
     * however few there are, where the others split by token and head. Measured, these with 2
     * and 4 column tiles / the others, us a launch. Groups of 8 of 32 heads of 128: at 0, 128
     * tokens 12.8, 18.7 / 12.3, 256 19.4, 27.7 / 26.6, 512 41.9, 46.7 / 61.5; at 4000, 128 tokens
     * 171, 262 / 131, 256 200, 271 / 257, 320 399, 325 / 328, 464 445, 353 / 498, 512 455, 367 /
     * 535; trees at 2047 of 85 103, 154 / 55, 512 305, 270 / 265. 32 single heads: at 0, 64 tokens
     * 11, 19 / 58, at 4000 196, 289 / 469; tree of 85 at 2047 108, 157 / 366. 128 latent heads: at
     * 4000, 9 tokens 195, 256 / 160, 32 386, 316 / 493. */
    const double t2 = values_many_ns(a, 2, wgs(2)), t4 = values_many_ns(a, 4, wgs(4));
    if (std::min(t2, t4) >= 0.97 * other_ns) return false;
    if (t2 < t4) k_values_many<2><<<(int)wgs(2), 256, 0, st>>>(a);
    else k_values_many<4><<<(int)wgs(4), 256, 0, st>>>(a);
    return true;
}

} // namespace hxl
