// s3d_elem.h -- the element kernel (strain rate, stress and memory-variable
// update, weak divergence; see s3d_kernels.hip for the step it belongs to)
// and the helpers it shares with the other kernels. Templates and inline
// functions only: the element-kernel launchers instantiate it once per GLL
// order in their own translation units (s3d_elem.hip), which build in
// parallel.
#pragma once

#include "s3d_internal.h"

namespace s3d {

// Element tile: EPB elements per workgroup, one lane per element-local node.
// EPB = 0 selects the default, as many elements as fit in 256 lanes.
template <int P>
constexpr int default_epb() { return (256 / ((P + 1) * (P + 1) * (P + 1))) > 0 ? (256 / ((P + 1) * (P + 1) * (P + 1))) : 1; }

template <int P, int E = 0>
struct Shape {
    static constexpr int P1 = P + 1;
    static constexpr int NP = P1 * P1 * P1;
    static constexpr int PB = P * P * P;
    static constexpr int EPB = E > 0 ? E : default_epb<P>();
    static constexpr int NT = ((EPB * NP + 63) / 64) * 64;
};

// Workgroup order of the element kernel: dispatch deals consecutive workgroups
// to the 8 XCDs in turn; with ORDER_CHUNKS, XCD x runs the tiles of chunks x, x + 8,
// x + 16, ... of XCD_CHUNK consecutive tiles each. Neighbours along theta
// (shared velocity and force nodes) still meet in one L2, and all XCDs work
// in one window of memory (8 chunks) that moves through the state block. With
// one contiguous range of tiles per XCD eight windows far apart compete for
// the DRAM rows: element kernel at order 4, 96x96x48, FP32 with five memory
// words, 2.43 ms with ranges, 2.28 ms with chunks; FP64 at 48x48x24 0.55 and
// 0.52 ms. Chunks of 4 to 64 tiles are within 3 % of each other at orders 2
// to 7, and 16 within 1 % of the best of each; alternating the tiles of two
// planes inside the order (so that the upper tile finds the shared velocity
// nodes in L2) costs 1 to 5 % and is not done. The workgroups past the last
// whole group of 8 chunks keep the plain order.
// A launch of at most XCD_RESIDENT workgroups is in flight as a whole, there
// is no moving window, and what its XCD wrote in the last step may still be in
// that L2: ranges (12x12x8, order 4, FP64: 12.8 us, 13.2 us with chunks; at
// 2048 workgroups 25.5 and 26.2 us, at 4608 60.0 and 55.2 us). A count that 8
// does not divide takes them too: 256 steps of 12x12x8, whose node kernel has
// 381 workgroups, 4.21 ms in plain order, 3.78 ms in ranges.
// On the largest meshes the ranges win again, most likely where a plane
// exceeds what the L2s and the Infinity Cache keep until the next one reads
// its velocity: FP64 from about 5e7 nodes on (chunks and ranges, ms: 96x96x48
// 4.51 4.41, 128x128x48 8.21 7.85, 160x160x96 24.6 22.6, 192x192x96 34.6 32.3;
// 48x48x24 0.53 0.55). In FP32 it goes by the mesh (192x192x96 17.0 16.2,
// 192x192x32 5.81 5.67, 128x128x96 8.05 7.97, but 160x160x96 11.9 12.5,
// 96x96x48 2.12 2.25, 96x96x192 8.02 8.95), so chunks unless s3d_autotune
// finds ranges faster.
constexpr int XCD_CHUNK = 16;
constexpr int XCD_RESIDENT = 2048;
constexpr long RANGE_NODES_FP64 = 50000000;
enum { ORDER_PLAIN, ORDER_CHUNKS, ORDER_RANGES };

__device__ inline int chunk_block(int b, int G, int on)
{
    constexpr int group = 8 * XCD_CHUNK;
    if (on == ORDER_PLAIN) return b;
    if (on == ORDER_RANGES || G <= XCD_RESIDENT) {
        const int q = G >> 3;   // the last G mod 8 workgroups keep their place
        return b < 8 * q ? (b & 7) * q + (b >> 3) : b;
    }
    if (b >= G / group * group) return b;
    const int g = b / group, r = b - g * group;
    return g * group + (r & 7) * XCD_CHUNK + (r >> 3);
}

template <int P>
__device__ inline long unique_index(int ex, int ey, int ez, int i, int j, int k,
                                    int nx, int ny)
{
    int bx = ex + (i == P), by = ey + (j == P), bz = ez + (k == P);
    int li = (i == P) ? 0 : i, lj = (j == P) ? 0 : j, lk = (k == P) ? 0 : k;
    long b = (long)bx + (long)(nx + 1) * ((long)by + (long)(ny + 1) * bz);
    return b * (P * P * P) + li + P * (lj + P * lk);
}

template <typename R>
__device__ inline void kahan_add(R &s, R &c, R inc)
{
    R y = inc - c;
    R t = s + y;
    c = (t - s) - y;
    s = t;
}

// ---------------------------------------------------------------------------
// element kernel
// ---------------------------------------------------------------------------
// Element-major block fields (the state block, lam/mu/tau, the displacement
// gradient; the element force has its own two-part layout, force_index):
// component c of element e occupies the NP entries at (e * nc + c) * NP.
// The state block's parts are addressed through pointers at their first
// components (sig, sig_lo, mem) with nc = state_components(KS, VM).
__device__ __forceinline__ long em_index(long e, int nc, int c, int NP, int node)
{
    return (e * nc + c) * NP + node;
}

// Element force layout: first the nodes with k < p of every element,
// [e][c][(p+1)^2 p], then the k = p layers, [e][c][(p+1)^2]. The node kernel
// reads each part once: an element's k = p layer is the z-1 copy of the
// owned block above it, gathered a plane of blocks after the rest of the
// element, and in the plain element-major layout it shared cache lines with
// what had already been read.
template <int P>
__device__ __forceinline__ long force_index(long e, int c, int node, long nel)
{
    constexpr int NL = (P + 1) * (P + 1), NM = NL * P;
    return node < NM ? (e * 3 + c) * NM + node : nel * 3 * NM + (e * 3 + c) * NL + (node - NM);
}

// Direct HBM -> LDS loads (global_load_lds): the lanes of a wave write
// consecutive LDS words or 16-byte vectors from byte address `lds` (the same in
// the wave) on. Written as inline assembly so the compiler's wait accounting
// never sees them: it would wait for all of them before any read of LDS.
// Vector memory operations complete in issue order, and wait_loads<N> waits
// until at most the N newest are outstanding. The statements write M0, so it
// is in their clobber list; LLVM reserves M0 and warns about the clobber.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_load_dword(const void *g, unsigned lds)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
                 :: "v"(g), "s"(__builtin_amdgcn_readfirstlane(lds)) : "m0");
}

__device__ __forceinline__ void lds_load_x4(const void *g, unsigned lds)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :: "v"(g), "s"(__builtin_amdgcn_readfirstlane(lds)) : "m0");
}
#pragma clang diagnostic pop

template <int N>
__device__ __forceinline__ void wait_loads()
{
    static_assert(N < 64, "vmcnt has 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

__device__ __forceinline__ unsigned lds_address(const void *p) { return (unsigned)(size_t)p; }

// The words [w0, w0 + n) of an element-major block into LDS, in 16-byte
// vectors by the workgroup's NT lanes, n at most W. The block starts on a
// 16-byte boundary and the vectors do too: word w0 arrives at lds[w0 & 3], and
// up to 3 words before and after the range come along (the blocks are
// allocated BLOCK_PAD bytes longer). lds holds lds_words(W).
constexpr int lds_words(int W) { return (W + 3 + 3) / 4 * 4; }

// loads that every wave issues for a whole run of W words (some issue more)
constexpr int run_loads(int W, int NT) { return W > 4 * NT - 256 ? (W - 4 * NT + 256 + 4 * NT - 1) / (4 * NT) : 0; }

template <int W, int NT>
__device__ __forceinline__ int lds_load_run(const float *block, long w0, int n, const float *lds)
{
    const int off = (int)(w0 & 3), end = n > 0 ? n + off : 0;
    const int lane = threadIdx.x & 63, first = (threadIdx.x >> 6) * 256;
    const float *src = block + (w0 - off);
#pragma unroll
    for (int q = 0; q < (W + 3 + 4 * NT - 1) / (4 * NT); ++q) {
        const int at = first + q * 4 * NT;
        if (at + 4 * lane < end) lds_load_x4(src + at + 4 * lane, lds_address(lds + at));
    }
    return off;
}

// Geometry rows per element (FP64): sin, 1/sin, cot of theta_q and the theta
// taper profile (ElemArgs::gx), the phi profile (py), r, 1/r, r^2 of r_q and the
// r profile (gz).
enum { G_SIN = 0, G_ISIN, G_COT, G_PX, G_PY, G_R, G_IR, G_R2, G_PZ, G_N };

// The tables of a tile into LDS, word by word: the coefficients (CoefTable
// order) and the geometry rows of its elements, [EPB][G_N][P1] doubles.
template <int P, int EPB, int NT, typename R>
__device__ __forceinline__ void load_tables(const ElemArgs<R> &a, int tile, const double *cf, const double *gtab)
{
    constexpr int P1 = P + 1, CW = 2 * coef_words(P1), GW = 2 * G_N * P1;
    const int t = threadIdx.x, w = t & ~63;
    const unsigned *coef = (const unsigned *)(const double *)a.coef;
#pragma unroll
    for (int q = 0; q < (CW + NT - 1) / NT; ++q)
        if (q * NT + t < CW) lds_load_dword(coef + q * NT + t, lds_address((const unsigned *)cf + q * NT + w));
#pragma unroll
    for (int q = 0; q < (EPB * GW + NT - 1) / NT; ++q) {
        const int at = q * NT + t;
        if (at < EPB * GW) {
            const int es = at / GW, m = at - es * GW, row = m / (2 * P1), m2 = m - row * 2 * P1;
            int e = tile * EPB + es;
            e = e < a.nel ? e : a.nel - 1;
            const int ex = e % a.nx, ey = (e / a.nx) % a.ny, ez = e / (a.nx * a.ny);
            const double *x = row < G_PY ? (const double *)a.gx + (ex * 4 + row) * P1
                              : row == G_PY ? (const double *)a.py + ey * P1
                                            : (const double *)a.gz + (ez * 4 + row - G_R) * P1;
            lds_load_dword((const unsigned *)x + m2, lds_address((const unsigned *)gtab + q * NT + w));
        }
    }
}

// Data of one tile. FP32 kernels keep it in LDS: the state [EPB][NS][NP], the
// moduli [EPB][NC][NP] (not BF16 ones), the velocity [3][NT]; FP64 kernels in
// registers, with LDS for the staged velocity, then effective stress.
template <int P, int E, typename R, int VM, bool S16, int KS>
struct Tile {
    using S = Shape<P, E>;
    static constexpr bool DMA = sizeof(R) == 4, MAT = DMA && !S16;
    static constexpr int NS = state_components(KS, VM), NC = VM ? 3 : 2;
    static constexpr int TW = S::EPB * NS * S::NP, MW = S::EPB * NC * S::NP;   // words
    static constexpr int SBUF = DMA ? lds_words(TW) : 6 * S::EPB * S::NP, MBUF = MAT ? lds_words(MW) : 1,
                         VBUF = DMA ? 3 * S::NT : 1;
    static constexpr int LDS = (int)sizeof(R) * (SBUF + MBUF + VBUF) +
                               8 * (coef_words(S::P1) + S::EPB * G_N * S::P1) + 4 * S::EPB;
};

// Where the kernel stores the new stress, compensation and memory variables:
// before the weak divergence, while other waves still compute, or after it.
// Early costs registers nothing (the values leave before the divergence needs
// its own) and starts the stores sooner, at orders up to 5 and for elastic
// order 6: order 5 383 us against 393 at 48x40x24 with five memory words,
// 260 against 295 elastic with FP32 compensation; order 3 elastic 108 against
// 117 at 61x53x31; order 2 698 against 725 at 100x100x64. The wide
// workgroups of orders 6 and 7 are few on a CU and wait for their own stores
// at the divergence's barrier: order 6 440 us late, 490 early at 40x36x20,
// order 7 397 and 421 at 36x30x18 (elastic 277 and 287).
template <int P, typename R, int VM>
constexpr bool stores_early() { return sizeof(R) == 4 && (P <= 5 || (P == 6 && VM == 0)); }

// Dynamic LDS of a launch, which the kernel does not use: it keeps the
// workgroups of a CU to about 130 KB of tiles in flight. More of them only
// widen the window of memory that is open at a time: order 4, 32 KB a tile, 5
// and 4 workgroups per CU: 2.25 and 2.16 ms at 96x96x48 with five memory
// words and BF16 compensation, 1.50 and 1.43 ms at 96x96x32 with six and none;
// 3 workgroups 2.22 ms.
template <int P, int E, typename R, int VM, bool S16, int KS>
constexpr unsigned spare_lds()
{
    constexpr int cu = 160 * 1024, lds = Tile<P, E, R, VM, S16, KS>::LDS;
    constexpr int fit = cu / lds, want = 130 * 1024 / lds > 2 ? 130 * 1024 / lds : 2;
    return Tile<P, E, R, VM, S16, KS>::DMA && fit > want ? cu / (want + 1) + 1 - lds : 0;
}

// Element kernel body: the workgroup advances tile `tile` (EPB elements, one
// lane per element-local node). S16: the static per-node fields are stored
// in BF16 (ElemArgs::s16). KS: stress compensation, 0 off, 1 FP32 words, 2
// BF16 words in pairs (a template parameter: a run-time choice leaves register
// joins that wait for every load in flight). VM: memory words per mechanism, 0
// elastic, 6 the six components, 5 their deviatoric part (see the stress rate
// below).
//
// FP32 kernels load everything straight into LDS: the tables and the velocity
// first, for the strain rate, behind them the tile's part of the state block
// and of the moduli, which are contiguous, in 16-byte vectors. They hold no
// state in registers until they use it, and the effective stress takes the
// place of the stress in LDS. HBM bounds them (the contractions only at order
// 6): one dword load per lane and component into registers, waiting for the
// lot, ran 2.46 ms at order 4, 96x96x48 with five memory words and BF16
// compensation (5.0 TB/s with the force), this 2.07 ms (5.9 TB/s; a copy
// reaches 6.2); order 2, 100x100x64 0.86 and 0.68 ms; order 3, 100x100x50 1.28
// and 1.15; order 5, 48x40x24 0.46 and 0.39; order 6, 40x36x20 0.55 and 0.48;
// order 7, 36x30x18 0.44 and 0.40. (The part of these gains that is the
// workgroup order's is at chunk_block.) FP64 kernels keep the tile in
// registers, since in LDS it would leave one workgroup per CU: 0.53 ms at
// order 4, 48x48x24, 5.8 TB/s.
template <int P, int E, typename R, int VM, bool S16, int KS>
__device__ __forceinline__ void elem_body(const ElemArgs<R> &a, int tile)
{
    using S = Shape<P, E>;
    using C = coef_t<R>;
    constexpr int P1 = S::P1, NP = S::NP, EPB = S::EPB, NT = S::NT;
    using T = Tile<P, E, R, VM, S16, KS>;
    constexpr int NS = T::NS;         // words per node of the state block
    constexpr bool VISCO = VM != 0;
    constexpr int NM = NRDISS * VM;   // memory words per node
    constexpr int NC = T::NC;         // lam, mu (, tau)
    constexpr bool DMA = T::DMA, MAT = T::MAT;
    constexpr int TW = T::TW, MW = T::MW;
    constexpr bool EARLY = stores_early<P, R, VM>();
    __shared__ __align__(16) R sbuf[T::SBUF];
    __shared__ __align__(16) R mbuf[T::MBUF];
    __shared__ R vbuf[T::VBUF];
    static_assert(sizeof(C) == 8, "tables are FP64");
    __shared__ __align__(16) C cf[coef_words(P1)];    // Dx, Dy, Dz, dl*w, weights
    __shared__ __align__(16) C gtab[EPB][G_N * P1];   // geometry rows of the tile's elements
    __shared__ int sst[EPB];                          // moment-tensor source slot per element

    const int t = threadIdx.x;
    const int slot = t / NP;
    const int node = t - slot * NP;
    const bool inside = slot < EPB;
    const int es = inside ? slot : 0;
    const int i = node % P1, j = (node / P1) % P1, k = node / (P1 * P1);
    // element of this lane; lanes without one (the tail of the last tile, or
    // past the tile's nodes) read element 0's addresses and store nothing
    const int e = tile * EPB + slot;
    const bool valid = inside && e < a.nel;
    const long ev = valid ? e : 0;
    const long eb = ev * NP + node;   // element-local address

    // ---- loads: what the strain rate needs first, the state behind it ----
    long u;
    {
        const int ee = (int)ev;
        u = unique_index<P>(ee % a.nx, (ee / a.nx) % a.ny, ee / (a.nx * a.ny), i, j, k, a.nx, a.ny);
    }
    load_tables<P, EPB, NT>(a, tile, cf, &gtab[0][0]);
    if (t < EPB) {
        const int se = tile * EPB + t;
        if (a.src_slot)
            lds_load_dword((const int *)a.src_slot + (se < a.nel ? se : a.nel - 1), lds_address(sst));
        else
            sst[t] = -1;
    }
    int soff = 0, moff = 0;   // LDS places of the tile's first words
    R v[3], sg[6], lo[6], M[!DMA && VISCO ? NM : 1], lam, mu, tau = R(0);
    const int ne = a.nel - tile * EPB < EPB ? a.nel - tile * EPB : EPB;   // elements of the tile
    if constexpr (DMA) {
        const int w = t & ~63;
        lds_load_dword((const R *)a.vx + u, lds_address(vbuf + w));
        lds_load_dword((const R *)a.vy + u, lds_address(vbuf + NT + w));
        lds_load_dword((const R *)a.vz + u, lds_address(vbuf + 2 * NT + w));
        soff = lds_load_run<TW, NT>((const float *)a.sig, (long)tile * TW, ne * NS * NP, sbuf);
        if constexpr (MAT) moff = lds_load_run<MW, NT>((const float *)a.lam, (long)tile * MW, ne * NC * NP, mbuf);
        if constexpr (S16) {
            const long mb = em_index(ev, NC, 0, NP, node);
            lam = (R)(float)a.s16.lam[mb];
            mu = (R)(float)a.s16.mu[mb];
            if constexpr (VISCO) tau = (R)(float)a.s16.tau[mb];
        }
    } else {
        v[0] = a.vx[u];
        v[1] = a.vy[u];
        v[2] = a.vz[u];
#pragma unroll
        for (int c = 0; c < 6; ++c) sg[c] = a.sig[em_index(ev, NS, c, NP, node)];
        const long mb = em_index(ev, NC, 0, NP, node);
        lam = a.lam[mb];
        mu = a.mu[mb];
        if constexpr (VISCO) tau = a.tau[mb];
#pragma unroll
        for (int c = 0; c < NM; ++c) M[c] = a.mem[em_index(ev, NS, c, NP, node)];
    }
    // iteration it = *it_dev + 1 uses the STF sample it-1 (zero for it = 1)
    const int it = *a.it_dev + 1;

    const C *gs = gtab[es];

    // LDS views: velocity component c of node n of this lane's element at
    // lv[c * VS + n], effective stress component c at ls[c * SS + n] (FP32: the
    // state block's component c)
    constexpr int VS = DMA ? NT : EPB * NP, SS = DMA ? NP : EPB * NP;
    R *const lv = (DMA ? vbuf : sbuf) + es * NP;
    R *const ls = DMA ? sbuf + soff + es * (NS * NP) : lv;
    const R *const lm = mbuf + moff + es * (NC * NP) + node;
    if constexpr (DMA) {
        // tables and velocity: all but the state's loads, which only a whole
        // tile issues in full
        if (ne == EPB)
            wait_loads<run_loads(TW, NT) + (MAT ? run_loads(MW, NT) : 0)>();
        else
            wait_loads<0>();
    } else if (inside) {
        // the tables' loads are older than those of v
#pragma unroll
        for (int c = 0; c < 3; ++c) lv[c * VS + node] = v[c];
        asm volatile("" ::: "memory");
    }
    __syncthreads();

    // ---- K1: tensor-product derivatives along theta, phi, r ----
    C dxv[3] = {0, 0, 0}, dyv[3] = {0, 0, 0}, dzv[3] = {0, 0, 0};
    {
        const C *Dxi = cf + i * P1;
        const C *Dyj = cf + P1 * P1 + j * P1;
        const C *Dzk = cf + 2 * P1 * P1 + k * P1;
#pragma unroll
        for (int q = 0; q < P1; ++q) {
            const R *vx = lv + q + P1 * (j + P1 * k);
            const R *vy = lv + i + P1 * (q + P1 * k);
            const R *vz = lv + i + P1 * (j + P1 * q);
            const C cx = Dxi[q], cy = Dyj[q], cz = Dzk[q];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                dxv[c] += (C)vx[c * VS] * cx;
                dyv[c] += (C)vy[c * VS] * cy;
                dzv[c] += (C)vz[c * VS] * cz;
            }
        }
    }

    // ---- K2: spherical completion, K4: symmetrisation ----
    R exx, eyy, ezz, exy, exz, eyz;
    {
        const C ux = DMA ? lv[node] : v[0], uy = DMA ? lv[VS + node] : v[1], uz = DMA ? lv[2 * VS + node] : v[2];
        const C inv_r = gs[G_IR * P1 + k];
        const C cot = gs[G_COT * P1 + i];
        const C inv_rs = inv_r * gs[G_ISIN * P1 + i];
        const C ezx = -dzv[0];
        const C exz_c = (dxv[2] - ux) * inv_r;
        const C ezy = -dzv[1];
        const C eyz_c = -uy * inv_r + dyv[2] * inv_rs;
        const C exy_c = dxv[1] * inv_r;
        const C eyx = -uy * cot * inv_r + dyv[0] * inv_rs;
        const C gxx = (uz + dxv[0]) * inv_r;
        const C gyy = dyv[1] * inv_rs + (uz + ux * cot) * inv_r;
        const C gzz = -dzv[2];
        const C gxy = (exy_c + eyx) * 0.5;
        const C gxz = (exz_c + ezx) * 0.5;
        const C gyz = (eyz_c + ezy) * 0.5;
        exx = (R)gxx;
        eyy = (R)gyy;
        ezz = (R)gzz;
        exy = (R)gxy;
        exz = (R)gxz;
        eyz = (R)gyz;
        // K3: the displacement gradient integrates the velocity gradient
        // (src/evolution.f90:179-187); kept as its symmetric part, the
        // only form the reference outputs (src/volume_snapshot.f90:220-236),
        // in FP64, and only when requested
        if (a.dgrad && valid) {
            double *g = a.dgrad + em_index(ev, 6, 0, NP, node);
            g[0 * NP] += a.dt * (double)gxx;
            g[1 * NP] += a.dt * (double)gxy;
            g[2 * NP] += a.dt * (double)gxz;
            g[3 * NP] += a.dt * (double)gyy;
            g[4 * NP] += a.dt * (double)gyz;
            g[5 * NP] += a.dt * (double)gzz;
        }
    }

    if constexpr (DMA) {
        // the state, of every wave
        wait_loads<0>();
        __syncthreads();
    }
    // memory variable c of this lane's node, as the step found it
    auto mem = [&](int c) -> R { return DMA ? ls[(NS - NM + c) * NP + node] : M[c]; };
    if constexpr (MAT) {
        lam = lm[0];
        mu = lm[NP];
        if constexpr (VISCO) tau = lm[2 * NP];
    }

    // ---- K5: stress rate times dt (lam, mu, A, B, C carry the dt) ----
    R rt[6];
    const R tmu = R(2) * mu;
    if constexpr (!VISCO) {
        const R Lr = lam * (exx + eyy + ezz);
        rt[XX] = Lr + tmu * exx;
        rt[YY] = Lr + tmu * eyy;
        rt[ZZ] = Lr + tmu * ezz;
        rt[XY] = tmu * exy;
        rt[XZ] = tmu * exz;
        rt[YZ] = tmu * eyz;
    } else {
        // SLS in the loop form of the commented-out src/evolution.f90:216-284:
        // lam holds kappa - 2 mu_tau / 3 and mu holds mu_tau = mu (1 + tau),
        // both formed in FP64; 2 mu itself only scales the memory variables
        const R tmut = tmu;                                    // 2 mu_tau
        const R tm = tmut / (R(1) + tau);                      // 2 mu
        if constexpr (VM == 6) {
            R Md[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) Md[c] = mem(c) + mem(6 + c) + mem(12 + c);
            const R Msum = Md[XX] + Md[YY] + Md[ZZ];
            const R Lr = lam * (exx + eyy + ezz) - tm * Msum * R(1.0 / 3.0);
            rt[XX] = Lr + tmut * exx + tm * Md[XX];
            rt[YY] = Lr + tmut * eyy + tm * Md[YY];
            rt[ZZ] = Lr + tmut * ezz + tm * Md[ZZ];
            rt[XY] = tmut * exy + tm * Md[XY];
            rt[XZ] = tmut * exz + tm * Md[XZ];
            rt[YZ] = tmut * eyz + tm * Md[YZ];
        } else {
            // The memory variables enter the stress rate only as
            // Md - tr(Md)/3 I, and every component relaxes at the same
            // rate with the same forcing (t3 e), so their deviatoric
            // part evolves on its own, driven by the deviatoric strain
            // rate: five words per mechanism hold it (xx xy xz yy yz,
            // zz = -(xx + yy)), and the trace is never formed.
            R Dd[5];
#pragma unroll
            for (int c = 0; c < 5; ++c) Dd[c] = mem(c) + mem(5 + c) + mem(10 + c);
            const R Dzz = -(Dd[XX] + Dd[YY]);
            const R Lr = lam * (exx + eyy + ezz);
            rt[XX] = Lr + tmut * exx + tm * Dd[XX];
            rt[YY] = Lr + tmut * eyy + tm * Dd[YY];
            rt[ZZ] = Lr + tmut * ezz + tm * Dzz;
            rt[XY] = tmut * exy + tm * Dd[XY];
            rt[XZ] = tmut * exz + tm * Dd[XZ];
            rt[YZ] = tmut * eyz + tm * Dd[YZ];
        }
    }
    if (S16 ? a.s16.ca != nullptr : a.ca != nullptr) {   // anisotropy (src/evolution.f90:290-296)
        R pa, pb, pc;
        if constexpr (S16) {
            pa = (R)(float)a.s16.ca[eb];
            pb = (R)(float)a.s16.cb[eb];
            pc = (R)(float)a.s16.cc[eb];
        } else {
            pa = a.ca[eb];
            pb = a.cb[eb];
            pc = a.cc[eb];
        }
        rt[XX] += pc * ezz + pa * (eyy + exx);
        rt[YY] += pc * ezz + pa * (eyy + exx);
        rt[ZZ] += pc * (eyy + exx);
        rt[XZ] += R(2) * pb * exz;
        rt[YZ] += R(2) * pb * eyz;
    }

    // ---- K6: integrate the stress ----
    if constexpr (DMA) {
#pragma unroll
        for (int c = 0; c < 6; ++c) sg[c] = ls[c * NP + node];
    }
    if constexpr (KS == 1) {
#pragma unroll
        for (int c = 0; c < 6; ++c) lo[c] = ls[(6 + c) * NP + node];
    } else if constexpr (KS == 2) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const unsigned w = __builtin_bit_cast(unsigned, (float)ls[(6 + q) * NP + node]);
            lo[2 * q] = (R)bf16_lo(w);
            lo[2 * q + 1] = (R)bf16_hi(w);
        }
    }
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        if constexpr (KS != 0)
            kahan_add(sg[c], lo[c], rt[c]);
        else
            sg[c] = sg[c] + rt[c];
    }

    // ---- K7: moment-tensor glut and single force of the previous add() ----
    R src[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int sl = sst[es];
    if (valid && sl >= 0 && it > 1 && it <= a.nt) {
#pragma unroll
        for (int c = 0; c < 9; ++c) {
            const int ch = a.src_chan[sl * 9 + c];
            if (ch >= 0) {
                const double d = a.stf[(long)ch * a.nt + (it - 2)];
                src[c] = (R)(-(d * a.src_coef[((long)sl * 9 + c) * NP + node]));
            }
        }
    }

    if constexpr (!DMA) __syncthreads();   // the staged velocity is no longer needed
    if (inside) {
        // effective stress, with the glut
#pragma unroll
        for (int c = 0; c < 6; ++c) ls[c * SS + node] = sg[c] + src[c];
    }

    // ---- taper factor of this node (K13) ----
    R dmp = R(0);   // 1 - taper
    {
        const C tx = gs[G_PX * P1 + i], ty = gs[G_PY * P1 + j], tz = gs[G_PZ * P1 + k];
        if (tx + ty + tz != C(0)) dmp = (R)taper_damp(tx, ty, tz, a.alpha);
    }

    // ---- tapered stress (K13) and its compensation ----
    unsigned lo2[3];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        sg[c] = sg[c] - sg[c] * dmp;
        if constexpr (KS != 0) lo[c] = lo[c] - lo[c] * dmp;
    }
    if constexpr (KS == 2) {
#pragma unroll
        for (int q = 0; q < 3; ++q) lo2[q] = pack_bf16((float)lo[2 * q], (float)lo[2 * q + 1]);
    }

    // ---- store them and the new memory variables (loop form of
    // src/evolution.f90:415-442) ----
    auto store_state = [&]() {
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            a.sig_w[em_index(ev, NS, c, NP, node)] = sg[c];
            if constexpr (KS == 1) a.sig_lo_w[em_index(ev, NS, c, NP, node)] = lo[c];
        }
        if constexpr (KS == 2) {
#pragma unroll
            for (int q = 0; q < 3; ++q) a.sig_lo2_w[em_index(ev, NS, q, NP, node)] = lo2[q];
        }
        if constexpr (VISCO) {
            // M (1 - dt/tau_p) - dt tau / (3 tau_p) e  ==  M - dt/tau_p (M + tau/3 e):
            // the decrement form keeps the FP32 relaxation rate exact to one
            // rounding of dt/tau_p (1 - dt/tau_p would lose its low bits)
            const R t3 = tau * R(1.0 / 3.0);
            R em[6] = {exx, exy, exz, eyy, eyz, ezz};
            if constexpr (VM == 5) {   // deviatoric strain rate
                const R tr3 = (exx + eyy + ezz) * R(1.0 / 3.0);
                em[XX] = exx - tr3;
                em[YY] = eyy - tr3;
            }
#pragma unroll
            for (int m = 0; m < NRDISS; ++m) {
#pragma unroll
                for (int c = 0; c < VM; ++c) {
                    const R x = mem(VM * m + c);
                    a.mem_w[em_index(ev, NS, VM * m + c, NP, node)] = x - a.rate[m] * (x + t3 * em[c]);
                }
            }
        }
    };
    if constexpr (EARLY) {
        if (valid) store_state();
    }

    __syncthreads();

    // ---- K8: weak divergence ----
    C Sx[3] = {0, 0, 0}, Sy[3] = {0, 0, 0}, Sz[3] = {0, 0, 0};
    {
        const C *dl = cf + 3 * P1 * P1;
        const C *dli = dl + i * P1, *dlj = dl + j * P1, *dlk = dl + k * P1;
        // x contraction: sxx, sxy, sxz feed sx, sy, sz; y: sxy, syy, syz;
        // z: sxz, syz, szz
        constexpr int comp[3][3] = {{XX, XY, XZ}, {XY, YY, YZ}, {XZ, YZ, ZZ}};
#pragma unroll
        for (int q = 0; q < P1; ++q) {
            const R *wx = ls + q + P1 * (j + P1 * k);
            const R *wy = ls + i + P1 * (q + P1 * k);
            const R *wz = ls + i + P1 * (j + P1 * q);
            const C ax = dli[q] * gs[G_SIN * P1 + q], ay = dlj[q], az = dlk[q] * gs[G_R2 * P1 + q];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                Sx[c] += ax * (C)wx[comp[0][c] * SS];
                Sy[c] += ay * (C)wy[comp[1][c] * SS];
                Sz[c] += az * (C)wz[comp[2][c] * SS];
            }
        }
    }
    const C rk = gs[G_R * P1 + k];
    const C *cw = cf + 4 * P1 * P1;
    const C Cx = cw[j] * cw[k] * rk * a.d1;
    const C Cy = cw[i] * cw[k] * rk * a.d2;
    const C Cz = cw[i] * cw[j] * gs[G_SIN * P1 + i] * a.d3;

    if (valid) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            a.force[force_index<P>(ev, c, node, a.nel)] = (R)((C)src[6 + c] + Cz * Sz[c] + Cy * Sy[c] + Cx * Sx[c]);
        if constexpr (!EARLY) store_state();
    }
}

// ---------------------------------------------------------------------------
// receivers: one wave per receiver, all its channels
// ---------------------------------------------------------------------------
// The curl formulas (src/config/channel_mod.f90:620-774 for receivers,
// src/volume_snapshot.f90:238-245 for snapshots) from the parts of a step's
// start velocity and the velocity vx, vy at its end; comp 0, 1, 2 =
// rot_vx, rot_vy, rot_vz.
__device__ inline double curl_formula(int comp, const double part[6], double vxn, double vyn, double r,
                                      double rs, double ct, double st)
{
    if (comp == 0) return -vyn / r + part[0] / rs + part[3];
    if (comp == 1) return -part[4] + (vxn - part[1]) / r;
    return (part[2] + vyn * ct - part[5] / st) / r;
}

template <typename R>
struct RecArgs {
    int n;      // receivers
    int pressure;   // some of them record the pressure (the only use of sig)
    int nx, ny, nel, nt;
    int ns;     // components of the state block
    gptr<const R> vx, vy, vz, lx, ly, lz, sig;
    gptr<const bf16> hx, hy, hz;  // BF16 velocity compensation (lx.. null) or null
    gptr<const int> rec_rot;      // curl slot per receiver, -1 none (null: no curl receivers)
    gptr<const double> rot_buf;   // per curl slot [10][NP], see curl_strain_kernel
    gptr<const int> rec_e, rec_nch, rec_off, rec_ch;  // channels of receiver r: rec_ch[rec_off[r] + q]
    gptr<const double> rec_vm;
    gptr<double> traces;          // [sum of channels][nt], receiver r's at rec_off[r]
    gptr<const int> it_dev;
    // sources, for the echo channels: slot per element (null: no sources),
    // channel row per slot and component, coefficients, source-time table
    gptr<const int> src_slot, src_chan;
    gptr<const double> src_coef, stf;
};

// Receiver r's samples of the iteration just completed, *it_dev (the node
// kernel has advanced the counter), by the 64 lanes of one wave. CURL: the
// receiver may have curl channels.
template <int P, typename R, bool CURL>
__device__ __forceinline__ void record_body(const RecArgs<R> &a, int r)
{
    constexpr int P1 = P + 1, NP = P1 * P1 * P1;
    const int it = *a.it_dev;
    if (it < 1 || it > a.nt) return;
    const int lane = threadIdx.x & 63;
    const int e = a.rec_e[r];
    const int ex = e % a.nx, ey = (e / a.nx) % a.ny, ez = e / (a.nx * a.ny);
    double acc[CURL ? 7 : 4] = {};   // vx, vy, vz, pressure, rot_vx, rot_vy, rot_vz
    const int rs = CURL && a.rec_rot ? a.rec_rot[r] : -1;
    for (int n = lane; n < NP; n += 64) {
        const int i = n % P1, j = (n / P1) % P1, k = n / (P1 * P1);
        const long u = unique_index<P>(ex, ey, ez, i, j, k, a.nx, a.ny);
        const double w = a.rec_vm[(long)r * NP + n];
        // compensated velocity: value = hi - lo
        const double vxn = (double)a.vx[u] - vel_lo(a.lx, a.hx, u);
        const double vyn = (double)a.vy[u] - vel_lo(a.ly, a.hy, u);
        acc[0] += w * vxn;
        acc[1] += w * vyn;
        acc[2] += w * ((double)a.vz[u] - vel_lo(a.lz, a.hz, u));
        if (a.pressure) {
            const double tr = (double)a.sig[em_index(e, a.ns, XX, NP, n)] + (double)a.sig[em_index(e, a.ns, YY, NP, n)] +
                              (double)a.sig[em_index(e, a.ns, ZZ, NP, n)];
            acc[3] += -((double)(1.0f / 3.0f) * tr) * w;
        }
        if constexpr (CURL) {
            if (rs >= 0) {
                // curl channels (src/config/channel_mod.f90:620-774): strain-rate
                // parts of the step's start velocity, this velocity at its end
                const double *b = a.rot_buf + (long)rs * 10 * NP + n;
                double part[6];
#pragma unroll
                for (int c = 0; c < 6; ++c) part[c] = b[c * NP];
                const double rr = b[6 * NP], rst = b[7 * NP], ct = b[8 * NP], st = b[9 * NP];
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[4 + c] += w * curl_formula(c, part, vxn, vyn, rr, rst, ct, st);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < (CURL ? 7 : 4); ++c)
        for (int off = 32; off > 0; off >>= 1) acc[c] += __shfl_down(acc[c], off, 64);
    // source-echo channels: add(it) of this step wrote, per component c with
    // a source in this element, src_c = -stf(it) * coef_c (an assignment: the
    // last source of the element wins, as in add_m** / add_f*,
    // src/config/channel_mod.f90:859-1095); record_m** / record_f* sum vm *
    // src_c (:871-1085). mxx .. mzz, fx, fy, fz; zero in other elements.
    const int slot = a.src_slot ? a.src_slot[e] : -1;
    auto echo = [&](int c) {
        double s = 0.0;
        const int ch = slot >= 0 ? a.src_chan[slot * 9 + c] : -1;
        if (ch < 0) return s;
        const double sd = a.stf[(long)ch * a.nt + (it - 1)];
        if (sd != 0.0)
            for (int n = lane; n < NP; n += 64)
                s += a.rec_vm[(long)r * NP + n] * -(sd * a.src_coef[((long)slot * 9 + c) * NP + n]);
        for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
        return s;
    };
    const int nch = a.rec_nch[r];
    const int off = a.rec_off[r];
    for (int q = 0; q < nch; ++q) {
        const int ch = a.rec_ch[off + q];
        double val = 0.0;
        switch (ch) {
        case 0: val = acc[0]; break;          // vx
        case 1: val = acc[1]; break;          // vy
        case 2: val = acc[2]; break;          // vz
        case 3: val = -acc[0]; break;         // n = -vx
        case 4: val = acc[1]; break;          // e = vy
        case 5: val = acc[2]; break;          // z = vz
        case 6: val = acc[3]; break;          // pressure
        case 7: if constexpr (CURL) val = acc[4]; break;   // rot_vx
        case 8: if constexpr (CURL) val = acc[5]; break;   // rot_vy
        case 9: if constexpr (CURL) val = acc[6]; break;   // rot_vz
        default:                              // mxx .. mzz, fx, fy, fz
            if (ch >= 10 && ch < 19) val = echo(ch - 10);
            break;
        }
        if (lane == 0) a.traces[((long)off + q) * a.nt + (it - 1)] = val;
    }
}

// Workgroups of an element launch that record the receivers of the iteration
// before it, one receiver per wave, ahead of the tiles: rounded up to a
// multiple of 8 so that the tiles' order on the XCDs stays. A receiver launch
// of its own takes 7 to 8 us of a 25 us step at 12x12x8, 13 to 20 us with 32
// to 256 receivers, almost all of it latency that the tiles hide here: with
// the step counter advanced by the node kernel a step at 12x12x8, order 4, FP64
// in captured chunks goes from 24.6 to 15.6 us.
__host__ __device__ inline int record_blocks(int receivers, int lanes)
{
    const int per = lanes / 64;
    return ((receivers + per - 1) / per + 7) / 8 * 8;
}

// Waves per SIMD that the registers must leave room for: one-element FP32
// workgroups of order 6 have 6 waves, and 3 of them fit a CU only at 5 waves
// per SIMD (96 VGPRs; with stress compensation they take 101 to 103 by
// themselves and ran 525 us at 40x36x20 with 2 workgroups per CU, 483 us with
// 3), those of order 7 have 8 waves, and 2 fit at 4 (128 VGPRs; one variant
// took 130: 566 us at 36x30x18 against 453).
template <int P, int E, typename R>
constexpr int min_waves() { return sizeof(R) == 4 && Shape<P, E>::EPB == 1 ? (P == 6 ? 5 : P == 7 ? 4 : 1) : 1; }

template <int P, int E, typename R, int VM, bool S16, int KS>
__global__ void __launch_bounds__((Shape<P, E>::NT), (min_waves<P, E, R>()))
elem_kernel(const ElemArgs<R> a, const RecArgs<R> rec)
{
    constexpr int NT = Shape<P, E>::NT;
    const int nb = record_blocks(rec.n, NT), b = (int)blockIdx.x - nb;
    if (b < 0) {
        const int r = (int)blockIdx.x * (NT / 64) + (int)(threadIdx.x >> 6);
        if (r < rec.n) record_body<P, R, false>(rec, r);
        return;
    }
    elem_body<P, E, R, VM, S16, KS>(a, chunk_block(b, gridDim.x - nb, a.remap));
}

template <int P, int E, typename R, int VM, int KS>
__global__ void __launch_bounds__((Shape<P, E>::NT), (min_waves<P, E, R>()))
elem_kernel_batch(const ElemArgs<R> *__restrict__ args, const int2 *__restrict__ own,
                  const RecArgs<R> *__restrict__ recs, const int2 *__restrict__ rown, int nrec)
{
    constexpr int NT = Shape<P, E>::NT;
    const int nb = record_blocks(nrec, NT), b = (int)blockIdx.x - nb;
    if (b < 0) {
        const int r = (int)blockIdx.x * (NT / 64) + (int)(threadIdx.x >> 6);
        if (r < nrec) record_body<P, R, false>(recs[rown[r].x], rown[r].y);
        return;
    }
    // (simulation, its workgroup index), in XCD-aware order over the whole
    // batch
    const int2 o = own[chunk_block(b, gridDim.x - nb, 1)];
    elem_body<P, E, R, VM, false, KS>(args[o.x], o.y);
}

}  // namespace s3d
