// s3d_kernels.hip -- gfx950 kernels of the forward time step.
//
// One time step (reference src/ses3d-nt.F90:240-270 around
// src/evolution.f90:87-444) is two kernels:
//
//   elem_kernel  one workgroup per EPB elements, one lane per element-local
//                node. Gathers the element's velocity into LDS, forms the
//                strain rate (K1-K4), the stress rate and the stress / memory
//                variable update (K5-K7, SLS), adds the moment-tensor glut,
//                stages the effective stress in LDS and contracts the weak
//                divergence (K8). Writes the element force, the tapered
//                stress and the memory variables; all HBM traffic coalesced.
//   node_kernel  one lane per unique node or row of them (node_rows). Sums the (up to 8) element copies
//                of the force in the reference's theta -> phi -> r order
//                (K10, src/communicate_fields.F90:48-79; deterministic, no
//                atomics), multiplies by 1/M (K9), integrates the velocity
//                (K12, optional compensated summation) and tapers it (K13).
//                Its first lane advances the step counter.
// and the receivers (one wave each: sum vm * field over the element), which
// ride in the next step's element kernel, or in record_kernel after the last
// step of a call.
//
// HBM bytes per element-local node and step (FP32, Kahan on v, visco):
//   stress 24 r + 24 w, memory variables 72 r + 72 w (60 + 60 in the
//   five-word deviatoric form), lambda/mu/tau 12 r,
//   force 12 w + 12 r, velocity ~(3 r gather) + unique-node v, lo, 1/M
//   (~24*u r + 24*u w with u = unique/element-local ~ 0.52).
#include "s3d_elem.h"

namespace s3d {

// ---------------------------------------------------------------------------
// node kernel: assembly, 1/M, velocity integration, taper
// ---------------------------------------------------------------------------
// Which form of the kernel: true for one lane per row of P nodes (row_body),
// false for one per node (node_body). Neither reaches the copy rate: the
// force copies of one node lie in up to 8 elements, 3.4 loads per node and
// component at order 2, 1.95 at order 4. A row needs P / 2 + 2.5 of them per
// node less address work, but keeps 3 P sums, velocities and compensation
// words in registers and its lanes read P words apart. Measured, lane per
// node and lane per row, in us:
//   order 2, 100x100x64, FP32 words    161  116    60x60x40, BF16  41.3 30.2
//   order 2, 60x60x30, FP64           41.5 36.4    60x60x40, none  23.5 18.7
//   order 3, 61x53x31, no words       42.4 37.5    FP32 words      58.1 62.0
//   order 4, 48x48x24, FP64            110   98    96x96x48, FP32   418  516
//   order 4, 64x60x28, no words       92.0 82.1    64x60x28, FP32   112  140
//   order 5, 37x29x19, FP64           76.1 70.9    48x40x24, FP32   106  121
//   order 6, 28x28x14, FP64           64.2 67.1    40x36x20, FP32   110  134
// Rows of few workgroups only wait longer: order 4, FP64, 6x6x4 6.4 and
// 8.6, 12x12x8 7.8 and 9.1, 20x20x14 (106 thousand rows) 15.5 and 15.5; order
// 5, 16x16x10 10.4 and 11.5, 28x28x16 (358 thousand) 24.0 and 23.9; order 3,
// 32x32x20 (206 thousand) 12.5 and 12.9; order 2, 42x42x24 (185 thousand) 13.3
// and 11.5. So rows from NODE_ROWS on, two workgroups for each CU.
constexpr long NODE_ROWS = 131072;
template <int P, typename R, int KV>
constexpr bool node_rows() { return P <= 2 || (KV == 0 && P <= 5); }

template <int P, typename R>
bool by_rows(int kv, long nblk)
{
    const bool rows = kv == 0   ? node_rows<P, R, 0>()
                      : kv == 1 ? node_rows<P, R, 1>()
                                : node_rows<P, R, 2>();
    return rows && nblk * (P * P) >= NODE_ROWS;
}

// Lanes of the node kernel of a mesh of nblk blocks.
template <int P, typename R>
long node_lanes(int kv, long nblk)
{
    return nblk * (by_rows<P, R>(kv, nblk) ? P * P : P * P * P);
}

// KV: compensated velocity integration, 0 off, 1 FP32 compensation words,
// 2 BF16 compensation words (the term carries the rounding error of the
// sum, below half an FP32 unit of it, so 8 bits of it keep the sum within
// a small fraction of that unit).
template <int P, typename R, int KV>
__device__ __forceinline__ void node_body(const NodeArgs<R> &a, long tid)
{
    constexpr int P1 = P + 1, PB = P * P * P;
    constexpr int NL = P1 * P1, NM = NL * P;   // force layout, see force_index
    if (tid >= a.nblk * PB) return;
    // the iteration is complete with this kernel: advance the step counter
    // (the element kernel has read it, the receivers read it afterwards). A
    // launch of its own for this took 4.5 us per step of a captured chunk.
    if (tid == 0) a.it_dev[0] = a.it_dev[0] + 1;
    // 32-bit index arithmetic (s3d_create keeps unique nodes below 2^32 and
    // elements below 2^31): 64-bit divisions by the run-time block counts
    // took about 40 % of the kernel's VALU instructions
    const unsigned t = (unsigned)tid;
    const unsigned b = t / PB;
    const unsigned o = t - b * PB;
    const unsigned li = o % P, lj = (o / P) % P, lk = o / (P * P);
    const unsigned nx = a.nx, ny = a.ny, nz = a.nz;
    const unsigned nbx = nx + 1, nby = ny + 1;
    const unsigned bq = b / nbx;
    const unsigned bx = b - bq * nbx, bz = bq / nby, by = bq - bz * nby;
    if ((bx == nx && li) || (by == ny && lj) || (bz == nz && lk)) return;

    // Copies: element (bx-dx, by-dy, bz-dz) at local (li+dx*P, lj+dy*P,
    // lk+dz*P), from clamped (always valid) addresses: dz = 0 in the k < p
    // part of the force, dz = 1 (lk = 0, local k = p) in the k = p layers
    // (force_index). Only present copies are loaded (lane-predicated loads:
    // an interior node, the common case, issues one load instead of eight);
    // absent ones are +0. Adding +0 is exact: the sum equals the reference's
    // theta -> phi -> r sweep.
    const bool px0 = bx < nx, px1 = li == 0 && bx > 0;
    const bool py0 = by < ny, py1 = lj == 0 && by > 0;
    const bool pz0 = bz < nz, pz1 = lk == 0 && bz > 0;
    const unsigned ex0 = bx < nx ? bx : nx - 1, ex1 = bx > 0 ? bx - 1 : 0;
    const unsigned ey0 = by < ny ? by : ny - 1, ey1 = by > 0 ? by - 1 : 0;
    const unsigned ez0 = bz < nz ? bz : nz - 1, ez1 = bz > 0 ? bz - 1 : 0;
    const long top = (long)a.nel * 3 * NM;   // start of the k = p layers
    long addr[8];
    bool pres[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const int dx = m & 1, dy = (m >> 1) & 1, dz = m >> 2;
        const unsigned e = (dx ? ex1 : ex0) + nx * ((dy ? ey1 : ey0) + ny * (dz ? ez1 : ez0));
        const unsigned i2 = li + dx * P < P ? li + dx * P : P;
        const unsigned j2 = lj + dy * P < P ? lj + dy * P : P;
        addr[m] = dz ? top + (long)e * (3 * NL) + (i2 + P1 * j2) : (long)e * (3 * NM) + (i2 + P1 * (j2 + P1 * lk));
        pres[m] = (dx ? px1 : px0) && (dy ? py1 : py0) && (dz ? pz1 : pz0);
    }
    R acc[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        R v[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) v[m] = R(0);
        v[0] = a.force[addr[0] + c * NM];   // clamped: in bounds also for a padding block
#pragma unroll
        for (int m = 1; m < 8; ++m)
            if (pres[m]) v[m] = a.force[addr[m] + c * (m < 4 ? NM : NL)];
        v[0] = pres[0] ? v[0] : R(0);
        acc[c] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    }
    const long u = tid;
    R im;
    if (a.dt_inv_mm)
        im = a.dt_inv_mm[u];
    else
        im = (R)(float)a.dt_inv_mm16[u];
    R dmp = R(0);   // 1 - taper
    if (a.taper_on) {
        const unsigned ex = bx < nx ? bx : nx - 1, i = bx < nx ? li : P;
        const unsigned ey = by < ny ? by : ny - 1, j = by < ny ? lj : P;
        const unsigned ez = bz < nz ? bz : nz - 1, k = bz < nz ? lk : P;
        dmp = (R)taper_damp(a.px[ex * P1 + i], a.py[ey * P1 + j], a.pz[ez * P1 + k], a.alpha);
    }
    R *v[3] = {a.vx, a.vy, a.vz};
    if constexpr (KV == 1) {
        R *l[3] = {a.lx, a.ly, a.lz};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            R s = v[c][u], cc = l[c][u];
            kahan_add(s, cc, acc[c] * im);
            v[c][u] = s - s * dmp;
            l[c][u] = cc - cc * dmp;
        }
    } else if constexpr (KV == 2) {
        bf16 *h[3] = {a.hx, a.hy, a.hz};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            R s = v[c][u], cc = (R)(float)h[c][u];
            kahan_add(s, cc, acc[c] * im);
            v[c][u] = s - s * dmp;
            h[c][u] = (bf16)(float)(cc - cc * dmp);
        }
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const R s = v[c][u] + acc[c] * im;
            v[c][u] = s - s * dmp;
        }
    }
}

// The same for one lane per row of P unique nodes along theta: no lane loads
// a dx = 1 copy for the first node of an element under a predicate that idles
// the rest of its wave, and the index arithmetic is done once per row. The
// lane holds the row's sums, so it only pays while these fit: see node_rows.
template <int P, typename R, int KV>
__device__ __forceinline__ void row_body(const NodeArgs<R> &a, long tid)
{
    constexpr int P1 = P + 1;
    constexpr int NL = P1 * P1, NM = NL * P;   // force layout, see force_index
    if (tid >= a.nblk * (P * P)) return;
    if (tid == 0) a.it_dev[0] = a.it_dev[0] + 1;
    const unsigned t = (unsigned)tid;
    const unsigned b = t / (P * P);
    const unsigned o = t - b * (P * P);
    const unsigned lj = o % P, lk = o / P;
    const unsigned nx = a.nx, ny = a.ny, nz = a.nz;
    const unsigned nbx = nx + 1, nby = ny + 1;
    const unsigned bq = b / nbx;
    const unsigned bx = b - bq * nbx, bz = bq / nby, by = bq - bz * nby;
    if ((by == ny && lj) || (bz == nz && lk)) return;

    // Copies of node li of the row: element (bx-dx, by-dy, bz-dz) at local
    // (li+dx*P, lj+dy*P, lk+dz*P); dx = 1 only for li = 0. dz = 0 lies in the
    // k < p part of the force, dz = 1 (lk = 0, local k = p) in the k = p layers
    // (force_index). Only present copies are loaded; absent ones are +0, and
    // adding +0 is exact: the sum equals the reference's theta -> phi -> r
    // sweep.
    const bool px0 = bx < nx, px1 = bx > 0;
    const bool py0 = by < ny, py1 = lj == 0 && by > 0;
    const bool pz0 = bz < nz, pz1 = lk == 0 && bz > 0;
    const long top = (long)a.nel * 3 * NM;   // start of the k = p layers
    R x[4][3][P], w[4][3];                   // (dy, dz): the row's values, dx = 1's
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int dy = m & 1, dz = m >> 1;
        const bool here = (dy ? py1 : py0) && (dz ? pz1 : pz0);
        const unsigned e = bx + nx * ((by - dy) + ny * (bz - dz)), j2 = dy ? P : lj;
        const long row = dz ? top + (long)e * (3 * NL) + P1 * j2 : (long)e * (3 * NM) + P1 * (j2 + P1 * lk);
        constexpr int step[2] = {NM, NL};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            w[m][c] = R(0);
#pragma unroll
            for (int i = 0; i < P; ++i) x[m][c][i] = R(0);
        }
        if (here && px0)
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int i = 0; i < P; ++i) x[m][c][i] = a.force[row + c * step[dz] + i];
        if (here && px1)   // element e - 1, the row's last node
#pragma unroll
            for (int c = 0; c < 3; ++c) w[m][c] = a.force[row - 3 * (dz ? NL : NM) + c * step[dz] + P];
    }
    const long u = (long)t * P;
    const int n = px0 ? P : 1;   // nodes of the row
    R im[P], vv[3][P], cc[3][P];
    R *v[3] = {a.vx, a.vy, a.vz};
    R *l[3] = {a.lx, a.ly, a.lz};
    bf16 *h[3] = {a.hx, a.hy, a.hz};
    // the whole row also of a padding block: its other entries exist
#pragma unroll
    for (int i = 0; i < P; ++i) im[i] = a.dt_inv_mm ? a.dt_inv_mm[u + i] : (R)(float)a.dt_inv_mm16[u + i];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int i = 0; i < P; ++i) {
            vv[c][i] = v[c][u + i];
            if constexpr (KV == 1) cc[c][i] = l[c][u + i];
            if constexpr (KV == 2) cc[c][i] = (R)(float)h[c][u + i];
        }
    R dmp[P];   // 1 - taper
#pragma unroll
    for (int i = 0; i < P; ++i) dmp[i] = R(0);
    if (a.taper_on) {
        const double py = a.py[by < ny ? by * P1 + lj : ny * P1 - 1], pz = a.pz[bz < nz ? bz * P1 + lk : nz * P1 - 1];
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const double px = a.px[px0 ? bx * P1 + i : nx * P1 - 1];
            if (px + py + pz != 0.0) dmp[i] = (R)taper_damp(px, py, pz, a.alpha);
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
#pragma unroll
        for (int i = 0; i < P; ++i) {
            R s[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) s[m] = i == 0 ? x[m][c][0] + w[m][c] : x[m][c][i];
            const R acc = (s[0] + s[1]) + (s[2] + s[3]);
            if constexpr (KV != 0)
                kahan_add(vv[c][i], cc[c][i], acc * im[i]);
            else
                vv[c][i] = vv[c][i] + acc * im[i];
            vv[c][i] = vv[c][i] - vv[c][i] * dmp[i];
            if constexpr (KV != 0) cc[c][i] = cc[c][i] - cc[c][i] * dmp[i];
        }
        if (n == P) {
#pragma unroll
            for (int i = 0; i < P; ++i) {
                v[c][u + i] = vv[c][i];
                if constexpr (KV == 1) l[c][u + i] = cc[c][i];
                if constexpr (KV == 2) h[c][u + i] = (bf16)(float)cc[c][i];
            }
        } else {
            v[c][u] = vv[c][0];
            if constexpr (KV == 1) l[c][u] = cc[c][0];
            if constexpr (KV == 2) h[c][u] = (bf16)(float)cc[c][0];
        }
    }
}

template <int P, typename R, int KV>
__device__ __forceinline__ void assemble(const NodeArgs<R> &a, long tid)
{
    if constexpr (node_rows<P, R, KV>())
        if (a.rows) return row_body<P, R, KV>(a, tid);
    node_body<P, R, KV>(a, tid);
}

// Workgroups in the element kernel's order (chunk_block), so that they read
// the force from the L2 that its XCD wrote it to, and walk HBM as one window:
// in plain order order 6, 40x36x20 took 115 us (now 109), order 7, 36x30x18
// 109 (103), order 3, 61x53x31 44.8 (41.9), order 4, 24x24x16 15.4 (14.0);
// order 4, 96x96x48 416 (418).
template <int P, typename R, int KV>
__global__ void __launch_bounds__(256)
node_kernel(const NodeArgs<R> a)
{
    const long tid = (long)chunk_block(blockIdx.x, gridDim.x, ORDER_CHUNKS) * blockDim.x + threadIdx.x;
    assemble<P, R, KV>(a, tid);
}

template <int P, typename R, int KV>
__global__ void __launch_bounds__(256)
node_kernel_batch(const NodeArgs<R> *__restrict__ args, const int2 *__restrict__ own)
{
    const int2 o = own[blockIdx.x];
    const long tid = (long)o.y * blockDim.x + threadIdx.x;
    assemble<P, R, KV>(args[o.x], tid);
}

// Strain-rate parts of the curl receiver channels (reference record_rot_v*,
// src/config/channel_mod.f90:620-774, which read the step's strain-rate
// arrays): for each curl receiver's element, from the velocity at the start
// of the step (hi - lo, FP64), the raw derivatives (src/evolution.f90:126-159),
// their spherical completion (:165-173) and the symmetrisation (:206-208) as
// the step forms them; stored per node: EYZ, EZY, EZX, EXZ, EXY, EYX (EYZ,
// EXZ, EXY symmetrised; EZY, EZX, EYX completed only), r, r sin(theta),
// cot(theta), sin(theta). Launched before the node kernel updates v.
template <typename R>
struct CurlArgs {
    int nx, ny, nrot;
    gptr<const R> vx, vy, vz, lx, ly, lz;
    gptr<const bf16> hx, hy, hz;   // BF16 velocity compensation (lx.. null) or null
    gptr<const ThTab<double>> tth;
    gptr<const RTab<double>> tr;
    gptr<const int> rot_e;       // element of each curl slot
    gptr<double> buf;            // [nrot][10][NP]
    double Dx[MAXP1 * MAXP1], Dy[MAXP1 * MAXP1], Dz[MAXP1 * MAXP1];   // D[i*P1 + q] = 2 l'_q(xi_i) / d
};

template <typename R>
__device__ __forceinline__ double curl_vel(gptr<const R> v, gptr<const R> l, gptr<const bf16> h, long u)
{
    return (double)v[u] - vel_lo(l, h, u);
}

// The strain-rate parts the curl formulas use, at node (i, j, k) of element
// (ex, ey, ez), from the current velocity: eyz, exz, exy as the step's
// symmetrisation leaves them and ezy, ezx, eyx as its spherical completion
// leaves them (src/evolution.f90:165-208), in that order in part[0..5].
template <int P, typename R>
__device__ inline void curl_parts(const CurlArgs<R> &a, int ex, int ey, int ez, int i, int j, int k,
                                  double part[6])
{
    constexpr int P1 = P + 1;
    double exy = 0.0, exz = 0.0, eyx = 0.0, eyz = 0.0, ezx = 0.0, ezy = 0.0;
    for (int q = 0; q < P1; ++q) {
        const double d1 = a.Dx[i * P1 + q];
        const long u = unique_index<P>(ex, ey, ez, q, j, k, a.nx, a.ny);
        exy = exy + curl_vel(a.vy, a.ly, a.hy, u) * d1;
        exz = exz + curl_vel(a.vz, a.lz, a.hz, u) * d1;
    }
    for (int q = 0; q < P1; ++q) {
        const double d2 = a.Dy[j * P1 + q];
        const long u = unique_index<P>(ex, ey, ez, i, q, k, a.nx, a.ny);
        eyx = eyx + curl_vel(a.vx, a.lx, a.hx, u) * d2;
        eyz = eyz + curl_vel(a.vz, a.lz, a.hz, u) * d2;
    }
    for (int q = 0; q < P1; ++q) {
        const double d3 = a.Dz[k * P1 + q];
        const long u = unique_index<P>(ex, ey, ez, i, j, q, a.nx, a.ny);
        ezx = ezx + curl_vel(a.vx, a.lx, a.hx, u) * d3;
        ezy = ezy + curl_vel(a.vy, a.ly, a.hy, u) * d3;
    }
    const long u = unique_index<P>(ex, ey, ez, i, j, k, a.nx, a.ny);
    const double vxn = curl_vel(a.vx, a.lx, a.hx, u), vyn = curl_vel(a.vy, a.ly, a.hy, u);
    const double r = a.tr[ez * P1 + k].r, st = a.tth[ex * P1 + i].sin_t, ct = a.tth[ex * P1 + i].cot;
    const double rs = r * st;
    ezx = -ezx;
    exz = (exz - vxn) / r;
    ezy = -ezy;
    eyz = -vyn / r + eyz / rs;
    exy = exy / r;
    eyx = -(vyn * ct) / r + eyx / rs;
    part[0] = (eyz + ezy) / 2.0;
    part[1] = (exz + ezx) / 2.0;
    part[2] = (exy + eyx) / 2.0;
    part[3] = ezy;
    part[4] = ezx;
    part[5] = eyx;
}

template <int P, typename R>
__global__ void __launch_bounds__(64) curl_strain_kernel(const CurlArgs<R> a)
{
    constexpr int P1 = P + 1, NP = P1 * P1 * P1;
    const int s = blockIdx.x;
    if (s >= a.nrot) return;
    const int e = a.rot_e[s];
    const int ex = e % a.nx, ey = (e / a.nx) % a.ny, ez = e / (a.nx * a.ny);
    for (int n = threadIdx.x; n < NP; n += 64) {
        const int i = n % P1, j = (n / P1) % P1, k = n / (P1 * P1);
        double part[6];
        curl_parts<P, R>(a, ex, ey, ez, i, j, k, part);
        const double r = a.tr[ez * P1 + k].r, st = a.tth[ex * P1 + i].sin_t, ct = a.tth[ex * P1 + i].cot;
        double *b = a.buf + (long)s * 10 * NP + n;
#pragma unroll
        for (int c = 0; c < 6; ++c) b[c * NP] = part[c];
        b[6 * NP] = r;
        b[7 * NP] = r * st;
        b[8 * NP] = ct;
        b[9 * NP] = st;
    }
}

// Volume curl fields, first half: the parts of every element-local node from
// the current velocity (the start velocity of the next step), element-major
// parts[e][6][NP]. One workgroup per element.
template <int P, typename R>
__global__ void __launch_bounds__(64) curl_parts_kernel(const CurlArgs<R> a, long nel, double *parts)
{
    constexpr int P1 = P + 1, NP = P1 * P1 * P1;
    const long e = blockIdx.x;
    if (e >= nel) return;
    const int ex = (int)(e % a.nx), ey = (int)((e / a.nx) % a.ny), ez = (int)(e / ((long)a.nx * a.ny));
    for (int n = threadIdx.x; n < NP; n += 64) {
        const int i = n % P1, j = (n / P1) % P1, k = n / (P1 * P1);
        double part[6];
        curl_parts<P, R>(a, ex, ey, ez, i, j, k, part);
#pragma unroll
        for (int c = 0; c < 6; ++c) parts[(e * 6 + c) * NP + n] = part[c];
    }
}

// Volume curl fields, second half: rot_v{x,y,z} (comp 0, 1, 2) of node n of
// element e from the stored parts and the current velocity (a source of
// export_field).
template <int P, typename R>
struct CurlSrc {
    CurlArgs<R> a;
    gptr<const double> parts;
    int comp;
    __device__ double operator()(long e, int n) const
    {
        constexpr int P1 = P + 1, NP = P1 * P1 * P1;
        const int ex = (int)(e % a.nx), ey = (int)((e / a.nx) % a.ny), ez = (int)(e / ((long)a.nx * a.ny));
        const int i = n % P1, j = (n / P1) % P1, k = n / (P1 * P1);
        double part[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) part[c] = parts[(e * 6 + c) * NP + n];
        const long u = unique_index<P>(ex, ey, ez, i, j, k, a.nx, a.ny);
        const double vxn = curl_vel(a.vx, a.lx, a.hx, u), vyn = curl_vel(a.vy, a.ly, a.hy, u);
        const double r = a.tr[ez * P1 + k].r, st = a.tth[ex * P1 + i].sin_t, ct = a.tth[ex * P1 + i].cot;
        return curl_formula(comp, part, vxn, vyn, r, r * st, ct, st);
    }
};

// The receivers' own launch: after the last step of a call, and after every
// step where the element kernel of the next one cannot record (curl channels,
// or a stress block updated in place).
template <int P, typename R>
__global__ void __launch_bounds__(64) record_kernel(const RecArgs<R> a)
{
    record_body<P, R, true>(a, blockIdx.x);
}

template <int P, typename R>
__global__ void __launch_bounds__(64) record_kernel_batch(const RecArgs<R> *__restrict__ args, const int2 *__restrict__ own)
{
    const int2 o = own[blockIdx.x];
    record_body<P, R, true>(args[o.x], o.y);
}

// ---------------------------------------------------------------------------
// setup and I/O kernels
// ---------------------------------------------------------------------------

// Fields to and from the host. The host side is the reference layout [n][e]
// (FP64, e fastest), the device fields are element-major or on unique nodes,
// so both directions transpose a tile of IO_E elements x IO_N nodes in LDS:
// device memory is read and written along the nodes of an element, the host
// image along the elements. The host image is one chunk of the field in
// pinned host memory (nodes n0 .. n0+nn-1, elements e0 .. e0+ne-1,
// chunk[(n - n0) * ne + (e - e0)]), which the kernels read and write directly,
// 256 B per half wave: no device copy of the field, no separate transfer. What
// bounds them is the host link. (With one lane per value in host order and a
// device buffer, at 96x96x48, order 4, the conversion alone took 1.0 ms for a
// stress component, 2.1 ms for a velocity component.)
constexpr int IO_E = 32, IO_N = 64;

// Sources: value of node n of element e.
// One component of an element-major block of nc components, less its FP32
// compensation words (lo null: none).
template <typename R>
struct BlockSrc {
    gptr<const R> p, lo;
    int nc, NP;
    __device__ double operator()(long e, int n) const
    {
        const long a = e * nc * NP + n;
        return lo ? (double)p[a] - (double)lo[a] : (double)p[a];
    }
};

// The same with BF16 compensation words in pairs.
struct PairSrc {
    gptr<const float> p;
    gptr<const unsigned> lo;
    int half, nc, NP;
    __device__ double operator()(long e, int n) const
    {
        const long a = e * nc * NP + n;
        const unsigned w = lo[a];
        return (double)p[a] - (double)(half ? bf16_hi(w) : bf16_lo(w));
    }
};

// zz of a deviatoric memory variable
template <typename R>
struct DeviatorSrc {
    gptr<const R> xx, yy;
    int nc, NP;
    __device__ double operator()(long e, int n) const
    {
        const long a = e * nc * NP + n;
        return -((double)xx[a] + (double)yy[a]);
    }
};

template <int P, typename R>
struct UniqueSrc {
    gptr<const R> v, lo;
    gptr<const bf16> lo16;
    int nx, ny;
    __device__ double operator()(long e, int n) const
    {
        constexpr int P1 = P + 1;
        const int i = n % P1, j = (n / P1) % P1, k = n / (P1 * P1);
        const int ex = (int)(e % nx), ey = (int)((e / nx) % ny), ez = (int)(e / ((long)nx * ny));
        const long u = unique_index<P>(ex, ey, ez, i, j, k, nx, ny);
        return (double)v[u] - vel_lo(lo, lo16, u);
    }
};

template <typename Src>
__global__ void __launch_bounds__(256) export_field(const Src src, long e0, int ne, int n0, int nn, double *chunk)
{
    __shared__ double tile[IO_N][IO_E + 1];
    const int eb = blockIdx.x * IO_E, nb = blockIdx.y * IO_N;
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int q = threadIdx.x >> 6; q < IO_E; q += 4)
        if (eb + q < ne && nb + l < nn) tile[l][q] = src(e0 + eb + q, n0 + nb + l);
    __syncthreads();
    const int e = eb + (threadIdx.x & 31);
#pragma unroll
    for (int q = threadIdx.x >> 5; q < IO_N; q += 8)
        if (e < ne && nb + q < nn) chunk[(long)(nb + q) * ne + e] = tile[q][threadIdx.x & 31];
}

// Destinations: store the value of node n of element e.
// One component of an element-major block of nc components; its FP32
// compensation word (lo not null) becomes zero.
template <typename R>
struct BlockDst {
    gptr<R> p, lo;
    int nc, NP;
    __device__ void operator()(long e, int n, double x) const
    {
        const long a = e * nc * NP + n;
        p[a] = (R)x;
        if (lo) lo[a] = R(0);
    }
};

// The same with BF16 compensation words in pairs: the component's half.
struct PairDst {
    gptr<float> p;
    gptr<unsigned> lo;
    int half, nc, NP;
    __device__ void operator()(long e, int n, double x) const
    {
        const long a = e * nc * NP + n;
        p[a] = (float)x;
        lo[a] &= half ? 0x0000ffffu : 0xffff0000u;
    }
};

// A unique-node field takes the owner element's copy of a node: the element
// whose block holds it, the last element on the far domain faces.
template <int P, typename R>
struct UniqueDst {
    gptr<R> v, lo;
    gptr<bf16> lo16;
    int nx, ny, nz;
    __device__ void operator()(long e, int n, double x) const
    {
        constexpr int P1 = P + 1;
        const int i = n % P1, j = (n / P1) % P1, k = n / (P1 * P1);
        const int ex = (int)(e % nx), ey = (int)((e / nx) % ny), ez = (int)(e / ((long)nx * ny));
        if ((i == P && ex < nx - 1) || (j == P && ey < ny - 1) || (k == P && ez < nz - 1)) return;
        const long u = unique_index<P>(ex, ey, ez, i, j, k, nx, ny);
        v[u] = (R)x;
        if (lo) lo[u] = (R)(x - (double)(R)x) * R(-1);
        if (lo16) lo16[u] = (bf16)(float)(-(x - (double)(R)x));
    }
};

template <typename Dst>
__global__ void __launch_bounds__(256) import_field(const Dst dst, long e0, int ne, int n0, int nn, const double *chunk)
{
    __shared__ double tile[IO_N][IO_E + 1];
    const int eb = blockIdx.x * IO_E, nb = blockIdx.y * IO_N;
    const int e = eb + (threadIdx.x & 31);
#pragma unroll
    for (int q = threadIdx.x >> 5; q < IO_N; q += 8)
        if (e < ne && nb + q < nn) tile[q][threadIdx.x & 31] = chunk[(long)(nb + q) * ne + e];
    __syncthreads();
    const int l = threadIdx.x & 63;
#pragma unroll
    for (int q = threadIdx.x >> 6; q < IO_E; q += 4)
        if (eb + q < ne && nb + l < nn) dst(e0 + eb + q, n0 + nb + l, tile[l][q]);
}

// Adjoint density sensitivity (reference ses3d_grad,
// src/SOURCE/ses3d_grad.F90:212-213): g += inc_dt * (fx*vx + fy*vy + fz*vz) / jac
// for the nodes and elements of one chunk of the forward snapshot in pinned
// host memory (three components, see import_field), the velocity (hi - lo)
// gathered from the unique nodes, g element-major [e][NP].
template <int P, typename R>
struct GradArgs {
    gptr<double> g;
    UniqueSrc<P, R> v[3];
    double inc_dt, jac;
};

template <int P, typename R>
__global__ void __launch_bounds__(256) grad_rho_kernel(const GradArgs<P, R> a, long e0, int ne, int n0, int nn,
                                                       const double *chunk)
{
    constexpr int NP = (P + 1) * (P + 1) * (P + 1);
    __shared__ double tile[3][IO_N][IO_E + 1];
    const int eb = blockIdx.x * IO_E, nb = blockIdx.y * IO_N;
    const int el = eb + (threadIdx.x & 31);
    for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int q = threadIdx.x >> 5; q < IO_N; q += 8)
            if (el < ne && nb + q < nn)
                tile[c][q][threadIdx.x & 31] = chunk[((long)c * nn + nb + q) * ne + el];
    __syncthreads();
    const int l = threadIdx.x & 63;
    for (int q = threadIdx.x >> 6; q < IO_E; q += 4)
        if (eb + q < ne && nb + l < nn) {
            const long e = e0 + eb + q;
            const int n = n0 + nb + l;
            const double ax = a.v[0](e, n), ay = a.v[1](e, n), az = a.v[2](e, n);
            a.g[e * NP + n] = a.g[e * NP + n] +
                              a.inc_dt * ((tile[0][l][q] * ax + tile[1][l][q] * ay) + tile[2][l][q] * az) / a.jac;
        }
}

// FP64 -> storage precision (BF16 through the nearest float)
template <typename S>
__device__ inline S narrow(double x)
{
    if constexpr (sizeof(S) == 2)
        return (S)(float)x;
    else
        return (S)x;
}

__global__ void __launch_bounds__(256) fill_kernel(double *p, long n, double x)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = x;
}

// Material from the FP64 staging arrays (element-major, as all that follow:
// the set-up kernels then read and write along the nodes; in the reference
// layout every lane fetched a line of its own): tau
// (= 6.0814 Q^-1.015, src/model_paras.F90:407), rho, dt*A, dt*B, dt*C and the
// moduli times dt, elastic: lambda, mu; visco-elastic (dtau non-null):
// kappa - 2 mu_tau / 3 = lambda - 2/3 tau mu and mu_tau = mu (1 + tau)
// (src/evolution.f90:216-284). All formed in FP64 and rounded once: a
// constant tau makes 1 + tau the same number in every node of a region, and
// an FP32 rounding of it would be a systematic modulus error.
template <typename R, typename S>
__global__ void material_kernel(const double *rhoinv, const double *lam, const double *mu,
                                const double *q, const double *A, const double *B, const double *C,
                                S *dlam, S *dmu, S *dtau, R *drho, S *dA, S *dB, S *dC,
                                long nel, int NP, int ncm, double dt)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nel * NP) return;
    long e = t / NP;
    int n = (int)(t - e * NP);
    const long s = t;
    long tm = em_index(e, ncm, 0, NP, n);   // lam/mu/tau: element-major block of ncm
    const double l = lam ? lam[s] : 0.0, m = mu ? mu[s] : 0.0;
    if (dtau) {
        double qq = q ? q[s] : 1.79769313486231570815e+308;
        const double tau = (double)6.0814f * pow(qq, (double)-1.015f);
        dtau[tm] = narrow<S>(tau);
        dlam[tm] = narrow<S>(dt * (l - (2.0 / 3.0) * tau * m));
        dmu[tm] = narrow<S>(dt * (m * (1.0 + tau)));
    } else {
        dlam[tm] = narrow<S>(dt * l);
        dmu[tm] = narrow<S>(dt * m);
    }
    double ri = rhoinv ? rhoinv[s] : 0.0;
    drho[t] = (R)(ri > 0.0 ? 1.0 / ri : 0.0);
    if (dA) {
        dA[t] = A ? narrow<S>(dt * A[s]) : narrow<S>(0.0);
        dB[t] = B ? narrow<S>(dt * B[s]) : narrow<S>(0.0);
        dC[t] = C ? narrow<S>(dt * C[s]) : narrow<S>(0.0);
    }
}

// Mass matrix -J r^2 sin(theta) rho W per copy (src/model_paras.F90:411),
// assembled with the same theta -> phi -> r summation tree as the force.
// Stores M (FP64) and dt/M (storage precision S).
template <int P, typename S>
__global__ void mass_kernel(const double *rhoinv, const double *sin_t, const double *rad,
                            const double *w, double jac, double dt, double *mm64, S *dt_inv_mm,
                            int nx, int ny, int nz, long nblk)
{
    constexpr int P1 = P + 1, PB = P * P * P;
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long b = t / PB;
    int o = (int)(t - b * PB);
    if (b >= nblk) return;
    int li = o % P, lj = (o / P) % P, lk = o / (P * P);
    int nbx = nx + 1, nby = ny + 1;
    int bx = (int)(b % nbx), by = (int)((b / nbx) % nby), bz = (int)(b / ((long)nbx * nby));
    if ((bx == nx && li) || (by == ny && lj) || (bz == nz && lk)) {
        dt_inv_mm[t] = narrow<S>(0.0);
        mm64[t] = 0.0;
        return;
    }
    bool px[2] = {bx < nx, li == 0 && bx > 0};
    bool py[2] = {by < ny, lj == 0 && by > 0};
    bool pz[2] = {bz < nz, lk == 0 && bz > 0};
    double zsum = 0;
    bool zhas = false;
    for (int dz = 0; dz < 2; ++dz) {
        if (!pz[dz]) continue;
        double ysum = 0;
        bool yhas = false;
        for (int dy = 0; dy < 2; ++dy) {
            if (!py[dy]) continue;
            double xsum = 0;
            bool xhas = false;
            for (int dx = 0; dx < 2; ++dx) {
                if (!px[dx]) continue;
                int ex = bx - dx, ey = by - dy, ez = bz - dz;
                int i = li + dx * P, j = lj + dy * P, k = lk + dz * P;
                long e = ex + (long)nx * (ey + (long)ny * ez);
                int n = i + P1 * (j + P1 * k);
                double ri = rhoinv ? rhoinv[e * (P1 * P1 * P1) + n] : 0.0;
                double rho = ri > 0.0 ? 1.0 / ri : 0.0;
                double r = rad[ez * P1 + k];
                double ww = w[i] * w[j] * w[k];
                double val = -(jac * (r * r) * sin_t[ex * P1 + i] * rho * ww);
                xsum = xhas ? xsum + val : val;
                xhas = true;
            }
            ysum = yhas ? ysum + xsum : xsum;
            yhas = true;
        }
        zsum = zhas ? zsum + ysum : ysum;
        zhas = true;
    }
    mm64[t] = zsum;
    dt_inv_mm[t] = narrow<S>(zsum != 0.0 ? dt / zsum : 0.0);
}

// Courant number partial maxima (src/model_paras.F90:529-561), FP64.
template <int P>
__global__ void cfl_kernel(const double *rhoinv, const double *lam, const double *mu,
                           const double *theta, const double *phi, const double *rad,
                           int nx, int ny, int nz, double *partial)
{
    constexpr int P1 = P + 1, NP = P1 * P1 * P1;
    const long nel = (long)nx * ny * nz;
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double m[3] = {0, 0, 0};
    if (t < nel * NP) {
        const long e = t / NP, n = t - e * NP;
        int i = (int)(n % P1), j = (int)((n / P1) % P1), k = (int)(n / (P1 * P1));
        int ex = (int)(e % nx), ey = (int)((e / nx) % ny), ez = (int)(e / ((long)nx * ny));
        double ri = rhoinv ? rhoinv[t] : 0.0;
        double l = lam ? lam[t] : 0.0, u = mu ? mu[t] : 0.0;
        double cp = sqrt((l + 2.0 * u) * ri), cs = sqrt(u * ri);
        double vmax = cs < cp ? cp : cs;
        double r = rad[ez * P1 + k];
        if (i >= 1) m[0] = vmax / (r * (theta[ex * P1 + i] - theta[ex * P1 + i - 1]));
        if (j >= 1) m[1] = vmax / (r * sin(theta[ex * P1 + i]) * (phi[ey * P1 + j] - phi[ey * P1 + j - 1]));
        if (k >= 1) m[2] = vmax / (rad[ez * P1 + k - 1] - r);
    }
    __shared__ double sm[3][256];
    for (int c = 0; c < 3; ++c) sm[c][threadIdx.x] = m[c];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int c = 0; c < 3; ++c)
                sm[c][threadIdx.x] = fmax(sm[c][threadIdx.x], sm[c][threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int c = 0; c < 3; ++c) partial[blockIdx.x * 3 + c] = sm[c][0];
}

// v range and kinetic energy partials over unique / element-local nodes
template <int P, typename R>
__global__ void vrange_kernel(const R *vx, const R *vy, const R *vz, int nx, int ny, int nz,
                              long nblk, double *partial)
{
    constexpr int PB = P * P * P;
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long b = t / PB;
    int o = (int)(t - b * PB);
    double mn = 1e308, mx = -1e308;
    if (b < nblk) {
        int li = o % P, lj = (o / P) % P, lk = o / (P * P);
        int nbx = nx + 1, nby = ny + 1;
        int bx = (int)(b % nbx), by = (int)((b / nbx) % nby), bz = (int)(b / ((long)nbx * nby));
        if (!((bx == nx && li) || (by == ny && lj) || (bz == nz && lk))) {
            double a0 = vx[t], a1 = vy[t], a2 = vz[t];
            mn = fmin(a0, fmin(a1, a2));
            mx = fmax(a0, fmax(a1, a2));
        }
    }
    __shared__ double s0[256], s1[256];
    s0[threadIdx.x] = mn;
    s1[threadIdx.x] = mx;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            s0[threadIdx.x] = fmin(s0[threadIdx.x], s0[threadIdx.x + s]);
            s1[threadIdx.x] = fmax(s1[threadIdx.x], s1[threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = s0[0];
        partial[2 * blockIdx.x + 1] = s1[0];
    }
}

// min and max over n partial (min, max) pairs, one workgroup of 256 lanes;
// the result pair goes to out[0], out[1]
__global__ void __launch_bounds__(256) range_reduce_kernel(const double *partial, int n, double *out)
{
    double mn = 1e308, mx = -1e308;
    for (int q = threadIdx.x; q < n; q += 256) {
        mn = fmin(mn, partial[2 * q]);
        mx = fmax(mx, partial[2 * q + 1]);
    }
    __shared__ double s0[256], s1[256];
    s0[threadIdx.x] = mn;
    s1[threadIdx.x] = mx;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            s0[threadIdx.x] = fmin(s0[threadIdx.x], s0[threadIdx.x + s]);
            s1[threadIdx.x] = fmax(s1[threadIdx.x], s1[threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = s0[0];
        out[1] = s1[0];
    }
}

template <int P, typename R>
__global__ void kinetic_kernel(const R *vx, const R *vy, const R *vz, const R *rho,
                               const ThTab<coef_t<R>> *tth, const RTab<coef_t<R>> *tr, const double *w,
                               int nx, int ny, int nz, double *partial)
{
    constexpr int P1 = P + 1, NP = P1 * P1 * P1;
    const long nel = (long)nx * ny * nz;
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double acc = 0.0;
    if (t < nel * NP) {
        long e = t / NP;
        int n = (int)(t - e * NP);
        int i = n % P1, j = (n / P1) % P1, k = n / (P1 * P1);
        int ex = (int)(e % nx), ey = (int)((e / nx) % ny), ez = (int)(e / ((long)nx * ny));
        long u = unique_index<P>(ex, ey, ez, i, j, k, nx, ny);
        double a0 = vx[u], a1 = vy[u], a2 = vz[u];
        double r = (double)tr[ez * P1 + k].r;
        acc = (a0 * a0 + a1 * a1 + a2 * a2) * (r * r * (double)tth[ex * P1 + i].sin_t) *
              (double)rho[t] * (w[i] * w[j] * w[k]);
    }
    __shared__ double s0[256];
    s0[threadIdx.x] = acc;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) s0[threadIdx.x] += s0[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = s0[0];
}

}  // namespace s3d
