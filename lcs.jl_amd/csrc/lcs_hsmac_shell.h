// The passes around the sweeps of HSMAC in divergence form (lcs_hsmac_div.h):
// refresh, face slabs of the overlap order, and the update of U, V, W, P.  Each
// function is one thread's work, tid its index in a workgroup of 256.
//
// __host__ __device__ so that a host harness runs the same code against the oracle.
#pragma once

#include "lcs_hsmac_div.h"

namespace lcs {

// ---- refresh --------------------------------------------------------------------
// one thread per cell of the shell (dv_refresh_cells)
template <typename T>
__host__ __device__ inline void dv_refresh_block(const Geom &g, const DvCoef<T> &c, const T *Do, const T *Fo, T *Dn, T *Fn, T *P,
                                        T *planes, T dti, int accumulate, int blk, int tid)
{
    long n[3];
    dv_refresh_cells(g, n);
    int t = blk * 256 + tid;
    if (t >= n[0] + n[1] + n[2]) return;
    const int h = g.h, sx = (int)g.sx, sy = (int)g.sy;
    auto layer = [h](int q, int m) { return q <= h ? q : m + q - 2; };  // 0..h, then m+h-1..m+2h-1
    int x, y, z;
    if (t < n[0]) {
        x = t % sx;
        t /= sx;
        y = t % sy;
        z = layer(t / sy, g.nz);
    } else if (t < n[0] + n[1]) {
        t -= (int)n[0];
        x = t % sx;
        t /= sx;
        y = layer(t % (2 * h + 2), g.ny);
        z = h + 1 + t / (2 * h + 2);
    } else {
        t -= (int)(n[0] + n[1]);
        x = layer(t % (2 * h + 2), g.nx);
        t /= 2 * h + 2;
        y = h + 1 + t % (g.ny - 2);
        z = h + 1 + t / (g.ny - 2);
    }
    dv_refresh_cell(g, c, dv_planes(g), Do, Fo, Dn, Fn, P, planes, dti, accumulate, x, y, z);
}

// ---- face slabs of the overlap order -----------------------------------------------
// Both colours over the two slabs of one axis (AXIS 0: z, 1: y, 2: x, in the
// reference's order), one thread per column across the slabs' three layers.
// dp goes to the axis's plane buffer; D is left as it is until k_dv_face_apply
// adds the corrections of all three axes, and the cells next to a slab of an
// earlier axis add that slab's corrections as they are read.
template <typename T>
struct DvFaces {
    Geom g;
    T *planes;
    DvPlanes pl;
    int px;  // row pitch of D and F
    __host__ __device__ long at(int i, int j, int k) const
    {
        return (long)(i + g.h - 1) + (long)px * ((j + g.h - 1) + g.sy * (long)(k + g.h - 1));
    }
    __host__ __device__ T *buf(int axis) const { return planes + pl.dp[2 - axis]; }
    // dp of the slab layers around a cell: layer t of slab s
    __host__ __device__ T z(int s, int t, int i, int j) const
    {
        return buf(0)[((long)(s * 3 + t) * (g.ny + 5) + (j + 1)) * (g.nx + 5) + (i + 1)];
    }
    __host__ __device__ T y(int s, int t, int i, int k) const
    {
        return buf(1)[((long)(s * 3 + t) * (g.nz - 1) + (k - 2)) * (g.nx + 5) + (i + 1)];
    }
    __host__ __device__ T x(int s, int t, int j, int k) const
    {
        return buf(2)[((long)(s * 3 + t) * (g.nz - 1) + (k - 2)) * (g.ny - 1) + (j - 2)];
    }
    // slab and layer of coordinate c on an axis of n cells; false in the core
    __host__ __device__ static bool layer(int c, int n, int &s, int &t)
    {
        s = c > 1;
        t = s ? c - n - 1 : c + 1;
        return c <= 1 || c >= n + 1;
    }
    // dp of any shell cell; 0 in the core and outside domain 1
    __host__ __device__ T dp(int i, int j, int k) const
    {
        if (i < -1 || i > g.nx + 3 || j < -1 || j > g.ny + 3 || k < -1 || k > g.nz + 3) return T(0);
        int s, t;
        if (layer(k, g.nz, s, t)) return z(s, t, i, j);
        if (layer(j, g.ny, s, t)) return y(s, t, i, k);
        if (layer(i, g.nx, s, t)) return x(s, t, j, k);
        return T(0);
    }
};

// STRIDE: nblk workgroups walk the columns; without it each column has its
// thread (a loop that ends after one turn cost the x slabs 0.8 of 4.9 us at 32^3).
template <typename T, int AXIS, bool STRIDE>
__host__ __device__ inline double dv_face_block(const DvFaces<T> &f, const T *D, const DvCoef<T> &c, int want_sum, int blk,
                                                int nblk, int tid)
{
    const Geom &g = f.g;
    // lateral ranges: l1 is the unit-stride index of the buffer
    const int lo1 = AXIS == 2 ? 2 : -1, hi1 = AXIS == 2 ? g.ny : g.nx + 3;
    const int lo2 = AXIS == 0 ? -1 : 2, hi2 = AXIS == 0 ? g.ny + 3 : g.nz;
    const int n1 = hi1 - lo1 + 1, n2 = hi2 - lo2 + 1, n = AXIS == 0 ? g.nz : (AXIS == 1 ? g.ny : g.nx);
    double acc = 0.0;
    for (int t0 = blk * 256 + tid; t0 < 2 * n1 * n2; t0 += nblk * 256) {
        const int s = t0 >= n1 * n2, u = s ? t0 - n1 * n2 : t0;
        const int l1 = lo1 + u % n1, l2 = lo2 + u / n1;
        const T ca = AXIS == 0 ? c.cz : (AXIS == 1 ? c.cy : c.cx);
        const T c1 = AXIS == 2 ? c.cy : c.cx, c2 = AXIS == 0 ? c.cy : c.cz;
        const int a0 = s ? n + 1 : -1;
        // Latency bounds this launch on small boxes: D of the three layers of the
        // column and of its four lateral neighbours (clamped into the slab) is loaded
        // at once, and so are the corrections of the slabs of earlier axes, which
        // only columns beside an edge have.  32^3 FP32, x, y, z slabs: 4.9, 3.7 and
        // 3.7 us; loaded by layer and parity, with a wait each: 9.7, 6.3 and 4.7 us.
        const int m1[5] = {l1, l1 > lo1 ? l1 - 1 : l1, l1 < hi1 ? l1 + 1 : l1, l1, l1};
        const int m2[5] = {l2, l2, l2, l2 > lo2 ? l2 - 1 : l2, l2 < hi2 ? l2 + 1 : l2};
        auto cell = [&](int t, int q, int &i, int &j, int &k) {
            i = AXIS == 2 ? a0 + t : m1[q];
            j = AXIS == 2 ? m1[q] : (AXIS == 1 ? a0 + t : m2[q]);
            k = AXIS == 0 ? a0 + t : m2[q];
        };
        T v[3][5];
#pragma unroll
        for (int t = 0; t < 3; t++)
#pragma unroll
            for (int q = 0; q < 5; q++) {
                int i, j, k;
                cell(t, q, i, j, k);
                v[t][q] = D[f.at(i, j, k)];
            }
        if (AXIS >= 1 && (l2 <= 3 || l2 >= g.nz - 1)) {
            T z[3][5];
#pragma unroll
            for (int t = 0; t < 3; t++)
#pragma unroll
                for (int q = 0; q < 5; q++) {
                    int i, j, k;
                    cell(t, q, i, j, k);
                    z[t][q] = k == g.nz ? f.z(1, 0, i, j) : f.z(0, 2, i, j);
                }
#pragma unroll
            for (int t = 0; t < 3; t++)
#pragma unroll
                for (int q = 0; q < 5; q++)
                    if (m2[q] == 2 || m2[q] == g.nz) v[t][q] -= c.cz * z[t][q];
        }
        if (AXIS == 2 && (l1 <= 3 || l1 >= g.ny - 1)) {
            T y[3][5];
#pragma unroll
            for (int t = 0; t < 3; t++)
#pragma unroll
                for (int q = 0; q < 5; q++) {
                    int i, j, k;
                    cell(t, q, i, j, k);
                    y[t][q] = j == g.ny ? f.y(1, 0, i, k) : f.y(0, 2, i, k);
                }
#pragma unroll
            for (int t = 0; t < 3; t++)
#pragma unroll
                for (int q = 0; q < 5; q++)
                    if (m1[q] == 2 || m1[q] == g.ny) v[t][q] -= c.cy * y[t][q];
        }
        const int par = (a0 + l1 + l2) & 1;  // layer t is red when (t + par) is even
        T d[3], lat[3];
#pragma unroll
        for (int t = 0; t < 3; t++) {  // lateral red corrections, used by the black layers
            d[t] = v[t][0];
            T s1 = T(0), s2 = T(0);
            if (l1 > lo1) s1 += c.k * v[t][1];
            if (l1 < hi1) s1 += c.k * v[t][2];
            if (l2 > lo2) s2 += c.k * v[t][3];
            if (l2 < hi2) s2 += c.k * v[t][4];
            lat[t] = c1 * s1 + c2 * s2;
        }
        T dp[3];
        for (int t = 0; t < 3; t++)
            if (!((t + par) & 1)) dp[t] = c.k * d[t];
        for (int t = 0; t < 3; t++)
            if ((t + par) & 1) {
                T axial = T(0);
                if (t > 0) axial += dp[t > 0 ? t - 1 : 0];
                if (t < 2) axial += dp[t < 2 ? t + 1 : 2];
                d[t] = (d[t] - ca * axial) - lat[t];
                dp[t] = c.k * d[t];
            }
        T *b = f.buf(AXIS);
        for (int t = 0; t < 3; t++) {
            b[((long)(s * 3 + t) * n2 + (l2 - lo2)) * n1 + (l1 - lo1)] = dp[t];
            const int i = AXIS == 2 ? a0 + t : l1, j = AXIS == 2 ? l1 : (AXIS == 1 ? a0 + t : l2);
            const int k = AXIS == 0 ? a0 + t : l2;
            if (want_sum && in_d3(g, i, j, k)) acc += (double)(d[t] * d[t]);
        }
        if (!STRIDE) break;
    }
    return acc;
}

// one thread per cell that a slab correction changes (dv_face_cells)
template <typename T>
__host__ __device__ inline void dv_apply_block(const DvFaces<T> &f, T *D, T *F, const DvCoef<T> &c, int blk, int tid)
{
    const Geom &g = f.g;
    long n[3];
    dv_face_cells(g, n);
    int t = blk * 256 + tid;
    if (t >= n[0] + n[1] + n[2]) return;
    int i, j, k;
    auto shell = [](int q, int m) { return q < 4 ? q - 1 : m + q - 4; };
    if (t < n[0]) {
        i = t % (g.nx + 5) - 1;
        t /= g.nx + 5;
        j = t % (g.ny + 5) - 1;
        k = shell(t / (g.ny + 5), g.nz);
    } else if (t < n[0] + n[1]) {
        t -= (int)n[0];
        i = t % (g.nx + 5) - 1;
        t /= g.nx + 5;
        j = shell(t % 8, g.ny);
        k = 3 + t / 8;
    } else {  // the four layers of a row share a line: layers fastest
        t -= (int)(n[0] + n[1]);
        i = shell(t % 8, g.nx);
        t /= 8;
        j = 3 + t % (g.ny - 3);
        k = 3 + t / (g.ny - 3);
    }
    const T own = f.dp(i, j, k);
    const T sx = f.dp(i - 1, j, k) + f.dp(i + 1, j, k);
    const T sy = f.dp(i, j - 1, k) + f.dp(i, j + 1, k);
    const T sz = f.dp(i, j, k - 1) + f.dp(i, j, k + 1);
    const long p = f.at(i, j, k);
    D[p] = ((dv_self(c, D[p], own) - c.cx * sx) - c.cy * sy) - c.cz * sz;
    F[p] += own;
}

// ---- final update -----------------------------------------------------------------
// U += dxi (F(i) - F(i+1)) and likewise V, W; P += F / dt; over the whole
// array, with the seam and edge planes.  FORCE applies the deferred linear
// forcing to the velocity first and sums its power over the interior.  Each
// thread marches a column of planes, F of the plane above in a register; a
// workgroup takes the tasks (column, chunk) t, t + nblk, ...
// when: 0 always, 1 only if the call has converged
template <typename T, bool FORCE>
__host__ __device__ inline double dv_finish_task(const Geom &g, T *U, T *V, T *W, T *P, const T *F, const T *planes,
                                        const DvCoef<T> &c, double d, const DevScalars *S, int seams, int zc, int gxy,
                                        int t, int tid)
{
    const T dti = T(1.0 / d);
    const DvPlanes pl = dv_planes(g);
    const int sx = (int)g.sx, sy = (int)g.sy, sz = g.nz + 2 * g.h, h = g.h;
    const int q = t % gxy * 256 + tid;
    const int z0 = t / gxy * zc, z1 = sz < z0 + zc ? sz : z0 + zc;
    double pw = 0.0;
    if (q < sx * sy) {
        const int x = q % sx, y = q / sx;
        const long sxy = g.sx * g.sy;
        const T A = FORCE ? T(S->lf[4]) : T(0), um = T(S->lf[1]), vm = T(S->lf[2]), wm = T(S->lf[3]), rdt = T(d);
        auto im = [](int v, int n, int hh) { return v < hh ? v + n - hh : (v >= n + hh ? v - n - hh : v - hh); };
        const int mi = im(x, g.nx, h), mj = im(y, g.ny, h);
        const bool seamx = seams && (x == h - 1 || x == g.nx + h - 1), seamy = seams && (y == h - 1 || y == g.ny + h - 1);
        const bool in_xy = x >= h && x < g.nx + h && y >= h && y < g.ny + h;
        const int px = dv_pitch(g, (int)sizeof(T));
        const long pxy = (long)px * g.sy;
        long p = q + sxy * z0, f = x + (long)px * y + pxy * z0;
        T fc = F[f];
        for (int z = z0; z < z1; z++, p += sxy, f += pxy) {
            const int mk = im(z, g.nz, h);
            // F of a group's start is zero until the first refresh
            T fx = T(0), fy = T(0), fz = T(0);
            if (x < sx - 1)
                fx = F[f + 1];
            else if (seams)
                fx = planes[pl.edge[0] + y + g.sy * (long)z];
            if (y < sy - 1)
                fy = F[f + px];
            else if (seams)
                fy = planes[pl.edge[1] + x + g.sx * (long)z];
            if (z < sz - 1)
                fz = F[f + pxy];
            else if (seams)
                fz = planes[pl.edge[2] + x + g.sx * (long)y];
            T u = U[p], v = V[p], w = W[p];
            const T pr = P[p];
            if (FORCE) {
                const T us = A * (u - um), vs = A * (v - vm), ws = A * (w - wm);
                if (in_xy && z >= h && z < g.nz + h) pw += (double)((u * us + v * vs) + w * ws);
                u += us * rdt;
                v += vs * rdt;
                w += ws * rdt;
            }
            T du = c.dxi * (fc - fx), dv = c.dyi * (fc - fy), dw = c.dzi * (fc - fz);
            if (seamx) du += planes[pl.seam[0] + mj + (long)g.ny * mk];
            if (seamy) dv += planes[pl.seam[1] + mi + (long)g.nx * mk];
            if (seams && (z == h - 1 || z == g.nz + h - 1)) dw += planes[pl.seam[2] + mi + (long)g.nx * mj];
            U[p] = u + du;
            V[p] = v + dv;
            W[p] = w + dw;
            P[p] = pr + fc * dti;
            fc = fz;
        }
    }
    return pw;
}

template <typename T, bool FORCE>
__host__ __device__ inline double dv_finish_block(const Geom &g, T *U, T *V, T *W, T *P, const T *F, const T *planes,
                                         const DvCoef<T> &c, double d, const DevScalars *S, int seams, int zc, int gxy,
                                         int blk, int nblk, int tid)
{
    const int ntask = gxy * ((g.nz + 2 * g.h + zc - 1) / zc);
    double pw = 0.0;
    for (int t = blk; t < ntask; t += nblk)
        pw += dv_finish_task<T, FORCE>(g, U, V, W, P, F, planes, c, d, S, seams, zc, gxy, t, tid);
    return pw;
}

}  // namespace lcs
