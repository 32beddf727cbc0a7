// HSMAC in divergence form: the red-black sweeps of a time-blocked group
// (src/flows/couples/hsmac.jl:1-35, 131-201) carried on two arrays instead of
// four.
//
// A cell's correction dp = -omega div dl moves its six faces, so it changes
// only its own divergence and that of its six neighbours:
//   D(c)   += 2 (dxi^2 + dyi^2 + dzi^2) dp(c),
//   D(c+-1) -= dxi^2 dp(c)  (and dyi^2, dzi^2 along y, z).
// The sweeps therefore need the divergence D alone, and the velocity and
// pressure follow at the end from the accumulated F = sum dp:
//   U(i) += dxi (F(i) - F(i+1)),  P += F / dt.
// A sweep moves D and F (read and write: 4 element passes) where the in-place
// form moves U, V, W, P (8), and two consecutive sweeps share one pass.
// D, F live in halo arrays of the field's shape with padded rows (dv_pitch);
// every visited cell, ghosts included, is the reference's cell in the
// reference's order, so the results agree to rounding.
//
// A group starts with a periodic fill of U, V, W.  In divergence form
// (the "refresh", dv_refresh_cell below):
//   * ghost D and F take their image's values;
//   * the low plane of each axis had used ghost face 0, which the fill
//     replaces by face n: D(1) += dxi^2 ((F0 - F1) - (Fn - Fn+1)), because both
//     faces had the same value when the group began;
//   * face n keeps the correction of ghost cell n+1, whose F now becomes
//     F(1): the difference dxi (F1 - Fn+1) goes to the "seam" plane of that
//     face, which the final update adds;
//   * the pressure of a ghost cell is not refilled: P += (F - F(image)) / dt;
//   * the last ghost face n+h has its upper cell outside the array: the F of
//     that cell's image is kept in the "edge" plane.
// A group's first sweep is the core (2:n), which reads D of core cells only,
// and the refresh changes only other cells.  So the sweep runs first, from one
// (D, F) set to the other, and the refresh then corrects ghosts and low planes
// of the sweep's output from the sweep's input: no thread reads what another
// one writes.
// The divergence a check sees is that of D, which the sweeps reduce far below
// what the velocity can show: U rounded to its type has an error of ulp / sqrt(12)
// a face, and ulp^2 averages 3/7 eps^2 U^2 over the mantissas, so a cell's
// div^2 has the mean eps^2 / 14 (dxi^2 U^2 + dyi^2 V^2 + dzi^2 W^2) even where
// D is zero.  The construct pass sums that term and every check adds it
// (dv_noise): a call whose epsp lies below it runs to itrmax, as the sweeps on
// the velocity do, and the logged divergence is one the velocity shows (64^3
// FP32, U in [0, 1): floor 3.2e-8 / dx, the returned velocity's 2.5e-8 to 3e-8).
#pragma once

#include "lcs_hsmac_plan.h"
#include "lcs_hsmac_tile.h"
#include "lcs_internal.h"

namespace lcs {

template <typename T>
struct DvCoef {
    T k;           // dp = k div = (-omega dl) div
    T cx, cy, cz;  // dxi^2, dyi^2, dzi^2
    // 2 (cx + cy + cz) in two parts: rounded to one T, it would differ from the
    // neighbours' coefficients by eps c0, and each correction would leave eps c0 F
    // behind in D.  F is smooth, D is k^2 F for its waves of number k, so that is
    // a relative error of eps c0 / k^2: 6e-4 in D of the longest wave at 256^3
    // FP32, which no later sweep corrects (fields 8e-5 off after 300-sweep calls,
    // 8e-7 with the two parts).
    T c0, c0l;
    T dxi, dyi, dzi;
};

template <typename T>
inline DvCoef<T> dv_coef(const Geom &g, double omega)
{
    DvCoef<T> c;
    c.dxi = T(1.0 / spacing(g.nx));
    c.dyi = T(1.0 / spacing(g.ny));
    c.dzi = T(1.0 / spacing(g.nz));
    c.cx = c.dxi * c.dxi;
    c.cy = c.dyi * c.dyi;
    c.cz = c.dzi * c.dzi;
    const long double s = 2.0L * (((long double)c.cx + (long double)c.cy) + (long double)c.cz);
    c.c0 = T(s);
    c.c0l = T(s - (long double)c.c0);
    c.k = -T(omega) * (T(1) / c.c0);
    return c;
}
// the factor of the construct pass's sum in div^2 (see above)
template <typename T>
inline double dv_noise(const Geom &g)
{
    const double eps = sizeof(T) == 8 ? 0x1p-52 : 0x1p-23;
    return eps * eps / 14.0 / (double)g.len;
}
// a batch record's coefficients (the T values, stored as doubles)
template <typename T>
__host__ __device__ inline DvCoef<T> dv_coef_rec(const BoxRec &B)
{
    DvCoef<T> c;
    c.k = T(B.dv_c[0]);
    c.cx = T(B.dv_c[1]);
    c.cy = T(B.dv_c[2]);
    c.cz = T(B.dv_c[3]);
    c.c0 = T(B.dv_c[4]);
    c.c0l = T(B.dv_c[5]);
    c.dxi = T(B.dv_c[6]);
    c.dyi = T(B.dv_c[7]);
    c.dzi = T(B.dv_c[8]);
    return c;
}
// D of a cell after its own correction
template <typename T>
__host__ __device__ inline T dv_self(const DvCoef<T> &c, T d, T dp)
{
    return std::fma(c.c0, dp, std::fma(c.c0l, dp, d));
}

enum { kDvPlain = 0, kDvConstruct = 1 };

template <typename T>
struct DvArgs {
    Geom g;
    const T *Ds, *Fs;       // input set (plain)
    T *Dd, *Fd;             // output set
    const T *U, *V, *W;     // construct: velocity with filled ghosts
    DvCoef<T> c;
    T dscale;               // construct: div of the forced velocity is (1 + A dt) times that of the loaded one
    int kind[2];            // region of each sweep (hs_region)
    int sum[2];             // form the sum of div^2 of that sweep
    int zc;                 // planes per chunk
    int px;                 // row pitch of D and F
};

// the refresh of one cell that is a ghost or lies on a low or high interior
// plane (array indices x, y, z): Do, Fo the set the core sweep read, Dn, Fn the
// one it wrote.  accumulate: seams of an earlier refresh of the call are kept.
template <typename T>
__host__ __device__ inline void dv_refresh_cell(const Geom &g, const DvCoef<T> &c, const DvPlanes &pl, const T *Do, const T *F,
                                       T *Dn, T *Fn, T *P, T *pn, T dti, int accumulate, int x, int y, int z)
{
    const int h = g.h, nx = g.nx, ny = g.ny, nz = g.nz;
    const int px = dv_pitch(g, (int)sizeof(T));
    const long sx = px, sxy = (long)px * g.sy;  // of D and F
    auto image = [h](int v, int n) { return v < h ? v + n : (v >= n + h ? v - n : v); };
    const int ix = image(x, nx), iy = image(y, ny), iz = image(z, nz);
    const long p = x + sx * (y + g.sy * (long)z), im = ix + sx * (iy + g.sy * (long)iz);
    // low planes: ghost face 0 becomes face n
    T fix = T(0);
    if (ix == h) fix += c.cx * ((F[im - 1] - F[im]) - (F[im + nx - 1] - F[im + nx]));
    if (iy == h) fix += c.cy * ((F[im - sx] - F[im]) - (F[im + (ny - 1) * sx] - F[im + ny * sx]));
    if (iz == h) fix += c.cz * ((F[im - sxy] - F[im]) - (F[im + (nz - 1) * sxy] - F[im + nz * sxy]));
    if (p == im) {
        if (ix == h || iy == h || iz == h) Dn[p] += fix;
        if (x == nx + h - 1) {
            T &t = pn[pl.seam[0] + (y - h) + (long)ny * (z - h)];
            const T v = c.dxi * (F[p - nx + 1] - F[p + 1]);
            t = accumulate ? t + v : v;
        }
        if (y == ny + h - 1) {
            T &t = pn[pl.seam[1] + (x - h) + (long)nx * (z - h)];
            const T v = c.dyi * (F[p - (ny - 1) * sx] - F[p + sx]);
            t = accumulate ? t + v : v;
        }
        if (z == nz + h - 1) {
            T &t = pn[pl.seam[2] + (x - h) + (long)nx * (y - h)];
            const T v = c.dzi * (F[p - (nz - 1) * sxy] - F[p + sxy]);
            t = accumulate ? t + v : v;
        }
        return;
    }
    // the sweep changed a ghost by its core neighbours' corrections: Dn - Do
    Dn[p] = (Do[im] + fix) + (Dn[p] - Do[p]);
    Fn[p] = F[im];
    P[x + g.sx * (y + g.sy * (long)z)] += (F[p] - F[im]) * dti;
    // the cell above the last ghost face: its image is one above this cell's
    if (x == (int)g.sx - 1) pn[pl.edge[0] + y + g.sy * (long)z] = F[im + 1];
    if (y == (int)g.sy - 1) pn[pl.edge[1] + x + g.sx * (long)z] = F[im + sx];
    if (z == nz + 2 * h - 1) pn[pl.edge[2] + x + g.sx * (long)y] = F[im + sxy];
}

// neighbouring lane's value across the wave; lanes past its ends read 0
#ifdef __HIPCC__
template <int UP>
__device__ inline float dv_lane(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), UP ? 0x130 : 0x138, 0xf, 0xf, true));
}
template <int UP>
__device__ inline double dv_lane(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), UP ? 0x130 : 0x138, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), UP ? 0x130 : 0x138, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
#endif
// member m of the neighbouring lane's state as it was before this step
#ifdef __HIP_DEVICE_COMPILE__
#define DV_LANE(UP, m) dv_lane<UP>(th.m)
#else
#define DV_LANE(UP, m) (th.lane[UP] ? th.lane[UP]->m : T(0))
#endif

template <typename T>
struct DvPair {
    T v[2];
};
// two neighbouring elements of a row (rows start at any element)
template <typename T>
__host__ __device__ inline DvPair<T> dv_load2(const T *p)
{
    DvPair<T> r;
    __builtin_memcpy(&r, p, sizeof(r));
    return r;
}

// NS fused sweeps (1 or 2) marching up in z.
//
// A lane owns two neighbouring cells of a row, (2l, 2l+1): one red and one
// black on every plane.  A block of LX lanes covers a row of W = 2 LX cells;
// it holds RW consecutive rows in registers, NB blocks make the workgroup.
// At step q sweep s works on plane z = q - 2s (its input is complete there):
//   red    dp on plane z;
//   black  dp on plane z-1, from its red neighbours on z-2, z-1, z;
//   final  red D of plane z-2, from its black neighbours on z-3, z-2, z-1.
// Red and black values of a plane are kept apart, so the y and z neighbours of
// a cell are the same lane's values and the x neighbours are the lane's own
// and one neighbouring lane's (a DPP move).  Rows at the ends of a block come
// from LDS, written one step earlier: one barrier per plane.  A sweep needs
// two more cells on each side in x and y (the window's halo) and two more
// planes at each end of a chunk.
// A tile owns the OWN cells in the middle of its window of W: a multiple of a
// 64-byte line, so stored row segments start and end on lines.
template <typename T, int NS, int MODE, int LX, int RW, int NB>
struct DvTile {
    using Win = DvWindow<(int)sizeof(T), NS, LX, RW, NB>;
    static constexpr int W = Win::W, OWN = Win::OWN, HX = Win::HX;
    static constexpr int ROWS = Win::ROWS, HY = Win::HY, HZ = 2 * NS, NT = NB * LX;
    static constexpr int EX = 2 * NS * 2 * NB * 2 * LX;  // exchange elements in LDS
    static_assert(RW % 2 == 0, "a block's first row keeps the parity of the tile's");
    // planes loaded ahead, one register set for steps of each parity (4 and 6
    // sets: no faster at 32^3, 256^3 or 1000^3)
    static constexpr int PF = 2;
    static_assert(HX >= 2 * NS && HX % 2 == 0, "halo of the window");

    __host__ __device__ static int tiles_x(const Geom &g) { return Win::tiles_x(g); }
    __host__ __device__ static int tiles_y(const Geom &g) { return Win::tiles_y(g); }

    struct Th {
#ifndef __HIP_DEVICE_COMPILE__
        const Th *lane[2];      // host harness: states of the lanes below and above before the step
#endif
        int X, xo, b, lx;       // first cell of the lane, clamped load offset, block, lane
        int Y;                  // first row of the block
        int wx0, wy0, ox0, ox1, oy0, oy1, zo0, zo1;
        unsigned reg[NS];       // bit 2r+s: cell (row r, slot s) is inside the sweep's region in x and y
        unsigned own, cnt;      // owned cells; owned cells inside (1:n+1) in x and y
        int zlo[NS], zhi[NS];   // region planes (array index)
        DvPair<T> d[PF][RW];    // loaded planes, by step
        DvPair<T> f[PF][RW];    // loaded F
        // construct: raw loads
        T um[MODE == kDvConstruct ? PF : 1][MODE == kDvConstruct ? RW : 1];
        DvPair<T> v[MODE == kDvConstruct ? PF : 1][MODE == kDvConstruct ? RW + 1 : 1];
        DvPair<T> w[MODE == kDvConstruct ? PF : 1][MODE == kDvConstruct ? RW : 1];
        DvPair<T> wp[MODE == kDvConstruct ? RW : 1];  // W of the plane below
        // pipeline
        T rq[NS][2][RW];        // red D after its own correction, planes z-1, z-2
        T bq0[RW], bq1[2][RW];  // black D waiting for sweep 0 (next step) and sweep 1 (two steps on)
        T rp[NS][RW], rpp[NS][RW], bp[NS][RW], bpp[NS][RW];  // dp of the last planes
        T bout[RW], fr[RW];     // black D of the next output plane, red F of the next F plane
        double acc[NS];
        T nse;  // construct: sum of dxi^2 U^2 + dyi^2 V^2 + dzi^2 W^2 (a lane that owns one of its rows counts both)
    };

    __host__ __device__ static inline int mini(int a, int b) { return a < b ? a : b; }
    __host__ __device__ static inline int maxi(int a, int b) { return a > b ? a : b; }
    __host__ __device__ static inline int clampi(int v, int hi) { return v < 0 ? 0 : (v > hi ? hi : v); }

    // returns whether any cell of the window lies outside the core (2:n) in x or y
    __host__ __device__ static bool init(const DvArgs<T> &a, int bx, int by, int bz, int tid, Th &th)
    {
        const Geom &g = a.g;
        const int gx = tiles_x(g), gy = tiles_y(g);
        th.b = tid / LX;
        th.lx = tid % LX;
        th.ox0 = bx * OWN;
        th.ox1 = bx == gx - 1 ? (int)g.sx : th.ox0 + OWN;
        th.wx0 = bx == 0 ? 0 : th.ox0 - HX;
        th.wy0 = by * (ROWS - 2 * HY);
        th.oy0 = by == 0 ? 0 : th.wy0 + HY;
        th.oy1 = by == gy - 1 ? (int)g.sy : th.wy0 + ROWS - HY;
        th.zo0 = bz * a.zc;
        th.zo1 = mini(g.nz + 2 * g.h, th.zo0 + a.zc);
        th.X = th.wx0 + 2 * th.lx;
        th.Y = th.wy0 + th.b * RW;
        th.xo = mini(th.X, (int)g.sx - 2);
        th.own = 0;
        th.cnt = 0;
        const int h = g.h;
        for (int s = 0; s < NS; s++) th.reg[s] = 0;
#pragma unroll
        for (int r = 0; r < RW; r++)
            for (int s = 0; s < 2; s++) {
                const int x = th.X + s, y = th.Y + r;
                const unsigned bit = 1u << (2 * r + s);
                if (x >= th.ox0 && x < th.ox1 && y >= th.oy0 && y < th.oy1) {
                    th.own |= bit;
                    if (x >= h && x <= g.nx + h && y >= h && y <= g.ny + h) th.cnt |= bit;
                }
                for (int q = 0; q < NS; q++) {
                    const Box3 R = hs_region(g, a.kind[q]);
                    if (x >= R.lo[0] + h - 1 && x <= R.hi[0] + h - 1 && y >= R.lo[1] + h - 1 && y <= R.hi[1] + h - 1)
                        th.reg[q] |= bit;
                }
            }
        for (int q = 0; q < NS; q++) {
            const Box3 R = hs_region(g, a.kind[q]);
            th.zlo[q] = R.lo[2] + h - 1;
            th.zhi[q] = R.hi[2] + h - 1;
        }
        const T z = T(0);
#pragma unroll
        for (int r = 0; r < RW; r++) {
            th.bout[r] = th.fr[r] = th.bq0[r] = th.bq1[0][r] = th.bq1[1][r] = z;
            for (int q = 0; q < NS; q++) {
                th.rq[q][0][r] = th.rq[q][1][r] = z;
                th.rp[q][r] = th.rpp[q][r] = th.bp[q][r] = th.bpp[q][r] = z;
            }
            if constexpr (MODE == kDvConstruct) th.wp[r].v[0] = th.wp[r].v[1] = z;
        }
        for (int q = 0; q < NS; q++) th.acc[q] = 0.0;
        th.nse = T(0);
        return !(th.wx0 >= h + 1 && th.wx0 + W - 1 <= g.nx + h - 1 && th.wy0 >= h + 1 &&
                 th.wy0 + ROWS - 1 <= g.ny + h - 1);
    }

    // element offset of row r's load in its plane of row pitch px
    template <bool EXY>
    __host__ __device__ static inline int row_off(const Geom &g, const Th &th, int r, int px)
    {
        const int y = EXY ? mini(th.Y + r, (int)g.sy - 1) : th.Y + r;
        return y * px + th.xo;
    }
    // a lane whose first cell is the row's last element loaded one element early
    template <bool EXY>
    __host__ __device__ static inline void fix_end(const Geom &g, const Th &th, DvPair<T> &p)
    {
        if (EXY && th.X == (int)g.sx - 1) p.v[0] = p.v[1];
    }

    template <bool EXY>
    __host__ __device__ static inline void load_d(const DvArgs<T> &a, Th &th, int q, int e)
    {
        const Geom &g = a.g;
        const int sz = g.nz + 2 * g.h;
        const int z = clampi(q, sz - 1);
        if constexpr (MODE == kDvConstruct) {
            const long base = (long)z * (g.sx * g.sy);
            const T *U = a.U + base, *V = a.V + base, *Wz = a.W + base;
            const int xm = maxi(mini(th.X, (int)g.sx) - 1, 0);
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const int o = row_off<EXY>(g, th, r, (int)g.sx);
                th.d[e][r] = dv_load2(U + o);
                fix_end<EXY>(g, th, th.d[e][r]);
                th.um[e][r] = U[o - th.xo + xm];
                th.v[e][r + 1] = dv_load2(V + o);
                fix_end<EXY>(g, th, th.v[e][r + 1]);
                th.w[e][r] = dv_load2(Wz + o);
                fix_end<EXY>(g, th, th.w[e][r]);
            }
            const int ym = mini(maxi(th.Y - 1, 0), (int)g.sy - 1);
            th.v[e][0] = dv_load2(V + ym * (int)g.sx + th.xo);
            fix_end<EXY>(g, th, th.v[e][0]);
        } else {
            const T *D = a.Ds + (long)z * ((long)a.px * g.sy);
#pragma unroll
            for (int r = 0; r < RW; r++) {
                th.d[e][r] = dv_load2(D + row_off<EXY>(g, th, r, a.px));
                fix_end<EXY>(g, th, th.d[e][r]);
            }
        }
    }

    // F of plane z: of every row of the window, though only the owned cells' is
    // used (24 of 32 rows in a two-sweep pass)
    template <bool EXY>
    __host__ __device__ static inline void load_f(const DvArgs<T> &a, Th &th, int z, int e)
    {
        if constexpr (MODE == kDvConstruct) return;
        const Geom &g = a.g;
        if (z < th.zo0 || z >= th.zo1) return;
        const T *F = a.Fs + (long)z * ((long)a.px * g.sy);
#pragma unroll
        for (int r = 0; r < RW; r++) {
            th.f[e][r] = dv_load2(F + row_off<EXY>(g, th, r, a.px));
            fix_end<EXY>(g, th, th.f[e][r]);
        }
    }

    // store a pair of owned cells
    __host__ __device__ static inline void store2(T *p, const Th &th, int r, const DvPair<T> &v)
    {
        const unsigned m = th.own >> (2 * r) & 3u;
        if (m == 3u)
            __builtin_memcpy(p, &v, sizeof(v));
        else if (m == 1u)
            *p = v.v[0];
    }

    // one plane; SET = E = the step's parity: the red slot of row r on plane q is (E + r) & 1
    template <int SET, bool EXY>
    __host__ __device__ static inline void step(const DvArgs<T> &a, T *lds, Th &th, int q)
    {
        constexpr int E = SET & 1;
        const Geom &g = a.g;
        const DvCoef<T> &c = a.c;
        T R[RW];
        // the loaded plane, red and black apart
        T bload[RW];
        T nse = T(0);
#pragma unroll
        for (int r = 0; r < RW; r++) {
            DvPair<T> d = th.d[SET][r];
            if constexpr (MODE == kDvConstruct) {
                const DvPair<T> v1 = th.v[SET][r + 1], v0 = th.v[SET][r], w1 = th.w[SET][r];
                const T um = th.um[SET][r];
                const T u0 = d.v[0], u1 = d.v[1];
                d.v[0] = ((c.dxi * (u0 - um) + c.dyi * (v1.v[0] - v0.v[0])) + c.dzi * (w1.v[0] - th.wp[r].v[0])) *
                         a.dscale;
                d.v[1] = ((c.dxi * (u1 - u0) + c.dyi * (v1.v[1] - v0.v[1])) + c.dzi * (w1.v[1] - th.wp[r].v[1])) *
                         a.dscale;
                th.wp[r] = w1;
                const T e = (c.cx * (u0 * u0 + u1 * u1) + c.cy * (v1.v[0] * v1.v[0] + v1.v[1] * v1.v[1])) +
                            c.cz * (w1.v[0] * w1.v[0] + w1.v[1] * w1.v[1]);
                nse += e;
            }
            const int sr = (E + r) & 1;
            R[r] = d.v[sr];
            bload[r] = d.v[1 - sr];
        }
        if constexpr (MODE == kDvConstruct)
            if (q >= th.zo0 && q < th.zo1) th.nse += nse;
        load_d<EXY>(a, th, q + PF, SET);
        // plane of F handled at this step
        const int zf = q - 2 * (NS - 1) - 1;
        DvPair<T> fin[RW];
#pragma unroll
        for (int r = 0; r < RW; r++) fin[r] = th.f[SET][r];
        load_f<EXY>(a, th, zf + PF, SET);
        T *xin = lds + E * (EX / 2), *xout = lds + (1 - E) * (EX / 2);
        T rn[NS][RW], bn[NS][RW], Bf[NS][RW], ra[NS][RW];  // dp; black D after its correction; red D after its own
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int zr = q - 2 * s;
            const T kr = zr >= th.zlo[s] && zr <= th.zhi[s] ? c.k : T(0);
            const T kb = zr - 1 >= th.zlo[s] && zr - 1 <= th.zhi[s] ? c.k : T(0);
            const bool sumr = a.sum[s] && kr != T(0) && zr >= th.zo0 && zr < th.zo1 && zr >= g.h && zr <= g.nz + g.h;
            const bool sumb = a.sum[s] && kb != T(0) && zr - 1 >= th.zo0 && zr - 1 < th.zo1 && zr - 1 >= g.h &&
                              zr - 1 <= g.nz + g.h;
            const unsigned cm = EXY ? th.cnt & th.reg[s] : th.cnt;
            // rows of the neighbouring blocks (dp of the last step)
            const T *ein = xin + s * (4 * NB * LX);
            T *eout = xout + s * (4 * NB * LX);
            const int bm = clampi(th.b - 1, NB - 1), bpl = clampi(th.b + 1, NB - 1);
            const T rdn = ein[(bm * 2 + 1) * LX + th.lx], rup = ein[bpl * 2 * LX + th.lx];
            const T bdn = ein[2 * NB * LX + (bm * 2 + 1) * LX + th.lx];
            const T bup = ein[2 * NB * LX + bpl * 2 * LX + th.lx];
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const int sr = (E + r) & 1;
                T dp = kr * R[r];
                if (EXY) dp = th.reg[s] >> (2 * r + sr) & 1u ? dp : T(0);
                rn[s][r] = dp;
                if (sumr && (cm >> (2 * r + sr) & 1u)) th.acc[s] += (double)(R[r] * R[r]);
                ra[s][r] = dv_self(c, R[r], dp);
            }
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const int sr = (E + r + 1) & 1;  // red slot on plane zr-1
                const T own = th.rp[s][r];
                const T oth = sr == 0 ? DV_LANE(1, rp[s][r]) : DV_LANE(0, rp[s][r]);
                const T dn = r > 0 ? th.rp[s][r > 0 ? r - 1 : 0] : rdn;
                const T up = r < RW - 1 ? th.rp[s][r < RW - 1 ? r + 1 : r] : rup;
                T B = s == 0 ? th.bq0[r] : th.bq1[1][r];
                B = ((B - c.cx * (own + oth)) - c.cy * (dn + up)) - c.cz * (th.rpp[s][r] + rn[s][r]);
                T dp = kb * B;
                if (EXY) dp = th.reg[s] >> (2 * r + 1 - sr) & 1u ? dp : T(0);
                bn[s][r] = dp;
                if (sumb && (cm >> (2 * r + 1 - sr) & 1u)) th.acc[s] += (double)(B * B);
                Bf[s][r] = dv_self(c, B, dp);
            }
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const int sr = (E + r) & 1;  // red slot on plane zr-2
                const T own = th.bp[s][r];
                const T oth = sr == 0 ? DV_LANE(0, bp[s][r]) : DV_LANE(1, bp[s][r]);
                const T dn = r > 0 ? th.bp[s][r > 0 ? r - 1 : 0] : bdn;
                const T up = r < RW - 1 ? th.bp[s][r < RW - 1 ? r + 1 : r] : bup;
                R[r] = ((th.rq[s][1][r] - c.cx * (own + oth)) - c.cy * (dn + up)) - c.cz * (th.bpp[s][r] + bn[s][r]);
            }
            // rows for the neighbouring blocks' next step
            eout[th.b * 2 * LX + th.lx] = rn[s][0];
            eout[(th.b * 2 + 1) * LX + th.lx] = rn[s][RW - 1];
            eout[2 * NB * LX + th.b * 2 * LX + th.lx] = bn[s][0];
            eout[2 * NB * LX + (th.b * 2 + 1) * LX + th.lx] = bn[s][RW - 1];
        }
        // F of the black cells of plane zf and of the red cells of plane zf + 1
        T fb[RW], frn[RW];
#pragma unroll
        for (int r = 0; r < RW; r++) {
            fb[r] = bn[NS - 1][r];
            frn[r] = rn[NS - 1][r];
            if (NS == 2) {  // sweep 0 corrected these cells two steps ago
                fb[r] = th.bpp[0][r] + fb[r];
                frn[r] = th.rpp[0][r] + frn[r];
            }
        }
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int r = 0; r < RW; r++) {
                th.rq[s][1][r] = th.rq[s][0][r];
                th.rq[s][0][r] = ra[s][r];
                th.rpp[s][r] = th.rp[s][r];
                th.rp[s][r] = rn[s][r];
                th.bpp[s][r] = th.bp[s][r];
                th.bp[s][r] = bn[s][r];
            }
#pragma unroll
        for (int r = 0; r < RW; r++) {
            th.bq0[r] = bload[r];
            th.bq1[1][r] = th.bq1[0][r];
            th.bq1[0][r] = Bf[0][r];
        }
        // output: D of plane q - 2 NS, F of plane zf
        const int zo = q - 2 * NS;
        const long sxy = (long)a.px * g.sy;
        if (zo >= th.zo0 && zo < th.zo1) {
            T *D = a.Dd + (long)zo * sxy;
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const int sr = (E + r) & 1;
                DvPair<T> v;
                v.v[sr] = R[r];
                v.v[1 - sr] = th.bout[r];
                store2(D + (th.Y + r) * a.px + th.X, th, r, v);
            }
        }
        if (zf >= th.zo0 && zf < th.zo1) {
            T *F = a.Fd + (long)zf * sxy;
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const int sr = (E + r + 1) & 1;
                DvPair<T> v;
                v.v[sr] = th.fr[r];
                v.v[1 - sr] = fb[r];
                if constexpr (MODE != kDvConstruct) {
                    v.v[0] += fin[r].v[0];
                    v.v[1] += fin[r].v[1];
                }
                store2(F + (th.Y + r) * a.px + th.X, th, r, v);
            }
        }
#pragma unroll
        for (int r = 0; r < RW; r++) {
            th.bout[r] = Bf[NS - 1][r];
            th.fr[r] = frn[r];
        }
    }

    // the first step's plane: red cells have even i+j+k, and it is chosen so that
    // the red slot of row r on plane q is (step parity + r) & 1
    __host__ __device__ static inline int first(const DvArgs<T> &a, const Th &th)
    {
        const int q = th.zo0 - HZ > 0 ? th.zo0 - HZ : 0;
        return (th.wx0 + th.wy0 + q + a.g.h + 1) & 1 ? q - 1 : q;
    }
    __host__ __device__ static inline int last(const Th &th) { return th.zo1 - 1 + HZ; }
    // loads ahead of step q
    template <bool EXY>
    __host__ __device__ static inline void prologue(const DvArgs<T> &a, Th &th, int q)
    {
        const Geom &g = a.g;
#pragma unroll
        for (int e = 0; e < PF; e++) load_d<EXY>(a, th, q + e, e);
        if constexpr (MODE == kDvConstruct) {  // W below the first plane
            const long base = (long)clampi(q - 1, g.nz + 2 * g.h - 1) * (g.sx * g.sy);
#pragma unroll
            for (int r = 0; r < RW; r++) {
                th.wp[r] = dv_load2(a.W + base + row_off<EXY>(g, th, r, (int)g.sx));
                fix_end<EXY>(g, th, th.wp[r]);
            }
        }
#pragma unroll
        for (int e = 0; e < PF; e++) load_f<EXY>(a, th, q - 2 * (NS - 1) - 1 + e, e);
    }
#ifdef __HIPCC__
    template <bool EXY>
    __device__ static inline void march(const DvArgs<T> &a, T *lds, Th &th)
    {
        int q = first(a, th);
        const int q1 = last(th);
        prologue<EXY>(a, th, q);
        for (; q <= q1; q += PF) {
            step<0, EXY>(a, lds, th, q);
            __syncthreads();
            step<1, EXY>(a, lds, th, q + 1);
            __syncthreads();
        }
    }

    // the tile's sweeps; sums of div^2 of the lane's cells in acc, and of the rounding term in nse
    __device__ static inline void run(const DvArgs<T> &a, int bx, int by, int bz, T *lds, double acc[NS], double &nse)
    {
        Th th;
        const bool edge = init(a, bx, by, bz, (int)threadIdx.x, th);
        for (int t = threadIdx.x; t < EX; t += NT) lds[t] = T(0);
        __syncthreads();
        if (edge)
            march<true>(a, lds, th);
        else
            march<false>(a, lds, th);
#pragma unroll
        for (int s = 0; s < NS; s++) acc[s] = th.acc[s];
        nse = th.own ? (double)th.nse : 0.0;
    }
#endif

    // One workgroup for a host harness, step by step in the kernel's barrier order:
    // th and was hold NT states each.
    template <bool EXY>
    static void emulate_march(const DvArgs<T> &a, T *lds, Th *th, Th *was)
    {
        const int q0 = first(a, th[0]), q1 = last(th[0]);
        for (int t = 0; t < NT; t++) prologue<EXY>(a, th[t], q0);
        for (int q = q0; q <= q1 + (q1 - q0 + 1) % PF; q++) {
            for (int t = 0; t < NT; t++) was[t] = th[t];
            for (int t = 0; t < NT; t++) {
                th[t].lane[0] = t % 64 > 0 ? was + t - 1 : nullptr;
                th[t].lane[1] = t % 64 < 63 && t + 1 < NT ? was + t + 1 : nullptr;
                if ((q - q0) % PF == 0)
                    step<0, EXY>(a, lds, th[t], q);
                else
                    step<1, EXY>(a, lds, th[t], q);
            }
        }
    }
    static void emulate_block(const DvArgs<T> &a, int bx, int by, int bz, T *lds, Th *th, Th *was, double acc[NS],
                              double &nse)
    {
        bool edge = false;
        for (int t = 0; t < NT; t++) edge = init(a, bx, by, bz, t, th[t]);
        for (int t = 0; t < EX; t++) lds[t] = T(0);
        if (edge)
            emulate_march<true>(a, lds, th, was);
        else
            emulate_march<false>(a, lds, th, was);
        for (int t = 0; t < NT; t++) {
            for (int s = 0; s < NS; s++) acc[s] += th[t].acc[s];
            if (th[t].own) nse += (double)th[t].nse;
        }
    }
};

}  // namespace lcs
