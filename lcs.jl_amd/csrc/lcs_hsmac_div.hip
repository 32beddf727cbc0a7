// HSMAC in divergence form (lcs_hsmac_div.h, lcs_hsmac_shell.h): kernels of the
// sweeps, of the shell passes and of the update, and the call that runs a whole
// couple! with them, for one box and for batches.
#include <algorithm>
#include <cmath>

#include "lcs_device.h"
#include "lcs_hsmac_div.h"
#include "lcs_hsmac_shell.h"

namespace lcs {

// Partial slots of a call: 0 and 1 the sums of div^2 of a pass's sweeps, 2 to 4
// those of the face slabs, 5 the rounding terms of the construct pass, which
// every check until the next one reads.
constexpr long kDvNoiseSlot = 5L * kMaxPartBlocks;

// ---- sweeps -------------------------------------------------------------------
// the two (D, F) sets; which one is current is known on the host until the
// call has converged
template <typename T>
struct DvSets {
    T *D[2], *F[2];
};

// (The FP32 construct pass would take a few registers over 128, at which two
// workgroups of 512 threads share a CU.)
template <typename T, int NS, int MODE, int LX, int RW, int NB>
__global__ void __launch_bounds__(LX *NB, MODE == kDvConstruct && sizeof(T) == 4 ? 4 : 1)
    k_dv_sweep(DvArgs<T> a, int gx, int gy, int force, DtRef dt, DevScalars *S, double *part)
{
    using Tile = DvTile<T, NS, MODE, LX, RW, NB>;
    __shared__ __align__(16) T lds[Tile::EX];
    __shared__ double red_lds[16];
    if (MODE != kDvConstruct && S->hs_done) return;
    a.dscale = T(1);
    if (MODE == kDvConstruct) {
        // the linear forcing U + (A (U - mean)) dt scales the divergence
        if (force) a.dscale = T(1) + T(S->lf[4]) * T(dt.factor * (*dt.src));
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            S->hs_done = 0;
            S->hs_itr = 0;
            S->hs_div = 0.0;
            S->hs_par = 0;
        }
    }
    const int t = xcd_linear(blockIdx.x, gridDim.x);
    double acc[NS], nse;
    Tile::run(a, t % gx, t / gx % gy, t / (gx * gy), lds, acc, nse);
    for (int s = 0; s < NS; s++)
        if (a.sum[s]) {
            const double v = block_sum(acc[s], red_lds);
            if (threadIdx.x == 0) part[(long)s * kMaxPartBlocks + blockIdx.x] = v;
        }
    if (MODE == kDvConstruct) {
        const double v = block_sum(nse, red_lds);
        if (threadIdx.x == 0) part[kDvNoiseSlot + blockIdx.x] = v;
    }
}

// ---- refresh --------------------------------------------------------------------
template <typename T>
__global__ void __launch_bounds__(256)
    k_dv_refresh(Geom g, DvCoef<T> c, const T *Do, const T *Fo, T *Dn, T *Fn, T *P, T *planes, DtRef dt, int accumulate,
                 const DevScalars *S)
{
    if (S->hs_done) return;
    dv_refresh_block(g, c, Do, Fo, Dn, Fn, P, planes, T(1.0 / (dt.factor * (*dt.src))), accumulate, (int)blockIdx.x,
                     (int)threadIdx.x);
}

// ---- face slabs of the overlap order -----------------------------------------------
template <typename T, int AXIS, bool STRIDE>
__global__ void __launch_bounds__(256)
    k_dv_face(DvFaces<T> f, const T *D, DvCoef<T> c, const DevScalars *S, int want_sum, double *part)
{
    __shared__ double lds[16];
    if (S->hs_done) return;
    const double acc = dv_face_block<T, AXIS, STRIDE>(f, D, c, want_sum, (int)blockIdx.x, (int)gridDim.x, (int)threadIdx.x);
    if (want_sum) {
        const double v = block_sum(acc, lds);
        if (threadIdx.x == 0) part[blockIdx.x] = v;
    }
}

template <typename T>
__global__ void __launch_bounds__(256) k_dv_face_apply(DvFaces<T> f, T *D, T *F, DvCoef<T> c, const DevScalars *S)
{
    if (S->hs_done) return;
    dv_apply_block(f, D, F, c, (int)blockIdx.x, (int)threadIdx.x);
}

// ---- convergence ----------------------------------------------------------------
struct DvCheck {
    int npass;
    int cnt[5];
    int nnoise;            // workgroups of the construct pass
    double noise;          // dv_noise
    double len3, dxmin, epsp;
    int itr;     // index of the sweep
    int par;     // set that holds its result
    int decide;  // the sweep may end the iteration
};

__global__ void k_dv_check(const double *part, DvCheck a, DevScalars *S)
{
    __shared__ double lds[16];
    // (the first rounding term is loaded ahead of the flag's wait)
    double acc = 0.0, nse = (int)threadIdx.x < a.nnoise ? part[kDvNoiseSlot + threadIdx.x] : 0.0;
    if (S->hs_done) return;
    for (int q = 0; q < a.npass; q++)
        for (int m = threadIdx.x; m < a.cnt[q]; m += blockDim.x) acc += part[(long)q * kMaxPartBlocks + m];
    for (int m = threadIdx.x + blockDim.x; m < a.nnoise; m += blockDim.x) nse += part[kDvNoiseSlot + m];
    const double s = block_sum(acc / a.len3 + a.noise * nse, lds);
    if (threadIdx.x == 0) {
        const double div = sqrt(s);
        S->hs_div = div;
        if (a.decide && div * a.dxmin < a.epsp) {
            S->hs_itr = a.itr;
            S->hs_par = a.par;
            S->hs_done = 1;
        } else
            S->hs_itr = a.itr + 1;
    }
}

// ---- final update -----------------------------------------------------------------
template <typename T, bool FORCE>
__global__ void __launch_bounds__(256)
    k_dv_finish(Geom g, T *U, T *V, T *W, T *P, DvSets<T> sets, const T *planes, DvCoef<T> c, DtRef dt,
                DevScalars *S, int when, int par, int slot, int seams, int zc, int gxy, double *part)
{
    __shared__ double lds[16];
    const bool done = S->hs_done != 0;
    if (when == 1 && !done) return;
    const double pw = dv_finish_block<T, FORCE>(g, U, V, W, P, sets.F[done ? S->hs_par : par], planes, c,
                                                dt.factor * (*dt.src), S, seams, zc, gxy,
                                                xcd_linear(blockIdx.x, gridDim.x), (int)gridDim.x, (int)threadIdx.x);
    if (FORCE) {
        const double v = block_sum(pw, lds);
        if (threadIdx.x == 0) part[blockIdx.x] = v;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0 && slot >= 0 && slot < 2) {
        S->itr[slot] = S->hs_itr;
        S->div[slot] = S->hs_div;
    }
}

__global__ void k_dv_power(const double *part, int nblk, double len, DevScalars *S, int when)
{
    __shared__ double lds[16];
    if (when == 1 && !S->hs_done) return;
    double s = 0.0;
    for (int q = threadIdx.x; q < nblk; q += blockDim.x) s += part[q];
    s = block_sum(s, lds);
    if (threadIdx.x == 0) S->p = s / len;
}

// ---- one call ------------------------------------------------------------------
template <typename T>
struct DvRun {
    Box &b;
    T *U, *V, *W, *P;
    T *planes;  // DvPlanes
    DvSets<T> sets;
    DvCoef<T> c;
    DtRef dt;
    int par = 0;       // current set
    int nrefresh = 0;  // refreshes so far
    bool force = false;
    DvCheck ck;

    template <int NS, int MODE, int LX, int RW, int NB>
    int sweep(int k0, int k1, int sum0, int sum1)
    {
        using Tile = DvTile<T, NS, MODE, LX, RW, NB>;
        const Geom &g = b.g;
        DvArgs<T> a;
        a.g = g;
        a.Ds = sets.D[par];
        a.Fs = sets.F[par];
        const int out = MODE == kDvConstruct ? par : 1 - par;
        a.Dd = sets.D[out];
        a.Fd = sets.F[out];
        a.U = U;
        a.V = V;
        a.W = W;
        a.c = c;
        a.px = dv_pitch(g, (int)sizeof(T));
        a.kind[0] = k0;
        a.kind[1] = k1;
        a.sum[0] = sum0;
        a.sum[1] = sum1;
        const int gx = Tile::tiles_x(g), gy = Tile::tiles_y(g), nplanes = g.nz + 2 * g.h;
        const long cols = (long)gx * gy;
        const void *k = (const void *)k_dv_sweep<T, NS, MODE, LX, RW, NB>;
        int per_cu = 1, rc = kernel_setup(k, Tile::NT, 0, &per_cu);
        if (rc) return rc;
        int nz = dv_chunks(cols, nplanes, 4 * NS, (long)b.cus * per_cu);
        a.zc = (nplanes + nz - 1) / nz;
        nz = (nplanes + a.zc - 1) / a.zc;
        const int blocks = (int)(cols * nz);
        const double cells = (double)g.cells() * sizeof(T);
        ProfScope ps(b, MODE == kDvConstruct ? "hsmac_construct" : (NS == 2 ? "hsmac_div_sweep2" : "hsmac_div_sweep"),
                     (MODE == kDvConstruct ? 5.0 : 4.0) * cells);
        hipLaunchKernelGGL((k_dv_sweep<T, NS, MODE, LX, RW, NB>), dim3(blocks), dim3(Tile::NT), 0, b.stream, a, gx,
                           gy, force ? 1 : 0, dt, b.S, b.part);
        LCS_HIP(hipGetLastError());
        if (MODE == kDvConstruct) ck.nnoise = blocks;
        ck.npass = 0;
        ck.cnt[ck.npass++] = sum0 ? blocks : 0;
        ck.cnt[ck.npass++] = sum1 ? blocks : 0;
        par = out;
        return LCS_OK;
    }
    template <int NS, int MODE>
    int sweep_shape(int k0, int k1, int sum0, int sum1)
    {
        // Shapes by size (lanes, rows a lane, blocks), measured at 1000^3, 256^3,
        // 128^3, 64^3 and 32^3 FP32 and 500^3, 64^3 FP64.  Tall tiles re-read
        // fewer halo rows: at 1000^3 one sweep takes 3.51 ms with 48 rows and
        // 3.86 with 32 (4.64 and 4.22 TB/s of a 5.4 TB/s copy of two arrays).
        // Where a box has few tiles, smaller ones fill more CUs and take
        // fewer instructions a step: at 128^3 18.8 us with windows of 64 cells
        // against 23.8 of 128.  The registers of two sweeps (and of FP64) bound
        // the rows a workgroup can hold.
        const long sy = b.g.sy;
        if constexpr (sizeof(T) == 8) {
            if constexpr (NS == 1 && MODE == kDvPlain)
                if (sy >= 256) return sweep<NS, MODE, 32, 2, 24>(k0, k1, sum0, sum1);
            return sweep<NS, MODE, 32, 2, 16>(k0, k1, sum0, sum1);
        } else {
            if (sy < 200) return sweep<NS, MODE, 32, 2, 16>(k0, k1, sum0, sum1);
            if constexpr (NS == 2)
                if (sy < 512) return sweep<NS, MODE, 64, 2, 12>(k0, k1, sum0, sum1);
            if constexpr (NS == 1 && MODE == kDvPlain)
                if (sy >= 512) return sweep<NS, MODE, 64, 4, 12>(k0, k1, sum0, sum1);
            return sweep<NS, MODE, 64, 2, 16>(k0, k1, sum0, sum1);
        }
    }
    // the fill at the start of a later group, after its core sweep
    int refresh(int accumulate)
    {
        const Geom &g = b.g;
        long n[3];
        dv_refresh_cells(g, n);
        ProfScope ps(b, "hsmac_refresh", 0.0);
        hipLaunchKernelGGL(k_dv_refresh<T>, dim3((unsigned)((n[0] + n[1] + n[2] + 255) / 256)), dim3(256), 0, b.stream,
                           g, c, sets.D[1 - par], sets.F[1 - par], sets.D[par], sets.F[par], P, planes, dt,
                           accumulate, b.S);
        LCS_HIP(hipGetLastError());
        nrefresh++;
        return LCS_OK;
    }
    int faces(int want_sum)
    {
        const Geom &g = b.g;
        DvFaces<T> f{g, planes, dv_planes(g), dv_pitch(g, (int)sizeof(T))};
        T *D = sets.D[par], *F = sets.F[par];
        long cols[3];
        dv_face_columns(g, cols);
        ProfScope ps(b, "hsmac_faces", 0.0);
        for (int ax = 0; ax < 3; ax++) {
            const int blocks = dv_blocks(cols[ax]);
            double *part = b.part + (long)ck.npass * kMaxPartBlocks;
            const bool stride = cols[ax] > 256L * blocks;
            auto *k = ax == 0   ? (stride ? k_dv_face<T, 0, true> : k_dv_face<T, 0, false>)
                      : ax == 1 ? (stride ? k_dv_face<T, 1, true> : k_dv_face<T, 1, false>)
                                : (stride ? k_dv_face<T, 2, true> : k_dv_face<T, 2, false>);
            hipLaunchKernelGGL(k, dim3(blocks), dim3(256), 0, b.stream, f, D, c, b.S, want_sum, part);
            LCS_HIP(hipGetLastError());
            ck.cnt[ck.npass++] = want_sum ? blocks : 0;
        }
        long n[3];
        dv_face_cells(g, n);
        hipLaunchKernelGGL(k_dv_face_apply<T>, dim3((unsigned)((n[0] + n[1] + n[2] + 255) / 256)), dim3(256), 0,
                           b.stream, f, D, F, c, b.S);
        LCS_HIP(hipGetLastError());
        return LCS_OK;
    }
    int check(int itr, int decide)
    {
        ck.itr = itr;
        ck.par = par;
        ck.decide = decide;
        ProfScope ps(b, "hsmac_check", 0.0);
        hipLaunchKernelGGL(k_dv_check, dim3(1), dim3(256), 0, b.stream, b.part, ck, b.S);
        LCS_HIP(hipGetLastError());
        return LCS_OK;
    }
    double finish_bytes() const { return 9.0 * sizeof(T) * (double)b.g.cells(); }
    int finish(int when, int slot)
    {
        const Geom &g = b.g;
        int gxy, zc, blocks;
        dv_finish_grid(g, b.cus, gxy, zc, blocks);
        double *part = b.part + kPowerSlot;
        {
            ProfScope ps(b, "hsmac_finish", finish_bytes());
            if (force)
                hipLaunchKernelGGL((k_dv_finish<T, true>), dim3(blocks), dim3(256), 0, b.stream, g, U, V, W, P, sets,
                                   (const T *)planes, c, dt, b.S, when, par, slot, nrefresh > 0 ? 1 : 0, zc, gxy, part);
            else
                hipLaunchKernelGGL((k_dv_finish<T, false>), dim3(blocks), dim3(256), 0, b.stream, g, U, V, W, P, sets,
                                   (const T *)planes, c, dt, b.S, when, par, slot, nrefresh > 0 ? 1 : 0, zc, gxy, part);
            LCS_HIP(hipGetLastError());
        }
        if (force) {
            hipLaunchKernelGGL(k_dv_power, dim3(1), dim3(256), 0, b.stream, part, blocks, (double)g.cells(), b.S, when);
            LCS_HIP(hipGetLastError());
        }
        return LCS_OK;
    }
    int poll(bool &done)
    {
        LCS_HIP(hipMemcpyAsync(b.S_host, b.S, sizeof(DevScalars), hipMemcpyDeviceToHost, b.stream));
        LCS_HIP(hipStreamSynchronize(b.stream));
        done = b.S_host->hs_done != 0;
        return LCS_OK;
    }
};

// the box's D and F sets and planes: one allocation, made by the first call
int dv_buffers(Box &b)
{
    if (b.dv) return LCS_OK;
    const size_t bytes = dv_bytes(b.g, b.esize);
    LCS_HIP(hipMalloc(&b.dv, bytes));
    b.bytes += bytes;
    return LCS_OK;
}

template <typename T>
static int hsmac_div_t(Box &b, void **Us, DtRef dt, const lcs_hsmac_params &prm, int slot, bool lf_deferred)
{
    const Geom &g = b.g;
    int rc;
    if ((rc = dv_buffers(b))) return rc;
    const double dx = spacing(g.nx), dy = spacing(g.ny), dz = spacing(g.nz);
    const size_t set = dv_elems(g, sizeof(T));
    T *dv = (T *)b.dv;
    DvRun<T> run{b, (T *)Us[0], (T *)Us[1], (T *)Us[2], (T *)b.f[LCS_FIELD_P], dv + 4 * set, {}, {}, dt};
    for (int q = 0; q < 2; q++) {
        run.sets.D[q] = dv + q * set;
        run.sets.F[q] = dv + (2 + q) * set;
    }
    run.c = dv_coef<T>(g, prm.omega);
    run.force = lf_deferred;
    run.ck.len3 = (double)(g.nx + 1) * (double)(g.ny + 1) * (double)(g.nz + 1);
    run.ck.dxmin = std::min(std::min(dx, dy), dz);
    run.ck.epsp = prm.epsp;
    run.ck.noise = dv_noise<T>(g);

    const int last = 3 * ((prm.itrmax + 2) / 3) - 1;  // index of the last sweep the call can run
    auto may_end = [&](int n) { return n >= prm.itrmin ? 1 : 0; };
    auto counts = [&](int n) { return may_end(n) || n == last ? 1 : 0; };
    bool done = false;
    for (int n = 0; n <= last && !done; n += 3) {
        // d1: the core, then the face slabs
        const int s0 = counts(n);
        const bool fresh = n % (3 * kDvGroups) == 0;
        if (fresh) {
            if (n > 0) {  // the groups so far go into U, V, W, P
                if ((rc = run.finish(0, -1))) return rc;
                run.force = false;
                run.nrefresh = 0;
            }
            if ((rc = launch_ghost_fill(b, Us, 3, g.h, 1, nullptr))) return rc;
        }
        rc = fresh ? run.template sweep_shape<1, kDvConstruct>(0, 0, s0, 0)
                   : run.template sweep_shape<1, kDvPlain>(0, 0, s0, 0);
        if (rc || (!fresh && (rc = run.refresh(run.nrefresh > 0))) || (rc = run.faces(s0))) return rc;
        if (s0) {
            if ((rc = run.check(n, may_end(n)))) return rc;
            if (may_end(n)) {
                // most calls end here (the first sweep past itrmin): the update
                // follows at once if so, and the host looks before it goes on
                if ((rc = run.finish(1, slot)) || (rc = run.poll(done))) return rc;
                if (done) return LCS_OK;
                prof_uncount(b, "hsmac_finish", 1, run.finish_bytes());  // it found the call not done
            }
        }
        // d2 and d3: one pass unless the d2 sweep may end the iteration
        if (!may_end(n + 1)) {
            const int s2 = counts(n + 2);
            if ((rc = run.template sweep_shape<2, kDvPlain>(2, 3, 0, s2))) return rc;
            if (s2 && (rc = run.check(n + 2, may_end(n + 2)))) return rc;
        } else {
            if ((rc = run.template sweep_shape<1, kDvPlain>(2, 2, 1, 0)) || (rc = run.check(n + 1, 1)) ||
                (rc = run.template sweep_shape<1, kDvPlain>(3, 3, 1, 0)) || (rc = run.check(n + 2, 1)))
                return rc;
        }
        if (may_end(n + 2)) {
            if ((rc = run.poll(done))) return rc;
            // the d3 sweep after a d2 sweep that ended the call did nothing
            if (done && may_end(n + 1) && b.S_host->hs_itr == n + 1)
                prof_uncount(b, "hsmac_div_sweep", 1, 4.0 * sizeof(T) * (double)g.cells());
        }
    }
    return run.finish(0, slot);
}

int launch_hsmac_div(Box &b, void **Us, DtRef dt, const lcs_hsmac_params &prm, int slot, bool lf_deferred)
{
    return b.esize == 8 ? hsmac_div_t<double>(b, Us, dt, prm, slot, lf_deferred)
                        : hsmac_div_t<float>(b, Us, dt, prm, slot, lf_deferred);
}

bool hsmac_takes_div(const Geom &g, int esize, const lcs_hsmac_params &prm)
{
    return prm.time_blocking && prm.overlap && prm.coloring == LCS_COLORING_RED_BLACK_FAST && prm.itrmax >= 1 &&
           dv_fits(g, esize);
}

// ---- batches -------------------------------------------------------------------
// The same per box, one launch per phase over the listed boxes.  A box's two
// sets are numbered relative to its parity S->hs_par, so that the launches of a
// group do not depend on how many groups ran before (they are captured once and
// replayed): the groups before itrmin change sets an even number of times, the
// later ones change the parity at their end.  Tiles and chunks follow from the
// box's size alone, so that its sums of div^2, and with them its log, do not
// depend on the other boxes.
constexpr int kDvBLx = 32, kDvBRw = 2, kDvBNb = 16;

template <typename T>
__device__ inline T *dv_b_set(const BoxRec &B, int which, int cur)  // which 0: D, 1: F
{
    return (T *)B.dv_mem + (long)(2 * which + ((B.S->hs_par ^ cur) & 1)) * B.dv_set;
}
template <typename T>
__device__ inline T *dv_b_planes(const BoxRec &B)
{
    return (T *)B.dv_mem + 4 * B.dv_set;
}

template <typename T, int NS, int MODE>
__global__ void __launch_bounds__(kDvBLx *kDvBNb)
    k_b_dv_sweep(const BoxRec *tab, const TileItem *tiles, int set, int in, int k0, int k1, int sum0, int sum1,
                 double dtfac, int force)
{
    using Tile = DvTile<T, NS, MODE, kDvBLx, kDvBRw, kDvBNb>;
    __shared__ __align__(16) T lds[Tile::EX];
    __shared__ double red_lds[16];
    const TileItem it = tiles[blockIdx.x];
    const BoxRec &B = tab[it.box];
    if (b_halted(B)) return;
    const DevScalars *S = B.S;
    if (S->hs_done) return;
    DvArgs<T> a;
    a.g = B.g;
    a.Ds = dv_b_set<T>(B, 0, in);
    a.Fs = dv_b_set<T>(B, 1, in);
    a.Dd = dv_b_set<T>(B, 0, 1 - in);
    a.Fd = dv_b_set<T>(B, 1, 1 - in);
    a.U = (const T *)B.f[3 * set];
    a.V = (const T *)B.f[3 * set + 1];
    a.W = (const T *)B.f[3 * set + 2];
    a.c = dv_coef_rec<T>(B);
    a.dscale = MODE == kDvConstruct && force && B.lf_force ? T(1) + T(S->lf[4]) * T(dtfac * S->dt) : T(1);
    a.kind[0] = k0;
    a.kind[1] = k1;
    a.sum[0] = sum0;
    a.sum[1] = sum1;
    a.zc = B.dv_zc[NS - 1];
    a.px = dv_pitch(B.g, (int)sizeof(T));
    double acc[NS], nse;
    Tile::run(a, it.bx, it.by, it.bz, lds, acc, nse);
    const int blk = (it.bz * B.dv_gy[NS - 1] + it.by) * B.dv_gx + it.bx;
    for (int s = 0; s < NS; s++)
        if (a.sum[s]) {
            const double v = block_sum(acc[s], red_lds);
            if (threadIdx.x == 0) B.part[(long)s * kMaxPartBlocks + blk] = v;
        }
    if (MODE == kDvConstruct) {
        const double v = block_sum(nse, red_lds);
        if (threadIdx.x == 0) B.part[kDvNoiseSlot + blk] = v;
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
    k_b_dv_refresh(const BoxRec *tab, const WorkItem *work, int in, double dtfac, int accumulate)
{
    const WorkItem w = work[blockIdx.x];
    const BoxRec &B = tab[w.box];
    if (b_halted(B) || B.S->hs_done) return;
    dv_refresh_block(B.g, dv_coef_rec<T>(B), dv_b_set<T>(B, 0, in), dv_b_set<T>(B, 1, in), dv_b_set<T>(B, 0, 1 - in),
                     dv_b_set<T>(B, 1, 1 - in), (T *)B.f[6], dv_b_planes<T>(B), T(1.0 / (dtfac * B.S->dt)), accumulate,
                     w.blk, (int)threadIdx.x);
}

template <typename T>
__device__ inline DvFaces<T> dv_b_faces(const BoxRec &B)
{
    return DvFaces<T>{B.g, dv_b_planes<T>(B), dv_planes(B.g), dv_pitch(B.g, (int)sizeof(T))};
}

template <typename T, int AXIS>
__global__ void __launch_bounds__(256) k_b_dv_face(const BoxRec *tab, const WorkItem *work, int cur, int sum)
{
    __shared__ double lds[16];
    const WorkItem w = work[blockIdx.x];
    const BoxRec &B = tab[w.box];
    if (b_halted(B) || B.S->hs_done) return;
    const double acc =
        dv_face_block<T, AXIS, false>(dv_b_faces<T>(B), dv_b_set<T>(B, 0, cur), dv_coef_rec<T>(B), sum, w.blk, 0,
                                      (int)threadIdx.x);
    if (sum) {
        const double v = block_sum(acc, lds);
        if (threadIdx.x == 0) B.part[(long)(2 + AXIS) * kMaxPartBlocks + w.blk] = v;
    }
}

template <typename T>
__global__ void __launch_bounds__(256) k_b_dv_apply(const BoxRec *tab, const WorkItem *work, int cur)
{
    const WorkItem w = work[blockIdx.x];
    const BoxRec &B = tab[w.box];
    if (b_halted(B) || B.S->hs_done) return;
    dv_apply_block(dv_b_faces<T>(B), dv_b_set<T>(B, 0, cur), dv_b_set<T>(B, 1, cur), dv_coef_rec<T>(B), w.blk,
                   (int)threadIdx.x);
}

__global__ void k_b_dv_check(const BoxRec *tab, const int *boxes, int slots, int cur, int itr_abs, double epsp,
                             int itrmin, int flip)
{
    __shared__ double lds[16];
    const BoxRec &B = tab[boxes[blockIdx.x]];
    if (b_halted(B)) return;
    DevScalars *S = B.S;
    double nse = (int)threadIdx.x < B.dv_tiles[0] ? B.part[kDvNoiseSlot + threadIdx.x] : 0.0;
    if (S->hs_done) return;
    const int cnt[5] = {B.dv_tiles[0], B.dv_tiles[1], B.dv_faces[0], B.dv_faces[1], B.dv_faces[2]};
    double acc = 0.0;
    for (int q = 0; q < 5; q++)
        if (slots >> q & 1)
            for (int m = threadIdx.x; m < cnt[q]; m += blockDim.x) acc += B.part[(long)q * kMaxPartBlocks + m];
    for (int m = threadIdx.x + blockDim.x; m < B.dv_tiles[0]; m += blockDim.x) nse += B.part[kDvNoiseSlot + m];
    const Geom &g = B.g;
    const double len3 = (double)(g.nx + 1) * (double)(g.ny + 1) * (double)(g.nz + 1);
    const double s = block_sum(acc / len3 + B.dv_noise * nse, lds);
    if (threadIdx.x == 0) {
        const double dxmin = fmin(fmin(B.dx, B.dy), B.dz);
        const double div = sqrt(s);
        const int itr = itr_abs >= 0 ? itr_abs : S->hs_itr;
        S->hs_div = div;
        if (div * dxmin < epsp && itrmin <= itr) {
            S->hs_itr = itr;
            S->hs_par ^= cur;
            S->hs_done = 1;
        } else {
            S->hs_itr = itr + 1;
            S->hs_par ^= flip;
        }
    }
}

// The groups whose corrections an update adds: all since the last one.  final:
// the box's last group is that of its last sweep; else ngroups - 1.
__device__ inline bool dv_b_update(const BoxRec &B, int final, int ngroups, int force, int &seams, int &forced)
{
    const bool done = B.S->hs_done != 0;
    if (b_halted(B) || (!final && done)) return false;
    const int last = final && done ? B.S->hs_itr / 3 : ngroups - 1;
    seams = last % kDvGroups > 0;
    forced = force && B.lf_force && last < kDvGroups;
    return true;
}

template <typename T>
__global__ void __launch_bounds__(256)
    k_b_dv_finish(const BoxRec *tab, const WorkItem *work, int set, double dtfac, int final, int ngroups, int force)
{
    __shared__ double lds[16];
    const WorkItem w = work[blockIdx.x];
    const BoxRec &B = tab[w.box];
    int seams, forced;
    if (!dv_b_update(B, final, ngroups, force, seams, forced)) return;
    T *U = (T *)B.f[3 * set], *V = (T *)B.f[3 * set + 1], *W = (T *)B.f[3 * set + 2], *P = (T *)B.f[6];
    const T *F = dv_b_set<T>(B, 1, 0), *planes = dv_b_planes<T>(B);
    const DvCoef<T> c = dv_coef_rec<T>(B);
    const double d = dtfac * B.S->dt;
    if (forced) {
        const double pw =
            dv_finish_block<T, true>(B.g, U, V, W, P, F, planes, c, d, B.S, seams, B.dv_fzc, B.dv_gxy, w.blk,
                                     B.dv_fin, (int)threadIdx.x);
        const double v = block_sum(pw, lds);
        if (threadIdx.x == 0) B.part[kPowerSlot + w.blk] = v;
    } else
        dv_finish_block<T, false>(B.g, U, V, W, P, F, planes, c, d, B.S, seams, B.dv_fzc, B.dv_gxy, w.blk, B.dv_fin,
                                  (int)threadIdx.x);
}

__global__ void k_b_dv_power(const BoxRec *tab, const int *boxes, int final, int ngroups, int force)
{
    __shared__ double lds[16];
    const BoxRec &B = tab[boxes[blockIdx.x]];
    int seams, forced;
    if (!dv_b_update(B, final, ngroups, force, seams, forced) || !forced) return;
    double v = 0.0;
    for (int q = threadIdx.x; q < B.dv_fin; q += blockDim.x) v += B.part[kPowerSlot + q];
    v = block_sum(v, lds);
    if (threadIdx.x == 0) B.S->p = v / (double)B.g.cells();
}

template <typename T>
static int dv_record_t(Box &b, const lcs_hsmac_params &prm, int i, BoxRec &r, DvWork &w)
{
    using T1 = DvTile<T, 1, kDvPlain, kDvBLx, kDvBRw, kDvBNb>;
    using T2 = DvTile<T, 2, kDvPlain, kDvBLx, kDvBRw, kDvBNb>;
    static_assert(T1::OWN == T2::OWN, "one tile count along x");
    const Geom &g = b.g;
    int rc = dv_buffers(b);
    if (rc) return rc;
    r.dv = 1;
    r.dv_mem = b.dv;
    r.dv_set = (long)dv_elems(g, sizeof(T));
    const DvCoef<T> c = dv_coef<T>(g, prm.omega);
    const T v[9] = {c.k, c.cx, c.cy, c.cz, c.c0, c.c0l, c.dxi, c.dyi, c.dzi};
    for (int q = 0; q < 9; q++) r.dv_c[q] = (double)v[q];
    r.dv_noise = dv_noise<T>(g);
    const int nplanes = g.nz + 2 * g.h;
    r.dv_gx = T1::tiles_x(g);
    r.dv_gy[0] = T1::tiles_y(g);
    r.dv_gy[1] = T2::tiles_y(g);
    for (int q = 0; q < 2; q++) {
        r.dv_zc[q] = dv_batch_zc(nplanes);
        const int nz = (nplanes + r.dv_zc[q] - 1) / r.dv_zc[q];
        r.dv_tiles[q] = r.dv_gx * r.dv_gy[q] * nz;
        for (int z = 0; z < nz; z++)
            for (int y = 0; y < r.dv_gy[q]; y++)
                for (int x = 0; x < r.dv_gx; x++) w.tiles[q].push_back({i, x, y, z});
    }
    auto blocks = [](long n) { return (int)((n + 255) / 256); };
    auto list = [&](std::vector<WorkItem> &l, int n) {
        for (int k = 0; k < n; k++) l.push_back({i, k});
    };
    long n[3];
    dv_refresh_cells(g, n);
    list(w.refresh, blocks(n[0] + n[1] + n[2]));
    dv_face_cells(g, n);
    list(w.apply, blocks(n[0] + n[1] + n[2]));
    long cols[3];
    dv_face_columns(g, cols);
    for (int a = 0; a < 3; a++) {
        r.dv_faces[a] = blocks(cols[a]);
        list(w.faces[a], r.dv_faces[a]);
    }
    dv_finish_grid(g, 8, r.dv_gxy, r.dv_fzc, r.dv_fin);
    list(w.fin, r.dv_fin);
    const long X = g.nx + 2L * g.h, Y = g.ny + 2L * g.h;
    list(w.ghost, blocks(2L * g.h * (X * Y + X * g.nz + (long)g.ny * g.nz)));
    w.boxes.push_back(i);
    int most = std::max(r.dv_tiles[0], r.dv_tiles[1]);
    for (int a = 0; a < 3; a++) most = std::max(most, r.dv_faces[a]);
    return most > kMaxPartBlocks ? fail(LCS_ERR_CAPACITY, "box too large for a batch") : LCS_OK;
}

int dv_batch_record(Box &b, const lcs_hsmac_params &prm, int i, BoxRec &r, DvWork &w)
{
    return b.esize == 8 ? dv_record_t<double>(b, prm, i, r, w) : dv_record_t<float>(b, prm, i, r, w);
}

#define DV_LAUNCH(kern, n, nt, ...)                                                     \
    do {                                                                                \
        if ((n) == 0) return LCS_OK;                                                    \
        if (esize == 8)                                                                 \
            hipLaunchKernelGGL((kern(double)), dim3(n), dim3(nt), 0, s, __VA_ARGS__);   \
        else                                                                            \
            hipLaunchKernelGGL((kern(float)), dim3(n), dim3(nt), 0, s, __VA_ARGS__);    \
        LCS_HIP(hipGetLastError());                                                     \
        return LCS_OK;                                                                  \
    } while (0)

int launch_b_dv_sweep(hipStream_t s, int esize, const BoxRec *tab, const TileItem *tiles, int n, int ns, int construct,
                      int set, int in, int k0, int k1, int sum0, int sum1, double dtfac, int force)
{
#define K2(T) k_b_dv_sweep<T, 2, kDvPlain>
#define KC(T) k_b_dv_sweep<T, 1, kDvConstruct>
#define K1(T) k_b_dv_sweep<T, 1, kDvPlain>
    if (ns == 2) DV_LAUNCH(K2, n, kDvBLx * kDvBNb, tab, tiles, set, in, k0, k1, sum0, sum1, dtfac, force);
    if (construct) DV_LAUNCH(KC, n, kDvBLx * kDvBNb, tab, tiles, set, in, k0, k1, sum0, sum1, dtfac, force);
    DV_LAUNCH(K1, n, kDvBLx * kDvBNb, tab, tiles, set, in, k0, k1, sum0, sum1, dtfac, force);
#undef K2
#undef KC
#undef K1
}

int launch_b_dv_refresh(hipStream_t s, int esize, const BoxRec *tab, const WorkItem *work, int n, int in, double dtfac,
                        int accumulate)
{
#define K(T) k_b_dv_refresh<T>
    DV_LAUNCH(K, n, 256, tab, work, in, dtfac, accumulate);
#undef K
}

int launch_b_dv_face(hipStream_t s, int esize, const BoxRec *tab, const WorkItem *work, int n, int axis, int cur,
                     int sum)
{
#define K0(T) k_b_dv_face<T, 0>
#define K1(T) k_b_dv_face<T, 1>
#define K2(T) k_b_dv_face<T, 2>
    if (axis == 0) DV_LAUNCH(K0, n, 256, tab, work, cur, sum);
    if (axis == 1) DV_LAUNCH(K1, n, 256, tab, work, cur, sum);
    DV_LAUNCH(K2, n, 256, tab, work, cur, sum);
#undef K0
#undef K1
#undef K2
}

int launch_b_dv_apply(hipStream_t s, int esize, const BoxRec *tab, const WorkItem *work, int n, int cur)
{
#define K(T) k_b_dv_apply<T>
    DV_LAUNCH(K, n, 256, tab, work, cur);
#undef K
}

int launch_b_dv_check(hipStream_t s, const BoxRec *tab, const int *boxes, int n, int slots, int cur, int itr,
                      double epsp, int itrmin, int flip)
{
    if (n == 0) return LCS_OK;
    hipLaunchKernelGGL(k_b_dv_check, dim3(n), dim3(256), 0, s, tab, boxes, slots, cur, itr, epsp, itrmin, flip);
    LCS_HIP(hipGetLastError());
    return LCS_OK;
}

static int b_dv_finish(hipStream_t s, int esize, const BoxRec *tab, const WorkItem *work, int n, int set, double dtfac,
                       int final, int ngroups, int force)
{
#define K(T) k_b_dv_finish<T>
    DV_LAUNCH(K, n, 256, tab, work, set, dtfac, final, ngroups, force);
#undef K
}

int launch_b_dv_finish(hipStream_t s, int esize, const BoxRec *tab, const WorkItem *work, int n, const int *boxes,
                       int nboxes, int set, double dtfac, int final, int ngroups, int force)
{
    int rc = b_dv_finish(s, esize, tab, work, n, set, dtfac, final, ngroups, force);
    if (rc || !force || nboxes == 0) return rc;
    hipLaunchKernelGGL(k_b_dv_power, dim3(nboxes), dim3(256), 0, s, tab, boxes, final, ngroups, force);
    LCS_HIP(hipGetLastError());
    return LCS_OK;
}

}  // namespace lcs
