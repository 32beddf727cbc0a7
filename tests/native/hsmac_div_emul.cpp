// Host execution of HSMAC in divergence form (lcs.jl_amd/csrc/lcs_hsmac_div.h,
// lcs_hsmac_shell.h): a whole couple! call, every workgroup of every pass run
// thread by thread in the kernels' barrier order, so that a test can compare the
// kernels' own code with the oracle.  D, F and the planes stand between margins
// that must come out untouched.
#include <cmath>
#include <vector>

#include "lcs_hsmac_div.h"
#include "lcs_hsmac_shell.h"

using namespace lcs;

namespace {

template <typename T>
struct Guarded {
    static constexpr size_t M = 4096;
    std::vector<T> v;
    explicit Guarded(size_t n) : v(n + 2 * M, T(NAN)) {}
    T *data() { return v.data() + M; }
    bool intact() const
    {
        for (size_t q = 0; q < M; q++)
            if (!std::isnan(v[q]) || !std::isnan(v[v.size() - 1 - q])) return false;
        return true;
    }
};

template <typename T>
void fill_ghosts(const Geom &g, T *A)
{
    auto image = [&](int v, int n) { return v < g.h ? v + n : (v >= n + g.h ? v - n : v); };
    for (int z = 0; z < g.nz + 2 * g.h; z++)
        for (int y = 0; y < g.sy; y++)
            for (int x = 0; x < g.sx; x++)
                A[x + g.sx * (y + g.sy * (long)z)] =
                    A[image(x, g.nx) + g.sx * (image(y, g.ny) + g.sy * (long)image(z, g.nz))];
}

template <typename T>
struct Call {
    Geom g;
    T *U, *V, *W, *P;
    double dt;
    DvCoef<T> c;
    const DevScalars *S;
    int shape, zc, cus;
    Guarded<T> D0, D1, F0, F1, planes;
    T *D[2], *F[2];
    int par = 0;
    double sum = 0, nse = 0;
    bool force;

    Call(const Geom &g, void *const *f, double dt, double omega, const DevScalars *S, int shape, int zc, int cus, bool force)
        : g(g), U((T *)f[0]), V((T *)f[1]), W((T *)f[2]), P((T *)f[3]), dt(dt), c(dv_coef<T>(g, omega)), S(S),
          shape(shape), zc(zc), cus(cus), D0(dv_elems(g, sizeof(T))), D1(dv_elems(g, sizeof(T))),
          F0(dv_elems(g, sizeof(T))), F1(dv_elems(g, sizeof(T))), planes(dv_planes(g).total),
          D{D0.data(), D1.data()}, F{F0.data(), F1.data()}, force(force)
    {
    }

    template <int NS, int MODE, int LX, int RW, int NB>
    double run(int k0, int k1)
    {
        using Tile = DvTile<T, NS, MODE, LX, RW, NB>;
        DvArgs<T> a;
        const int out = MODE == kDvConstruct ? par : 1 - par;
        a.g = g;
        a.Ds = D[par];
        a.Fs = F[par];
        a.Dd = D[out];
        a.Fd = F[out];
        a.U = U;
        a.V = V;
        a.W = W;
        a.c = c;
        a.dscale = MODE == kDvConstruct && force ? T(1) + T(S->lf[4]) * T(dt) : T(1);
        a.kind[0] = k0;
        a.kind[1] = k1;
        a.sum[0] = a.sum[1] = 1;
        a.zc = zc;
        a.px = dv_pitch(g, sizeof(T));
        std::vector<T> lds(Tile::EX);
        std::vector<typename Tile::Th> th(Tile::NT), was(Tile::NT);
        double acc[NS] = {};
        if (MODE == kDvConstruct) nse = 0;
        double n = 0;
        for (int bz = 0; bz < (g.nz + 2 * g.h + zc - 1) / zc; bz++)
            for (int by = 0; by < Tile::tiles_y(g); by++)
                for (int bx = 0; bx < Tile::tiles_x(g); bx++)
                    Tile::emulate_block(a, bx, by, bz, lds.data(), th.data(), was.data(), acc, n);
        if (MODE == kDvConstruct) nse = n;
        par = out;
        return acc[NS - 1];
    }
    // the windows of the size rule's classes: 0 small boxes, 1 tall ones, 2 (FP32) taller ones
    template <int NS, int MODE>
    double sweep(int k0, int k1)
    {
        if constexpr (sizeof(T) == 8) {
            if constexpr (NS == 1 && MODE == kDvPlain)
                if (shape > 0) return run<NS, MODE, 32, 2, 24>(k0, k1);
            return run<NS, MODE, 32, 2, 16>(k0, k1);
        } else {
            if (shape == 0) return run<NS, MODE, 32, 2, 16>(k0, k1);
            if constexpr (NS == 2)
                if (shape == 1) return run<NS, MODE, 64, 2, 12>(k0, k1);
            if constexpr (NS == 1 && MODE == kDvPlain)
                if (shape == 2) return run<NS, MODE, 64, 4, 12>(k0, k1);
            return run<NS, MODE, 64, 2, 16>(k0, k1);
        }
    }
    void refresh(int accumulate)
    {
        long n[3];
        dv_refresh_cells(g, n);
        for (int b = 0; b < (n[0] + n[1] + n[2] + 255) / 256; b++)
            for (int t = 0; t < 256; t++)
                dv_refresh_block(g, c, D[1 - par], F[1 - par], D[par], F[par], P, planes.data(), T(1.0 / dt), accumulate, b, t);
    }
    template <int AXIS>
    double face(const DvFaces<T> &f, long cols, bool stride)
    {
        double s = 0;
        const int blocks = stride ? 3 : (int)((cols + 255) / 256);
        for (int b = 0; b < blocks; b++)
            for (int t = 0; t < 256; t++)
                s += stride ? dv_face_block<T, AXIS, true>(f, D[par], c, 1, b, blocks, t)
                            : dv_face_block<T, AXIS, false>(f, D[par], c, 1, b, blocks, t);
        return s;
    }
    double faces(bool stride)
    {
        DvFaces<T> f{g, planes.data(), dv_planes(g), dv_pitch(g, sizeof(T))};
        long cols[3], n[3];
        dv_face_columns(g, cols);
        const double s = (face<0>(f, cols[0], stride) + face<1>(f, cols[1], stride)) + face<2>(f, cols[2], stride);
        dv_face_cells(g, n);
        for (int b = 0; b < (n[0] + n[1] + n[2] + 255) / 256; b++)
            for (int t = 0; t < 256; t++) dv_apply_block(f, D[par], F[par], c, b, t);
        return s;
    }
    double finish(int seams, bool stride)
    {
        int gxy, fzc, blocks;
        dv_finish_grid(g, cus, gxy, fzc, blocks);
        if (stride) blocks = 3;
        double pw = 0;
        for (int b = 0; b < blocks; b++)
            for (int t = 0; t < 256; t++)
                pw += force ? dv_finish_block<T, true>(g, U, V, W, P, F[par], planes.data(), c, dt, S, seams, fzc, gxy, b, blocks, t)
                            : dv_finish_block<T, false>(g, U, V, W, P, F[par], planes.data(), c, dt, S, seams, fzc, gxy, b, blocks, t);
        return pw / (double)g.cells();
    }
    bool intact() const { return D0.intact() && D1.intact() && F0.intact() && F1.intact() && planes.intact(); }

    // the call of hsmac_div_t
    int couple(double epsp, int itrmin, int itrmax, bool stride, int *itr, double *div, double *power)
    {
        const int last = 3 * ((itrmax + 2) / 3) - 1;
        const double len3 = (double)(g.nx + 1) * (g.ny + 1) * (g.nz + 1);
        const double dxmin = std::min({spacing(g.nx), spacing(g.ny), spacing(g.nz)});
        int seams = 0;
        auto ends = [&](int n, double s) {
            *div = std::sqrt(s / len3 + dv_noise<T>(g) * nse);
            *itr = n >= itrmin && *div * dxmin < epsp ? n : n + 1;
            return *itr == n;
        };
        auto update = [&]() {
            const double p = finish(seams, stride);
            if (force) *power = p;
            force = false;
        };
        for (int n = 0; n <= last; n += 3) {
            const bool fresh = n % (3 * kDvGroups) == 0;
            if (fresh) {
                if (n > 0) update();
                seams = 0;
                for (T *A : {U, V, W}) fill_ghosts(g, A);
            }
            double s = fresh ? sweep<1, kDvConstruct>(0, 0) : sweep<1, kDvPlain>(0, 0);
            if (!fresh) {
                refresh(seams);
                seams = 1;
            }
            s += faces(stride);
            bool done = ends(n, s);
            if (!done && n + 1 < itrmin)
                done = ends(n + 2, sweep<2, kDvPlain>(2, 3));
            else if (!done)
                done = ends(n + 1, sweep<1, kDvPlain>(2, 2)) || ends(n + 2, sweep<1, kDvPlain>(3, 3));
            if (done) break;
        }
        update();
        return intact() ? 0 : -2;
    }
};

template <typename T>
int run(const Geom &g, void *const *f, double dt, double omega, double epsp, int itrmin, int itrmax, const double *lf,
        int shape, int zc, int stride, int *itr, double *div, double *power)
{
    if (!dv_fits(g, sizeof(T))) return -1;
    DevScalars S = {};
    if (lf)
        for (int q = 0; q < 5; q++) S.lf[q] = lf[q];
    Call<T> c(g, f, dt, omega, &S, shape, zc, 8, lf != nullptr);
    return c.couple(epsp, itrmin, itrmax, stride != 0, itr, div, power);
}

}  // namespace

// lf: null, or the deferred linear forcing {-, mean U, mean V, mean W, A}
extern "C" int hsmac_div_emul(int esize, int nx, int ny, int nz, int h, void *const *f, double dt, double omega,
                              double epsp, int itrmin, int itrmax, const double *lf, int shape, int zc, int stride,
                              int *itr, double *div, double *power)
{
    const Geom g = make_geom(nx, ny, nz, h);
    return esize == 8 ? run<double>(g, f, dt, omega, epsp, itrmin, itrmax, lf, shape, zc, stride, itr, div, power)
                      : run<float>(g, f, dt, omega, epsp, itrmin, itrmax, lf, shape, zc, stride, itr, div, power);
}
