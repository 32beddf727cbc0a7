// The launch counts of HSMAC in divergence form (lcs.jl_amd/csrc/lcs_hsmac_plan.h)
// for a box, as the launchers form them.
#include "lcs_hsmac_plan.h"

using namespace lcs;

template <int ESIZE>
static void counts(const Geom &g, long *out)
{
    out[0] = kMaxPartBlocks;
    long cols[3];
    dv_face_columns(g, cols);
    for (int a = 0; a < 3; a++) out[1 + a] = dv_blocks(cols[a]);
    int gxy, zc, blocks;
    const int nplanes = g.nz + 2 * g.h;
    dv_finish_grid(g, 256, gxy, zc, blocks);
    out[4] = blocks;
    out[5] = (long)gxy * ((nplanes + zc - 1) / zc);  // tasks
    dv_finish_grid(g, 8, gxy, zc, blocks);
    out[6] = blocks;
    const long c1 = DvWindow<ESIZE, 1, 32, 2, 16>::columns(g), c2 = DvWindow<ESIZE, 2, 32, 2, 16>::columns(g);
    // sweeps in the windows of the size class, one and two a pass
    const long s1 = ESIZE == 8 ? (g.sy >= 256 ? DvWindow<ESIZE, 1, 32, 2, 24>::columns(g) : c1)
                    : g.sy < 200 ? c1
                                 : (g.sy >= 512 ? DvWindow<ESIZE, 1, 64, 4, 12>::columns(g)
                                                : DvWindow<ESIZE, 1, 64, 2, 16>::columns(g));
    const long s2 = ESIZE == 8 || g.sy < 200 ? c2
                    : g.sy < 512 ? DvWindow<ESIZE, 2, 64, 2, 12>::columns(g)
                                 : DvWindow<ESIZE, 2, 64, 2, 16>::columns(g);
    out[7] = s1 * dv_chunks(s1, nplanes, 4, 1024);
    out[8] = s2 * dv_chunks(s2, nplanes, 8, 1024);
    long r[3], f[3];
    dv_refresh_cells(g, r);
    dv_face_cells(g, f);
    out[9] = r[0] + r[1] + r[2];
    out[10] = f[0] + f[1] + f[2];
    out[11] = (long)dv_pitch(g, ESIZE) * g.sy;
    out[12] = (long)dv_bytes(g, ESIZE);
}

extern "C" int hsmac_div_plan(int nx, int ny, int nz, int h, int esize, long *out)
{
    const Geom g = make_geom(nx, ny, nz, h);
    if (!dv_fits(g, esize)) return 0;
    if (esize == 8)
        counts<8>(g, out);
    else
        counts<4>(g, out);
    return 1;
}
