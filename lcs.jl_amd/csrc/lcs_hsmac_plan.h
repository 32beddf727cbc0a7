// Sizes and work counts of HSMAC in divergence form (lcs_hsmac_div.h), and the
// rule that sends a box to it.  No kernels: a host test checks the counts
// against their limits at sizes that no test runs.
#pragma once

#include <algorithm>
#include <climits>

#include "lcs_internal.h"

namespace lcs {

// Row pitch of D and F in elements: rows start on 64-byte lines, and the pitch
// is an odd number of lines, so that the rows of a tile spread over the memory
// channels (a pitch of 4096 bytes ran a marching copy at 3.4 TB/s, 4032 bytes
// at 4.7, the field's own 4024 at 3.5: 1006^3 FP32, 112-wide tiles).
__host__ __device__ inline int dv_pitch(const Geom &g, int esize)
{
    if (g.sx < 256) return (int)g.sx;  // small boxes run from cache
    const int line = 64 / esize, n = ((int)g.sx + line - 1) / line;
    return (n | 1) * line;
}

// seam and edge planes of a box, one allocation: U, V, W seam planes over
// the interior, then U, V, W edge planes over the whole cross-section
struct DvPlanes {
    long seam[3], edge[3], dp[3];
    long total;
};
__host__ __device__ inline DvPlanes dv_planes(const Geom &g)
{
    DvPlanes p;
    const long nx = g.nx, ny = g.ny, nz = g.nz, sz = nz + 2 * g.h;
    long at = 0;
    const long s[3] = {ny * nz, nx * nz, nx * ny}, e[3] = {g.sy * sz, g.sx * sz, g.sx * g.sy};
    // corrections of the face slabs of the overlap order, x, y, z: 2 slabs x 3 layers
    const long d[3] = {6 * (ny - 1) * (nz - 1), 6 * (nx + 5) * (nz - 1), 6 * (nx + 5) * (ny + 5)};
    for (int a = 0; a < 3; a++) {
        p.seam[a] = at;
        at += s[a];
    }
    for (int a = 0; a < 3; a++) {
        p.edge[a] = at;
        at += e[a];
    }
    for (int a = 0; a < 3; a++) {
        p.dp[a] = at;
        at += d[a];
    }
    p.total = at;
    return p;
}

// elements of one D or F array
inline size_t dv_elems(const Geom &g, int esize)
{
    return (size_t)dv_pitch(g, esize) * (size_t)g.sy * (size_t)(g.nz + 2 * g.h);
}
// the two (D, F) sets and the planes
inline size_t dv_bytes(const Geom &g, int esize)
{
    return (4 * dv_elems(g, esize) + (size_t)dv_planes(g).total) * (size_t)esize;
}

// The window of a sweep's workgroup (DvTile) and the part of it that a tile owns
template <int ESIZE, int NS, int LX, int RW, int NB>
struct DvWindow {
    static constexpr int LINE = 64 / ESIZE;
    static constexpr int W = 2 * LX, OWN = (W - 4 * NS) / LINE * LINE, HX = (W - OWN) / 2;
    static constexpr int ROWS = NB * RW, HY = 2 * NS;

    // one element of padding at the end keeps the last window's edge outside the array
    __host__ __device__ static int tiles_x(const Geom &g)
    {
        return g.sx + 1 <= W ? 1 : ((int)g.sx + OWN - 1) / OWN;
    }
    __host__ __device__ static int tiles_y(const Geom &g)
    {
        const int s = (int)g.sy + 1, own = ROWS - 2 * HY;
        return s <= ROWS ? 1 : 1 + (s - ROWS + own - 1) / own;
    }
    static long columns(const Geom &g) { return (long)tiles_x(g) * tiles_y(g); }
};

// cells of the shell a refresh visits: z planes 0..h and nz+h-1.., then rows y
// 0..h and ny+h-1.., then x 0..h and nx+h-1..  (2h+2 layers on each axis)
__host__ __device__ inline void dv_refresh_cells(const Geom &g, long n[3])
{
    const long L = 2 * g.h + 2;
    n[0] = L * g.sx * g.sy;
    n[1] = L * g.sx * (g.nz - 2);
    n[2] = L * (g.ny - 2) * (long)(g.nz - 2);
}

// columns across the two slabs of the z, y and x axis
__host__ __device__ inline void dv_face_columns(const Geom &g, long n[3])
{
    n[0] = 2L * (g.nx + 5) * (g.ny + 5);
    n[1] = 2L * (g.nx + 5) * (g.nz - 1);
    n[2] = 2L * (g.ny - 1) * (g.nz - 1);
}

// cells a slab correction changes, each handled once: layers -1..2 and n..n+3
// of z over domain 1, then of y for k in 3..nz-1, then of x for j, k inside
__host__ __device__ inline void dv_face_cells(const Geom &g, long n[3])
{
    n[0] = 8L * (g.nx + 5) * (g.ny + 5);
    n[1] = 8L * (g.nx + 5) * (g.nz - 3);
    n[2] = 8L * (g.ny - 3) * (g.nz - 3);
}

// Workgroups of a pass that leaves one partial sum each: at most a partial
// slot's; where there is more work they stride over it.
inline int dv_blocks(long items)
{
    return (int)std::min<long>((items + 255) / 256, kMaxPartBlocks);
}

// Columns of planes of the update: gxy columns of 256 cells in chunks of zc
// planes.  Short chunks where the grid is small, so that the chip is filled, at
// most 32 planes while the tasks fit a partial slot, longer ones beyond that
// (1000^3: 252 planes).
inline void dv_finish_grid(const Geom &g, int cus, int &gxy, int &zc, int &blocks)
{
    const int nplanes = g.nz + 2 * g.h;
    gxy = (int)((g.sx * g.sy + 255) / 256);
    int nz = (int)std::min<long>(nplanes, std::max<long>(1, (8L * cus + gxy - 1) / gxy));
    nz = std::max(nz, (nplanes + 31) / 32);
    nz = std::min<int>(nz, std::max(1, kMaxPartBlocks / gxy));
    zc = (nplanes + nz - 1) / nz;
    blocks = (int)std::min<long>((long)gxy * ((nplanes + zc - 1) / zc), kMaxPartBlocks);
}

// z-chunks of a single box's sweep: the count with the fewest plane-steps on
// the busiest CU, a chunk paying `halo` planes, among chunks of at most
// kDvMaxChunk planes: workgroups end at different times, and short chunks
// even that out (1000^3, two sweeps: 4.17 ms with 2 chunks, 3.92 with 8)
constexpr int kDvMaxChunk = 128;
inline int dv_chunks(long cols, int nplanes, int halo, long slots)
{
    const int n0 = (nplanes + kDvMaxChunk - 1) / kDvMaxChunk;
    int best_n = std::max(1, (int)std::min<long>(n0, kMaxPartBlocks / cols));
    double best = 1e300;
    for (int n = best_n; n <= nplanes && cols * n <= kMaxPartBlocks; n++) {
        const int zc = (nplanes + n - 1) / n;
        const double cost = (double)((cols * n + slots - 1) / slots) * (zc + halo + 2);
        if (cost < best * 0.999) {
            best = cost;
            best_n = n;
        }
    }
    return best_n;
}

// planes per chunk of a batched sweep: about eight chunks for small boxes, of
// about 28 planes for others (each re-reads 4 NS planes; the launch fills the
// chip with the tiles of many boxes)
inline int dv_batch_zc(int nplanes)
{
    const int n = nplanes <= 80 ? 8 : std::max(1, (nplanes + 14) / 28);
    return (nplanes + n - 1) / n;
}

// Boxes the divergence form takes: one image per ghost, face slabs of one axis
// (with the ring of cells they change) that do not meet, columns of tiles that
// fit a partial slot in every window the sweeps use, and cell counts of the
// shell kernels within their 32-bit indices (less the stride of a capped grid).
inline bool dv_fits(const Geom &g, int esize)
{
    const int m = g.h > 8 ? g.h : 8;
    if (g.h < 3 || g.nx < m || g.ny < m || g.nz < m) return false;
    const long cols =
        esize == 8 ? std::max({DvWindow<8, 1, 32, 2, 16>::columns(g), DvWindow<8, 1, 32, 2, 24>::columns(g),
                               DvWindow<8, 2, 32, 2, 16>::columns(g)})
                   : std::max({DvWindow<4, 1, 32, 2, 16>::columns(g), DvWindow<4, 1, 64, 4, 12>::columns(g),
                               DvWindow<4, 1, 64, 2, 16>::columns(g), DvWindow<4, 2, 32, 2, 16>::columns(g),
                               DvWindow<4, 2, 64, 2, 12>::columns(g), DvWindow<4, 2, 64, 2, 16>::columns(g)});
    if (cols > kMaxPartBlocks) return false;
    long r[3], f[3];
    dv_refresh_cells(g, r);
    dv_face_cells(g, f);
    const long most = std::max({r[0] + r[1] + r[2], f[0] + f[1] + f[2], (long)dv_pitch(g, esize) * g.sy});
    return most < (long)INT_MAX - 256L * kMaxPartBlocks;
}

}  // namespace lcs
