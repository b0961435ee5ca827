// march_check.cpp -- CPU enumeration of every device address the whole-grid fused step
// (march.hip) forms, checked against the sizes of the arrays a shot allocates, and of its
// stores: each cell and each memory variable exactly once.  Test infrastructure (run by
// tests/test_march_index.py).
//
// The launch geometry comes from the library (make_plan, geometry) and every per-lane
// quantity from the functions the kernel calls (geom.hpp: xcd_block, tile_of,
// segment_planes, march_tile, layer_index, cell_offset,
// x/y/zmem_offset).  What this file restates is which planes a wave of each role loads.
//
// usage: march_check nx ny nz npml storage tile zseg strips free_surface [mutation]
// mutation 1: a memory variable's array is one element shorter; 2: a chunk owns one column less.
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

#include "core.hpp"
#include "geom.hpp"
#include "shot.hpp"

using namespace ela3d;

static long long g_acc = 0, g_bad = 0;
static void check(long long o, long long n, long long lim, const char* what)
{
    ++g_acc;
    if (o < 0 || o + n > lim) {
        if (g_bad++ < 8) std::printf("  out of bounds: %s [%lld, %lld) limit %lld\n", what, o, o + n, lim);
    }
}

int main(int argc, char** argv)
{
    if (argc < 10) return 2;
    int a[10] = {};
    for (int q = 0; q < 10 && q + 1 < argc; ++q) a[q] = std::atoi(argv[q + 1]);
    ela3d_config c;
    ela3d_config_default(&c);
    c.nx = a[0]; c.ny = a[1]; c.nz = a[2]; c.npoints_pml = a[3];
    c.storage = a[4];
    c.free_surface = a[8];
    c.isrc = c.nx / 2; c.jsrc = c.ny / 2; c.ksrc = c.nz / 2;
    c.nstep = 1;
    const int mutation = a[9];
    ShotPlan P;
    try {
        P = make_plan(c);
    } catch (const Error& e) {
        std::printf("refused %s\n", e.msg.c_str());
        return 0;
    }
    Tuning t;
    t.fused = 2; t.dbuf = 1; t.tile = a[5]; t.zseg_interior = a[6]; t.strips = a[7];
    const std::string why = march_unsupported(P, t);
    if (!why.empty()) {
        std::printf("refused %s\n", why.c_str());
        return 0;
    }
    LaunchGeom slab, G;
    geometry(P, t, slab, G);
    const int nx = c.nx, ny = c.ny, nz = c.nz;
    const int nxyp = int(plane_stride(nx, ny)), g0 = int(guard_elems(nx));
    const int lo[3] = {P.ax[0].lo, P.ax[1].lo, P.ax[2].lo}, hi[3] = {P.ax[0].hi, P.ax[1].hi, P.ax[2].hi};
    const int w[3] = {P.ax[0].width(), P.ax[1].width(), P.ax[2].width()};
    const long long field = (long long)nxyp * nz + 2ll * g0;
    const long long cut = mutation == 1 ? 1 : 0;
    const long long mem[3] = {(long long)nz * ny * w[0] - cut, (long long)nz * w[1] * nx - cut,
                              (long long)w[2] * ny * nx - cut};
    std::vector<unsigned char> cells(size_t(nx) * ny * nz, 0), ms[3];
    for (int q = 0; q < 3; ++q) ms[q].assign(size_t(mem[q] + cut), 0);
    // walked backwards, an XCD's blocks are the same ones in reverse
    for (int n = 1; n <= G.nblocks; n = n < 40 || n == G.nblocks ? n + 1 : G.nblocks) {
        std::vector<unsigned char> seen(size_t(n), 0);
        for (int b = 0; b < n; ++b) {
            const int x = b % 8, len = n / 8 + (x < n % 8 ? 1 : 0), t = turned(b, n, 1);
            if (turned(b, n, 0) != b || t < 0 || t >= n || seen[size_t(t)]++) {
                ++g_bad;
                break;
            }
            if (xcd_block(t, n) - xcd_block(x, n) != len - 1 - b / 8) ++g_bad;
        }
    }
    for (int b = 0; b < G.nblocks; ++b) {
        int chunk, zs, kb, ke;
        tile_of(G.box[0], xcd_block(b, G.nblocks), chunk, zs);
        segment_planes(G.box[0], zs, kb, ke);
        MarchTile T = march_tile(nx, ny, G.rows, G.xch, G.xw, chunk);
        if (mutation == 2) --T.x1;
        if (T.xe - T.xs > 64 || T.n < 1 || T.x1 <= T.x0) ++g_bad;  // lanes, rows, columns
        for (int wave = 0; wave < G.block / 64; ++wave) {
          if (wave >= T.n && wave != G.rows) continue;  // no row
          for (int half = 0; half < (wave == G.rows ? 2 : 1); ++half) {  // the last wave holds both halo rows
            const int role = wave == G.rows ? 1 + half : 0;
            const int slot = role == 0 ? wave + 1 : role == 1 ? 0 : T.n + 1;
            const int j = T.j0 - 1 + slot;
            if (j < 0 || j >= ny) continue;
            if (slot >= G.rows + 2) ++g_bad;
            for (int lane = 0; lane < 64; ++lane) {
                const int i = T.xs + lane, ic = i < T.xe ? i : T.xe - 1;
                const bool own = i >= T.x0 && i < T.x1;
                const int cx = layer_index(i, lo[0], hi[0]), cy = layer_index(j, lo[1], hi[1]);
                const bool inx = i < T.xe && cx >= 0;
                const unsigned o0 = cell_offset(g0, nxyp, 0, j * nx + ic);
                const unsigned ox = inx ? xmem_offset(0, j, cx, ny, w[0]) : 0u;
                for (int m = kb > 0 ? kb - 1 : kb; m <= ke && m < nz; ++m) {
                    const long long o = o0 + unsigned(m) * unsigned(nxyp);
                    check(o, 1, field, "field");
                    if (m < nz - 1 && m < ke) check(o + nxyp, 1, field, "field above");
                    const int cz = layer_index(m, lo[2], hi[2]);
                    const long long x = inx ? ox + unsigned(m * ny * w[0]) : 0u;
                    const long long y = cy >= 0 ? ymem_offset(m, cy, ic, nx, w[1]) : 0;
                    const long long z = cz >= 0 ? zmem_offset(cz, j, ic, nx, ny) : 0;
                    if (w[0] > 0) check(x, 1, mem[0], "x memory");
                    if (cy >= 0) check(y, 1, mem[1], "y memory");
                    if (cz >= 0) check(z, 1, mem[2], "z memory");
                    if (role != 0 || m < kb || m >= ke || !own) continue;
                    if (o != cell_offset(g0, nxyp, m, j * nx + i)) ++g_bad;
                    if (cells[(size_t(m) * ny + j) * nx + i]++) ++g_bad;
                    if (inx) {
                        if (x != xmem_offset(m, j, cx, ny, w[0])) ++g_bad;
                        if (x < mem[0] && ms[0][size_t(x)]++) ++g_bad;
                    }
                    if (cy >= 0 && y < mem[1] && ms[1][size_t(y)]++) ++g_bad;
                    if (cz >= 0 && z < mem[2] && ms[2][size_t(z)]++) ++g_bad;
                }
            }
          }
        }
    }
    for (unsigned char v : cells) g_bad += v != 1;
    for (const auto& m : ms)
        for (unsigned char v : m) g_bad += v != 1;
    std::printf("blocks %d accesses %lld violations %lld\n", G.nblocks, g_acc, g_bad);
    return 0;
}
