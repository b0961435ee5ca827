// tune.cpp -- launch-shape autotuner and its process-wide cache.
//
// Each pass is two launches (interior box, absorbing-layer boxes).  The tuner
// first times the interior candidates (threads per workgroup x z planes per
// workgroup x xy positions per lane) on the interior launches, then the
// absorbing-layer candidates on the absorbing-layer launches, then re-checks the
// interior z segment and its neighbours jointly with the z-layer segment over
// all four launches (the y absorbing-layer boxes march with the interior z
// segment), all on a scratch shot of the same grid (source amplitude 0, so the
// traffic is identical and nothing is perturbed).  The winner is cached keyed by
// (nx, ny, nz, storage, npoints_pml); shots created with block = 0 and
// zseg = 0 take the cached shape.  Then come overlapped and merged launches, and the two
// fused schedules (interior, whole grid).
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "shot.hpp"

namespace ela3d {

typedef std::tuple<int, int, int, int, int, int> TuneKey;

static std::mutex& tune_mutex()
{
    static std::mutex m;
    return m;
}

static std::map<TuneKey, std::pair<Tuning, double>>& tune_cache()
{
    static std::map<TuneKey, std::pair<Tuning, double>> c;
    return c;
}

static TuneKey key_of(const ela3d_config& c)
{
    // the free surface changes the box split (plane 0 is a box of its own)
    return TuneKey(c.nx, c.ny, c.nz, c.storage, c.npoints_pml, c.free_surface ? 1 : 0);
}

bool cached_tuning(const ela3d_config& c, Tuning& out)
{
    std::lock_guard<std::mutex> g(tune_mutex());
    auto it = tune_cache().find(key_of(c));
    if (it == tune_cache().end()) return false;
    out = it->second.first;
    return true;
}

void store_tuning(const ela3d_config& c, const Tuning& t, double ms)
{
    std::lock_guard<std::mutex> g(tune_mutex());
    tune_cache()[key_of(c)] = std::make_pair(t, ms);
}

}  // namespace ela3d

using ela3d::Error;
using ela3d::Tuning;

extern "C" {

int ela3d_autotune(const ela3d_config* cfg, const float* cp, const float* cs, const float* rho,
                   int32_t steps, ela3d_tuning* out)
{
    try {
        if (!cfg || !cp || !cs || !rho || steps < 1) throw Error{ELA3D_E_INVALID, "bad argument"};
        ela3d_config c = *cfg;
        c.factor = 0.0;  // scratch shot: same traffic, no wavefield
        c.nrec = 0;
        c.rec = nullptr;
        c.use_graph = 0;
        c.nstep = std::max(c.nstep, steps * 256 + 8192);  // energy steps come to the last candidate
        c.block = 256;
        c.zseg = 0;
        ela3d::ShotPlan plan = ela3d::make_plan(c);
        int n = 0;
        if (hipGetDeviceCount(&n) != hipSuccess || n <= c.device) throw Error{ELA3D_E_NODEVICE, "no HIP device"};
        // a second field set lets the scratch shot also try the fused schedules; its two-pass
        // candidates update the first one in place, cached as they are in the shots they are for
        const bool fusable = ela3d::fused_unsupported(plan, 1024).empty() || ela3d::fused_unsupported(plan, 512).empty();
        Tuning whole;
        whole.fused = 2;
        whole.dbuf = 1;
        whole.tile = 256;
        bool marchable = ela3d::march_unsupported(plan, whole).empty();
        std::unique_ptr<ela3d::Shot> shot;
        try {
            shot = ela3d::make_shot(plan, cp, cs, rho, nullptr, fusable || marchable);
        } catch (const Error& e) {
            if (e.code != ELA3D_E_OOM || fusable) throw;
            marchable = false;  // one set fits
            shot = ela3d::make_shot(plan, cp, cs, rho, nullptr, false);
        }
        static const int blocks[] = {64, 128, 256};
        static const int zsi[] = {1, 2, 4, 8, 16, 32};  // 1: more workgroups for small grids
        static const int zss[] = {1, 2, 4, 8};
        static const int vecs[] = {1, 2, 4};
        static const int vecs_slab[] = {1, 2};
        const bool verbose = std::getenv("ELA3D_TUNE_VERBOSE") != nullptr;
        Tuning best = ela3d::choose_tuning(plan);
        int tried = 0;
        std::vector<ela3d_kernel_stats> st;
        // launch times of the stress and velocity passes: [0] interior, [1] absorbing layers
        shot->set_overlap(false);  // per-launch times of launches run one after another
        auto measure = [&](const Tuning& t, double ms[2]) {
            shot->retune(t);
            double wall = 0.0;
            shot->profile(1, st, wall);  // warm
            shot->profile(steps, st, wall);
            ms[0] = (st[1].total_ms + st[3].total_ms) / steps;
            ms[1] = (st[0].total_ms + st[2].total_ms) / steps;
            ++tried;
        };
        double ms[2];
        // each stage times every candidate once over `steps` steps, then re-times
        // its best few over four times as many and keeps the fastest of those
        auto refine = [&](std::vector<std::pair<double, Tuning>>& c, int which) {
            std::sort(c.begin(), c.end(),
                      [](const std::pair<double, Tuning>& a, const std::pair<double, Tuning>& b) {
                          return a.first < b.first;
                      });
            const int keep = std::min<int>(5, int(c.size()));
            Tuning win = c[0].second;
            double win_ms = 1e300;
            for (int q = 0; q < keep; ++q) {
                shot->retune(c[q].second);
                double wall = 0.0;
                shot->profile(1, st, wall);
                shot->profile(4 * steps, st, wall);
                ++tried;
                const double t = which == 0 ? (st[1].total_ms + st[3].total_ms) / (4 * steps)
                                            : (st[0].total_ms + st[2].total_ms) / (4 * steps);
                if (t < win_ms) {
                    win_ms = t;
                    win = c[q].second;
                }
            }
            return win;
        };
        std::vector<std::pair<double, Tuning>> cands;
        for (int vv : vecs)
            for (int b : blocks)
                for (int zi : zsi) {
                    Tuning t = best;
                    t.block = b;
                    t.zseg_interior = zi;
                    t.vec = vv;
                    measure(t, ms);
                    if (verbose)
                        std::fprintf(stderr, "[tune] interior vec %d block %3d zseg %3d: %.4f ms\n", vv, b, zi,
                                     ms[0]);
                    cands.emplace_back(ms[0], t);
                }
        best = refine(cands, 0);
        cands.clear();
        for (int vv : vecs_slab)
            for (int b : blocks)
                for (int zs : zss) {
                    Tuning t = best;
                    t.block_slab = b;
                    t.zseg_slab = zs;
                    t.vec_slab = vv;
                    measure(t, ms);
                    if (verbose)
                        std::fprintf(stderr, "[tune] layers   vec %d block %3d zseg %3d: %.4f ms\n", vv, b, zs,
                                     ms[1]);
                    cands.emplace_back(ms[1], t);
                }
        best = refine(cands, 1);
        // The interior z segment also sets how the y absorbing-layer boxes march (they
        // run in the absorbing-layer launch), so re-check it and its neighbours in zsi
        // jointly with the z-layer segment, scored by all four stencil launches.
        {
            auto stencil_ms = [&](const Tuning& t) {
                shot->retune(t);
                double wall = 0.0;
                shot->profile(1, st, wall);
                shot->profile(4 * steps, st, wall);
                ++tried;
                return (st[0].total_ms + st[1].total_ms + st[2].total_ms + st[3].total_ms) / (4 * steps);
            };
            const int nz = int(sizeof(zsi) / sizeof(zsi[0]));
            int at = 0;
            while (at < nz && zsi[at] != best.zseg_interior) ++at;
            const Tuning centre = best;
            double best_ms = stencil_ms(centre);
            for (int d : {-1, 0, 1}) {
                if (at + d < 0 || at + d >= nz) continue;
                for (int zs : zss) {
                    Tuning t = centre;
                    t.zseg_interior = zsi[at + d];
                    t.zseg_slab = zs;
                    if (t.zseg_interior == centre.zseg_interior && zs == centre.zseg_slab) continue;
                    const double w = stencil_ms(t);
                    if (verbose)
                        std::fprintf(stderr, "[tune] interior zseg %2d, z-layer zseg %d: %.4f ms (chosen so far %.4f ms)\n",
                                     t.zseg_interior, zs, w, best_ms);
                    if (w < 0.995 * best_ms) {
                        best_ms = w;
                        best = t;
                    }
                }
            }
        }
        // schedule: the two launches in sequence, overlapped (pays off when neither
        // fills the GPU), or one mixed launch per pass (one kernel boundary less).
        // Timed as steps one after the other between two events: events around every launch
        // cost more than a small grid's kernels, the same for every schedule, and hid what
        // its launches and their gaps take.  Long enough to last milliseconds, and
        // whole energy cycles where those are short.
        struct Events {
            hipEvent_t at[2] = {nullptr, nullptr};
            ~Events()
            {
                for (auto& e : at)
                    if (e) (void)hipEventDestroy(e);
            }
        } ev;
        for (auto& e : ev.at) HIP_CHECK(hipEventCreate(&e));
        int n_wall = steps;
        auto wall_of = [&](const Tuning& t) {
            shot->retune(t);
            shot->enqueue_steps(std::max(1, n_wall / 8));
            (void)shot->sync();
            HIP_CHECK(hipEventRecord(ev.at[0], shot->stream()));
            shot->enqueue_steps(n_wall);
            HIP_CHECK(hipEventRecord(ev.at[1], shot->stream()));
            HIP_CHECK(hipEventSynchronize(ev.at[1]));
            float wall = 0.f;
            HIP_CHECK(hipEventElapsedTime(&wall, ev.at[0], ev.at[1]));
            ++tried;
            return double(wall) / n_wall;
        };
        if (wall_of(best) < 0.3) n_wall = std::max(steps, 48);
        if (c.energy_every > 0 && c.energy_every <= 16)
            n_wall = (n_wall + c.energy_every - 1) / c.energy_every * c.energy_every;
        double wall3[3] = {0.0, 0.0, 1e300};
        Tuning cand[3] = {best, best, best};
        cand[1].overlap = 1;
        wall3[0] = wall_of(cand[0]);
        wall3[1] = wall_of(cand[1]);
        static const int mblocks[] = {128, 256};
        static const int mzi[] = {4, 8, 16};
        static const int mzs[] = {2, 4};
        static const int mvec[] = {1, 2};
        for (int vv : mvec)
            for (int b : mblocks)
                for (int zi : mzi)
                    for (int zs : mzs) {
                        Tuning t = best;
                        t.merged = 1;
                        t.block = b;
                        t.zseg_interior = zi;
                        t.zseg_slab = zs;
                        t.vec = vv;
                        const double w = wall_of(t);
                        if (verbose)
                            std::fprintf(stderr, "[tune] merged vec %d block %3d zseg %2d/%d: %.4f ms\n", vv, b, zi,
                                         zs, w);
                        if (w < wall3[2]) {
                            wall3[2] = w;
                            cand[2] = t;
                        }
                    }
        int pick = 0;
        if (wall3[2] < 0.99 * wall3[pick]) pick = 2;
        if (wall3[1] < 0.97 * wall3[pick]) pick = 1;
        best = cand[pick];
        double best_wall = wall3[pick];
        if (fusable || marchable) {  // fused interior step: tile x z segment; whole-grid fused step:
                                     // workgroup x z segment; the fastest of them replaces the
                                     // two-pass pick if it is at least 1 % faster
            static const int tiles[] = {512, 768, 1024};
            static const int fzs[] = {4, 8, 12, 16, 24, 32};
            std::vector<std::pair<double, Tuning>> fc;
            for (int tl : tiles) {
                if (!ela3d::fused_unsupported(plan, tl).empty()) continue;
                for (int z : fzs) {
                    Tuning t = best;
                    t.overlap = 0;
                    t.merged = 0;
                    t.fused = 1;
                    t.dbuf = 1;
                    t.tile = tl;
                    t.zseg_interior = z;
                    const double w = wall_of(t);
                    if (verbose) std::fprintf(stderr, "[tune] fused tile %4d zseg %2d: %.4f ms\n", tl, z, w);
                    fc.emplace_back(w, t);
                }
            }
            static const int mtiles[] = {256, 512, 1024};
            static const int mzs2[] = {1, 2, 3, 4, 6, 8};
            for (int tl : mtiles)
                for (int z : mzs2) {
                    Tuning t = best;
                    t.overlap = 0;
                    t.merged = 0;
                    t.fused = 2;
                    t.dbuf = 1;
                    t.tile = tl;
                    t.zseg_interior = z;
                    t.strips = 4;
                    if (!marchable || !ela3d::march_unsupported(plan, t).empty()) continue;
                    const double w = wall_of(t);
                    if (verbose) std::fprintf(stderr, "[tune] whole-grid workgroup %4d zseg %2d: %.4f ms\n", tl, z, w);
                    fc.emplace_back(w, t);
                }
            // the three fastest again, three rounds in turn with the two-pass pick,
            // each kept at its best round: their differences (under 1 %) are below
            // one short timing's noise
            std::sort(fc.begin(), fc.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
            if (fc.size() > 3) fc.resize(3);
            const Tuning split = best;
            for (int r = 0; r < 3 && !fc.empty(); ++r) {
                best_wall = std::min(best_wall, wall_of(split));
                for (auto& c : fc) c.first = std::min(c.first, wall_of(c.second));
            }
            Tuning fbest = best;
            double fwall = 1e300;
            for (const auto& c : fc) {
                if (verbose)
                    std::fprintf(stderr, "[tune] fused finalist (%s) tile %4d zseg %2d: %.4f ms\n",
                                 c.second.fused == 2 ? "whole grid" : "interior", c.second.tile,
                                 c.second.zseg_interior, c.first);
                if (c.first < fwall) {
                    fwall = c.first;
                    fbest = c.second;
                }
            }
            if (fwall < 0.99 * best_wall) {
                best_wall = fwall;
                best = fbest;
            }
        }
        if (verbose)
            std::fprintf(stderr, "[tune] step wall: split %.4f ms, overlapped %.4f ms, merged %.4f ms\n",
                         wall3[0], wall3[1], wall3[2]);
        shot->retune(best);
        const double best_ms = wall_of(best);
        ela3d::store_tuning(*cfg, best, best_ms);
        if (out) {
            out->block = best.block;
            out->zseg_interior = best.zseg_interior;
            out->zseg_slab = best.zseg_slab;
            out->vec = best.vec;
            out->block_slab = best.block_slab;
            out->vec_slab = best.vec_slab;
            out->overlap = best.overlap;
            out->merged = best.merged;
            out->dbuf = best.dbuf;
            out->fused = best.fused;
            out->tile = best.tile;
            out->strips = best.strips;
            out->ms_per_step = best_ms;
            out->candidates = tried;
        }
        return ELA3D_OK;
    } catch (const Error& e) {
        ela3d::set_last_error(e.msg);
        return e.code;
    } catch (const std::exception& e) {
        ela3d::set_last_error(e.what());
        return ELA3D_E_INVALID;
    }
}

int ela3d_tuning_set(const ela3d_config* cfg, const ela3d_tuning* t)
{
    if (!cfg || !t || t->block <= 0 || t->zseg_interior <= 0 || t->zseg_slab <= 0) return ELA3D_E_INVALID;
    auto ok_block = [](int b) { return b == 64 || b == 128 || b == 256; };
    const int bs = t->block_slab ? t->block_slab : t->block;
    const int vs = t->vec_slab ? t->vec_slab : 1;
    if (!ok_block(t->block) || !ok_block(bs)) return ELA3D_E_INVALID;
    if (t->vec != 1 && t->vec != 2 && t->vec != 4) return ELA3D_E_INVALID;
    if (vs != 1 && vs != 2) return ELA3D_E_INVALID;
    Tuning u;
    u.block = t->block;
    u.zseg_interior = t->zseg_interior;
    u.vec = t->vec;
    u.block_slab = bs;
    u.zseg_slab = t->zseg_slab;
    u.vec_slab = vs;
    u.overlap = t->overlap ? 1 : 0;
    u.merged = t->merged ? 1 : 0;
    u.dbuf = t->dbuf ? 1 : 0;
    u.fused = t->fused == 2 ? 2 : t->fused ? 1 : 0;
    u.tile = t->tile > 0 ? t->tile : 1024;
    if (t->strips < 0 || t->strips > 64) return ELA3D_E_INVALID;
    u.strips = t->strips;
    if (u.fused) u.dbuf = 1;
    ela3d::store_tuning(*cfg, u, t->ms_per_step);
    return ELA3D_OK;
}

int ela3d_tuning_get(const ela3d_config* cfg, ela3d_tuning* t)
{
    if (!cfg || !t) return ELA3D_E_INVALID;
    Tuning u;
    if (!ela3d::cached_tuning(*cfg, u)) return ELA3D_E_NOTFOUND;
    t->block = u.block;
    t->zseg_interior = u.zseg_interior;
    t->zseg_slab = u.zseg_slab;
    t->vec = u.vec;
    t->block_slab = u.block_slab;
    t->vec_slab = u.vec_slab;
    t->overlap = u.overlap;
    t->merged = u.merged;
    t->dbuf = u.dbuf;
    t->fused = u.fused;
    t->tile = u.tile;
    t->strips = u.strips;
    t->ms_per_step = 0.0;
    t->candidates = 0;
    return ELA3D_OK;
}

}  // extern "C"
