// runs.hpp -- how an advance is cut into runs of steps that replay one captured graph each,
// and which runs a shot keeps graphs of.  Host code without HIP calls, so that a CPU program
// can count what a call pattern captures and launches.
#pragma once

#include <algorithm>
#include <cstddef>
#include <vector>

namespace ela3d {

// Consecutive steps from field set `par`; bit s of `energy`: step s sums the energy.
struct StepRun {
    int par, steps;
    unsigned energy;
    bool operator==(const StepRun& r) const { return par == r.par && steps == r.steps && energy == r.energy; }
};

// Between two graphs the GPU idles for 4 to 8 us (64^3, kernels 19 us a step: 24 us with one
// step per graph, 20 with 16), a graph's own nodes follow each other at once: runs of about 16
// steps, where the gap has become small.  Capturing costs about 5 us a step, what a run's gaps
// cost once: a run is captured when it comes up for the second time, and made of single steps
// or shorter runs before.
//
// Nothing is given back while a shot steps (its graphs may be running, and waiting for them
// would hold up the caller), so the runs a call pattern needs have to be few:
//  * long advances are cut where energy cycles start, into blocks that are the same from cycle
//    to cycle: whole cycles of up to 16 steps together, longer ones in equal parts of 16 to 31;
//  * what is left before the first and after the last block, and advances shorter than one,
//    are runs of their own, up to kOwn of them (cadence 13, 50 steps a call: 13 phases times 2
//    field sets of each);
//  * past that they are put together from runs of 1, 2, 4, 8 and 16 steps that hold no energy
//    step or end on one, of which there are 20.
// 64^3, 50 steps a call, us a step and of the caller's time: cadence 7 15.1 and 1.0, 17 14.8 and
// 1.0, none 14.6 and 1.0.  With the 16 runs used last kept, and waits where one gives way to
// another, cadence 7 took 20.9 and 20.9, 17 19.3 and 19.1, none the same.
template <typename Exec>
class StepRuns {
public:
    static constexpr size_t kOwn = 32;   // graphs of runs that belong to one call pattern
    static constexpr size_t kSeen = 32;  // runs remembered that came up once

    void set_energy(int every)
    {
        every_ = std::max(0, every);
        if (every_ == 0)
            block_ = last_ = 16;
        else if (every_ <= 16)
            block_ = last_ = 16 / every_ * every_;
        else {  // 16 to 31 steps
            const int parts = every_ / 16;
            block_ = (every_ + parts - 1) / parts;
            last_ = every_ - (every_ - 1) / block_ * block_;
        }
    }

    // steps of the first run of an advance of n steps after `done` steps
    int first(int done, int n) const
    {
        if (n <= std::max(16, block_)) return n;
        if (every_ == 0) return 16;
        const int at = done % every_;
        if (every_ <= 16) return block_ - at;
        const int from = at / block_ * block_;
        return std::min(from + block_, every_) - at;
    }

    // The run's graph, from capture() where it is to have one and has none yet; none (null):
    // the run is made of parts.
    template <typename Capture>
    Exec graph(const StepRun& r, Capture capture)
    {
        for (const Held& h : held_)
            if (h.run == r) return h.exec;
        const bool shared = common(r);
        if (!shared && own_ >= kOwn) return Exec();
        if (r.steps > 1 && !seen(r)) return Exec();
        held_.reserve(held_.size() + 1);
        held_.push_back(Held{r, capture()});
        if (!shared) ++own_;
        return held_.back().exec;
    }

    // part(steps) for every part of a run without a graph, in order
    template <typename Part>
    void parts(StepRun r, Part part) const
    {
        const bool ones = simple(r) && (r.steps & (r.steps - 1)) == 0;
        while (r.steps > 0) {
            int n = 1;
            if (!ones) {
                n = r.steps & -r.steps;
                if (!simple(r)) {  // up to the first energy step
                    int e = 0;
                    while (!(r.energy >> e & 1u)) ++e;
                    n = (e + 1) & -(e + 1);
                }
            }
            part(n);
            r.steps -= n;
            r.energy >>= n;
        }
    }

    template <typename Destroy>
    void clear(Destroy destroy)
    {
        for (Held& h : held_) destroy(h.exec);
        held_.clear();
        seen_.clear();
        own_ = 0;
    }
    size_t held() const { return held_.size(); }

private:
    struct Held {
        StepRun run;
        Exec exec;
    };
    // no energy step, or only the last one
    static bool simple(const StepRun& r) { return (r.energy & ~(1u << (r.steps - 1))) == 0; }
    // a block, or a run that others are put together from
    bool common(const StepRun& r) const
    {
        if (simple(r) && (r.steps <= 16 && (r.steps & (r.steps - 1)) == 0)) return true;
        if (every_ > 16) return simple(r) && (r.steps == block_ || r.steps == last_);
        return r.steps == block_ && (r.energy == 0 || r.energy >> (r.steps - 1) & 1u);
    }
    bool seen(const StepRun& r)
    {
        if (std::find(seen_.begin(), seen_.end(), r) != seen_.end()) return true;
        if (seen_.size() == kSeen) seen_.erase(seen_.begin());
        seen_.push_back(r);
        return false;
    }

    int every_ = 0, block_ = 16, last_ = 16;
    size_t own_ = 0;
    std::vector<Held> held_;
    std::vector<StepRun> seen_;
};

}  // namespace ela3d
