// CPU: counts what call patterns capture and launch through the run cutting of
// ela3d_amd/csrc/runs.hpp.  Arguments: energy cadence, steps a call, calls.  Prints
//   held H launches L covered C wrong W
// H graphs held at the end, L launches and C steps of the second half of the calls, W runs
// whose steps, field set or energy steps are not those of the step count they start from.
#include <cstdio>
#include <cstdlib>

#include "runs.hpp"

using ela3d::StepRun;

struct Shot {
    ela3d::StepRuns<int> runs;
    int every = 0, done = 0, next = 0, launches = 0, wrong = 0;
    std::vector<StepRun> made{StepRun{}};  // by graph number

    StepRun at(int n) const
    {
        StepRun r{done & 1, n, 0};
        for (int s = 0; s < n; ++s)
            if (every > 0 && (done + 1 + s) % every == 0) r.energy |= 1u << s;
        return r;
    }
    void run(int n)
    {
        const StepRun r = at(n);
        const int g = runs.graph(r, [&] {
            made.push_back(r);
            return int(made.size()) - 1;
        });
        if (!g) {
            if (n < 2) ++wrong;
            const int to = done + n;
            runs.parts(r, [&](int part) { run(part); });
            if (done != to) ++wrong;
            return;
        }
        if (!(made[size_t(g)] == r)) ++wrong;
        ++launches;
        done += n;
    }
    void step(int n)
    {
        while (n > 0) {
            const int r = runs.first(done, n);
            if (r < 1 || r > n || r > 31) {
                ++wrong;
                return;
            }
            run(r);
            n -= r;
        }
    }
};

int main(int argc, char** argv)
{
    if (argc < 4) return 2;
    Shot s;
    s.every = std::atoi(argv[1]);
    const int n = std::atoi(argv[2]), calls = std::atoi(argv[3]);
    s.runs.set_energy(s.every);
    int half = 0, from = 0;
    for (int c = 0; c < calls; ++c) {
        if (c == calls / 2) {
            half = s.launches;
            from = s.done;
        }
        s.step(n > 0 ? n : 1 + (c * 37 + c * c) % 61);  // 0: a length of its own for each call
    }
    std::printf("held %zu launches %d covered %d wrong %d\n", s.runs.held(), s.launches - half, s.done - from, s.wrong);
    return 0;
}
