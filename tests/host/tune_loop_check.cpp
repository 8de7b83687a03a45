// The autotuner's candidates where batches take the one-launch slice loop,
// which has no column tiles: one per batch, chain count and plans, with the
// automatic tile; batches that take the passes keep one per column tile.
#include "../../ms-stem-fem_amd/csrc/msf_host.hpp"

#include <cstdio>
#include <set>

using namespace msf;

int main()
{
    long loop_bad = 0, tiles_bad = 0, loops = 0;
    for (int64_t P : {2, 16, 120, 256, 300, 1024})
        for (int64_t B : {1, 2, 16, 120, 256, 496})
            for (int64_t from : {1, 64, 128}) {
                if (B > P) continue;
                TuneSpace t;
                t.P = P;
                t.B = B;
                t.plane = 128 * 96;
                t.plans = {0, 3};
                t.tile = [](int64_t b, int, bool beside) { return b < 200 && !beside ? 8 : 16; };
                t.loop = [&](int64_t b, int pv) { return b >= from && pv == 0; };
                t.fused = [](int, int) { return false; };
                const std::vector<TunedShape> c = tune_candidates(t);
                for (const TunedShape& s : c) {
                    std::set<int> w;
                    long n = 0;
                    for (const TunedShape& o : c)
                        if (o[0] == s[0] && o[2] == s[2] && o[3] == s[3]) {
                            w.insert(o[1]);
                            ++n;
                        }
                    if (t.loop(s[0], s[3])) {
                        ++loops;
                        loop_bad += n != 1 || *w.begin() != t.tile(s[0], s[3], s[2] == 2);
                    } else {
                        tiles_bad += n != 3 || w != std::set<int>{4, 8, 16};
                    }
                }
            }
    std::printf("loop %ld tiles %ld loops %d\n", loop_bad, tiles_bad, loops > 0);
    return 0;
}
