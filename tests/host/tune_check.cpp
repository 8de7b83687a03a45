// The autotuner's candidates (msf_host.cpp tune_candidates) over many runs:
// the shape a run of the rules takes is among them once, with the automatic
// tile of its batch and chains; one candidate per batch, chain count and column
// tile; several chains only with several batches.  Prints the violations of each.
#include "../../ms-stem-fem_amd/csrc/msf_host.hpp"

#include <algorithm>
#include <cstdio>
#include <set>

using namespace msf;

int main()
{
    long rule_bad = 0, twice = 0, tiles_bad = 0, one_batch = 0, fused_bad = 0;
    for (int64_t P : {2, 3, 16, 100, 120, 256, 300, 1024, 5000})
        for (int64_t B : {1, 2, 16, 40, 64, 120, 256, 496})
            for (int np : {1, 2, 3}) {
                    if (B > P) continue;
                    TuneSpace t;
                    t.P = P;
                    t.B = B;
                    t.plane = 45056; // 256 x 176
                    for (int k = 0; k < np; ++k) t.plans.push_back(3 - k);
                    t.tile = [](int64_t b, int, bool beside) {
                        return b < 24 ? 1 : b < 200 && !beside ? 8 : 16;
                    };
                    t.fused = [](int w, int) { return w == 16; };
                    const std::vector<TunedShape> c = tune_candidates(t);
                    const TunedShape r = tune_rule(t);
                    const bool two = B * t.plane >= kTwoChainPixels && B < P;
                    rule_bad += r != TunedShape{(int)B, t.tile(B, 3, two), two ? 2 : 1, 3};
                    rule_bad += std::count(c.begin(), c.end(), r) != 1;
                    twice += std::set<TunedShape>(c.begin(), c.end()).size() != c.size();
                    for (const TunedShape& s : c) {
                        std::set<int> w;
                        for (const TunedShape& o : c)
                            if (o[0] == s[0] && o[2] == s[2] && o[3] == s[3]) w.insert(o[1]);
                        if (s[2] == 3) {
                            fused_bad += s[1] != 16;
                        } else {
                            w.erase(1);
                            tiles_bad += w != std::set<int>{4, 8, 16};
                        }
                        one_batch += s[2] > 1 && s[0] >= P;
                    }
                }
    std::printf("rule %ld twice %ld tiles %ld one batch %ld fused %ld\n", rule_bad, twice,
                tiles_bad, one_batch, fused_bad);
    return 0;
}
