// Batches of a run by the rule (msf_host.cpp batch_rule), over every position
// count up to 1024 on square grids and some rectangles: the batches cover the
// positions in order and stay within 96 MiB of waves; where two chains of
// batches ask for one batch more than the fewest, their number is even and
// they differ by a row workgroup's positions and a partial workgroup at most;
// elsewhere the chains change nothing.  Prints the violations of each.
#include "../../ms-stem-fem_amd/csrc/msf_host.hpp"

#include <algorithm>
#include <cstdio>

using namespace msf;

int main()
{
    // unit: positions of a row-pass workgroup of the automatic radix plan
    const struct { int nx, ny, unit; } grids[] = {{256, 256, 16}, {384, 384, 8}, {512, 512, 8},
                                                  {768, 768, 4}, {1024, 1024, 2}, {1024, 512, 8},
                                                  {384, 1024, 2}};
    long cover = 0, room = 0, odd = 0, uneven = 0, changed = 0, fired = 0;
    for (const auto& g : grids) {
        const Domain d = make_domain(g.nx, g.ny, g.nx * 0.08, g.ny * 0.08, 0.0, 0.0, 200e3);
        const RowRanges keep = slice_keep_ranges(d);
        const int64_t plane = (int64_t)g.nx * ((keep.amax + keep.bmax + 15) / 16 * 16);
        const int64_t pixels = (int64_t)g.nx * g.ny;
        for (int64_t P = 1; P <= 1024; ++P) {
            const BatchSplit one = batch_rule(P, plane, pixels, false, g.unit);
            const BatchSplit s = batch_rule(P, plane, pixels, true, g.unit);
            for (const BatchSplit* b : {&one, &s}) {
                bool ok = b->n >= 1 && b->begin(0) == 0 && b->begin(b->n) == P;
                for (int64_t k = 0; k < b->n; ++k) {
                    const int64_t nb = b->begin(k + 1) - b->begin(k);
                    ok = ok && nb >= 1 && nb <= b->depth;
                }
                cover += !ok;
                room += b->depth > 1 && b->depth * plane * 8 > 96ll << 20;
            }
            // fewest batches within the room, as one chain takes them
            int64_t bmax = std::max<int64_t>(1, (96ll << 20) / (plane * 8));
            if (bmax >= 32) bmax -= bmax % 16;
            const int64_t few = (P + bmax - 1) / bmax, more = (P + few) / (few + 1);
            if (pixels >= 384 * 384 && few >= 3 && few % 2 && more * plane >= kTwoChainPixels) {
                ++fired;
                int64_t lo = P, hi = 0;
                for (int64_t k = 0; k < s.n; ++k) {
                    const int64_t nb = s.begin(k + 1) - s.begin(k);
                    lo = std::min(lo, nb);
                    hi = std::max(hi, nb);
                }
                odd += s.n % 2;
                uneven += hi - lo > 2 * g.unit - 1 || 2 * lo < hi;
            } else {
                changed += s.depth != one.depth || s.n != one.n || s.unit != one.unit;
            }
        }
    }
    std::printf("cover %ld room %ld odd %ld uneven %ld changed %ld fired %d\n", cover, room, odd,
                uneven, changed, fired > 0);
    return 0;
}
