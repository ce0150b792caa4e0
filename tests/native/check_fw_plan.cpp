// The forward's tile plan over rounds of re-runs with random outcomes: in one
// launch no tile reads a boundary slot that another writes, slots never overlap,
// and every tile's start is checked against, and re-run from, the column that
// the tile before it last ran to.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>

#include "fw_plan.h"

using namespace aw;

#define REQUIRE(x)                                              \
    do {                                                        \
        if (!(x)) {                                             \
            printf("%s:%d: %s\n", __FILE__, __LINE__, #x);      \
            exit(1);                                            \
        }                                                       \
    } while (0)

int main()
{
    std::mt19937 rng(7);
    const int Rs[] = {1, 2, 4, 6, 8, 12, 16, 32};
    for (int trial = 0; trial < 400; trial++) {
        FwPlan plan;
        std::vector<int> R;
        const int n = 1 + rng() % 4;
        for (int i = 0; i < n; i++) {
            const int L = 1 + rng() % 500, W = 1 + rng() % 20;
            const int C = rng() % 4 ? W + 1 + rng() % 60 : 0;
            const size_t k0 = plan.tiles.size();
            plan.add(i, L, Rs[rng() % 8], C, W);
            R.push_back(0);
            int end = 0;   // the tiles cover the columns, each after its warm-up
            for (size_t k = k0; k < plan.tiles.size(); k++) {
                const FwTile &t = plan.tiles[k];
                REQUIRE(t.inst == i && t.cs == end && t.c1 > t.cs && t.c0 == (t.cs ? t.cs - W : 0));
                REQUIRE(t.mode == (t.cs ? 1 : 0) && (t.bin >= 0) == (t.cs > 0) && (t.bout >= 0) == (t.c1 < L));
                if (t.bin >= 0) REQUIRE(t.bin == plan.tiles[k - 1].bout);
                end = t.c1;
            }
            REQUIRE(end == L);
        }
        std::vector<int> last(plan.tiles.size(), 0);   // what tile k last ran to its end as
        std::map<int, int> slot;                       // what a slot holds
        int stamp = 0;
        const auto launch = [&](const std::vector<FwTile> &ts) {
            for (const FwTile &a : ts)
                for (const FwTile &b : ts) {
                    if (a.bin >= 0 && b.mode == 2) REQUIRE(a.bin != b.bout);
                    if (&a != &b && a.bout >= 0) REQUIRE(a.bout != b.bout);
                }
        };
        for (size_t k = 0; k < plan.tiles.size(); k++)
            if (plan.tiles[k].bout >= 0) slot[plan.tiles[k].bout] = last[k] = ++stamp;
        std::vector<int> chk = plan.started();
        for (int round = 0; round < 30 && !chk.empty(); round++) {
            std::vector<int> redo;
            for (int k : chk) {
                REQUIRE(slot.at(plan.tiles[k].bin) == last[k - 1]);
                if (rng() % 3) redo.push_back(k);
            }
            const std::vector<FwTile> sub = plan.rerun(redo);
            REQUIRE(sub.size() == redo.size());
            launch(sub);
            std::vector<int> early;
            for (size_t x = 0; x < sub.size(); x++) {
                const FwTile &t = sub[x], &p = plan.tiles[redo[x]];
                REQUIRE(t.mode == 2 && t.c0 == t.cs && t.cs == p.cs && t.c1 == p.c1 && t.bin == p.bin);
                REQUIRE(slot.at(t.bin) == last[redo[x] - 1]);
                early.push_back(rng() % 3 ? 0 : t.cs + 1);
            }
            for (size_t x = 0; x < sub.size(); x++)
                if (!early[x] && sub[x].bout >= 0) slot[sub[x].bout] = last[redo[x]] = ++stamp;
            chk = plan.finished(redo, sub, early);
            size_t want = 0;
            for (size_t x = 0; x < sub.size(); x++) want += !early[x] && sub[x].bout >= 0;
            REQUIRE(chk.size() == want);
        }
        for (const FwTile &t : plan.tiles)
            if (t.bin >= 0) REQUIRE(slot.at(t.bin) == last[&t - plan.tiles.data() - 1]);
        // slots lie in the planned units, a row apart
        FwPlan one;
        one.add(0, 400, 16, 50, 10);
        std::vector<FwTile> re = one.rerun({1, 2});
        REQUIRE(re[0].bout - one.tiles[1].bout == 16 && re[1].bout + 16 <= one.units);
        REQUIRE(one.tiles[2].bout - one.tiles[1].bout == 32);
    }
    printf("ok\n");
}
