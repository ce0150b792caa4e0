// fw_plan.h -- the forward's tiles, and the boundary columns they pass on.
#pragma once

#include <algorithm>
#include <vector>

namespace aw {

// A forward tile: columns [c0, c1) of an instance computed by one workgroup.
// mode 0 starts from the prior at column 0.  mode 1 starts at c0 from a
// uniform vector and stores nothing before cs (a warm-up: the filter
// forgets its start).  mode 2 starts at c0 from the column held in boundary
// slot bin (written by the tile before).  A tile with bout >= 0 also
// computes column c1 into boundary slot bout, for the check of the next
// tile's start.
struct FwTile {
    int inst;
    int c0, cs, c1;
    int mode;
    int bout, bin;
};

// Boundary slots are counted in units of 64 entries, a slot taking the R units
// of its instance's row; its normaliser is stored at the slot's first unit.
constexpr int BND_UNIT = 64;

// The tiles of a forward and the rounds of their re-runs.  Tiles that fail
// their check in one round are re-run in one launch, neighbours among them, and
// a workgroup may start when the one before it is already done.  So a boundary
// column has two slots: a launch reads the one that the launches before it
// left and writes the other, and which of them holds depends on no timing.
class FwPlan {
public:
    std::vector<FwTile> tiles;   // bin, bout: the slots that hold the column now
    int units = 0;               // of all slots

    // the columns of instance i (R states per lane) in tiles of C columns, of
    // which all but the first spend W on their warm-up; one tile where C is 0
    // or the instance no longer
    void add(int i, int L, int R, int C, int W)
    {
        if (!C || L <= C || C <= W) {
            put(FwTile{i, 0, 0, L, 0, -1, -1}, 0);
            return;
        }
        for (int s = 0, e = C, bin = -1;; s = e, e += C - W) {
            const bool last = e >= L;
            const int bout = last ? -1 : units;
            put(FwTile{i, s ? s - W : 0, s, std::min(e, L), s ? 1 : 0, bout, bin}, R);
            if (last) return;
            units += 2 * R;
            bin = bout;
        }
    }
    // the tiles whose start is checked after the first launch
    std::vector<int> started() const
    {
        std::vector<int> chk;
        for (int k = 0; k < (int)tiles.size(); k++)
            if (tiles[k].bin >= 0) chk.push_back(k);
        return chk;
    }
    // the re-runs of the tiles `redo`, one launch
    std::vector<FwTile> rerun(const std::vector<int> &redo) const
    {
        std::vector<FwTile> sub;
        for (int k : redo) {
            FwTile t = tiles[k];
            t.mode = 2;
            t.c0 = t.cs;
            if (t.bout >= 0) t.bout += t.bout == first_[k] ? size_[k] : -size_[k];
            sub.push_back(t);
        }
        return sub;
    }
    // After that launch: a tile that rejoined its stored columns (early) kept
    // its boundary column; the tile after one that ran to its end takes the new
    // one, and is in the list returned, to be checked again.
    std::vector<int> finished(const std::vector<int> &redo, const std::vector<FwTile> &sub,
                              const std::vector<int> &early)
    {
        std::vector<int> chk;
        for (size_t x = 0; x < redo.size(); x++) {
            if (early[x] || sub[x].bout < 0) continue;
            tiles[redo[x]].bout = tiles[redo[x] + 1].bin = sub[x].bout;
            chk.push_back(redo[x] + 1);
        }
        return chk;
    }

private:
    std::vector<int> first_, size_;   // of each tile's bout: its first slot, units per slot
    void put(const FwTile &t, int R)
    {
        tiles.push_back(t);
        first_.push_back(t.bout);
        size_.push_back(R);
    }
};

}  // namespace aw
