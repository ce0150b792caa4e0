"""The traceback's parallel walk at the sizes where it can go wrong: columns
around the length of a unit, one block and many blocks per window, every
states-per-lane count up to 16, the finest time grid, and recombination rates
at which most columns change state or end a block.  FP64 threads against the
oracle's, and tiles of both precisions against one tile per instance."""
import numpy as np
import pytest

from workloads import instance

pytestmark = pytest.mark.gpu

# (haplotypes, columns, time points, bases per column): bases per column scale
# the recombination and mutation rates of a column
CASES = [(3, 1, 20, 10), (3, 2, 20, 10), (3, 47, 20, 1), (3, 49, 20, 1), (4, 97, 20, 1),
         (5, 65, 12, 10), (6, 300, 32, 10), (8, 600, 20, 2000), (12, 900, 20, 500),
         (24, 700, 20, 200), (30, 400, 28, 100), (48, 500, 20, 100), (70, 300, 20, 100),
         (100, 260, 20, 50)]


@pytest.mark.parametrize("k,L,T,c", CASES)
def test_walk_matches_oracle_and_untiled(aw, k, L, T, c):
    print("traceback walk k=%d L=%d T=%d c=%d" % (k, L, T, c), flush=True)
    tr, seqs, inst, model = instance(aw, k, L, 70 + k, ntimes=T, c=c)
    u = np.random.RandomState(L).uniform(size=L)
    fw, _ = inst.forward()
    ref = inst.traceback(fw, u)
    b = aw.Batch()
    b.add(tr, seqs, *model, k - 1, u)
    b.upload()
    b.run(0, 0)
    assert np.array_equal(b.path(0), ref)
    for prec in (0, 1):
        b.run(prec, 0)
        whole = b.path(0)
        for tile, warm in ((64, 0), (64, 30), (150, 256)):
            b.set_traceback(warm, 1)
            b.run(prec, tile)
            assert np.array_equal(b.path(0), whole), (prec, tile, warm)
    aw.delete_local_trees(tr)


@pytest.mark.parametrize("k,L,T,c", [(4, 400, 20, 10), (8, 900, 20, 200), (24, 1200, 20, 50),
                                     (60, 900, 28, 100), (100, 600, 20, 50)])
def test_walk_over_tile_starts(aw, k, L, T, c):
    """FP32 tables in forward tiles with short warm-ups and loose checks, so that
    the columns at the tiles' starts (and where a re-run rejoins) do not follow
    from the column stored before them: the thread is the sequential sample of
    the table as it is stored."""
    print("traceback of tiles k=%d L=%d T=%d c=%d" % (k, L, T, c), flush=True)
    tr, seqs, inst, model = instance(aw, k, L, 40 + k, ntimes=T, c=c)
    u = np.random.RandomState(L + 1).uniform(size=L)
    b = aw.Batch()
    b.add(tr, seqs, *model, k - 1, u)
    b.upload()
    for tile, warm, tol in ((40, 1, 10.0), (100, 2, 0.5), (300, 4, 1e-2)):
        for tb in (0, 128):
            b.run(1, tb, fw_tile=tile, fw_warm=warm, fw_tol=tol)
            assert np.array_equal(b.path(0), inst.traceback(b.alpha(0), u)), (tile, warm, tol, tb)
    aw.delete_local_trees(tr)
