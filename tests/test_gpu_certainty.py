"""What the FP32 traceback rests on where it decides a column without its row: an
entry of the next column, taken back through normaliser and emission, is the row's
total of entry times weight within n + 13 roundings of 2^-24 (n time bins: n + 6 in
the recursion's sums, or 13 in its product, 3 to the column, 3 through the
normaliser, 1 in the row), at the finest grid and the largest blocks; and the thread
is the sequential sample of the table as it is stored, whole and in tiles."""
import numpy as np
import pytest

from workloads import instance

pytestmark = pytest.mark.gpu

# (haplotypes, columns, time points, bases per column, population size)
CASES = [(5, 400, 32, 10, 1e4), (24, 900, 32, 50, 1e4), (60, 500, 32, 50, 1e4),
         (16, 600, 12, 100, 1e4), (110, 500, 20, 50, 3e4), (128, 400, 20, 50, 3e4)]


@pytest.mark.parametrize("k,L,T,c,N", CASES)
def test_totals_of_rows_and_sequential_sample(aw, k, L, T, c, N):
    print("certainty k=%d L=%d T=%d" % (k, L, T), flush=True)
    tr, seqs, inst, model = instance(aw, k, L, 60 + k, ntimes=T, c=c, popsizes=np.full(T, N))
    nst, offs = inst.nstates(), inst.block_offsets()
    if k == 128:
        assert nst.max() > 1024
    u = np.random.RandomState(L + 2).uniform(size=L)
    b = aw.Batch()
    b.add(tr, seqs, *model, k - 1, u)
    b.upload()
    b.run(1, 0)
    a, norms = b.alpha(0), b.norms(0)
    bound = (max(T - 1 + 6, 13) + 7) * 2.0 ** -24
    lens, col = np.asarray(inst.blocklens), 0
    checked = 0
    for t, n in enumerate(lens):
        if n > 1 and checked < 2000000:
            rows = a[offs[t]:offs[t + 1]].reshape(n, nst[t])
            tot = rows[:-1] @ inst.trans_dense(t) * inst.emissions(t)[1:]
            v1 = rows[1:] * norms[col + 1:col + n, None]
            big = v1 >= 1e-30
            assert big.any()
            assert np.abs(v1[big] / tot[big] - 1).max() <= bound
            checked += big.sum()
        col += n
    assert checked > 1000
    assert np.array_equal(b.path(0), inst.traceback(a, u))
    for tile, warm, tol in ((60, 1, 10.0), (150, 4, 1e-2)):
        for tb in (0, 100):
            b.run(1, tb, fw_tile=tile, fw_warm=warm, fw_tol=tol)
            assert np.array_equal(b.path(0), inst.traceback(b.alpha(0), u)), (tile, warm, tol, tb)
    aw.delete_local_trees(tr)
