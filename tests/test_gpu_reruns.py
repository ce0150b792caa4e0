"""Forward tiles whose re-runs follow one another: short tiles, a warm-up of
one column and a tight tolerance, so that neighbouring tiles fail together and run to
their ends in the same launch, in rounds until the last tile's start is right.
The result depends on no timing (tables, normalisers and likelihoods of two runs
are the same) and is the untiled run's within the FP32 mode's 2e-4."""
import numpy as np
import pytest

from workloads import instance

pytestmark = pytest.mark.gpu


def test_neighbouring_reruns_repeat(aw):
    made = [instance(aw, k, L, 20 + k, c=10) for k, L in ((24, 1200), (6, 900), (60, 700))]
    print("re-runs of neighbouring tiles", flush=True)
    b = aw.Batch()
    for (k, L), (tr, seqs, _, model) in zip(((24, 1200), (6, 900), (60, 700)), made):
        b.add(tr, seqs, *model, k - 1, np.random.RandomState(L).uniform(size=L))
    b.upload()

    def run(**kw):
        st = b.run(1, 0, **kw)
        return st, [(b.alpha(i), b.norms(i), b.lnl(i), b.path(i)) for i in range(3)]

    _, whole = run()
    tiled = dict(fw_tile=60, fw_warm=1, fw_tol=1e-7)
    st, first = run(**tiled)
    print("tiles %d re-runs %d" % (st["fw_tiles"], st["fw_reruns"]), flush=True)
    assert st["fw_reruns"] >= st["fw_tiles"] // 2
    _, second = run(**tiled)
    for (a, n, l, p), (a2, n2, l2, p2), (a0, n0, l0, _) in zip(first, second, whole):
        assert np.array_equal(a, a2) and np.array_equal(n, n2) and l == l2 and np.array_equal(p, p2)
        assert np.abs(n / n0 - 1).max() <= 2e-4 and abs(l - l0) <= 2e-4 * abs(l0)
        assert np.abs(a - a0).max() <= 2e-4 * np.abs(a0).max()
    for tr, _, _, _ in made:
        aw.delete_local_trees(tr)
