"""The forward's two-wave tiles at the sizes where they can go wrong: one and
two columns, the ends of the 64-column and 64-block windows, switches in most
columns, every states-per-lane count up to 16, and the coarsest and finest time
grids.  FP64 tables against the oracle's within 1e-12, FP32 ones (whole and in
tiles that are re-run) within the FP32 mode's 2e-4 on normalised columns."""
import numpy as np
import pytest

from workloads import instance

pytestmark = pytest.mark.gpu

# (haplotypes, columns, time points, bases per column)
CASES = [(3, 1, 20, 10), (3, 2, 20, 10), (3, 64, 20, 1), (4, 65, 20, 10), (6, 129, 12, 10),
         (8, 300, 20, 2000), (12, 500, 20, 1000), (16, 257, 32, 100), (30, 300, 28, 100),
         (24, 400, 20, 200), (40, 300, 20, 100), (64, 200, 20, 100), (90, 150, 20, 100),
         (110, 120, 20, 100)]


def _columns(inst, a):
    offs, nst = inst.block_offsets(), inst.nstates()
    for blk in range(len(offs) - 1):
        yield a[int(offs[blk]):int(offs[blk + 1])].reshape(-1, int(nst[blk]))


@pytest.mark.parametrize("k,L,T,c", CASES)
def test_forward_tables(aw, k, L, T, c):
    print("forward k=%d L=%d T=%d c=%d" % (k, L, T, c), flush=True)
    tr, seqs, inst, model = instance(aw, k, L, 90 + k, ntimes=T, c=c,
                                     popsizes=np.full(T, 3e4 if k > 100 else 1e4))
    fw, lnl = inst.forward()
    b = aw.Batch()
    b.add(tr, seqs, *model, k - 1, np.random.RandomState(L).uniform(size=L))
    b.upload()
    b.run(0, 0)
    rel = np.abs(b.alpha(0) - fw) / np.maximum(np.abs(fw), 1e-300)
    assert rel.max() <= 1e-12, rel.max()
    assert abs(b.lnl(0) - lnl) <= 1e-12 * max(abs(lnl), 1e-300)
    for kw in ({}, dict(fw_tile=100, fw_warm=2, fw_tol=1e-5)):
        b.run(1, 0, **kw)
        for got, ref in zip(_columns(inst, b.alpha(0)), _columns(inst, fw)):
            got = got / got.sum(axis=1, keepdims=True)
            assert np.abs(got - ref / ref.sum(axis=1, keepdims=True)).max() <= 2e-4
    aw.delete_local_trees(tr)
