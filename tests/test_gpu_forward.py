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


@pytest.mark.parametrize("prec", [0, 1])
def test_table_copied_in_pieces(aw, prec):
    """Tables of several staging halves, and ranges of them from odd columns
    on: every entry is the whole table's, which agrees with the oracle."""
    k, L = 30, 5000
    print("table copy prec=%d k=%d L=%d" % (prec, k, L), flush=True)
    tr, seqs, inst, model = instance(aw, k, L, 5, ntimes=20, c=20)
    nst = np.asarray(inst.nstates())
    fw, _ = inst.forward()
    assert fw.size > 3 * (2 << 20) // 8
    b = aw.Batch()
    b.add(tr, seqs, *model, k - 1, np.random.RandomState(L).uniform(size=L))
    b.upload()
    b.run(prec, 0)
    whole = b.alpha(0)
    for got, ref in zip(_columns(inst, whole), _columns(inst, fw)):
        got = got / got.sum(axis=1, keepdims=True)
        assert np.abs(got - ref / ref.sum(axis=1, keepdims=True)).max() <= (2e-4 if prec else 1e-12)
    per_col = np.concatenate([[n] * (int(y - x) // int(n)) for n, x, y in
                              zip(nst, inst.block_offsets(), inst.block_offsets()[1:])])
    off = np.concatenate([[0], np.cumsum(per_col)])
    for c0, c1 in ((0, 1), (L - 1, L), (1, L), (777, 2778), (1234, 1235)):
        part = b.alpha_range(0, c0, c1, per_col)
        assert np.array_equal(part, whole[off[c0]:off[c1]])
    aw.delete_local_trees(tr)


def test_forward_tables_of_the_largest_blocks(aw):
    """32 states per lane: blocks of more than 1024 states."""
    test_forward_tables(aw, 128, 150, 20, 100)
