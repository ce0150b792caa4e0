"""Uploads pass through pinned memory in pieces of 2 MB: instances of several
pieces, placed so that the pieces' ends fall elsewhere in each, give the thread
and likelihood that they give alone."""
import numpy as np
import pytest

from workloads import instance

pytestmark = pytest.mark.gpu


def test_batch_of_several_pieces(aw):
    print("upload of several pieces", flush=True)
    sizes = ((5, 777), (24, 120001), (11, 90000))
    made = [instance(aw, k, L, 3 + k, ntimes=20, c=10) for k, L in sizes]
    us = [np.random.RandomState(i).uniform(size=L) for i, (_, L) in enumerate(sizes)]

    def run(order):
        b = aw.Batch()
        for i in order:
            tr, seqs, _, model = made[i]
            b.add(tr, seqs, *model, sizes[i][0] - 1, us[i])
        b.upload()
        b.run(1, 8192)
        return {i: (b.path(x), b.lnl(x)) for x, i in enumerate(order)}

    alone = {i: run([i])[i] for i in range(3)}
    for order in ((0, 1, 2), (2, 1, 0)):
        for i, (path, lnl) in run(order).items():
            assert np.array_equal(path, alone[i][0]) and lnl == alone[i][1], (order, i)
    for m in made:
        aw.delete_local_trees(m[0])
