"""Performance cases of the threading HMM, through the Python binding's entry points.

A case is a dict of plain values.  ``kind`` says which call it stands for:

  thread    awamd_thread_forward: one lineage threaded into an ARG (forward
            and stochastic traceback from given uniforms), results in the
            caller's buffers
  sample    argweaverc.sample_thread on a copy of a partial ARG: the drop-in
            call of a resample_arg step, recombinations and insertion included
  region    argweaverc.resample_arg_region on a copy of a full ARG: internal
            branches re-threaded over a window, conditioned at its ends
  batch     argweaverc.Batch: independent instances, inputs resident
  serve     argweaverc.Server: requests submitted together, then waited for
  stats     argweaverc.arg_likelihood_device / arg_prior_device, the two
            statistics a chain records after every step

Inputs come from the package's seeded coalescent simulator under the model of
the repository's benchmark (20 time points to 200e3 generations, N = 1e4, or a
piecewise N(t), 1.6e-8 and 1.8e-8 per base at 10 bases per column).  Sizes follow from the case alone; the seed chooses the
ARG, the sequences and the uniforms.
"""
import ctypes
import math

import numpy as np

import argweaver_amd.argweaverc as A

C = 10                      # bases per column
RHO, MU = 1.6e-8 * C, 1.8e-8 * C
TILE = 4096                 # traceback tile of a single long instance
BATCH_TILE, TAIL = 14000, 4000
FW_BATCH = (100000, 40000)  # forward tile / warm-up of the mixed batch
FW_TOL = 1e-4


def listed():
    return [
        # the smallest call: 4 haplotypes, 700 columns, everything returned
        dict(name="thread_tiny", kind="thread", k=4, L=700, ntimes=20, pops="const", precision=0,
             table=True, noalloc=False),
        # 8 haplotypes over 100 kb in the fixed workspace, for callers that
        # must not allocate
        dict(name="thread_100kb_noalloc", kind="thread", k=8, L=10000, ntimes=20, pops="const",
             precision=0, table=True, noalloc=True),
        # FP32 with its table, a mid-sized region
        dict(name="thread_fp32_table", kind="thread", k=20, L=20011, ntimes=20, pops="const",
             precision=1, table=True, noalloc=False),
        # a finer time grid than the usual one
        dict(name="thread_28_times", kind="thread", k=16, L=6001, ntimes=28, pops="const",
             precision=0, table=True, noalloc=False),
        # blocks of more than 1024 states: 128 haplotypes under N = 3e4
        dict(name="thread_big_blocks", kind="thread", k=128, L=3001, ntimes=20, pops="large",
             precision=1, table=False, noalloc=False),
        # one Gibbs step of a chain in FP32: 100 haplotypes, 5 Mb
        dict(name="thread_5mb_fp32", kind="thread", k=100, L=500000, ntimes=20, pops="piecewise",
             precision=1, table=False, noalloc=False),
        # the drop-in call on 50 haplotypes over 1 Mb
        dict(name="sample_1mb", kind="sample", k=50, L=100000, ntimes=20, pops="const"),
        # internal branches of 16 haplotypes re-threaded in a window
        dict(name="region_16", kind="region", k=16, L=20000, start=5000, end=15000, niters=3),
        # the mixed batch: 256 instances, 8..64 haplotypes, 50 kb .. 2 Mb
        dict(name="batch_256_fp32", kind="batch", n=256, kmin=8, kmax=64, lmin=5000, lmax=200000,
             precision=1),
        # a smaller batch in the drop-in precision
        dict(name="batch_32_fp64", kind="batch", n=32, kmin=8, kmax=50, lmin=5000, lmax=100000,
             precision=0),
        # a burst of requests to the server
        dict(name="serve_24_fp32", kind="serve", n=24, kmin=8, kmax=50, lmin=5000, lmax=100000,
             precision=1),
        # chain statistics of a 100-haplotype ARG over 1 Mb
        dict(name="stats_1mb", kind="stats", k=100, L=100000, pops="piecewise"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["thread", "thread", "thread", "sample", "region", "batch", "serve", "stats"])
    if kind == "thread":
        L = _logint(rng, 500, 400000)
        precision = rng.choice([0, 1])
        k = rng.randint(3, 64 if precision == 0 else 100)
        ntimes = rng.choice([20, 20, 20, 12, 28, 32])
        # a table of at most about 10^7 entries, in the fixed workspace only
        # where it fits with room to spare
        table = L * k * 12 <= 10000000 and rng.random() < 0.6
        noalloc = L * k <= 90000 and k <= 12 and rng.random() < 0.5
        return dict(kind=kind, k=k, L=L, ntimes=ntimes, pops=rng.choice(["const", "piecewise"]),
                    precision=precision, table=table, noalloc=noalloc)
    if kind == "sample":
        return dict(kind=kind, k=rng.randint(4, 64), L=_logint(rng, 1000, 150000), ntimes=20,
                    pops=rng.choice(["const", "piecewise"]))
    if kind == "region":
        L = _logint(rng, 2000, 40000)
        start = rng.randint(0, L // 2)
        return dict(kind=kind, k=rng.randint(4, 24), L=L, start=start,
                    end=rng.randint(start + L // 8, L), niters=rng.randint(1, 3))
    if kind == "stats":
        return dict(kind=kind, k=rng.randint(4, 128), L=_logint(rng, 2000, 200000),
                    pops=rng.choice(["const", "piecewise"]))
    precision = rng.choice([0, 1])
    lmin = _logint(rng, 1000, 10000)
    return dict(kind=kind, n=_logint(rng, 2, 160 if kind == "batch" else 48), kmin=rng.randint(3, 12),
                kmax=rng.randint(16, 64), lmin=lmin,
                lmax=lmin * rng.randint(2, 20 if precision else 10), precision=precision)


# ---------------------------------------------------------------------------
# inputs


def _pops(name, ntimes, rng):
    if name == "piecewise":
        return np.exp(rng.uniform(np.log(5e3), np.log(5e4), size=ntimes))
    return np.full(ntimes, 3e4 if name == "large" else 1e4)


def _arg(k, L, ntimes, pops, seed):
    """(trees with k leaves, sequences, model, uniforms)"""
    rng = np.random.RandomState(seed % (1 << 31))
    times = np.array(A.get_time_points(ntimes, 200e3), np.float64)
    p = _pops(pops, ntimes, rng)
    tr, seqs = A.simulate(k, L, times, p, RHO, MU, int(seed))
    return tr, seqs, (times, p, RHO, MU), rng.uniform(size=L)


class _Trees(object):
    """An ARG handle freed with its state."""

    def __init__(self, ptr):
        self.ptr = ptr

    def __del__(self):
        A.delete_local_trees(self.ptr)


def _mix(case, seed):
    sizes = np.random.RandomState(case["n"] * 1000 + case["kmin"] * 100 + case["kmax"])
    out = []
    for i in range(case["n"]):
        k = int(sizes.randint(case["kmin"], case["kmax"] + 1))
        L = int(np.exp(sizes.uniform(np.log(case["lmin"]), np.log(case["lmax"]))))
        tr, seqs, model, u = _arg(k, L, 20, "const", (seed % 1000003) * 1009 + i)
        A.remove_thread(tr, k - 1)
        out.append((_Trees(tr), A.CSeqs(seqs), model, k - 1, u))
    return out


def _table_size(case):
    """Room for any table of the case: every column with the most states a
    tree of k - 1 leaves has (no coalescence before the last time)."""
    return case["L"] * (case["k"] - 1) * case["ntimes"]


def _tree_cap(case):
    """Room for the local trees of an ARG: well over their expected number."""
    N = 3e4 if case.get("pops") == "piecewise" else 1e4
    return int(100 + 2.0 * case["L"] * RHO * 4.0 * N * sum(1.0 / i for i in range(1, case["k"])))


def prepare(case, seed):
    """What a program holds before the call."""
    kind = case["kind"]
    if kind in ("batch", "serve"):
        items = _mix(case, seed)
        if kind == "serve":
            srv = A.Server(hbm_budget_gb=48.0, precision=case["precision"], tile_cols=2000,
                           max_batch=64)
            return dict(case=case, items=items, server=srv)
        b = A.Batch()
        for tr, seqs, model, chrom, u in items:
            b.add(tr.ptr, seqs, *model, chrom, u)
        b.upload()
        b.set_tail_tiles(TAIL)
        return dict(case=case, batch=b, n=len(items))
    if kind == "region":
        tr, seqs, model, _ = _arg(case["k"], case["L"], 20, "const", seed)
        return dict(case=case, trees=_Trees(tr), seqs=A.CSeqs(seqs), model=model, seed=seed)
    ntimes = case.get("ntimes", 20)
    tr, seqs, model, u = _arg(case["k"], case["L"], ntimes, case["pops"], seed)
    if kind != "stats":
        A.remove_thread(tr, case["k"] - 1)
    s = dict(case=case, trees=_Trees(tr), seqs=A.CSeqs(seqs), model=model, u=u, seed=seed)
    if kind == "thread":
        s["path"], s["ms"] = np.zeros(case["L"], np.int32), np.zeros(4)
        s["alpha"] = None
        if case["table"]:
            n = _table_size(case)
            s["W"] = A.num_column_states(tr, ntimes)[0]
            s["alpha"] = np.zeros(n, np.float64)
            s["alpha32"] = np.zeros(n, np.float32) if case["precision"] else None
    return s


def _arrays(case, trees):
    """The ARG's arrays, with room to spare at the end of each."""
    out = {}
    for name, a in zip(("ptrees", "ages", "sprs", "blocklens"), A.trees_arrays(trees)):
        out[name] = np.full((_tree_cap(case),) + a.shape[1:], -1, np.int32)
        out[name][:len(a)] = a
    return out


def run(state):
    """One pass; returns what the path computes."""
    case = state["case"]
    kind = case["kind"]
    if kind == "thread":
        times, pops, rho, mu = state["model"]
        alpha, lnl = state["alpha"], ctypes.c_double(0.0)
        call = A.awamd_thread_forward_noalloc if case["noalloc"] else A.awamd_thread_forward
        if call(state["trees"].ptr, _dp(times), len(times), _dp(pops), rho, mu, state["seqs"].ptr,
                case["k"] - 1, _dp(state["u"]), case["precision"],
                None if alpha is None else _dp(alpha),
                state["path"].ctypes.data_as(A.c_int_p), ctypes.byref(lnl), _dp(state["ms"])):
            raise RuntimeError("thread_forward failed")
        out = dict(path=state["path"], lnl=lnl.value)
        if alpha is not None and case["precision"]:
            # an FP32 run's entries are 32-bit values
            out["alpha"] = state["alpha32"]
            out["alpha"][:state["W"]] = alpha[:state["W"]]
        elif alpha is not None:
            out["alpha"] = alpha
        return out
    if kind == "sample":
        tr = _Trees(A.argweaver_copy_trees(state["trees"].ptr))
        A.set_random_seed(state["seed"] % (1 << 31))
        A.sample_thread(tr.ptr, state["seqs"], *state["model"])
        return _arrays(case, tr.ptr)
    if kind == "region":
        tr = _Trees(A.argweaver_copy_trees(state["trees"].ptr))
        A.set_random_seed(state["seed"] % (1 << 31))
        A.resample_arg_region(tr.ptr, state["seqs"], *state["model"], case["start"], case["end"],
                              niters=case["niters"])
        return _arrays(case, tr.ptr)
    if kind == "batch":
        b = state["batch"]
        if case["precision"]:
            b.run(1, BATCH_TILE, fw_tile=FW_BATCH[0], fw_warm=FW_BATCH[1], fw_tol=FW_TOL)
        else:
            b.run(0, TILE)
        return dict(path=np.concatenate([b.path(i) for i in range(state["n"])]),
                    lnl=_lnls(case, [b.lnl(i) for i in range(state["n"])]))
    if kind == "serve":
        srv = state["server"]
        ids = [srv.submit(tr.ptr, seqs, *model, chrom, u)
               for tr, seqs, model, chrom, u in state["items"]]
        res = [srv.wait(i, timeout=60) for i in ids]
        return dict(path=np.concatenate([r["path"] for r in res]),
                    lnl=_lnls(case, [r["lnl"] for r in res]))
    times, pops, rho, mu = state["model"]
    return dict(likelihood=A.arg_likelihood_device(state["trees"].ptr, state["seqs"], times, mu),
                prior=A.arg_prior_device(state["trees"].ptr, times, pops, rho))


def _dp(a):
    return a.ctypes.data_as(A.c_double_p)


def _lnls(case, v):
    return np.array(v, np.float32 if case["precision"] else np.float64)


# ---------------------------------------------------------------------------
# work: the expected number of states of a k-1 leaf local tree under the
# coalescent (lineages at each time point, plus the shared end of a branch)


def _states(k, ntimes, N):
    n = max(k - 1, 2)
    times = A.get_time_points(ntimes, 200e3)
    s = sum(1.0 / (1.0 - (1.0 - 1.0 / n) * math.exp(-t / (4.0 * N))) for t in times[:ntimes - 1])
    return s + n


def _one(k, L, ntimes, N, precision, table):
    S = _states(k, ntimes, N)
    e = 4 if precision else 8
    blocks = 1 + L * RHO * 4.0 * N * sum(1.0 / i for i in range(1, max(k - 1, 2)))
    # the table written once and read once by the traceback, sequences, trees
    # (parent, children, age, mapping), uniforms, path, and the table returned
    by = L * S * 2 * e + L * k + blocks * (2 * k) * 20 + 12 * L + (8 * L * S if table else 0)
    # forward: scans, emission and scaling of a state, the time-bin product;
    # traceback: weight and cumulative sum of a state
    fl = L * (S * 16 + 2 * ntimes * ntimes)
    return by, fl


def work(case):
    kind = case["kind"]
    N = 3e4 if case.get("pops") == "large" else 2e4 if case.get("pops") == "piecewise" else 1e4
    if kind in ("batch", "serve"):
        a, b = math.log(case["lmin"]), math.log(case["lmax"])
        L = (math.exp(b) - math.exp(a)) / (b - a) if b > a else math.exp(a)
        ks = range(case["kmin"], case["kmax"] + 1)
        each = [_one(k, L, 20, N, case["precision"], False) for k in ks]
        m = case["n"] / len(each)
        return dict(bytes=m * sum(x[0] for x in each), flops=m * sum(x[1] for x in each))
    if kind == "stats":
        L, k = case["L"], case["k"]
        blocks = 1 + L * RHO * 4.0 * N * sum(1.0 / i for i in range(1, k))
        # sequences and trees read once; a pruning per variant column (about
        # 3 %) and per tree, 4 x 4 products on every branch
        return dict(bytes=L * k + blocks * 2 * k * 16, flops=(0.03 * L + blocks) * 2 * k * 32)
    if kind == "region":
        by, fl = _one(case["k"], case["end"] - case["start"], 20, N, 0, False)
        return dict(bytes=by * case["niters"], flops=fl * case["niters"])
    by, fl = _one(case["k"], case["L"], case["ntimes"], N, case.get("precision", 0),
                  case.get("table", False))
    return dict(bytes=by, flops=fl)


# ---------------------------------------------------------------------------
# the same values from dense matrices in numpy, 64 bits


class _Model(object):
    def __init__(self, times, pops, rho, mu):
        self.T = len(times)
        self.times, self.pop, self.rho, self.mu = times, pops, rho, mu
        self.step = np.append(np.diff(times), np.inf)
        mid = np.sqrt((times[1:] + 1.0) * (times[:-1] + 1.0))
        half = np.empty(2 * self.T - 1)
        half[0::2], half[1::2] = times, mid
        self.half = np.append(np.diff(half), [np.inf, np.inf])
        self.hpop = np.repeat(pops, 2)     # population size of each half interval
        self.mintime = times[1] * .1


class _Tree(object):
    """One local tree: lineage counts, branch lengths, states in node order."""

    def __init__(self, par, age, m):
        self.par, self.age, self.n = par, age, len(par)
        T = m.T
        self.root = int(np.nonzero(par == -1)[0][0])
        self.kids = [[] for _ in range(self.n)]
        for i, p in enumerate(par):
            if p >= 0:
                self.kids[p].append(i)
        self.top = np.where(par >= 0, age[np.maximum(par, 0)], T - 2)
        self.nb, self.nr = np.zeros(T, int), np.zeros(T, int)
        for i in range(self.n):
            self.nb[age[i]:self.top[i]] += 1
            self.nr[age[i]:self.top[i] + 1] += 1
        self.nb[self.top[self.root]] += 1
        self.nb[T - 1] = 1
        self.node = np.repeat(np.arange(self.n), self.top - age + 1)
        self.first = np.concatenate([[0], np.cumsum(self.top - age + 1)])
        self.time = np.arange(len(self.node)) - self.first[self.node] + age[self.node]
        b = np.where(par >= 0, m.times[self.top] - m.times[age], 0.0)
        self.length = b.sum()
        self.blen = np.where(par >= 0, np.maximum(b, m.mintime), 0.0)

    def index(self, node, time):
        if node < 0 or time < self.age[node] or time > self.top[node]:
            return -1
        return int(self.first[node] + time - self.age[node])


def _rates(t, m):
    """coalescence rate of the half intervals, and its running sum C[i + 2]"""
    r = m.half[:2 * m.T - 1] * np.repeat(t.nb, 2)[:2 * m.T - 1] / (2.0 * m.hpop[:2 * m.T - 1])
    return r, np.concatenate([[0.0, 0.0], np.cumsum(r)])


def _within(t, m):
    """dense transition matrix of one block"""
    n = m.T - 1
    r, Cs = _rates(t, m)
    i = np.arange(n)
    ra = t.age[t.root]
    above = i > ra
    ln = t.length + m.times[i] + np.where(above, m.times[i] - m.times[ra], 0.0)
    lnb = ln + np.where(above, m.step[i], m.step[ra])
    nb, nr = t.nb[i], t.nr[i]
    up = (nb + 1.0) / (nr + 1.0)
    lo = nb / (nr + 1.0 + (i < ra))
    eC = np.exp(Cs[2 * i + 1])             # to the start of interval i
    B = np.cumsum(eC * m.step[i] * up)
    NG = -eC * m.step[i] * (lo - up)
    last = i == n - 1
    rm1 = np.concatenate([[0.0], r])[2 * i]
    E2 = np.exp(-Cs[2 * i]) * np.where(last, 1.0, -np.expm1(-r[2 * i] - rm1))
    q = np.where(last, 1.0, -np.expm1(-r[2 * i]))
    G2, G3 = q * m.step[i] * up, q * m.step[i] * lo
    D = -np.expm1(-m.rho * ln) / lnb
    Bm = np.concatenate([[0.0], B])        # B[b - 1]
    a, b = i[:, None], i[None, :]
    base = np.where(a < b, E2[None, :] * (B - NG)[:, None],
                    (E2 * Bm[:n])[None, :] + np.where(a == b, G3[None, :], G2[None, :]))
    scale = D[:, None] / t.nr[i][None, :]
    stay = np.exp(-np.maximum(m.rho * ln, m.rho))
    P = (scale * base)[t.time[:, None], t.time[None, :]]
    for x in range(t.n):
        s = slice(t.first[x], t.first[x + 1])
        u = t.time[s]
        c = t.age[x]
        same = scale * (2 * base - (E2 * Bm[c])[None, :]) + np.diag(stay)
        P[s, s] = same[np.ix_(u, u)]
    return P


def _p_recomb(t, m, k, node, a):
    ra = t.age[t.root]
    ln = t.length + m.times[a] + (m.times[a] - m.times[ra] if node == t.root else 0.0)
    at = a if node == t.root else ra
    full = ln + m.times[at + 1] - m.times[at]
    nb = t.nb[k] + (k < a)
    nr = t.nr[k] + (k <= a) + (k == a) - (k >= max(ra, a))
    return nb * m.step[k] / (nr * full) * -np.expm1(-max(m.rho * ln, m.rho))


def _p_coal(t, m, k, j, a, pa):
    """the branch broken at time k joins the rest at time j (thread at a)"""
    rate = lambda x: m.half[x] * (t.nb[x // 2] - (x // 2 < pa) + (x // 2 < a)) / (2.0 * m.hpop[x])  # noqa: E731
    p = math.exp(-sum(rate(x) for x in range(2 * k, 2 * j - 1)))
    p /= t.nr[j] - (j <= pa) - (j == pa) + (j <= a) + (j == a)
    if j < m.T - 2:
        p *= -np.expm1(-rate(2 * j) - (rate(2 * j - 1) if j > k else 0.0))
    return p


def _switch(t1, t2, spr, mp, m):
    """dense transition matrix across an SPR (block t1 to block t2)"""
    rn, rt, cn, ct = (int(x) for x in spr)
    P = np.zeros((len(t1.node), len(t2.node)))
    pa = int(t1.age[t1.par[rn]])
    broke = int(t1.par[rn])
    other = [x for x in t1.kids[broke] if x != rn][0]
    for j, (n1, a) in enumerate(zip(t1.node.tolist(), t1.time.tolist())):
        if (n1, a) in ((rn, rt), (cn, ct)):
            continue
        to = (n1, a)
        if n1 != rn:
            if not t1.kids[n1]:
                n2, gone = n1, False
            elif n1 == broke:
                n2, gone = int(mp[other]), True
            else:
                n2, gone = int(mp[n1]), False
            if (cn == n1 and ct < a) or (mp[cn] == n2 and (ct < a or (gone and ct <= a))):
                n2 = int(t2.par[n2])
            to = (n2, a)
        elif rt > a:
            to = (int(mp[rn]), a)
        else:
            to = (int(t2.par[mp[other]]) if other == cn else int(mp[other]), pa)
        k = t2.index(*to)
        if k >= 0:
            # a state on the broken branch above the break takes its place
            eff = a if (n1 == rn and a > rt) else pa
            P[j, k] = _p_recomb(t1, m, rt, n1, a) * _p_coal(t1, m, rt, ct, a, eff)
    w = lambda j, n, a, q: _p_recomb(t1, m, rt, n, a) * _p_coal(t1, m, rt, j, a, q)  # noqa: E731
    js = t1.index(rn, rt)
    if js >= 0:
        stay = t2.index(int(mp[rn]), rt)
        esc = t2.index(int(t2.par[mp[other]]) if other == cn else int(mp[other]), pa)
        if stay >= 0:
            P[js, stay] = w(ct, rn, rt, pa)
        if esc >= 0:
            P[js, esc] = w(ct, rn, rt, rt)
    jc = t1.index(cn, ct)
    if jc >= 0:
        n3 = int(mp[other]) if broke == cn else int(mp[cn])
        mr = int(mp[rn])
        for k, (n2, b) in enumerate(zip(t2.node.tolist(), t2.time.tolist())):
            if (n2 == mr and b >= rt) or (n2 in (n3, int(t2.par[mr])) and b == ct):
                P[jc, k] = w(b, cn, ct, pa)
    return P


def _prior(t, m):
    r, Cs = _rates(t, m)
    p = np.zeros(m.T - 1)
    for b in range(m.T - 1):
        p[b] = math.exp(-r[:max(2 * b - 1, 0)].sum()) / t.nr[b]
        if b < m.T - 2:
            p[b] *= -np.expm1(-r[2 * b] - (r[2 * b - 1] if b else 0.0))
    return p[t.time]


def _jc(d, mu):
    """(4, 4) or (n, 4, 4) Jukes-Cantor probabilities of branches of length d"""
    e = np.exp(-4. / 3. * mu * np.asarray(d))[..., None, None]
    return .25 * (1.0 - e) + np.eye(4) * e


def _partials(t, cols, mu):
    """inner partial likelihoods [node, 4, column] of leaf bases cols"""
    J = _jc(t.blen, mu)
    inner = np.zeros((t.n, 4, cols.shape[1]))
    done, todo = set(), list(range(t.n))
    while todo:      # children before their parents
        rest = []
        for i in todo:
            if not t.kids[i]:
                for x, ch in enumerate(b"ACGT"):
                    inner[i, x] = cols[i] == ch
            elif all(c in done for c in t.kids[i]):
                a, b = t.kids[i]
                inner[i] = (J[a] @ inner[a]) * (J[b] @ inner[b])
            else:
                rest.append(i)
                continue
            done.add(i)
        todo = rest
    return J, inner


def _emit_variant(t, cols, new, m):
    """[column, state] emissions of variant columns"""
    J, inner = _partials(t, cols, m.mu)
    outer = np.ones_like(inner)
    stack = [t.root]
    while stack:
        p = stack.pop()
        for i in t.kids[p]:
            s = [x for x in t.kids[p] if x != i][0]
            outer[i] = J[s] @ inner[s]
            if p != t.root:
                outer[i] = outer[i] * (J[p] @ outer[p])
            stack.append(i)
    leaf = np.array([new == ch for ch in b"ACGT"], float)
    top = m.times[np.minimum(t.top, m.T - 1)]
    E = np.zeros((cols.shape[1], len(t.node)))
    here = m.times[t.time]
    J0 = _jc(np.maximum(here, m.mintime), m.mu)
    J1 = _jc(np.maximum(here - m.times[t.age[t.node]], m.mintime), m.mu)
    J2 = _jc(np.maximum(top[t.node] - here, m.mintime), m.mu)
    for k, n in enumerate(t.node):
        v = (J0[k] @ leaf) * (J1[k] @ inner[n])
        if n != t.root:
            v = v * (J2[k] @ outer[n])
        E[:, k] = .25 * v.sum(0)
    return E


def _emit_invariant(t, m):
    here = m.times[t.time]
    ln = t.blen.sum() + np.maximum(here, m.mintime)
    ln = ln + np.where(t.node == t.root, np.maximum(here - m.times[t.age[t.root]], m.mintime), 0.0)
    return .25 * np.exp(-m.mu * ln)


def _exact_thread(case, seed):
    s = prepare(dict(case), seed)
    P, G, S, bl = A.trees_arrays(s["trees"].ptr)
    maps, ids = A.trees_internal(s["trees"].ptr)
    m = _Model(*s["model"])
    seqs = s["seqs"].arr
    leaf, new = seqs[ids], seqs[case["k"] - 1]
    var = (leaf != new).any(0)
    rows, lnl, col, t0, x = [], 0.0, 0, None, None
    for b in range(len(bl)):
        t = _Tree(P[b], G[b], m)
        M = _within(t, m)
        end = col + int(bl[b])
        vc = np.nonzero(var[col:end])[0] + col
        E = dict(zip(vc.tolist(), _emit_variant(t, leaf[:, vc], new[vc], m))) if len(vc) else {}
        inv = _emit_invariant(t, m)
        for c in range(col, end):
            if c == 0:
                x = _prior(t, m)
            else:
                x = x @ (M if c > col else _switch(t0, t, S[b], maps[b], m)) * E.get(c, inv)
                z = x.sum()
                x = x / z
                lnl += math.log(z)
            rows.append(x)
        col, t0 = end, t
    out = dict(path=None, lnl=lnl)
    if case["table"]:
        out["alpha"] = np.zeros(_table_size(case))
        v = np.concatenate(rows)
        out["alpha"][:len(v)] = v
    return out


def _exact_stats(case, seed):
    s = prepare(dict(case), seed)
    P, G, S, bl = A.trees_arrays(s["trees"].ptr)
    _, ids = A.trees_internal(s["trees"].ptr)
    m = _Model(*s["model"])
    seqs = s["seqs"].arr[ids]
    var = (seqs != seqs[0]).any(0)
    lk, pr, col = 0.0, 0.0, 0
    for b in range(len(bl)):
        t = _Tree(P[b], G[b], m)
        n, end = int(bl[b]), col + int(bl[b])
        vc = np.nonzero(var[col:end])[0] + col
        ic = np.nonzero(~var[col:end])[0] + col
        cols = np.concatenate([vc, ic[:1]])
        v = np.log(.25 * _partials(t, seqs[:, cols], m.mu)[1][t.root].sum(0))
        lk += v[:len(vc)].sum() + (v[-1] * len(ic) if len(ic) else 0.0)
        rate = max(m.rho * t.length, m.rho)
        pr -= rate * n
        if b + 1 < len(bl):
            rn, rt, cn, ct = (int(x) for x in S[b + 1])
            ra, pa = t.age[t.root], int(t.age[t.par[rn]])
            nr = t.nr[rt] - (rt == ra)
            pr += math.log(rate) + math.log(t.nb[rt] * m.step[rt] / (nr * (t.length + m.step[ra])))
            rl = lambda x: m.half[x] * (t.nb[x // 2] - (x // 2 < pa)) / (2.0 * m.hpop[x])  # noqa: E731
            pr -= math.log(t.nr[ct] - (ct <= pa) - (ct == pa))
            if ct < m.T - 2:
                pr += math.log(-np.expm1(-rl(2 * ct) - (rl(2 * ct - 1) if ct > rt else 0.0)))
            pr -= sum(rl(x) for x in range(2 * rt, 2 * ct - 1))
        col = end
    return dict(likelihood=lk, prior=pr)


def exact(case, seed):
    """The floating outputs of run() in 64 bits, for sizes dense matrices
    reach in a few seconds."""
    if case["kind"] == "stats" and case["L"] * case["k"] <= 10000000:
        return _exact_stats(case, seed)
    if case["kind"] == "thread" and case["L"] * case["k"] * case["ntimes"] <= 9000000:
        return _exact_thread(case, seed)
    return None
