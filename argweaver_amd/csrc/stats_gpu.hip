// stats_gpu.hip -- the chain statistics an MCMC run reports every iteration,
// on the device: log P(sequences | ARG) (calc_arg_likelihood,
// src/argweaver/total_prob.cpp:19-45, with likelihood_tree,
// src/argweaver/emit.cpp:399-449).
//
// The reference walks the columns of every local tree, prunes each variant
// column through the tree (JC69, uniform root, branch lengths floored at a
// tenth of the first time step) and reuses the first invariant column's
// likelihood for every later invariant column of the same tree.  Here:
//   k_lnl_class  one thread per column: is every row equal at the column
//   k_lnl_first  one thread per local tree: its first invariant column
//   k_lnl_eval   one wave per column that needs a pruning (variant, or its
//                tree's first invariant column): level-synchronous pruning
//                with the four partial likelihoods of every node in LDS,
//                one node per lane and level
//   k_lnl_sum    one workgroup per 256 columns: the column's log-likelihood
//                (its own, or its tree's first invariant column's) summed in
//                a fixed order; the host adds the workgroup sums in order.
// The terms are the reference's; only the summation order differs.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <vector>

#include "../../include/argweaver_amd.h"
#include "aw_math.h"
#include "host_stage.h"
#include "local_trees.h"

namespace aw {
namespace {

struct LnlArgs {
    int B, N, L, nrows;
    double mintime, mu;
    const double *times;            // [T]
    const int *parent, *c0, *c1, *age;            // [B*N]
    const int *bstart;              // [B+1] column of each tree's start, then L
    const char *rows;               // [nrows*L]: row j is leaf j's sequence
    int *invariant;                 // [L]
    int *first;                     // [B] first invariant column, -1 for none
    double *lk;                     // [L] likelihood of the pruned columns
    double *part;                   // [ceil(L/256)] workgroup sums
};

__device__ int owner_block(const int *bstart, int B, int col)
{
    int lo = 0, hi = B - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (bstart[mid] <= col) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(256) void k_lnl_class(LnlArgs a)
{
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= a.L) return;
    const char r0 = a.rows[c];
    int inv = 1;
    for (int j = 1; j < a.nrows && inv; j++) inv = a.rows[(size_t)j * a.L + c] == r0;
    a.invariant[c] = inv;
}

__global__ __launch_bounds__(256) void k_lnl_first(LnlArgs a)
{
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= a.B) return;
    int f = -1;
    for (int c = a.bstart[b]; c < a.bstart[b + 1]; c++)
        if (a.invariant[c]) {
            f = c;
            break;
        }
    a.first[b] = f;
}

constexpr int LNL_MAXN = MAXN;

// one wave per column
__global__ __launch_bounds__(64) void k_lnl_eval(LnlArgs a)
{
    __shared__ double inner[LNL_MAXN][4];
    __shared__ double mut[LNL_MAXN], nomut[LNL_MAXN];
    __shared__ int hg[LNL_MAXN];   // node heights: leaves 0, a node one more than its higher child
    const int c = blockIdx.x, lane = threadIdx.x;
    const int b = owner_block(a.bstart, a.B, c);
    // an invariant column other than its tree's first takes that one's value
    if (a.invariant[c] && a.first[b] != c) return;   // uniform per wave
    const int N = a.N;
    const int *par = a.parent + (size_t)b * N, *ch0 = a.c0 + (size_t)b * N;
    const int *ch1 = a.c1 + (size_t)b * N, *ag = a.age + (size_t)b * N;
    int root = -1;
    for (int i = lane; i < N; i += 64) hg[i] = 0;
    __syncthreads();
    for (int i = lane; i < N; i += 64) {
        const int p = par[i];
        // every leaf raises its ancestors to their distance from it
        if (ch0[i] == -1) {
            int h = 1;
            for (int q = p; q != -1 && h <= N; q = par[q]) atomicMax(&hg[q], h++);
        }
        if (p == -1) {
            root = i;
            mut[i] = nomut[i] = 0.0;
        } else {
            const double t = fmax(a.times[ag[p]] - a.times[ag[i]], a.mintime);
            mut[i] = prob_branch(t, a.mu, true);
            nomut[i] = prob_branch(t, a.mu, false);
        }
    }
    // the root's index from whichever lane found it
    for (int off = 32; off > 0; off >>= 1) root = max(root, __shfl_xor(root, off));
    __syncthreads();
    const int H = hg[root];
    for (int h = 0; h <= H; h++) {
        for (int i = lane; i < N; i += 64) {
            if (hg[i] != h) continue;
            if (ch0[i] == -1) {
                const int code = base_code(a.rows[(size_t)i * a.L + c]);   // -1: 'N'
                for (int x = 0; x < 4; x++) inner[i][x] = (code < 0 || x == code) ? 1.0 : 0.0;
            } else {
                const int u = ch0[i], v = ch1[i];
                for (int x = 0; x < 4; x++) {
                    double p1 = 0.0, p2 = 0.0;
                    for (int y = 0; y < 4; y++) {
                        p1 += inner[u][y] * (x == y ? nomut[u] : mut[u]);
                        p2 += inner[v][y] * (x == y ? nomut[v] : mut[v]);
                    }
                    inner[i][x] = p1 * p2;
                }
            }
        }
        __syncthreads();
    }
    if (lane == 0) {
        double lk = 0.0;
        for (int x = 0; x < 4; x++) lk += inner[root][x] * .25;
        a.lk[c] = lk;
    }
}

__global__ __launch_bounds__(256) void k_lnl_sum(LnlArgs a)
{
    __shared__ double s[256];
    const int c = blockIdx.x * 256 + threadIdx.x;
    double v = 0.0;
    if (c < a.L) {
        const int b = owner_block(a.bstart, a.B, c);
        v = log(a.invariant[c] ? a.lk[a.first[b]] : a.lk[c]);
    }
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) a.part[blockIdx.x] = s[0];
}

// The device arrays of one call in one allocation: every take() before
// allocate() sizes it, the same calls after it place the arrays.
struct DevBufs {
    char *base = nullptr;
    size_t used = 0;
    int allocate(HostStage &s)
    {
        base = s.device(used);
        used = 0;
        return base == nullptr;
    }
    template <class T>
    void take(T *&p, size_t n)
    {
        p = reinterpret_cast<T *>(base + used);
        used += (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~size_t(255);
    }
};

int arg_loglik_device(const ArgTrees &tr, const double *times, int ntimes, double mu, char **seqs,
                      int nseqs, int seqlen, double *out)
{
    FlatTrees ft;
    flatten(tr, ft);
    const int B = ft.nblocks, N = ft.nnodes, L = seqlen;
    if (tr.length() != seqlen) {
        fprintf(stderr, "argweaver_amd: awamd_arg_likelihood: ARG length %d, %d columns\n",
                tr.length(), seqlen);
        return 1;
    }
    if (N > LNL_MAXN) {
        fprintf(stderr, "argweaver_amd: awamd_arg_likelihood: %d nodes (limit %d)\n", N, LNL_MAXN);
        return 1;
    }
    std::vector<int> bstart(B + 1);
    for (int b = 0; b < B; b++) bstart[b] = ft.start[b];
    bstart[B] = L;
    // row j is leaf j's sequence (seqids) for the tree's leaves, then the rest
    std::vector<const char *> rowp(nseqs);
    for (int j = 0; j < nseqs; j++) rowp[j] = seqs[j < (int)tr.seqids.size() ? tr.seqids[j] : j];

    DevBufs m;
    LnlArgs a{};
    a.B = B; a.N = N; a.L = L; a.nrows = nseqs;
    a.mintime = times[1] * .1;
    a.mu = mu;
    double *dt;
    int *dp, *dc0, *dc1, *dag, *dbs, *dinv, *dfirst;
    char *drows;
    double *dlk, *dpart;
    const int nwg = (L + 255) / 256;
    const auto place = [&] {
        m.take(dt, ntimes);
        m.take(dp, (size_t)B * N);
        m.take(dc0, (size_t)B * N);
        m.take(dc1, (size_t)B * N);
        m.take(dag, (size_t)B * N);
        m.take(dbs, B + 1);
        m.take(drows, (size_t)nseqs * L);
        m.take(dinv, L);
        m.take(dfirst, B);
        m.take(dlk, L);
        m.take(dpart, nwg);
    };
    place();
    const StageUse use;
    if (!use.s) return 1;
    if (m.allocate(*use.s)) {
        fprintf(stderr, "argweaver_amd: awamd_arg_likelihood: device allocation failed\n");
        return 1;
    }
    place();
    Uploader up(*use.s, 0);
    const size_t nodes = sizeof(int) * B * N;
    if (up.put(dt, times, sizeof(double) * ntimes) || up.put(dp, ft.parent.data(), nodes) ||
        up.put(dc0, ft.child0.data(), nodes) || up.put(dc1, ft.child1.data(), nodes) ||
        up.put(dag, ft.age.data(), nodes) ||
        up.put(dbs, bstart.data(), sizeof(int) * (B + 1)))
        return 1;
    for (int j = 0; j < nseqs; j++)
        if (up.put(drows + (size_t)j * L, rowp[j], L)) return 1;
    if (up.flush()) return 1;
    a.times = dt; a.parent = dp; a.c0 = dc0; a.c1 = dc1; a.age = dag; a.bstart = dbs; a.rows = drows; a.invariant = dinv; a.first = dfirst;
    a.lk = dlk; a.part = dpart;
    hipLaunchKernelGGL(k_lnl_class, dim3(nwg), dim3(256), 0, 0, a);
    hipLaunchKernelGGL(k_lnl_first, dim3((B + 255) / 256), dim3(256), 0, 0, a);
    hipLaunchKernelGGL(k_lnl_eval, dim3(L), dim3(64), 0, 0, a);
    hipLaunchKernelGGL(k_lnl_sum, dim3(nwg), dim3(256), 0, 0, a);
    HIP_OK(hipGetLastError());
    std::vector<double> part(nwg);
    HIP_OK(hipMemcpy(part.data(), dpart, sizeof(double) * nwg, hipMemcpyDeviceToHost));
    double s = 0.0;
    for (double x : part) s += x;
    *out = s;
    return 0;
}

// log P(ARG) (calc_arg_prior, src/argweaver/total_prob.cpp:262-299): a
// term per local tree, each on a wave of its own: the probability of the
// tree's recombination-free stretch and, when a tree follows, of the SPR
// into it (calc_spr_prob, total_prob.cpp:210-257).  The sums over nodes and time
// steps take a lane each (on one thread per tree, 0.50 ms for 100 haplotypes x
// 100000 columns; 0.035 so).
struct PriorArgs {
    int B, N;
    const Model *m;
    const int *parent, *age;             // [B*N]
    const int *spr;                      // [4B] the SPR into block b
    const int *len;                      // [B]
    const int *has_next;                 // [B] a block follows before the end
    double *term;                        // [B]
    double *part;                        // [ceil(B/256)]
};

__device__ double wave_sum(double x)
{
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    return x;
}

__global__ __launch_bounds__(64) void k_prior_block(PriorArgs a)
{
    __shared__ int nb[MAXT], nr[MAXT], nc[MAXT];
    const int b = blockIdx.x, lane = threadIdx.x, N = a.N;
    const int *par = a.parent + (size_t)b * N, *age = a.age + (size_t)b * N;
    const Model &m = *a.m;
    const int T = m.T;
    const bool spr = a.has_next[b];   // uniform over the wave
    for (int i = lane; i < T; i += 64) nb[i] = nr[i] = nc[i] = 0;
    __syncthreads();
    // tree length without the basal stub; the lineage counts (count_lineages)
    double len = 0.0;
    int root = N;
    for (int i = lane; i < N; i += 64) {
        const int p = par[i], page = p == -1 ? T - 2 : age[p];
        if (p == -1) root = min(root, i);
        else len += m.times[page] - m.times[age[i]];
        if (!spr) continue;
        for (int j = age[i]; j < page; j++) {
            atomicAdd(&nb[j], 1);
            atomicAdd(&nr[j], 1);
            atomicAdd(&nc[j], 1);
        }
        atomicAdd(&nr[page], 1);
        atomicAdd(&nc[page], 1);
        if (p == -1) atomicAdd(&nb[page], 1);
    }
    for (int off = 32; off > 0; off >>= 1) root = min(root, __shfl_xor(root, off));
    __syncthreads();
    const double treelen = wave_sum(len), rr = fmax(m.rho * treelen, m.rho);
    double v = -rr * a.len[b];
    if (spr) {
        const int *sp = a.spr + 4 * (size_t)(b + 1);
        const int rn = sp[0], k = sp[1], j = sp[3];
        const int root_age = age[root], broken_age = age[par[rn]];
        const auto rate = [&](int i) {
            const int n = (i / 2 == T - 1 ? 1 : nb[i / 2]) - int(i / 2 < broken_age);
            return m.csteps[i] * n / (2.0 * m.pop[i / 2]);
        };
        // the coalescence rates passed on the way from k up to j
        double passed = 0.0;
        for (int x = 2 * k + lane; x < 2 * j - 1; x += 64) passed += rate(x);
        v += log(rr) - wave_sum(passed);
        v += log(nb[k] * m.steps[k] /
                 ((nr[k] - int(k == root_age)) * (treelen + m.steps[root_age])));
        v -= log((double)(nc[j] - int(j <= broken_age) - int(j == broken_age)));
        if (j < T - 2) v += log(1.0 - exp(-rate(2 * j) - (j > k ? rate(2 * j - 1) : 0.0)));
    }
    if (lane == 0) a.term[b] = v;
}

__global__ __launch_bounds__(256) void k_sum_terms(const double *term, int n, double *part)
{
    __shared__ double s[256];
    const int i = blockIdx.x * 256 + threadIdx.x;
    s[threadIdx.x] = i < n ? term[i] : 0.0;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

int arg_logprior_device(const ArgTrees &tr, const Model &model, double *out)
{
    FlatTrees ft;
    flatten(tr, ft);
    const int B = ft.nblocks, N = ft.nnodes;
    std::vector<int> has_next(B);
    long long end = tr.start_coord;
    for (int b = 0; b < B; b++) {
        end += ft.len[b];
        has_next[b] = end < tr.end_coord ? 1 : 0;
    }
    DevBufs m;
    Model *dm;
    int *dp, *dag, *dspr, *dlen, *dnext;
    double *dterm, *dpart;
    const int nwg = (B + 255) / 256;
    const auto place = [&] {
        m.take(dm, 1);
        m.take(dp, (size_t)B * N);
        m.take(dag, (size_t)B * N);
        m.take(dspr, 4 * (size_t)B);
        m.take(dlen, B);
        m.take(dnext, B);
        m.take(dterm, B);
        m.take(dpart, nwg);
    };
    place();
    const StageUse use;
    if (!use.s) return 1;
    if (m.allocate(*use.s)) {
        fprintf(stderr, "argweaver_amd: awamd_arg_prior: device allocation failed\n");
        return 1;
    }
    place();
    Uploader up(*use.s, 0);
    const size_t nodes = sizeof(int) * B * N;
    if (up.put(dm, &model, sizeof(Model)) || up.put(dp, ft.parent.data(), nodes) ||
        up.put(dag, ft.age.data(), nodes) || up.put(dspr, ft.spr.data(), sizeof(int) * 4 * B) ||
        up.put(dlen, ft.len.data(), sizeof(int) * B) ||
        up.put(dnext, has_next.data(), sizeof(int) * B) || up.flush())
        return 1;
    PriorArgs a{B, N, dm, dp, dag, dspr, dlen, dnext, dterm, dpart};
    hipLaunchKernelGGL(k_prior_block, dim3(B), dim3(64), 0, 0, a);
    hipLaunchKernelGGL(k_sum_terms, dim3(nwg), dim3(256), 0, 0, (const double *)dterm, B, dpart);
    HIP_OK(hipGetLastError());
    std::vector<double> part(nwg);
    HIP_OK(hipMemcpy(part.data(), dpart, sizeof(double) * nwg, hipMemcpyDeviceToHost));
    double s = 0.0;
    for (double x : part) s += x;
    *out = s;
    return 0;
}

}  // namespace
}  // namespace aw

using namespace aw;

extern "C" double awamd_arg_likelihood(LocalTrees *trees, const double *times, int ntimes,
                                       double mu, char **seqs, int nseqs, int seqlen)
{
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
        fprintf(stderr, "argweaver_amd: awamd_arg_likelihood needs a HIP device\n");
        return NAN;
    }
    if (ntimes < 3 || ntimes > MAXT) {
        fprintf(stderr, "argweaver_amd: awamd_arg_likelihood: ntimes %d outside 3..%d\n", ntimes,
                MAXT);
        return NAN;
    }
    const ArgTrees &tr = *reinterpret_cast<ArgTrees *>(trees);
    if (tr.nnodes < 3) return log(.25) * seqlen;
    double v = NAN;
    if (arg_loglik_device(tr, times, ntimes, mu, seqs, nseqs, seqlen, &v)) return NAN;
    return v;
}

extern "C" double awamd_arg_prior(LocalTrees *trees, const double *times, int ntimes,
                                  const double *popsizes, double rho)
{
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
        fprintf(stderr, "argweaver_amd: awamd_arg_prior needs a HIP device\n");
        return NAN;
    }
    if (ntimes < 3 || ntimes > MAXT) {
        fprintf(stderr, "argweaver_amd: awamd_arg_prior: ntimes %d outside 3..%d\n", ntimes, MAXT);
        return NAN;
    }
    std::vector<double> pops(ntimes, 1.0);
    if (popsizes)
        for (int i = 0; i < ntimes; i++) pops[i] = popsizes[i];
    Model m;
    model_init(m, ntimes, times, pops.data(), rho, 0.0);
    double v = NAN;
    if (arg_logprior_device(*reinterpret_cast<ArgTrees *>(trees), m, &v)) return NAN;
    return v;
}
