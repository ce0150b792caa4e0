// engine.hip -- gfx950 kernels of the threading HMM and their host driver.
//
// Everything runs on one HIP stream over a Batch of independent instances
// whose inputs (local trees, sequences, uniforms) are resident in HBM.
//
//   k_classify_b   one lane per column: masked / invariant / variant
//   k_scan_b       one workgroup per instance: variant-column numbering, the
//                  mutation probabilities of branches by their times
//   k_prep_b       one workgroup per local-tree block: state space, lineage
//                  counts, TransMatrix vectors and tables, the switch matrix
//                  from the previous block, invariant emissions, first-column
//                  prior, and the per-state coefficient planes of the
//                  lane-run layout (engine.h)
//   k_var_emit_b   one wave per variant column: Felsenstein partials and the
//                  emission row over the block's states
//   k_fw_all       two waves per tile (an instance, or a part of a long one
//                  in FP32) over all its columns, every tile of a batch in
//                  one launch (forward_kernels.h).  Lane l owns states l*R ..
//                  l*R+R-1 (node-major).  The same-branch part of the
//                  transition is a per-branch prefix and suffix sum (in-lane
//                  scan plus a DPP wave-shift carry chain across the few
//                  lanes a branch spans), run by one wave; the other-branch
//                  part goes through the per-time sums (FP64 LDS atomics) and
//                  the (a,b) table, run by the other; a column costs
//                  O(S + T^2) and rows are written coalesced.
//   k_lnl_b        per-instance sum of log normalisers (FP64)
//   traceback      one workgroup per column tile (traceback.hip).  A tile
//                  before the last runs a speculative chain (a state sampled
//                  from a column past its end and a warm-up); a tile whose
//                  true state at its end proves to be another is re-run from
//                  it until it meets the chain's path (identical from there
//                  on)
//
// The forward kernel is a template over the table type: double is the
// drop-in arithmetic (the reference's forward table to ~1e-15), float keeps
// the table and the recursion in FP32 with per-column rescaling while the
// normalisers, the log-likelihood and the traceback CDF stay FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstdlib>
#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <numeric>
#include <thread>
#include <vector>

#include "engine.h"
#include "forward.h"
#include "host_stage.h"
#include "kernel_util.h"
#include "traceback.h"

namespace aw {

//===========================================================================
// column classification

__global__ void k_classify_b(const DevInst *__restrict__ D, const long long *coloff, int ninst)
{
    long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= coloff[ninst]) return;
    int i = find_owner(coloff, ninst, g);
    const DevInst &d = D[i];
    if (d.hostprep) return;
    int col = (int)(g - coloff[i]);
    char c0 = gp(d.seq)[col];
    bool inv = true;
    for (int r = 1; r < d.nrows; r++)
        if (gp(d.seq)[(size_t)r * d.L + col] != c0) { inv = false; break; }
    gp(d.vflag)[col] = inv ? 0 : 1;
    gp(d.cls)[col] = inv ? (c0 == 'N' ? -2 : -1) : 0;
}

// variant-column numbering of one instance: each of 16 waves owns a contiguous
// run of columns and counts them 64 at a time, a load of 8 times that in flight
// (runs of single threads, uncoalesced, took 0.77 ms for 500000 columns, this
// 0.28).  Also the instance's table of branch mutation probabilities.
__global__ __launch_bounds__(1024) void k_scan_b(const DevInst *__restrict__ D, int *nvar_out)
{
    __shared__ int part[16];
    const DevInst &d = D[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63;
    for (int x = tid; x < d.L / 32 + 1; x += 1024) gp(d.cut)[x] = 0;
    if (d.hostprep) {   // the whole workgroup leaves: the host knows the count
        if (tid == 0) nvar_out[blockIdx.x] = 0;
        return;
    }
    {
        const Model &M = *d.model;
        const int T = d.T;
        const double mintime = M.times[1] * .1;
        for (int x = tid; x < (T + 1) * T; x += 1024) {
            const int i = x / T, j = x % T;
            const double t = i < T ? M.times[i] - M.times[j] : M.times[j] - 0.0;
            gp(d.pmut)[2 * x] = prob_branch(fmax(t, mintime), M.mu, true);
            gp(d.pmut)[2 * x + 1] = prob_branch(fmax(t, mintime), M.mu, false);
        }
    }
    const int per = (d.L + 16 * 64 - 1) / (16 * 64) * 64;
    const int s0 = min(d.L, (tid >> 6) * per), e0 = min(d.L, s0 + per);
    constexpr int U = 8;
    const auto walk = [&](int run, bool store) {
        for (int c0 = s0; c0 < e0; c0 += 64 * U) {
            int f[U];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int c = c0 + 64 * u + lane;
                f[u] = c < e0 ? gp(d.vflag)[c] : 0;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const unsigned long long m = __ballot(f[u] != 0);
                if (store && f[u]) {
                    const int c = c0 + 64 * u + lane;
                    const int k = run + __popcll(m & ((1ull << lane) - 1));
                    gp(d.cls)[c] = k;
                    gp(d.vcol)[k] = c;
                }
                run += __popcll(m);
            }
        }
        return run;
    };
    const int cnt = walk(0, false);
    if (lane == 0) part[tid >> 6] = cnt;
    __syncthreads();
    int base = 0, total = 0;
    for (int w = 0; w < 16; w++) {
        if (w < (tid >> 6)) base += part[w];
        total += part[w];
    }
    walk(base, true);
    if (tid == 0) nvar_out[blockIdx.x] = total;
}

//===========================================================================
// per-block preparation

struct PrepShared {
    Model M;
    int par[MAXN], ch0[MAXN], ch1[MAXN], ag[MAXN];
    int ppar[MAXN], pch0[MAXN], pch1[MAXN], pag[MAXN];
    int map[MAXN];
    int root, proot;
    Lineages L, PL;
    TransVec tv;
    NodeIndex ni, pni;
    SwitchCtx cx;
    double mainlen;
    int recombsrc, recoalsrc;
    int node3, rparent;
    int wsum[8];
    int hgt[MAXN], dep[MAXN];
    double rates[2 * MAXT + 1], Cs[2 * MAXT + 2], lnBt[MAXT], eexp[MAXT];
    double red[3 * 4];
    // per-time factors of the state planes
    double eB[MAXT], eN[MAXT], eE2[MAXT], low[MAXT];
    double inv[MAXT], inv_root[MAXT];   // emission of an invariant column, off and on the root
};

// Lineage counts (count_lineages) with one thread per node and integer LDS
// atomics: the single-thread loop is a chain of dependent LDS updates.
// The counts must be zero on entry; the caller synchronises after.
__device__ inline void lineages_par(const TreeView &t, int T, Lineages &L, int tid, int NT)
{
    for (int i = tid; i < t.n; i += NT) {
        const int p = t.parent[i];
        const int page = (p == -1) ? T - 2 : t.age[p];
        for (int j = t.age[i]; j < page; j++) {
            atomicAdd(&L.nb[j], 1);
            atomicAdd(&L.nr[j], 1);
            atomicAdd(&L.nc[j], 1);
        }
        atomicAdd(&L.nr[page], 1);
        atomicAdd(&L.nc[page], 1);
        if (p == -1) atomicAdd(&L.nb[page], 1);
    }
}

// the node index (first state and top time of every node's branch,
// states.cpp:53-75) over the workgroup, one node per thread (blockDim.x ==
// MAXN == 256): a shuffle scan of the branch state counts in each wave,
// then the totals of the waves before (wsum[4], one per call); the caller
// synchronises before ni is read
__device__ inline void node_index_par(const TreeView &t, int T, NodeIndex &ni, int *wsum, int tid)
{
    int len = 0;
    if (tid < t.n) {
        ni.hi[tid] = t.top(tid, T);
        len = ni.hi[tid] - t.age[tid] + 1;
    }
    const int lane = tid & 63;
    int v = len;
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(v, off);
        if (lane >= off) v += u;
    }
    if (lane == 63) wsum[tid >> 6] = v;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < (tid >> 6); w++) base += wsum[w];
    if (tid < t.n) ni.first[tid] = base + v - len;
}

__device__ inline int node_of_state(const NodeIndex &ni, int n, int k)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (ni.first[mid] <= k) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// The coefficient planes of one block, written in the run's precision:
// FP32 runs keep only the FP32 planes (the same values as an FP64 plane
// rounded once)
struct PlaneOut {
    AW_GLOBAL double *p64;
    AW_GLOBAL float *p32;
    int RW;
    __device__ void put(int plane, int p, double v) const
    {
        if (p32) p32[(size_t)plane * RW + p] = (float)v;
        else p64[(size_t)plane * RW + p] = v;
    }
};

// Three sums over a 256-thread workgroup in a fixed order (a butterfly in
// each wave, then the four wave sums in wave order), so that every run adds
// the same terms in the same order; every thread gets the totals.
__device__ inline void block_sums3(double (&v)[3], double *red)
{
#pragma unroll
    for (int x = 0; x < 3; x++)
        for (int off = 32; off > 0; off >>= 1) v[x] += __shfl_xor(v[x], off);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int x = 0; x < 3; x++) red[4 * x + w] = v[x];
    __syncthreads();
#pragma unroll
    for (int x = 0; x < 3; x++) v[x] = ((red[4 * x] + red[4 * x + 1]) + red[4 * x + 2]) + red[4 * x + 3];
}

// Bound by its vector instructions (half of the cycles) and the barriers between
// its short phases; what it writes is 25 KB a block.  A table of all same-branch
// entries (20 KB) and emission terms per state (48 bytes) took it from 11.2 to
// 16.4 ms on the 256-instance batch (407000 blocks): the traceback forms the
// entries from X (engine.h), the emission terms depend on times only.
// At most 95 VGPRs: five waves per SIMD, without a spill.
__global__ __launch_bounds__(256, 5) void k_prep_b(const DevInst *__restrict__ D,
                                                const int *__restrict__ blkoff, int ninst)
{
    __shared__ PrepShared sh;
    const int inst = find_owner(blkoff, ninst, (int)blockIdx.x);
    const DevInst &d = D[inst];
    if (d.hostprep) return;   // uniform over the workgroup
    const int b = blockIdx.x - blkoff[inst];
    const int tid = threadIdx.x, NT = blockDim.x;
    const int T = d.T, N = d.N, T1 = T - 1;
    const int R = d.R, RW = 64 * R;

    if (tid == 0) sh.M = *d.model;
    for (int i = tid; i < N; i += NT) {
        size_t x = (size_t)b * N + i;
        sh.par[i] = gp(d.parent)[x];
        sh.ch0[i] = gp(d.c0)[x];
        sh.ch1[i] = gp(d.c1)[x];
        sh.ag[i] = gp(d.age)[x];
        if (b > 0) {
            size_t y = (size_t)(b - 1) * N + i;
            sh.ppar[i] = gp(d.parent)[y];
            sh.pch0[i] = gp(d.c0)[y];
            sh.pch1[i] = gp(d.c1)[y];
            sh.pag[i] = gp(d.age)[y];
            sh.map[i] = gp(d.map)[x];
        }
    }
    __syncthreads();
    TreeView t{N, -1, sh.par, sh.ch0, sh.ch1, sh.ag};
    TreeView pt{N, -1, sh.ppar, sh.pch0, sh.pch1, sh.pag};
    Spr spr{0, 0, 0, 0};
    if (b > 0) spr = Spr{gp(d.spr)[4 * b], gp(d.spr)[4 * b + 1], gp(d.spr)[4 * b + 2], gp(d.spr)[4 * b + 3]};
    // roots, zeroed lineage counts
    for (int i = tid; i < N; i += NT) {
        if (sh.par[i] == -1) sh.root = i;
        if (b > 0 && sh.ppar[i] == -1) sh.proot = i;
    }
    for (int i = tid; i < MAXT; i += NT) {
        sh.L.nb[i] = sh.L.nr[i] = sh.L.nc[i] = 0;
        sh.PL.nb[i] = sh.PL.nr[i] = sh.PL.nc[i] = 0;
    }
    __syncthreads();
    t.root = sh.root;
    pt.root = (b > 0) ? sh.proot : -1;
    lineages_par(t, T, sh.L, tid, NT);
    if (b > 0) lineages_par(pt, T, sh.PL, tid, NT);
    node_index_par(t, T, sh.ni, sh.wsum, tid);
    if (b > 0) node_index_par(pt, T, sh.pni, sh.wsum + 4, tid);
    if (tid == 0) {
        sh.L.nb[T - 1] = 1;
        sh.PL.nb[T - 1] = 1;
    }
    // node levels for the level-synchronous pruning of the emissions: depth
    // (root 0) by walking up to the root, height (leaves 0) by walking up
    // from every leaf and raising each ancestor's height to its distance
    // (integer LDS atomics); every walk is bounded by N
    for (int i = tid; i < N; i += NT) sh.hgt[i] = 0;
    __syncthreads();
    for (int j = tid; j < N; j += NT) {
        int dd = 0;
        for (int p = sh.par[j]; p != -1 && dd < N; p = sh.par[p]) dd++;
        sh.dep[j] = dd;
        if (sh.ch0[j] == -1) {
            int k = 1;
            for (int p = sh.par[j]; p != -1 && k <= N; p = sh.par[p], k++) atomicMax(&sh.hgt[p], k);
        }
    }
    // the block's tree lengths, fixed-order sums over the workgroup (one
    // node per thread): get_treelen of this tree (calc_trans) and of the
    // tree before (the switch), and the emissions' branch-length sum with
    // its minimum branch length (emit.cpp:778-819)
    double lens[3] = {0.0, 0.0, 0.0};
    {
        const double *tm_ = sh.M.times;
        const double mintime = tm_[1] * .1;
        if (tid < N) {
            const int p = sh.par[tid];
            if (p != -1) {
                lens[0] = tm_[sh.ag[p]] - tm_[sh.ag[tid]];
                lens[1] = fmax(tm_[sh.ag[p]] - tm_[sh.ag[tid]], mintime);
            }
            const int pp = (b > 0) ? sh.ppar[tid] : -1;
            if (pp != -1) lens[2] = tm_[sh.pag[pp]] - tm_[sh.pag[tid]];
        }
        block_sums3(lens, sh.red);   // also completes the levels
    }
    for (int i = tid; i < N; i += NT) gp(d.order)[(size_t)b * N + i] = sh.hgt[i] | (sh.dep[i] << 16);
    __syncthreads();
    // TransMatrix vectors (calc_trans) split over the workgroup with the
    // sequential version's expressions: the rate prefix in time order on
    // one thread, the per-time terms one thread each, the running logadd of
    // lnB as a prefix sum of exponentials.  Meanwhile one thread computes
    // the switch context's sums (calc_recoal_sums and friends).
    if (tid == 0) sh.mainlen = lens[1];
    if (tid == 128) gp(d.roots)[b] = sh.root;
    if (tid == 192 && b > 0) switch_ctx_sums(pt, sh.M, sh.PL, spr, lens[2], sh.cx);
    {
        const Model &M = sh.M;
        double *rates = sh.rates + 1, *C = sh.Cs + 2;
        if (tid == 64) rates[-1] = 0.0;
        for (int i = tid; i < 2 * T - 1; i += NT)
            rates[i] = M.csteps[i] * sh.L.nb[i / 2] / (2.0 * M.pop[i / 2]);
        __syncthreads();
        if (tid == 64) {
            C[-2] = 0.0;
            C[-1] = 0.0;
            double c = 0.0;
            for (int b2 = 0; b2 < 2 * T - 1; b2++) {
                c = c + rates[b2];
                C[b2] = c;
            }
        }
        __syncthreads();
        TransVec &tv = sh.tv;
        const int ri = t.age[t.root];
        const double root_age = M.times[ri];
        const double len = lens[0];
        for (int bb = tid; bb < T; bb += NT) {
            tv.D[bb] = tv.E[bb] = tv.lnB[bb] = tv.lnE2[bb] = tv.lnNegG1[bb] = 0.0;
            tv.G2[bb] = tv.G3[bb] = tv.lnG4[bb] = tv.norecombs[bb] = 0.0;
            if (bb >= T - 1) continue;
            const int nb = sh.L.nb[bb], nr = sh.L.nr[bb], nc = sh.L.nc[bb];
            double len2 = len + M.times[bb];
            double len2_b;
            if (bb > ri) {
                len2 += M.times[bb] - root_age;
                len2_b = len2 + M.steps[bb];
            } else {
                len2_b = len2 + M.steps[ri];
            }
            sh.lnBt[bb] = C[2 * bb - 1] + log(M.steps[bb] * (nb + 1.0) / (nr + 1.0));
            double e2 = -C[2 * bb - 2] + (bb < T - 2 ? log(1 - exp(-rates[2 * bb] - rates[2 * bb - 1])) : 0.0);
            tv.lnE2[bb] = e2;
            tv.lnG4[bb] = e2;
            tv.lnNegG1[bb] = C[2 * bb - 1] +
                log(-M.steps[bb] * ((nb / (nr + 1.0 + int(bb < ri))) - (nb + 1.0) / (nr + 1.0)));
            double q = (bb < T - 2 ? 1.0 - exp(-rates[2 * bb]) : 1.0);
            tv.G2[bb] = q * M.steps[bb] * (nb + 1.0) / (nr + 1.0);
            tv.G3[bb] = q * M.steps[bb] * (nb / (nr + 1.0 + int(bb < ri)));
            tv.D[bb] = (1.0 - exp(-M.rho * len2)) / len2_b;
            tv.E[bb] = 1.0 / nc;
            tv.norecombs[bb] = exp(-fmax(M.rho * len2, M.rho));
        }
        // the switch context's per-time recoalescence terms
        if (b > 0)
            for (int a = tid - 128; a >= 0 && a < T; a += NT)
                sh.cx.recoals[a] = sw_recoal(M, sh.PL, spr.rt, spr.ct, a, sh.cx.rpa);
        __syncthreads();
        // lnB[b] = logadd(lnB[b-1], term_b) (trans.cpp:26-115) as
        // tmax + log(sum of exp(term_k - tmax), k <= b): the same value up to
        // rounding; the running logadd on one thread when the terms span
        // more than exp's range
        double tmax = -INFINITY, tmin = INFINITY;
        for (int k = 0; k < T - 1; k++) {
            tmax = fmax(tmax, sh.lnBt[k]);
            tmin = fmin(tmin, sh.lnBt[k]);
        }
        if (tmax - tmin < 600.0) {
            for (int k = tid; k < T - 1; k += NT) sh.eexp[k] = exp(sh.lnBt[k] - tmax);
            __syncthreads();
            for (int bb = tid; bb < T - 1; bb += NT) {
                double sum = 0.0;
                for (int k = 0; k <= bb; k++) sum += sh.eexp[k];
                tv.lnB[bb] = tmax + log(sum);
            }
        } else if (tid == 0) {
            double lb = sh.lnBt[0];
            tv.lnB[0] = lb;
            for (int bb = 1; bb < T - 1; bb++) {
                lb = logadd(lb, sh.lnBt[bb]);
                tv.lnB[bb] = lb;
            }
        }
    }
    __syncthreads();
    t.root = sh.root;
    pt.root = (b > 0) ? sh.proot : -1;
    const Model &M = sh.M;
    const TransVec &tv = sh.tv;
    const int so = cp(d.soff)[b], S = cp(d.soff)[b + 1] - so;
    const PlaneOut coef{d.fp32 ? nullptr : gp(d.lcoef) + (size_t)b * NCOEF * RW,
                        d.fp32 ? gp(d.lcoef32) + (size_t)b * NCOEF * RW : nullptr, RW};
    auto info = gp(d.linfo) + (size_t)b * RW;
    auto det = gp(d.ldet) + (size_t)b * RW;

    // the factors of the planes that depend on the state's time only, each
    // the expression the per-state formulas below would evaluate
    for (int a = tid; a < T1; a += NT) {
        sh.eB[a] = exp(tv.lnB[a]);
        sh.eN[a] = exp(tv.lnNegG1[a]);
        sh.eE2[a] = exp(tv.lnE2[a]);
        sh.low[a] = a > 0 ? exp(tv.lnE2[a] + tv.lnB[a - 1]) : 0.0;
        emit_invariant(t, M, sh.mainlen, a, sh.inv[a], sh.inv_root[a]);
    }
    __syncthreads();   // per-time factors complete

    // Per-state planes.  For a target state (n, b) with c = age(n), the
    // reference's same-branch entry tmatrix2[a][k] = get_time(a,b,c,same) -
    // get_time(a,b,0,other) (sample_thread.cpp:210-226, trans.h:89-128)
    // factorises as
    //   a <  b:  D[a] (exp(lnB[a]) - exp(lnNegG1[a]) - B_{c-1}) * E[b] exp(lnE2[b])
    //   a >  b:  D[a] * E[b] (low_b + G2[b] - ct_b)
    //   a == b:  D[b] E[b] (low_b + G3[b] - ct_b) + norecombs[b]
    // with B_{c-1} = exp(lnB[c-1]), low_b = exp(lnE2[b] + lnB[b-1]) and
    // ct_b = exp(lnG4[b] + lnB[c-1]) (lnG4 = lnE2), so the branch-local
    // sum is a prefix sum (a < b) and a suffix sum (a > b) along the branch.
    for (int p = tid; p < RW; p += NT) {
        const int s = pos_state(p, R);
        double cf = 0, cd = 0, cg = 0, ck = 0, cj = 0, ce = 0, pr = 0;
        int inf = INFO_FIRST | INFO_LAST | 31;   // padding: time bin 31, whose TF is 0
        if (s < S) {
            const int n = node_of_state(sh.ni, N, s);
            const int a = sh.ag[n] + s - sh.ni.first[n];
            const int c = sh.ag[n], h = sh.ni.hi[n];
            const double Bc = c > 0 ? sh.eB[c - 1] : 0.0;
            const double low = sh.low[a];
            const double ct = c > 0 ? exp(tv.lnG4[a] + tv.lnB[c - 1]) : 0.0;
            cf = tv.D[a] * (sh.eB[a] - sh.eN[a] - Bc);
            cd = tv.D[a];
            cg = tv.E[a] * sh.eE2[a];
            ck = tv.E[a] * (low + tv.G2[a] - ct);
            // the diagonal (stay) entry dominates every state's value: it is
            // get_time(a, a, c, true) - get_time(a, a, 0, false), the
            // reference's tmatrix2 entry, in get_time's own expressions (its
            // low and c_term are low and ct above)
            const double term1 = tv.D[a] * tv.E[a];
            cj = (term1 * ((2 * (low + tv.G3[a])) - ct) + tv.norecombs[a]) -
                 term1 * (low + tv.G3[a]);
            ce = n == sh.root ? sh.inv_root[a] : sh.inv[a];
            if (b == 0) pr = prior_time(a, sh.L, M);
            inf = a | (a == c ? INFO_FIRST : 0) | (a == h ? INFO_LAST : 0) | INFO_VALID |
                  (c << 11) | (n << 16);
        }
        coef.put(CF, p, cf);
        coef.put(CD, p, cd);
        coef.put(CG, p, cg);
        coef.put(CK, p, ck);
        coef.put(CJ, p, cj);
        coef.put(CE, p, ce);
        coef.put(CRR, p, 0.0);
        coef.put(CCR, p, 0.0);
        coef.put(CDP, p, 0.0);
        det[p] = -1;
        info[p] = inf;
        if (b == 0) gp(d.lprior)[p] = pr;
    }

    // P(a -> b) on another branch (get_time), and the terms the traceback forms
    // the same-branch entries from (a table of all of those, 20 KB a block, was
    // a quarter of this kernel's time)
    auto vec = gp(d.tvec) + (size_t)b * time_vecs(T1);
    for (int x = tid; x < T1 * T1; x += NT) {
        const int a = x / T1, bb = x % T1;
        gp(d.tm)[(size_t)b * T1 * T1 + x] = tv.get_time(a, bb, 0, false);
        if (a < bb) vec[tv_x(T1) + x] = exp(tv.lnE2[bb] + tv.lnB[a]);
    }
    for (int a = tid; a < T1; a += NT) {
        vec[TV_D * T1 + a] = tv.D[a];
        vec[TV_E * T1 + a] = tv.E[a];
        vec[TV_NORECOMBS * T1 + a] = tv.norecombs[a];
        vec[TV_Y * T1 + a] = 0.0;
        if (a == 0) vec[tv_minage(T1)] = 0.0;
    }

    if (b == 0) return;
    __syncthreads();   // planes cleared before the switch entries are set

    // switch matrix from block b-1 (calc_transition_probs_switch), entries
    // of the previous block's states at their lane-run positions
    const int so1 = cp(d.soff)[b - 1], S1 = so - so1;
    for (int j = tid; j < S1; j += NT) {
        int n1 = node_of_state(sh.pni, N, j);
        int t1 = sh.pag[n1] + j - sh.pni.first[n1];
        int tgt = sw_determ(pt, t, sh.ni, spr, sh.map, n1, t1);
        const int p = lane_pos(j, R);
        det[p] = tgt;
        coef.put(CDP, p, tgt >= 0 ? sw_determprob(pt, M, sh.PL, spr, sh.cx, n1, t1) : 0.0);
    }
    if (tid == 0) {
        int rs = lookup(pt, sh.pni, spr.rn, spr.rt);
        int cs = lookup(pt, sh.pni, spr.cn, spr.ct);
        sh.recombsrc = rs;
        sh.recoalsrc = cs;
        gp(d.srcs)[2 * b] = rs;
        gp(d.srcs)[2 * b + 1] = cs;
        if (cs != -1) {
            int node1 = spr.cn;
            int last_parent = sh.ppar[spr.rn];
            if (last_parent == node1) {
                int other = (sh.pch1[last_parent] == spr.rn) ? sh.pch0[last_parent] : sh.pch1[last_parent];
                sh.node3 = sh.map[other];
            } else {
                sh.node3 = sh.map[node1];
            }
            sh.rparent = sh.par[sh.map[spr.rn]];
        }
    }
    __syncthreads();
    if (tid == 0 && sh.recombsrc != -1) {
        // get_recomb_transition_switch: stay and escape targets
        int parent = sh.ppar[spr.rn];
        int time2 = sh.pag[parent];
        int other = pt.sibling(spr.rn);
        int node2 = (other == spr.cn) ? sh.par[sh.map[other]] : sh.map[other];
        int stay = lookup(t, sh.ni, sh.map[spr.rn], spr.rt);
        int esc = lookup(t, sh.ni, node2, time2);
        if (stay != -1)
            coef.put(CRR, lane_pos(stay, R), sw_recomb_recoal(
                pt, M, sh.PL, spr, spr.ct, spr.rn, spr.rt, sh.cx.rpa, sh.cx.last_len));
        if (esc != -1)
            coef.put(CRR, lane_pos(esc, R), sw_recomb_recoal(
                pt, M, sh.PL, spr, spr.ct, spr.rn, spr.rt, spr.rt, sh.cx.last_len));
    }
    if (sh.recoalsrc != -1) {
        const int time1 = spr.ct;
        const int mrn = sh.map[spr.rn];
        for (int k = tid; k < S; k += NT) {
            int n2 = node_of_state(sh.ni, N, k);
            int t2 = sh.ag[n2] + k - sh.ni.first[n2];
            if (!((n2 == mrn && t2 >= spr.rt) || (n2 == sh.node3 && t2 == time1) ||
                  (n2 == sh.rparent && t2 == time1)))
                continue;
            coef.put(CCR, lane_pos(k, R), sw_recomb_recoal(pt, M, sh.PL, spr, t2, spr.cn, spr.ct,
                                                           sh.cx.rpa, sh.cx.last_len));
        }
    }
}

//===========================================================================
// emissions of variant columns, written as lane-run rows

// Felsenstein pruning (pruning) by one wave, level by level: the inner
// partials of all nodes of one height at once (children first), then the
// outer partials of all nodes of one depth (parents first).  Every node's
// arithmetic is the sequential version's, so the results are identical;
// one wave's LDS operations run in order, so a level sees the one before.
__device__ inline void pruning_wave(const TreeView &t, const int *lvl, const char *bases,
                                    const double *muts, const double *nomuts, double *inner,
                                    double *outer)
{
    const int lane = threadIdx.x;
    int hmax = 0, dmax = 0;
    for (int j = lane; j < t.n; j += 64) {
        hmax = max(hmax, lvl[j] & 0xffff);
        dmax = max(dmax, lvl[j] >> 16);
    }
    for (int off = 32; off > 0; off >>= 1) {
        hmax = max(hmax, __shfl_xor(hmax, off));
        dmax = max(dmax, __shfl_xor(dmax, off));
    }
    for (int h = 0; h <= hmax; h++) {
        for (int j = lane; j < t.n; j += 64) {
            if ((lvl[j] & 0xffff) != h) continue;
            if (t.c0[j] == -1) {
                leaf_partial(bases[j], inner + 4 * j);
                continue;
            }
            const int c1 = t.c0[j], c2 = t.c1[j];
            for (int a = 0; a < 4; a++) {
                double p1 = 0.0, p2 = 0.0;
                for (int b = 0; b < 4; b++) {
                    if (a == b) {
                        p1 += inner[4 * c1 + b] * nomuts[c1];
                        p2 += inner[4 * c2 + b] * nomuts[c2];
                    } else {
                        p1 += inner[4 * c1 + b] * muts[c1];
                        p2 += inner[4 * c2 + b] * muts[c2];
                    }
                }
                inner[4 * j + a] = p1 * p2;
            }
        }
        __syncthreads();
    }
    for (int dd = 0; dd <= dmax; dd++) {
        for (int j = lane; j < t.n; j += 64) {
            if ((lvl[j] >> 16) != dd) continue;
            if (j == t.root) {
                for (int a = 0; a < 4; a++) outer[4 * j + a] = 1.0;
                continue;
            }
            const int sib = t.sibling(j);
            const int parent = t.parent[j];
            for (int a = 0; a < 4; a++) {
                double p1 = 0.0, p2 = 0.0;
                for (int b = 0; b < 4; b++) {
                    const double ms = (a == b) ? nomuts[sib] : muts[sib];
                    p1 += inner[4 * sib + b] * ms;
                    if (parent != t.root) {
                        const double mp = (a == b) ? nomuts[parent] : muts[parent];
                        p2 += outer[4 * parent + b] * mp;
                    }
                }
                outer[4 * j + a] = (parent != t.root) ? p1 * p2 : p1;
            }
        }
        __syncthreads();
    }
}

// LDS of k_var_emit_b for trees of up to n nodes: the partials and branch
// probabilities (FP64), the tree arrays and levels, the leaf bases.  Sized
// by the batch's largest tree, so that small trees leave room for more
// waves on a CU.
inline size_t var_emit_lds(int n)
{
    return sizeof(double) * (10 * (size_t)n + 4) + sizeof(int) * 5 * (size_t)n + n;
}

__global__ __launch_bounds__(64) void k_var_emit_b(const DevInst *__restrict__ D,
                                                   const int *__restrict__ voff, int ninst,
                                                   int nmax)
{
    extern __shared__ double ve_dyn[];
    double *inner = ve_dyn, *outer = inner + 4 * nmax;
    double *muts = outer + 4 * nmax, *nomuts = muts + nmax, *in2 = nomuts + nmax;
    int *par = (int *)(in2 + 4), *ch0 = par + nmax, *ch1 = ch0 + nmax, *ag = ch1 + nmax,
        *lvl = ag + nmax;
    char *bases = (char *)(lvl + nmax);
    const int inst = find_owner(voff, ninst, (int)blockIdx.x);
    const DevInst &d = D[inst];
    if (d.hostprep) return;   // uniform over the wave
    const int v = blockIdx.x - voff[inst];
    const int lane = threadIdx.x;
    const int N = d.N, R = d.R, RW = 64 * R;
    const int col = gp(d.vcol)[v];
    const int b = find_owner(cp(d.bstart), d.B, col);
    const int nleaves = (N + 1) / 2;
    for (int i = lane; i < N; i += 64) {
        size_t x = (size_t)b * N + i;
        par[i] = gp(d.parent)[x];
        ch0[i] = gp(d.c0)[x];
        ch1[i] = gp(d.c1)[x];
        ag[i] = gp(d.age)[x];
        lvl[i] = gp(d.order)[x];
        if (i < nleaves) bases[i] = gp(d.seq)[(size_t)i * d.L + col];
    }
    __syncthreads();
    const int root = gp(d.roots)[b], T = d.T;
    // branch mutation probabilities for the pruning (prob_tree_mutation)
    const auto pm = gp(d.pmut);
    for (int i = lane; i < N; i += 64) {
        const auto e = pm + (i != root ? mut_entry(min(ag[par[i]], T - 1), ag[i], T) : 0);
        muts[i] = i != root ? e[0] : 0.0;
        nomuts[i] = i != root ? e[1] : 0.0;
    }
    __syncthreads();
    {
        TreeView t{N, root, par, ch0, ch1, ag};
        pruning_wave(t, lvl, bases, muts, nomuts, inner, outer);
        if (lane == 0) leaf_partial(gp(d.seq)[(size_t)nleaves * d.L + col], in2);
    }
    __syncthreads();
    const int S = cp(d.soff)[b + 1] - cp(d.soff)[b];
    auto row = gp(d.vemit) + (size_t)v * RW;
    const auto info = gp(d.linfo) + (size_t)b * RW;
    for (int p = lane; p < RW; p += 64) {
        const int k = pos_state(p, R);
        double e = 0.0;
        if (k < S) {
            // the new leaf's branch, and the two parts of the node's branch
            const int x = info[p], n = info_node(x), a = x & INFO_TIME;
            const int top = n != root ? min(ag[par[n]], T - 1) : a;
            const auto e0 = pm + mut_entry(T, a, T), e1 = pm + mut_entry(a, ag[n], T),
                       e2 = pm + mut_entry(top, a, T);
            const double mut[3] = {e0[0], e1[0], e2[0]}, nomut[3] = {e0[1], e1[1], e2[1]};
            e = emit_variant(in2, inner + 4 * n, outer + 4 * n, n == root, mut, nomut);
        }
        row[p] = e;
    }
}

// log-likelihood: sum of log column normalisers (16 waves: 0.42 ms for 500000
// columns; 4 waves took 1.1)
__global__ __launch_bounds__(1024) void k_lnl_b(const DevInst *__restrict__ D,
                                               const int *__restrict__ list)
{
    __shared__ double part[1024];
    const DevInst &d = D[list[blockIdx.x]];
    double s = 0.0;
    for (int c = threadIdx.x; c < d.L; c += 1024) s += log(gp(d.norms)[c]);
    part[threadIdx.x] = s;
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if (threadIdx.x < off) part[threadIdx.x] += part[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) *d.lnl = part[0];
}

//===========================================================================
// host driver

namespace {

// supported states-per-lane counts (one kernel instantiation each)
constexpr int NRV = 8;
constexpr int RVALS[NRV] = {1, 2, 4, 6, 8, 12, 16, 32};

// Device-wide state, initialised once per process.
struct Ctx {
    bool init = false;
    int dev = 0;
    hipDeviceProp_t prop{};
};

Ctx &ctx()
{
    static Ctx c;
    return c;
}

int ctx_init()
{
    static std::mutex mu;
    std::lock_guard<std::mutex> lk(mu);
    Ctx &c = ctx();
    if (c.init) return 0;
    HIP_OK(hipGetDevice(&c.dev));
    HIP_OK(hipGetDeviceProperties(&c.prop, c.dev));
    c.init = true;
    return 0;
}

// The upload, run, tuning and copy-out methods of a Batch hold a lock for
// their whole device work.  By default it is one process-wide lock, so
// batches driven from different host threads run one after another; a
// batch set concurrent (the server's) holds a lock of its own and runs
// beside the others.  Concurrent batches are safe because no stream ever
// waits on another stream's event (streams are joined by the host), so no
// hardware queue can hold a wait ahead of the work it waits for, and the
// kernels' dynamic-LDS limits only rise (set_lds_limit).  Recursive because
// run() uploads a batch that is not yet uploaded.
std::recursive_mutex &device_mutex()
{
    static std::recursive_mutex mu;
    return mu;
}
#define DEVICE_LOCK std::lock_guard<std::recursive_mutex> device_lock_(device_mutex())

//===========================================================================
// table rows for the host: columns [c0, c0 + n) of a lane-run table, `pitch`
// states each, in state order and FP64, one wave per column.  `out` is pinned
// host memory, which the stores reach over the link in whole lines (a lane's
// states lie apart in the row instead, whose second reader finds it in cache);
// the host then copies rows of S states.  Copying the padded rows out and
// picking the states on the host took 18 ms of a call's 23 (20011 columns, 19
// haplotypes, FP32); this way the call takes 11.7 ms.
template <class Real>
__global__ __launch_bounds__(256) void k_rows_out(const void *alpha, int c0, int n, int R, int pitch,
                                                  double *__restrict__ out)
{
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (c >= n) return;
    const Real *row = (const Real *)alpha + (size_t)(c0 + c) * (64 * R);
    double *o = out + (size_t)c * pitch;
    for (int s = threadIdx.x & 63; s < pitch; s += 64) o[s] = (double)row[lane_pos(s, R)];
}

// The batch's streams: main carries every stage; side carries only the
// traceback of the instances whose forward is final (their chains and
// re-runs, driven by a helper host thread) while the forward
// re-runs of others continue on main.  The two are joined by the host
// (stream synchronisation), never by a stream waiting on an event.
struct Streams {
    bool init = false;
    int dev = 0;   // theirs
    hipStream_t main = nullptr, side = nullptr;
    hipEvent_t ev[10];
    int create()
    {
        if (init) return 0;
        HIP_OK(hipGetDevice(&dev));
        HIP_OK(hipStreamCreateWithFlags(&main, hipStreamNonBlocking));
        HIP_OK(hipStreamCreateWithFlags(&side, hipStreamNonBlocking));
        for (auto &e : ev) HIP_OK(hipEventCreate(&e));
        init = true;
        return 0;
    }
    void destroy()
    {
        if (!init) return;
        (void)hipStreamSynchronize(main);
        (void)hipStreamSynchronize(side);
        for (auto &e : ev) (void)hipEventDestroy(e);
        (void)hipStreamDestroy(main);
        (void)hipStreamDestroy(side);
        init = false;
    }
};

// A caller-provided device region that buffers are carved from instead of
// hipMalloc (the no-allocation entry point); reset() before each use.
struct Arena {
    char *base = nullptr;
    size_t cap = 0, used = 0;
    void reset() { used = 0; }
};

// grow-only device buffer; with an arena it takes its memory from the arena
// (and never frees it)
struct DevBuf {
    char *p = nullptr;
    size_t cap = 0;
    Arena *arena = nullptr;
    int ensure(size_t n)
    {
        if (n <= cap) return 0;
        if (arena) {
            const size_t off = (arena->used + 255) & ~size_t(255);
            if (off + n > arena->cap) {
                fprintf(stderr,
                        "argweaver_amd: the instance needs more than the %zu bytes of the "
                        "no-allocation workspace\n",
                        arena->cap);
                return 1;
            }
            p = arena->base + off;
            cap = n;
            arena->used = off + n;
            return 0;
        }
        if (p) HIP_OK(hipFree(p));
        p = nullptr;
        cap = 0;
        HIP_OK(device_malloc((void **)&p, n));
        cap = n;
        return 0;
    }
    void release()
    {
        if (p && !arena) (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
};

// bump allocator over a size plan: first pass counts, second pass assigns
struct Plan {
    size_t used = 0;
    char *base = nullptr;
    template <class X>
    X *take(size_t n)
    {
        size_t off = (used + 255) & ~size_t(255);
        used = off + std::max<size_t>(n, 1) * sizeof(X);
        return base ? reinterpret_cast<X *>(base + off) : nullptr;
    }
};

// smallest supported states-per-lane count covering Smax states
int lanes_per_state_r(int Smax)
{
    for (int R : RVALS)
        if (64 * R >= Smax) return R;
    return -1;
}

}  // namespace

// The dynamic-LDS limit of a kernel only ever rises, under one lock: a
// batch on another host thread that set a larger limit for the same kernel
// is never undercut between its attribute call and its launch.
int set_lds_limit(const void *kern, size_t sh)
{
    static std::mutex mu;
    static std::map<const void *, size_t> cur;
    std::lock_guard<std::mutex> lk(mu);
    size_t &c = cur[kern];
    if (sh <= c) return 0;
    HIP_OK(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh));
    c = sh;
    return 0;
}

namespace {
std::mutex stage_mu;
std::vector<HostStage *> &stage_pool()
{
    // never destroyed (see run_instance)
    static auto *v = new std::vector<HostStage *>();
    return *v;
}
void free_stage(HostStage *s)
{
    for (auto &e : s->filled) (void)hipEventDestroy(e);
    if (s->dbuf) (void)hipFree(s->dbuf);
    (void)hipHostFree(s->p);
    delete s;
}
}  // namespace

HostStage *take_stage()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    {
        std::lock_guard<std::mutex> lk(stage_mu);
        auto &v = stage_pool();
        for (size_t i = 0; i < v.size(); i++)
            if (v[i]->dev == dev) {
                HostStage *s = v[i];
                v.erase(v.begin() + i);
                return s;
            }
    }
    HostStage *s = new HostStage();
    s->dev = dev;
    hipError_t e = hipHostMalloc((void **)&s->p, 2 * HostStage::HALF, hipHostMallocDefault);
    int events = 0;
    while (e == hipSuccess && events < 2) {
        e = hipEventCreateWithFlags(&s->filled[events], hipEventDisableTiming);
        if (e == hipSuccess) events++;
    }
    if (e == hipSuccess) return s;
    fprintf(stderr, "argweaver_amd: pinned staging memory: %s\n", hipGetErrorString(e));
    while (events > 0) (void)hipEventDestroy(s->filled[--events]);
    if (s->p) (void)hipHostFree(s->p);
    delete s;
    return nullptr;
}

void give_stage(HostStage *s)
{
    s->trim();
    {
        std::lock_guard<std::mutex> lk(stage_mu);
        if (stage_pool().size() < STAGE_KEEP) {
            stage_pool().push_back(s);
            return;
        }
    }
    free_stage(s);
}

size_t idle_stage_bytes()
{
    std::lock_guard<std::mutex> lk(stage_mu);
    size_t n = 0;
    for (const HostStage *s : stage_pool()) n += s->dcap;
    return n;
}

bool free_idle_stage_memory()
{
    std::lock_guard<std::mutex> lk(stage_mu);
    bool any = false;
    for (HostStage *s : stage_pool()) any |= s->drop();
    return any;
}

struct Batch::Impl {
    std::vector<HostInstance> hosts;
    std::vector<std::vector<double>> us, priors;
    std::vector<std::vector<int>> Sv;
    std::vector<std::vector<int>> soff;
    std::vector<DevInst> h;
    std::vector<long long> W;
    std::vector<double> lnl;
    std::vector<int> nvar;
    std::vector<Chunk> chunks;
    std::vector<int> tlist0, tlist1;   // host tile lists of the two launches
    DevBuf in, work, tab, aux, vbuf, tiles, fwb;
    Arena arena;   // base == nullptr: buffers come from hipMalloc
    Streams st;
    HostStage *stage = nullptr;   // a workspace batch's own
    DevInst *dD = nullptr;
    long long *d_coloff = nullptr;
    double *d_lnl = nullptr;   // [n] the instances' log-likelihoods
    int *d_blkoff = nullptr, *d_voff = nullptr, *d_nvar = nullptr, *d_list = nullptr;
    // traceback tiles: start / end states of their chains, re-run lists and
    // results
    int *d_ostart = nullptr, *d_oend = nullptr;
    int *d_ridx = nullptr, *d_rk1 = nullptr, *d_rres = nullptr;
    int *d_tlist = nullptr;   // [2 nch] tile lists of the two launches
    // instances with 32 states per lane run in kernel symbols of their own;
    // the LDS bytes of those symbols' forward and traceback launches
    bool any_big = false;
    size_t shf_big = 0, sht = 0, sht_big = 0;
    Chunk *d_chunks = nullptr;
    FwTile *d_fwt = nullptr, *d_fwre = nullptr;
    char *d_bnd = nullptr;
    double *d_bnorm = nullptr;
    int *d_fidx = nullptr, *d_fflag = nullptr;
    bool uploaded = false;
    Precision prec_done = Precision::FP64;
    bool own_lock = false;     // set_concurrent: this batch's own lock
    std::recursive_mutex mu;

    ~Impl()
    {
        st.destroy();
        if (stage) give_stage(stage);
        in.release();
        work.release();
        tab.release();
        aux.release();
        vbuf.release();
        tiles.release();
        fwb.release();
    }
};

// the lock of a batch's device work (see device_mutex)
#define BATCH_LOCK \
    std::lock_guard<std::recursive_mutex> batch_lock_(impl_->own_lock ? impl_->mu : device_mutex())

Batch::Batch() : impl_(new Impl) {}
void Batch::set_concurrent(bool on) { impl_->own_lock = on; }
Batch::~Batch() { delete impl_; }
int Batch::size() const { return (int)impl_->hosts.size(); }

void Batch::use_workspace(void *base, size_t cap)
{
    Impl &m = *impl_;
    m.arena.base = static_cast<char *>(base);
    m.arena.cap = cap;
    m.arena.reset();
    for (DevBuf *b : {&m.in, &m.work, &m.tab, &m.aux, &m.vbuf, &m.tiles, &m.fwb}) {
        b->release();
        b->arena = &m.arena;
    }
}

int Batch::init_streams()
{
    if (ctx_init()) return 1;
    if (impl_->st.create()) return 1;
    if (impl_->arena.base && !impl_->stage) impl_->stage = take_stage();
    return impl_->arena.base && !impl_->stage;
}

void Batch::clear()
{
    Impl &m = *impl_;
    if (m.arena.base) {
        // a workspace batch carves its buffers again from the start
        m.arena.reset();
        for (DevBuf *b : {&m.in, &m.work, &m.tab, &m.aux, &m.vbuf, &m.tiles, &m.fwb}) {
            b->p = nullptr;
            b->cap = 0;
        }
    }
    m.hosts.clear();
    m.us.clear();
    m.priors.clear();
    m.Sv.clear();
    m.soff.clear();
    m.h.clear();
    m.W.clear();
    m.lnl.clear();
    m.nvar.clear();
    m.chunks.clear();
    m.uploaded = false;
}
double Batch::lnl(int i) const { return impl_->lnl[i]; }
long long Batch::W(int i) const { return impl_->W[i]; }

int Batch::add(const HostInstance &hi, const double *u, const double *prior)
{
    return add(HostInstance(hi), u, prior);
}

int Batch::add(HostInstance &&hin, const double *u, const double *prior)
{
    Impl &m = *impl_;
    // upload() releases the host rows of the instances it copied, so a batch
    // that was uploaded takes no more instances until clear()
    if (m.uploaded) {
        fprintf(stderr, "argweaver_amd: Batch::add after upload (clear() the batch first)\n");
        return -1;
    }
    std::string why;
    if (instance_supported(hin, &why)) {
        fprintf(stderr, "argweaver_amd: Batch::add refused the instance: %s\n", why.c_str());
        return -1;
    }
    m.hosts.push_back(std::move(hin));
    const HostInstance &hi = m.hosts.back();
    m.us.emplace_back();
    if (u) m.us.back().assign(u, u + hi.ft.seqlen);
    m.priors.emplace_back();
    std::vector<int> Sv;
    long long W = 0;
    if (hi.prep) {
        Sv = hi.prep->S;
        for (int b = 0; b < hi.ft.nblocks; b++) W += (long long)Sv[b] * hi.ft.len[b];
    } else {
        W = instance_states(hi.ft, hi.model.T, &Sv);
    }
    if (prior) m.priors.back().assign(prior, prior + Sv[0]);
    m.W.push_back(W);
    m.Sv.push_back(Sv);
    m.uploaded = false;
    return (int)m.hosts.size() - 1;
}

// an instance's sizes, Sv its states per block
static int shape_instance(const HostInstance &hi, const std::vector<int> &Sv, DevInst &d)
{
    const FlatTrees &ft = hi.ft;
    d.hostprep = hi.prep ? 1 : 0;
    d.last_state = hi.last_state;
    d.T = hi.model.T; d.N = ft.nnodes; d.B = ft.nblocks; d.L = ft.seqlen;
    d.nrows = (int)hi.rows.size();
    d.Smax = 1;
    for (int S : Sv) d.Smax = std::max(d.Smax, S);
    d.R = lanes_per_state_r(d.Smax);
    if (d.R > 0) return 0;
    fprintf(stderr, "argweaver_amd: %d states per block exceed the %d of one wave\n", d.Smax,
            64 * RVALS[NRV - 1]);
    return 1;
}

// An instance's device arrays: what is uploaded, what a run fills, its forward
// table, and its variant rows, whose number a run finds.  instance_bytes adds
// the same plans up.
static void plan_inputs(Plan &p, DevInst &d)
{
    const int B = d.B, N = d.N, L = d.L;
    d.model = p.take<Model>(1);
    d.parent = p.take<int>((size_t)B * N);
    d.c0 = p.take<int>((size_t)B * N);
    d.c1 = p.take<int>((size_t)B * N);
    d.age = p.take<int>((size_t)B * N);
    d.map = p.take<int>((size_t)B * N);
    d.spr = p.take<int>(4 * (size_t)B);
    d.bstart = p.take<int>(B);
    d.blen = p.take<int>(B);
    d.soff = p.take<int>(B + 1);
    d.seq = p.take<char>((size_t)d.nrows * L);
    d.u = p.take<double>(L);
}

static void plan_work(Plan &p, DevInst &d, bool fp32)
{
    const int B = d.B, N = d.N, L = d.L, T1 = d.T - 1, RW = 64 * d.R;
    d.vflag = p.take<int>(L);
    d.cls = p.take<int>(L);
    d.vcol = p.take<int>(L);
    d.order = p.take<int>((size_t)B * N);
    d.roots = p.take<int>(B);
    d.pmut = p.take<double>(mut_entry(d.T + 1, 0, d.T));
    d.tm = p.take<double>((size_t)B * T1 * T1);
    d.tvec = p.take<double>((size_t)B * time_vecs(T1));
    d.srcs = p.take<int>(2 * (size_t)B);
    d.linfo = p.take<int>((size_t)B * RW);
    // coefficient planes in the run's precision only
    d.fp32 = fp32 ? 1 : 0;
    d.lcoef = fp32 ? nullptr : p.take<double>((size_t)B * NCOEF * RW);
    d.lcoef32 = fp32 ? p.take<float>((size_t)B * NCOEF * RW) : nullptr;
    d.ldet = p.take<int>((size_t)B * RW);
    d.pred = p.take<unsigned short>((size_t)B * RW);
    d.lprior = p.take<double>(RW);
    d.norms = p.take<double>(L);
    d.cut = p.take<unsigned>(L / 32 + 1);
    d.path = p.take<int>(L);
}

static void plan_table(Plan &p, DevInst &d)
{
    d.alpha = p.take<char>((size_t)d.L * 64 * d.R * (d.fp32 ? sizeof(float) : sizeof(double)));
}

static void plan_variants(Plan &p, DevInst &d)
{
    d.vemit = p.take<double>((size_t)std::max(d.nvar, 1) * 64 * d.R);
}

size_t instance_bytes(const HostInstance &hi, Precision prec, int nvar)
{
    DevInst d{};
    std::vector<int> Sv;
    if (hi.prep) Sv = hi.prep->S;
    else instance_states(hi.ft, hi.model.T, &Sv);
    if (shape_instance(hi, Sv, d)) return 0;
    d.nvar = nvar;
    Plan p;
    plan_inputs(p, d);
    plan_work(p, d, prec == Precision::FP32);
    plan_table(p, d);
    plan_variants(p, d);
    return p.used;
}

// Inputs: trees, sequences, uniforms and the model of every instance.
int Batch::upload()
{
    BATCH_LOCK;
    if (ctx_init()) return 1;
    Impl &m = *impl_;
    if (m.st.create()) return 1;
    Streams &c = m.st;
    const OnDevice on(c.dev);
    const int n = (int)m.hosts.size();
    m.h.assign(n, DevInst{});
    m.soff.assign(n, {});
    m.lnl.assign(n, 0.0);
    m.nvar.assign(n, 0);
    const StageUse use(m.stage);
    if (!use.s) return 1;
    Uploader up(*use.s, c.main);
    for (int pass = 0; pass < 2; pass++) {
        Plan p;
        p.base = pass ? m.in.p : nullptr;
        for (int i = 0; i < n; i++) {
            const HostInstance &hi = m.hosts[i];
            const FlatTrees &ft = hi.ft;
            const int B = ft.nblocks, N = ft.nnodes, L = ft.seqlen, T = hi.model.T;
            DevInst &d = m.h[i];
            if (pass == 0) {
                if (N > MAXN || T > MAXT) {
                    fprintf(stderr, "argweaver_amd: instance exceeds nnodes<=%d / ntimes<=%d\n",
                            MAXN, MAXT);
                    return 1;
                }
                std::vector<int> &so = m.soff[i];
                so.assign(B + 1, 0);
                for (int b = 0; b < B; b++) so[b + 1] = so[b] + m.Sv[i][b];
                if (shape_instance(hi, m.Sv[i], d)) return 1;
                d.W = m.W[i];
            }
            plan_inputs(p, d);
            if (pass == 1) {
                if (up.put((void *)d.model, &hi.model, sizeof(Model))) return 1;
                if (up.put((void *)d.parent, ft.parent.data(), sizeof(int) * B * N)) return 1;
                if (up.put((void *)d.c0, ft.child0.data(), sizeof(int) * B * N)) return 1;
                if (up.put((void *)d.c1, ft.child1.data(), sizeof(int) * B * N)) return 1;
                if (up.put((void *)d.age, ft.age.data(), sizeof(int) * B * N)) return 1;
                if (up.put((void *)d.map, ft.mapping.data(), sizeof(int) * B * N)) return 1;
                if (up.put((void *)d.spr, ft.spr.data(), sizeof(int) * 4 * B)) return 1;
                if (up.put((void *)d.bstart, ft.start.data(), sizeof(int) * B)) return 1;
                if (up.put((void *)d.blen, ft.len.data(), sizeof(int) * B)) return 1;
                if (up.put((void *)d.soff, m.soff[i].data(), sizeof(int) * (B + 1))) return 1;
                for (int r = 0; r < d.nrows; r++)
                    if (up.put((char *)d.seq + (size_t)r * L, hi.rows[r], L)) return 1;
                if (!m.us[i].empty())
                    if (up.put((void *)d.u, m.us[i].data(), sizeof(double) * L)) return 1;
            }
        }
        if (pass == 0 && m.in.ensure(p.used + 4096)) return 1;
    }
    if (up.flush()) return 1;
    HIP_OK(hipStreamSynchronize(c.main));
    // host rows may be released now
    for (auto &hi : m.hosts) hi.rows.clear();
    m.uploaded = true;
    return 0;
}

// Traceback tiles of every instance: tile_cols columns (0: one per
// instance), tail_cols for the instances with tail[inst] set, the instances
// with the most states per lane first.  Copies the tile list to the device
// on the main stream.
static int plan_tiles(Batch::Impl &m, int tile_cols, int warm,
                      const std::vector<char> *tail = nullptr, int tail_cols = 0)
{
    const int n = (int)m.h.size();
    std::vector<Chunk> &chs = m.chunks;
    chs.clear();
    // The tail instances' tiles run when the rest of the device is idle:
    // tail_cols long, or longer when that would give more workgroups than
    // the device has CUs
    if (tail && tail_cols > 0) {
        double cols = 0;
        for (int i = 0; i < n; i++)
            if ((*tail)[i]) cols += m.h[i].L;
        const double cus = std::max(1, ctx().prop.multiProcessorCount);
        tail_cols = std::max(tail_cols, (int)std::ceil(cols / cus));
    }
    std::vector<int> byr(n);
    std::iota(byr.begin(), byr.end(), 0);
    std::stable_sort(byr.begin(), byr.end(), [&](int a, int b) { return m.h[a].R > m.h[b].R; });
    m.sht = m.sht_big = 0;
    for (int i : byr) {
        const DevInst &d = m.h[i];
        const int tc = (tail && (*tail)[i] && tail_cols > 0) ? tail_cols : tile_cols;
        const int tile = tc > 0 ? std::max(64, tc) : d.L;
        const int nt = (d.L + tile - 1) / tile;
        for (int t = 0; t < nt; t++) {
            Chunk k;
            k.inst = i;
            k.c0 = t * tile;
            k.c1 = std::min(d.L, (t + 1) * tile);
            k.first = (t == 0);
            k.last = (t == nt - 1);
            k.cw = k.last ? d.L - 1 : std::min(d.L - 1, k.c1 + std::max(warm, 0));
            chs.push_back(k);
        }
        size_t &sh = d.R > 16 ? m.sht_big : m.sht;
        sh = std::max(sh, tb_lds_bytes(d.R));
    }
    const int nch = (int)chs.size();
    for (int pass = 0; pass < 2; pass++) {
        Plan p;
        p.base = pass ? m.tiles.p : nullptr;
        m.d_chunks = p.take<Chunk>(nch);
        m.d_ostart = p.take<int>(nch);
        m.d_oend = p.take<int>(nch);
        m.d_ridx = p.take<int>(2 * (size_t)nch);
        m.d_rk1 = p.take<int>(2 * (size_t)nch);
        m.d_rres = p.take<int>(4 * (size_t)nch);
        m.d_tlist = p.take<int>(2 * (size_t)nch);
        if (pass == 0 && m.tiles.ensure(p.used + 4096)) return 1;
    }
    HIP_OK(hipMemcpyAsync(m.d_chunks, chs.data(), sizeof(Chunk) * nch, hipMemcpyHostToDevice,
                          m.st.main));
    return 0;
}

// The chains of the tiles of the instances with take[inst] set (all when
// take is null) on stream s; slot 0 or 1 of the device tile lists.
static int launch_chains(Batch::Impl &m, bool fp32, const std::vector<char> *take, int slot,
                         hipStream_t s)
{
    const int nch = (int)m.chunks.size();
    std::vector<int> &list = slot ? m.tlist1 : m.tlist0;
    list.clear();
    // the tiles of the 32-states-per-lane instances after the others (a
    // launch of their own symbol)
    int nn = 0;
    for (int big = 0; big < 2; big++) {
        for (int j = 0; j < nch; j++)
            if ((!take || (*take)[m.chunks[j].inst]) && (m.h[m.chunks[j].inst].R > 16) == (big == 1))
                list.push_back(j);
        if (!big) nn = (int)list.size();
    }
    const int nl = (int)list.size();
    if (!nl) return 0;
    int *dl = m.d_tlist + (size_t)slot * nch;
    HIP_OK(hipMemcpyAsync(dl, list.data(), sizeof(int) * nl, hipMemcpyHostToDevice, s));
    if (nn > 0 && launch_tb_spec(fp32, false, m.dD, m.d_chunks, dl, nn, m.sht, m.d_ostart, m.d_oend, s))
        return 1;
    return nl > nn && launch_tb_spec(fp32, true, m.dD, m.d_chunks, dl + nn, nl - nn, m.sht_big,
                                     m.d_ostart, m.d_oend, s);
}

// Resolution of the tiles, right to left within each instance.  A tile
// whose true state at c1 is the start of its chain keeps that chain's path
// and passes the chain's end state on as the true state of the tile before.
// The first tile that does not fit is re-run from its true state, and in the
// same pass every tile before it whose predicted start (the end of the next
// tile's chain) is not its own is re-run from that prediction.  A re-run
// replaces the tile's chain by the one from its start (the samples until it
// meets the stored path, then that path), so a right prediction leaves the
// tile decided for the next pass.
// take: the instances to resolve (all when null); slot 0 or 1 of the
// device lists, so that two resolutions of disjoint instances can run at
// once on two streams.
static int resolve_tiles(Batch::Impl &m, bool fp32, RunStats &rs, hipStream_t s,
                         const std::vector<char> *take, int slot)
{
    const std::vector<Chunk> &chs = m.chunks;
    const int nch = (int)chs.size();
    // per instance: its first tile, the rightmost undecided tile and the
    // true state at that tile's column c1
    struct Walk {
        int f, r, b;
    };
    std::vector<Walk> ws;
    for (int j = 0; j < nch; j++)
        if (chs[j].last && !chs[j].first && (!take || (*take)[chs[j].inst])) {
            int f = j;
            while (!chs[f].first) f--;
            ws.push_back(Walk{f, j - 1, 0});
        }
    if (ws.empty()) return 0;
    int *ridx = m.d_ridx + (size_t)slot * nch, *rk1 = m.d_rk1 + (size_t)slot * nch;
    int *rres = m.d_rres + (size_t)slot * 2 * nch;
    std::vector<int> os(nch), oe(nch);
    HIP_OK(hipMemcpyAsync(os.data(), m.d_ostart, sizeof(int) * nch, hipMemcpyDeviceToHost, s));
    HIP_OK(hipMemcpyAsync(oe.data(), m.d_oend, sizeof(int) * nch, hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    for (Walk &w : ws) w.b = oe[w.r + 1];
    std::vector<int> pj, pk, res;
    while (true) {
        pj.clear();
        pk.clear();
        for (Walk &w : ws) {
            while (w.r >= w.f && os[w.r] == w.b) w.b = oe[w.r--];
            if (w.r < w.f) continue;
            int g = w.b;
            for (int j = w.r; j >= w.f; j--) {
                if (os[j] != g) {
                    pj.push_back(j);
                    pk.push_back(g);
                }
                g = oe[j];
            }
        }
        if (pj.empty()) break;
        const int np = (int)pj.size();
        HIP_OK(hipMemcpyAsync(ridx, pj.data(), sizeof(int) * np, hipMemcpyHostToDevice, s));
        HIP_OK(hipMemcpyAsync(rk1, pk.data(), sizeof(int) * np, hipMemcpyHostToDevice, s));
        if (m.sht && launch_tb_rerun(fp32, false, m.dD, m.d_chunks, ridx, rk1, np, m.sht, rres, s))
            return 1;
        if (m.sht_big &&
            launch_tb_rerun(fp32, true, m.dD, m.d_chunks, ridx, rk1, np, m.sht_big, rres, s))
            return 1;
        res.resize(2 * (size_t)np);
        HIP_OK(hipMemcpyAsync(res.data(), rres, sizeof(int) * res.size(), hipMemcpyDeviceToHost, s));
        HIP_OK(hipStreamSynchronize(s));
        rs.tb_passes++;
        for (int x = 0; x < np; x++) {
            const int j = pj[x];
            rs.tb_rerun_cols += chs[j].c1 - (res[2 * x] < 0 ? chs[j].c0 : res[2 * x]);
            os[j] = pk[x];
            oe[j] = res[2 * x + 1];
        }
    }
    return 0;
}

// The traceback of every instance whose forward table is resident: the
// chains of every tile in one launch, then the resolution (re-runs of the
// tiles that do not fit).  opt.fixup = false leaves the speculative paths
// (diagnostics).
static int traceback_stage(Batch::Impl &m, bool fp32, const BatchOptions &opt, RunStats &rs)
{
    if (plan_tiles(m, opt.tile_cols, opt.tile_warm)) return 1;
    if (launch_chains(m, fp32, nullptr, 0, m.st.main)) return 1;
    return opt.fixup ? resolve_tiles(m, fp32, rs, m.st.main, nullptr, 0) : 0;
}

int Batch::tune_tiles(Precision prec, const int *cand, int ncand, double *ms_out, int warm)
{
    BATCH_LOCK;
    BatchOptions opt;
    opt.prec = prec;
    opt.traceback = false;
    if (run(opt)) return -1;
    Impl &m = *impl_;
    Streams &c = m.st;
    const OnDevice on(c.dev);
    const bool fp32 = prec == Precision::FP32;
    int best = cand[0];
    float best_ms = 0;
    for (int i = 0; i < ncand; i++) {
        RunStats rs;
        (void)hipEventRecord(c.ev[6], c.main);
        BatchOptions topt;
        topt.prec = prec;
        topt.tile_cols = cand[i];
        topt.tile_warm = warm;
        if (traceback_stage(m, fp32, topt, rs)) return -1;
        (void)hipEventRecord(c.ev[7], c.main);
        HIP_OK(hipStreamSynchronize(c.main));
        float ms = 0;
        (void)hipEventElapsedTime(&ms, c.ev[6], c.ev[7]);
        if (ms_out) ms_out[i] = ms;
        if (i == 0 || ms < best_ms) {
            best_ms = ms;
            best = cand[i];
        }
    }
    return best;
}

int Batch::tune_forward(const int *tiles, const int *warms, int ncand, double tol, double *ms_out)
{
    BATCH_LOCK;
    int best = -1;
    double best_ms = 0;
    for (int i = 0; i < ncand; i++) {
        BatchOptions opt;
        opt.prec = Precision::FP32;
        opt.traceback = false;
        opt.fw_tile = tiles[i];
        opt.fw_warm = warms[i] > 0 ? warms[i] : opt.fw_warm;
        if (tol > 0) opt.fw_tol = tol;
        RunStats rs;
        if (run(opt, &rs)) return -1;
        if (ms_out) ms_out[i] = rs.ms_forward;
        if (best < 0 || rs.ms_forward < best_ms) {
            best_ms = rs.ms_forward;
            best = i;
        }
    }
    return best;
}

// FP32 forward column cost (us) by states per lane that tiles are planned with:
// medians of the tiles of the 256-instance batch (20 time points) on MI355X with
// one wave per tile.  With two a column takes 33 % of it at R = 2, 38-41 % at 4 to
// 12 and 46 % at 16, so that an instance's tiles end up to a fifth apart from those of
// another R; the plan stays, because it defines the FP32 tables.  Small R pays for a
// longer carry chain of the same-branch scan, so the cost is nearly flat up to R = 6.
constexpr double FW_CREF = 0.94;
inline double fw_cost_model(int R)
{
    return R <= 2 ? 0.94 : R == 4 ? 0.90 : R == 6 ? 0.98 : R == 8 ? 1.09 : R == 12 ? 1.34 : 1.60;
}

// The forward of every instance.  FP32 runs may split long instances into
// speculative tiles (BatchOptions::fw_tile); each tile's start is then
// checked against the boundary column of the tile before, and tiles that
// fail are re-run from that column until every check passes (a re-run
// changes the boundary column of the next tile, which is checked again).
// AWAMD_TRACE_TILES=1 in the environment: the forward re-runs are printed
// to stderr (diagnostics)
static bool trace_tiles()
{
    static const bool on = [] {
        const char *e = getenv("AWAMD_TRACE_TILES");
        return e && e[0] == '1';
    }();
    return on;
}

static int forward_stage(Batch::Impl &m, bool fp32, const BatchOptions &opt,
                         const std::vector<int> &order, size_t shf, int t1max, RunStats &rs,
                         const std::function<int(const std::vector<char> &)> &first_check)
{
    Streams &c = m.st;
    hipStream_t s = c.main;
    const size_t rsz = fp32 ? sizeof(float) : sizeof(double);
    FwPlan plan;
    const int C0 = (fp32 && opt.fw_tile > 0) ? opt.fw_tile : 0;
    const int W = std::max(opt.fw_warm, 1);
    for (int i : order) {
        // tiles of C0 columns at a column cost of FW_CREF us; an instance
        // whose columns cost more gets proportionally shorter tiles, so that
        // the tiles of every instance take about the same time
        const int C = C0 ? std::max(W + W / 4, (int)(C0 * FW_CREF / fw_cost_model(m.h[i].R))) : 0;
        plan.add(i, m.h[i].L, m.h[i].R, C, W);
    }
    const std::vector<FwTile> &tl = plan.tiles;
    const int nt = (int)tl.size();
    rs.fw_tiles = nt;
    for (int pass = 0; pass < 2; pass++) {
        Plan p;
        p.base = pass ? m.fwb.p : nullptr;
        m.d_fwt = p.take<FwTile>(nt);
        m.d_fwre = p.take<FwTile>(nt);
        m.d_bnd = p.take<char>((size_t)plan.units * BND_UNIT * rsz);
        m.d_bnorm = p.take<double>(plan.units);
        m.d_fidx = p.take<int>(nt);
        m.d_fflag = p.take<int>(nt);
        if (pass == 0 && m.fwb.ensure(p.used + 4096)) return 1;
    }
    HIP_OK(hipMemcpyAsync(m.d_fwt, tl.data(), sizeof(FwTile) * nt, hipMemcpyHostToDevice, s));
    const auto t_fw = std::chrono::steady_clock::now();
    // the 32-states-per-lane tiles run on the side stream, beside the
    // others: the host joins the main stream first (preparation, emissions
    // and the tile list done), and the side stream before the checks
    if (m.any_big) {
        HIP_OK(hipStreamSynchronize(s));
        if (fp32 ? launch_fw<float, true>(m.dD, m.d_fwt, nt, m.d_bnd, m.d_bnorm, m.shf_big, c.side,
                                          t1max)
                 : launch_fw<double, true>(m.dD, m.d_fwt, nt, m.d_bnd, m.d_bnorm, m.shf_big, c.side,
                                           t1max))
            return 1;
    }
    (void)hipEventRecord(c.ev[6], s);
    if (fp32 ? launch_fw<float, false>(m.dD, m.d_fwt, nt, m.d_bnd, m.d_bnorm, shf, s, t1max)
             : launch_fw<double, false>(m.dD, m.d_fwt, nt, m.d_bnd, m.d_bnorm, shf, s, t1max))
        return 1;
    (void)hipEventRecord(c.ev[7], s);
    if (m.any_big) HIP_OK(hipStreamSynchronize(c.side));
    // tiles whose start is to be checked: those with a boundary slot in
    std::vector<int> chk = plan.started();
    std::vector<int> flags;
    bool first = true;
    while (!chk.empty()) {
        const int nc = (int)chk.size();
        HIP_OK(hipMemcpyAsync(m.d_fidx, chk.data(), sizeof(int) * nc, hipMemcpyHostToDevice, s));
        if (launch_fw_check(m.dD, m.d_fwt, m.d_fidx, nc, m.d_bnd, m.d_bnorm, opt.fw_tol, m.d_fflag, s))
            return 1;
        flags.resize(nc);
        HIP_OK(hipMemcpyAsync(flags.data(), m.d_fflag, sizeof(int) * nc, hipMemcpyDeviceToHost, s));
        HIP_OK(hipStreamSynchronize(s));
        std::vector<int> redo;
        for (int x = 0; x < nc; x++)
            if (flags[x]) redo.push_back(chk[x]);
        if (first) {
            // the instances that will be re-run; the others are final
            first = false;
            std::vector<char> busy(m.h.size(), 0);
            for (int k : redo) busy[tl[k].inst] = 1;
            if (first_check(busy)) return 1;
        }
        if (redo.empty()) break;
        // re-run from the boundary column, then check the tiles after them
        const std::vector<FwTile> sub = plan.rerun(redo);
        rs.fw_reruns += (int)redo.size();
        if (trace_tiles()) {
            for (int k : redo)
                fprintf(stderr, "fw re-run: inst %d (L %d, R %d) tile [%d, %d)\n", tl[k].inst,
                        m.h[tl[k].inst].L, m.h[tl[k].inst].R, tl[k].cs, tl[k].c1);
        }
        // the tile list keeps every tile's index for the checks; the re-run
        // tiles are launched from a list of their own
        const int nr = (int)sub.size();
        HIP_OK(hipMemcpyAsync(m.d_fwre, sub.data(), sizeof(FwTile) * nr, hipMemcpyHostToDevice, s));
        if (launch_fw<float, false>(m.dD, m.d_fwre, nr, m.d_bnd, m.d_bnorm, shf, s, t1max,
                                    opt.fw_tol, m.d_fflag))
            return 1;
        if (m.any_big && launch_fw<float, true>(m.dD, m.d_fwre, nr, m.d_bnd, m.d_bnorm, m.shf_big,
                                                s, t1max, opt.fw_tol, m.d_fflag))
            return 1;
        std::vector<int> early(nr);
        HIP_OK(hipMemcpyAsync(early.data(), m.d_fflag, sizeof(int) * nr, hipMemcpyDeviceToHost, s));
        HIP_OK(hipStreamSynchronize(s));
        chk = plan.finished(redo, sub, early);
        if (!chk.empty())
            HIP_OK(hipMemcpyAsync(m.d_fwt, tl.data(), sizeof(FwTile) * nt, hipMemcpyHostToDevice, s));
        if (trace_tiles()) {
            for (int x = 0; x < nr; x++)
                fprintf(stderr, "  inst %d tile [%d, %d): %s %d\n", sub[x].inst, sub[x].cs,
                        sub[x].c1, early[x] ? "rejoined at" : "ran to", early[x] ? early[x] - 1 : sub[x].c1);
            fprintf(stderr, "fw re-run round: %d tiles, %.1f ms since the forward was queued\n", nr,
                    std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_fw).count());
        }
    }
    if (first) return first_check(std::vector<char>(m.h.size(), 0));
    return 0;
}

int Batch::run(const BatchOptions &opt, RunStats *st)
{
    BATCH_LOCK;
    if (ctx_init()) return 1;
    Impl &m = *impl_;
    if (!m.uploaded && upload()) return 1;
    Streams &c = m.st;
    const OnDevice on(c.dev);
    const int n = (int)m.hosts.size();
    hipStream_t s = c.main;
    const bool fp32 = opt.prec == Precision::FP32;

    std::vector<long long> coloff(n + 1, 0);
    std::vector<int> blkoff(n + 1, 0);
    for (int i = 0; i < n; i++) {
        coloff[i + 1] = coloff[i] + m.h[i].L;
        blkoff[i + 1] = blkoff[i] + m.h[i].B;
    }
    // per-instance work arrays
    for (int pass = 0; pass < 2; pass++) {
        Plan p;
        p.base = pass ? m.work.p : nullptr;
        for (int i = 0; i < n; i++) plan_work(p, m.h[i], fp32);
        if (pass == 0 && m.work.ensure(p.used + 4096)) return 1;
    }
    // forward tables
    for (int pass = 0; pass < 2; pass++) {
        Plan p;
        p.base = pass ? m.tab.p : nullptr;
        for (int i = 0; i < n; i++) plan_table(p, m.h[i]);
        if (pass == 0 && m.tab.ensure(p.used + 4096)) return 1;
    }
    // auxiliary arrays
    for (int pass = 0; pass < 2; pass++) {
        Plan p;
        p.base = pass ? m.aux.p : nullptr;
        m.dD = p.take<DevInst>(n);
        m.d_coloff = p.take<long long>(n + 1);
        m.d_blkoff = p.take<int>(n + 1);
        m.d_voff = p.take<int>(n + 1);
        m.d_nvar = p.take<int>(n);
        m.d_list = p.take<int>(n);
        m.d_lnl = p.take<double>(n);
        if (pass == 0 && m.aux.ensure(p.used + 4096)) return 1;
    }
    for (int i = 0; i < n; i++) m.h[i].lnl = m.d_lnl + i;

    (void)hipEventRecord(c.ev[0], s);
    HIP_OK(hipMemcpyAsync(m.d_coloff, coloff.data(), sizeof(long long) * (n + 1), hipMemcpyHostToDevice, s));
    HIP_OK(hipMemcpyAsync(m.d_blkoff, blkoff.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, s));
    HIP_OK(hipMemcpyAsync(m.dD, m.h.data(), sizeof(DevInst) * n, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_classify_b, dim3((unsigned)((coloff[n] + 255) / 256)), dim3(256), 0, s,
                       m.dD, m.d_coloff, n);
    hipLaunchKernelGGL(k_scan_b, dim3(n), dim3(1024), 0, s, m.dD, m.d_nvar);
    HIP_OK(hipGetLastError());
    HIP_OK(hipMemcpyAsync(m.nvar.data(), m.d_nvar, sizeof(int) * n, hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    for (int i = 0; i < n; i++)
        if (m.hosts[i].prep) m.nvar[i] = m.hosts[i].prep->nvar;

    // variant rows, allocated now that the counts are known
    std::vector<int> voff(n + 1, 0);
    for (int pass = 0; pass < 2; pass++) {
        Plan p;
        p.base = pass ? m.vbuf.p : nullptr;
        for (int i = 0; i < n; i++) {
            m.h[i].nvar = m.nvar[i];
            plan_variants(p, m.h[i]);
            voff[i + 1] = voff[i] + m.nvar[i];
        }
        if (pass == 0 && m.vbuf.ensure(p.used + 4096)) return 1;
    }
    HIP_OK(hipMemcpyAsync(m.d_voff, voff.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, s));
    HIP_OK(hipMemcpyAsync(m.dD, m.h.data(), sizeof(DevInst) * n, hipMemcpyHostToDevice, s));

    (void)hipEventRecord(c.ev[1], s);
    hipLaunchKernelGGL(k_prep_b, dim3(blkoff[n]), dim3(256), 0, s, m.dD, m.d_blkoff, n);
    HIP_OK(hipGetLastError());
    // caller-given first-column priors, in the lane-run layout
    std::vector<std::vector<double>> lpri(n);
    for (int i = 0; i < n; i++) {
        if (m.priors[i].empty()) continue;
        const int R = m.h[i].R;
        lpri[i].assign(64 * R, 0.0);
        for (size_t k = 0; k < m.priors[i].size(); k++) lpri[i][lane_pos((int)k, R)] = m.priors[i][k];
        HIP_OK(hipMemcpyAsync(m.h[i].lprior, lpri[i].data(), sizeof(double) * lpri[i].size(),
                              hipMemcpyHostToDevice, s));
    }
    // host-prepared instances: their per-block inputs, column classes and
    // variant rows (the device kernels above skipped them)
    if (std::any_of(m.hosts.begin(), m.hosts.end(), [](const HostInstance &hi) { return hi.prep != nullptr; })) {
        const StageUse use(m.stage);
        if (!use.s) return 1;
        Uploader up(*use.s, s);
        const auto put = [&](auto *dst, const auto &v) { return up.put(dst, v.data(), sizeof(v[0]) * v.size()); };
        std::vector<float> planes32;
        for (int i = 0; i < n; i++) {
            const HostPrep *hp = m.hosts[i].prep.get();
            if (!hp) continue;
            const DevInst &d = m.h[i];
            if (fp32) planes32.assign(hp->planes.begin(), hp->planes.end());
            if (fp32 ? put(d.lcoef32, planes32) : put(d.lcoef, hp->planes)) return 1;
            if (put(d.linfo, hp->info) || put(d.ldet, hp->det) || put(d.tm, hp->tm) ||
                put(d.tvec, hp->tvec) || put(d.srcs, hp->srcs) || put(d.lprior, hp->prior) ||
                put(d.cls, hp->cls) || put(d.vemit, hp->vemit))
                return 1;
        }
        if (up.flush()) return 1;
    }
    (void)hipEventRecord(c.ev[2], s);
    if (voff[n] > 0) {
        int nmax = 1;
        for (int i = 0; i < n; i++) nmax = std::max(nmax, m.h[i].N);
        hipLaunchKernelGGL(k_var_emit_b, dim3(voff[n]), dim3(64), var_emit_lds(nmax), s, m.dD,
                           m.d_voff, n, nmax);
    }
    HIP_OK(hipGetLastError());
    int rmax = 1;
    for (int i = 0; i < n; i++) rmax = std::max(rmax, m.h[i].R);
    if (launch_tb_pred(m.dD, m.d_blkoff, n, blkoff[n], rmax, s)) return 1;
    (void)hipEventRecord(c.ev[3], s);

    // forward: one workgroup per tile, all tiles in one launch, the longest
    // instances first
    std::vector<int> order(n);
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        const double ca = (double)m.h[a].L * m.h[a].R, cb = (double)m.h[b].L * m.h[b].R;
        return ca > cb;
    });
    HIP_OK(hipMemcpyAsync(m.d_list, order.data(), sizeof(int) * n, hipMemcpyHostToDevice, s));
    size_t shf = 0;
    int t1max = 0;
    m.any_big = false;
    m.shf_big = 0;
    for (int i = 0; i < n; i++) {
        const DevInst &d = m.h[i];
        t1max = std::max(t1max, d.T - 1);
        size_t &sh = d.R > 16 ? m.shf_big : shf;
        sh = std::max(sh, fw_lds_bytes(fp32, d.R));
        m.any_big |= d.R > 16;
    }
    RunStats rs;
    // Once the first check of the forward tiles has shown which instances
    // are re-run, the traceback chains of all the others go to the side
    // stream and run while the re-runs continue on the main stream.
    // A helper host thread then resolves those instances' tiles on the side
    // stream (its re-runs too), while this thread drives the forward re-runs
    // and then the re-run instances' traceback on the main stream.
    std::vector<char> busy, done;
    std::thread helper;
    RunStats rs_side;
    int rc_side = 0;
    auto early_tb = [&](const std::vector<char> &b) -> int {
        if (!opt.traceback || std::find(b.begin(), b.end(), 1) == b.end()) return 0;
        busy = b;
        if (plan_tiles(m, opt.tile_cols, opt.tile_warm, &b, opt.tail_tile_cols))
            return 1;
        HIP_OK(hipStreamSynchronize(s));   // the tile list is on the device
        done.assign(n, 0);
        for (int i = 0; i < n; i++) done[i] = !b[i];
        if (launch_chains(m, fp32, &done, 0, c.side)) return 1;
        if (opt.fixup)
            helper = std::thread([&] {
                const OnDevice side(c.dev);
                rc_side = resolve_tiles(m, fp32, rs_side, c.side, &done, 1);
                (void)hipEventRecord(c.ev[8], c.side);
            });
        return 0;
    };
    // the helper is joined on every path out of run()
    struct Joiner {
        std::thread &t;
        ~Joiner()
        {
            if (t.joinable()) t.join();
        }
    } joiner{helper};
    if (forward_stage(m, fp32, opt, order, shf, t1max, rs, early_tb)) return 1;
    (void)hipEventRecord(c.ev[4], s);
    hipLaunchKernelGGL(k_lnl_b, dim3(n), dim3(1024), 0, s, m.dD, m.d_list);
    HIP_OK(hipGetLastError());
    // traceback tiles: the chains of every tile, then their resolution
    if (opt.traceback) {
        if (busy.empty()) {
            if (traceback_stage(m, fp32, opt, rs)) return 1;
        } else {
            if (launch_chains(m, fp32, &busy, 1, s)) return 1;
            if (opt.fixup && resolve_tiles(m, fp32, rs, s, &busy, 0)) return 1;
            (void)hipEventRecord(c.ev[9], s);
            if (helper.joinable()) helper.join();
            HIP_OK(hipStreamSynchronize(c.side));
            if (rc_side) return 1;
            rs.tb_passes = std::max(rs.tb_passes, rs_side.tb_passes);
            rs.tb_rerun_cols += rs_side.tb_rerun_cols;
        }
    }
    (void)hipEventRecord(c.ev[5], s);
    // side by side, so that they come in one copy (256 copies took 3.4 ms)
    HIP_OK(hipMemcpyAsync(m.lnl.data(), m.d_lnl, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    m.prec_done = opt.prec;
    float ms;
    (void)hipEventElapsedTime(&ms, c.ev[1], c.ev[2]); rs.ms_prep = ms;
    (void)hipEventElapsedTime(&ms, c.ev[2], c.ev[3]); rs.ms_emit = ms;
    // forward: until the forward kernel ends; traceback: from there to the
    // end of the fix-up passes
    float fwd = 0;
    (void)hipEventElapsedTime(&fwd, c.ev[3], c.ev[4]);
    rs.ms_forward = fwd;
    (void)hipEventElapsedTime(&ms, c.ev[6], c.ev[7]);
    rs.ms_fw_main = ms;
    (void)hipEventElapsedTime(&ms, c.ev[3], c.ev[5]);
    rs.ms_traceback = opt.traceback ? std::max(0.f, ms - fwd) : 0.f;
    (void)hipEventElapsedTime(&ms, c.ev[0], c.ev[5]); rs.ms_total = ms;
    if (opt.traceback && opt.fixup && !busy.empty()) {
        // the two halves of the overlapped traceback, from the end of the
        // forward: the re-run instances' (main stream) and the others' (side)
        (void)hipEventElapsedTime(&ms, c.ev[4], c.ev[9]); rs.ms_tb_tail = ms;
        (void)hipEventElapsedTime(&ms, c.ev[4], c.ev[8]); rs.ms_tb_side = ms;
    }
    for (int i = 0; i < n; i++) {
        rs.W += m.W[i];
        rs.nvar += m.nvar[i];
    }
    if (st) *st = rs;
    return 0;
}

int Batch::copy_path(int i, int *path) const
{
    BATCH_LOCK;
    const Impl &m = *impl_;
    HIP_OK(hipMemcpy(path, m.h[i].path, sizeof(int) * m.h[i].L, hipMemcpyDeviceToHost));
    return 0;
}

int Batch::copy_norms(int i, double *norms) const
{
    BATCH_LOCK;
    const Impl &m = *impl_;
    HIP_OK(hipMemcpy(norms, m.h[i].norms, sizeof(double) * m.h[i].L, hipMemcpyDeviceToHost));
    return 0;
}

// block-major view (block b holds blocklen_b rows of S_b states, the
// reference's table layout) of columns [c0, c1) of the lane-run table.  While
// the kernel fills one half of the staging memory, the host copies the rows of
// the other half out.
int Batch::copy_alpha_range(int i, int c0, int c1, double *alpha) const
{
    BATCH_LOCK;
    Impl &m = *impl_;
    const DevInst &d = m.h[i];
    const FlatTrees &ft = m.hosts[i].ft;
    const std::vector<int> &Sv = m.Sv[i];
    if (c0 < 0 || c1 > d.L || c0 >= c1) return 1;
    const bool fp32 = m.prec_done == Precision::FP32;
    // no table before a run, or only part of one after a run that failed
    const size_t bytes = (size_t)d.L * 64 * d.R * (fp32 ? sizeof(float) : sizeof(double));
    if (!d.alpha || (char *)d.alpha + bytes > m.tab.p + m.tab.cap) return 1;
    const OnDevice on(m.st.dev);
    const StageUse use(m.stage);
    if (!use.s) return 1;
    const HostStage &stage = *use.s;
    const int pitch = *std::max_element(Sv.begin(), Sv.end());
    const int rows = (int)(HostStage::HALF / sizeof(double) / pitch);
    const auto fill = [&](int c, int half) {
        const int n = std::min(rows, c1 - c);
        hipLaunchKernelGGL(fp32 ? k_rows_out<float> : k_rows_out<double>, dim3((n + 3) / 4),
                           dim3(256), 0, m.st.main, d.alpha, c, n, d.R, pitch, stage.half(half));
        HIP_OK(hipGetLastError());
        HIP_OK(hipEventRecord(stage.filled[half], m.st.main));
        return 0;
    };
    const auto copy = [&] {
        int b = 0;
        if (fill(c0, 0)) return 1;
        for (int c = c0, half = 0; c < c1; c += rows, half ^= 1) {
            if (c + rows < c1 && fill(c + rows, half ^ 1)) return 1;
            HIP_OK(hipEventSynchronize(stage.filled[half]));
            const double *row = stage.half(half);
            for (int x = c; x < std::min(c + rows, c1); x++, row += pitch) {
                while (ft.start[b] + ft.len[b] <= x) b++;
                memcpy(alpha, row, sizeof(double) * Sv[b]);
                alpha += Sv[b];
            }
        }
        return 0;
    };
    if (!copy()) return 0;
    // a kernel may still write to the staging memory, which is given back
    (void)hipStreamSynchronize(m.st.main);
    return 1;
}

int Batch::copy_alpha(int i, double *alpha) const
{
    BATCH_LOCK;
    return copy_alpha_range(i, 0, impl_->h[i].L, alpha);
}

long long instance_states(const FlatTrees &ft, int T, std::vector<int> *Sv)
{
    long long W = 0;
    if (Sv) Sv->resize(ft.nblocks);
    for (int b = 0; b < ft.nblocks; b++) {
        const int N = ft.nnodes;
        const int *par = &ft.parent[(size_t)b * N];
        const int *age = &ft.age[(size_t)b * N];
        int S = 0;
        for (int i = 0; i < N; i++) {
            int top = par[i] == -1 ? T - 2 : age[par[i]];
            S += top - age[i] + 1;
        }
        if (Sv) (*Sv)[b] = S;
        W += (long long)S * ft.len[b];
    }
    return W;
}

int instance_supported(const HostInstance &hi, std::string *msg)
{
    char buf[160];
    buf[0] = 0;
    const FlatTrees &ft = hi.ft;
    if (ft.nnodes > MAXN || hi.model.T > MAXT) {
        snprintf(buf, sizeof buf, "instance has %d nodes and %d time points (limits %d and %d)",
                 ft.nnodes, hi.model.T, MAXN, MAXT);
    } else if (!hi.prep) {
        std::vector<int> Sv;
        instance_states(ft, hi.model.T, &Sv);
        int Smax = 1;
        for (int S : Sv) Smax = std::max(Smax, S);
        if (lanes_per_state_r(Smax) < 0)
            snprintf(buf, sizeof buf, "a block has %d states (limit %d per block)", Smax,
                     64 * RVALS[NRV - 1]);
    }
    if (msg) *msg = buf;
    return buf[0] ? 1 : 0;
}

bool device_available()
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return false;
    return n > 0;
}

const char *device_name()
{
    if (ctx_init()) return "unavailable";
    return ctx().prop.gcnArchName;
}

int device_info(char *buf, int n)
{
    if (ctx_init()) return 1;
    const hipDeviceProp_t &p = ctx().prop;
    snprintf(buf, n, "%s %s CUs=%d lds_per_block=%zu lds_per_cu=%zu clock_khz=%d mem_gb=%.1f",
             p.name, p.gcnArchName, p.multiProcessorCount, (size_t)p.sharedMemPerBlock,
             (size_t)p.maxSharedMemoryPerMultiProcessor, p.clockRate,
             p.totalGlobalMem / 1073741824.0);
    return 0;
}

// one instance on the given batch (cleared first)
static int run_one(Batch &bt, const HostInstance &hi, const double *u, int *path, double *alpha,
                   double *lnl, RunStats *stats, Precision prec, const double *prior,
                   int tile_cols)
{
    bt.clear();
    if (bt.add(hi, u, prior) < 0) return 1;
    if (bt.upload()) return 1;
    BatchOptions opt;
    opt.prec = prec;
    opt.traceback = (u != nullptr);
    // long instances trace back in tiles (the thread is the same as with one
    // tile: fix-up passes re-sample until the chains coalesce)
    // (500000 columns in tiles of 4096 / 8192 / 16384 / none: 3.3 / 3.1 / 3.2 / 22
    // ms; 100000 in FP64: 1.4 / 1.2 / 0.9 / 2.4; 20000: 0.33 / 0.33 / - / 0.38)
    opt.tile_cols = (tile_cols == 0 && hi.ft.seqlen >= 16384) ? 8192 : tile_cols;
    // FP32 forwards of long instances run as tiles (FP64 keeps the
    // sequential forward: its contract is the reference's table)
    if (prec == Precision::FP32) {
        opt.fw_tile = 50000;
        opt.fw_warm = 20000;
        opt.fw_tol = 1e-4;
    }
    if (bt.run(opt, stats)) return 1;
    if (path && u && bt.copy_path(0, path)) return 1;
    if (alpha && bt.copy_alpha(0, alpha)) return 1;
    if (lnl) *lnl = bt.lnl(0);
    return 0;
}

// one instance = a batch of one; the batch (its device buffers and streams)
// is kept per host thread, so repeated calls (every re-threading of
// resample_arg) reuse the allocations
int run_instance(const HostInstance &hi, const double *u, int *path, double *alpha, double *lnl,
                 RunStats *stats, Precision prec, const double *prior, int tile_cols)
{
    // never destroyed: releasing HIP objects from exit-time destructors can
    // run after the runtime itself has shut down
    static thread_local Batch *btp = new Batch();
    return run_one(*btp, hi, u, path, alpha, lnl, stats, prec, prior, tile_cols);
}

// The no-allocation workspace: one fixed device array, of which every GPU
// the library runs on holds its own copy until the process ends.  Host code
// never uses the name `scratch` as an address (on the host it is a stand-in
// symbol, not device memory): the copy on each device is found once, with
// that device current, by hipGetSymbolAddress, and that pointer is what the
// batch's buffers are carved from.
static __device__ __align__(256) char scratch[kNoAllocBytes];

namespace {
struct NoAllocDevice {
    char *ptr = nullptr;     // device address of this GPU's scratch
    Batch *batch = nullptr;  // never destroyed (see run_instance)
};
}  // namespace

// Set-up of the current device, once: the scratch address and a batch whose
// buffers live in it, with its stream and events created here, so that the
// calls after it allocate nothing.
static int noalloc_device(NoAllocDevice *&out)
{
    static std::mutex mu;
    static std::map<int, NoAllocDevice> devs;
    int dev = 0;
    HIP_OK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    auto it = devs.find(dev);
    if (it == devs.end()) {
        NoAllocDevice d;
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            fprintf(stderr, "argweaver_amd: hipGetSymbolAddress(scratch) failed on device %d: %s\n",
                    dev, hipGetErrorString(e));
            return 1;
        }
        d.ptr = static_cast<char *>(p);
        d.batch = new Batch();
        d.batch->use_workspace(d.ptr, kNoAllocBytes);
        if (d.batch->init_streams()) return 1;
        it = devs.emplace(dev, d).first;
    }
    out = &it->second;
    return 0;
}

int run_instance_noalloc(const HostInstance &hi, const double *u, int *path, double *alpha,
                         double *lnl, RunStats *stats, Precision prec)
{
    NoAllocDevice *d = nullptr;
    if (noalloc_device(d)) return 1;
    DEVICE_LOCK;   // calls on one GPU share its scratch: one at a time
    return run_one(*d->batch, hi, u, path, alpha, lnl, stats, prec, nullptr, 0);
}

}  // namespace aw

