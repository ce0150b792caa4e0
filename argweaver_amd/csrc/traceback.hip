// traceback.hip -- stochastic traceback (stochastic_traceback,
// sample_thread.cpp:522-569; sample_hmm_posterior_step :506-519; sample,
// common.h:272-290).
//
// The sample of a column depends on the state sampled at the column to its
// right, so one wave walking the columns pays the latency of a column's scan
// and sampling for every one of them.  But the state hardly ever changes
// inside a local-tree block (0.03-0.2 % of the columns), and across a switch
// it follows the likeliest source state in 94-99.8 % of the cases.  So a
// workgroup walks one tile, its waves working on consecutive runs of columns
// (units, about a block each) at once: the entry state of every unit is
// predicted by chasing the blocks' source tables from the true state, each
// wave samples its unit from the predicted entry state, and the units up to
// the first one whose outcome was not what the next one assumed are kept.
// Every stored sample is the sample of its column given its right neighbour,
// whatever was predicted, so the thread is that of a column-by-column walk.
//
// Inside a unit a wave decides its columns at once, a lane each, without
// reading their rows.  The total that a column's pick is a fraction of is what
// the forward recursion computed the next column's entry from: entry * normaliser
// / emission.  The state j assumed for the column has the share entry *
// weight of it; the sums below j are unknown, but lie between 0 and the rest, so
// a uniform that is off both ends by more than that and a guard of 2^-13 picks j
// wherever j stands.  The guard covers the FP32 recursion's rounding: its terms are
// all positive (and its planes normal numbers), and with n = T-1 time bins an entry
// passes at most n + 6 roundings (units of 2^-24) in the same-branch sum (planes 2,
// running sum and carry n + 1, products 3) or 13 in the other-branch product, 3 from
// there to the column, 3 through scale and normaliser, 1 in the row before, and 2 in
// the products that are sampled from: n + 15, so that the guard is 60 times the bound
// at 20 time points and 44 times at 32.
// Only the other columns, about twice the share that is not j's, are sampled from
// their rows, with the FP64 cumulative sums; so are those whose next column
// was not computed from the stored one (DevInst::cut).  The columns at switches go
// the same way, j being the likeliest source.
//
// Reading every row, a CU's bandwidth bound the walk (33 GB/s: 0.03 / 0.06 / 0.12
// us per column at 4 / 8 FP32 and 8 FP64 states per lane); now the latency of
// about six dependent loads per round of units does.  On MI355X: 10000 columns of
// 96 states, FP64, 5.1 ms column by column, 0.39 by rows, 0.24; 500k columns of
// 700 states, FP32, in tiles, 76, 16.6, 4.4; 256 instances (14.9M columns, FP32)
// after the forward 49.6, 8.3, 3.1.
#include "traceback.h"

#include "kernel_util.h"

namespace aw {

namespace {

// waves of a tile's workgroup.  BIG: 32 states per lane, whose rows need the
// registers of twice the waves
template <bool BIG>
constexpr int tb_waves()
{
    return BIG ? 8 : 16;
}

// columns per unit, at most 63: one lane each, and one for the switch after
// them.  Blocks average 10-55 columns; 48 and 32 are 2-10 % slower.
constexpr int TB_SEG = 63;
constexpr unsigned TB_NONE = 0xffff;   // no predicted source

// LDS: per-unit results, then the units' source tables
constexpr int TB_RES = 6;
enum : int { RES_OUT = 0, RES_HYP, RES_FLAG, RES_NEXT, RES_BLK, RES_MATCH };
enum : int { UNIT_LIVE = 1, UNIT_FINAL = 2 };

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// inclusive prefix sum over the 64 lanes: Hillis-Steele inside each 16-lane
// row, then the totals of the rows before
__device__ __forceinline__ double incl_scan(double v)
{
    v += dpp_r<DPP_ROW_SHR1>(v);
    v += dpp_r<DPP_ROW_SHR2>(v);
    v += dpp_r<DPP_ROW_SHR4>(v);
    v += dpp_r<DPP_ROW_SHR8>(v);
    const double t0 = readlane_d(v, 15), t1 = readlane_d(v, 31), t2 = readlane_d(v, 47);
    const int row = lane_id() >> 4;
    double off = 0.0;
    if (row >= 1) off = t0;
    if (row >= 2) off += t1;
    if (row >= 3) off += t2;
    return v + off;
}

// First index k of the lane-run weights (lane l holds states l*R..l*R+R-1)
// whose cumulative sum reaches u * total; S-1 if none does.  The products
// are in the table's precision, the cumulative sums FP64.  Branch-free: the
// owner lane counts the prefixes below the pick.
template <class Real, int R>
__device__ __forceinline__ int sample_state(const Real (&rv)[R], const Real (&tr)[R], int S, double u)
{
    const int lane = lane_id();
    double pre[R];
    double acc = 0.0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        acc += (double)(rv[r] * tr[r]);
        pre[r] = acc;
    }
    const double inc = incl_scan(acc);
    const double excl = dpp_r<DPP_WAVE_SHR1>(inc);
    const double pick = u * readlane_d(inc, 63);
    const unsigned long long m = __ballot(lane * R < S && excl + acc >= pick);
    const int owner = m ? (int)__ffsll((long long)m) - 1 : (S - 1) / R;
    const int nloc = min(R, S - lane * R);
    const double thr = pick - excl;
    int cnt = 0;
#pragma unroll
    for (int r = 0; r < R; r++) cnt += (pre[r] < thr) ? 1 : 0;
    const int rsel = m ? min(cnt, nloc - 1) : nloc - 1;
    return __builtin_amdgcn_readlane(lane * R + rsel, owner);
}

template <class Real, int R>
__device__ __forceinline__ void row_load(const AW_GLOBAL Real *alpha, int col, Real (&rv)[R])
{
    slots_load<R>(alpha + (size_t)col * (64 * R), lane_id(), rv);
}

// state sampled from column col alone (the last column, or the speculative
// start of a tile); every wave of the workgroup computes it
template <class Real, int R>
__device__ __forceinline__ int sample_alone(const DevInst &d, int col, int b, double u)
{
    Real rv[R], one[R];
    row_load<Real, R>((const AW_GLOBAL Real *)d.alpha, col, rv);
#pragma unroll
    for (int r = 0; r < R; r++) one[r] = Real(1);   // padding slots hold 0
    return sample_state<Real, R>(rv, one, cp(d.soff)[b + 1] - cp(d.soff)[b], u);
}

// The transition into state k within block b, as one register: lane a < 32
// holds P(a -> time of k) from another branch, lane 32 + a from k's own.
// (lk, rk) are k's lane and slot, node its branch.
template <class Real>
struct Target {
    int k, lk, rk, node, time;
    Real tab;
};

template <class Real, int R>
__device__ __forceinline__ Target<Real> tb_target(const DevInst &d, int b, int k)
{
    const int lane = lane_id(), T1 = d.T - 1, TT = T1 * T1;
    Target<Real> t;
    t.k = k;
    t.lk = k / R;
    t.rk = k % R;
    const int info = cp(d.linfo)[(size_t)b * (64 * R) + lane_pos(k, R)];
    t.node = info_node(info);
    t.time = info & INFO_TIME;
    const int c = info_age(info), a = min(lane & 31, T1 - 1);
    const AW_GLOBAL double *tm = gp(d.tm) + (size_t)b * TT;
    const AW_GLOBAL double *vec = gp(d.tvec) + (size_t)b * time_vecs(T1);
    const AW_GLOBAL double *other = tm + (a * T1 + t.time);
    const double same = same_entry(vec, T1, a, t.time, c, other);
    t.tab = (Real)(lane < 32 ? *other : same);
    return t;
}

// per-slot weights P(state -> k); padding slots carry time bin 31 and meet
// zeros of the table: their index is clamped into it
template <class Real, int R>
__device__ __forceinline__ void tb_weights(const DevInst &d, const int (&ti)[R],
                                           const Target<Real> &t, Real (&tr)[R])
{
    const int T1 = d.T - 1;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int a = min(ti[r] & INFO_TIME, T1 - 1);
        tr[r] = bperm_r(t.tab, 4 * (a + (info_node(ti[r]) == t.node ? 32 : 0)));
    }
}

// Table entries below this may have lost bits to underflow: such columns are
// sampled from their rows.
template <class Real>
constexpr double tb_small()
{
    return sizeof(Real) == 4 ? 1e-30 : 1e-280;
}

// Whether the state j of column c, with entry a0 and transition weight w into
// state k of column c+1, is certainly the sample for the uniform u.  v1: the
// entry of k in column c+1 before normalisation, which by the recursion is
// e * (sum over the states of column c of entry * weight), e being k's emission
// there.  Cumulative sums below j lie between 0 and the total less j's share.
template <class Real>
__device__ __forceinline__ bool tb_certain(double a0, double w, double v1, double e, double u)
{
    const double at = a0 * w * e, guard = v1 * 0x1p-13;
    return v1 >= tb_small<Real>() && u * v1 > (v1 - at) + guard && u * v1 < at - guard;
}

// One unit: the state of column ce is k; sample the n columns ce-1 .. ce-n
// of block b, and with sw the column ce-n-1 of block b-1.  uw: lane j holds
// the uniform of column ce-1-j.  pv receives the sampled states, lane j that
// of column ce-1-j; returns the last one.
template <class Real, int R>
__device__ __forceinline__ int tb_unit(const DevInst &d, int b, int ce, int n, bool sw, int k,
                                       double uw, int &pv)
{
    constexpr int RW = 64 * R;
    const int lane = lane_id();
    const AW_GLOBAL Real *alpha = (const AW_GLOBAL Real *)d.alpha;
    const AW_GLOBAL Real *pl = planes<Real>(d, b, RW);
    const int S = cp(d.soff)[b + 1] - cp(d.soff)[b];
    // lane j: the transition from column ce-1-j to the next, the switch last
    const int c = max(ce - 1 - min(lane, n), 0);
    const double norm = gp(d.norms)[c + 1];
    const int cls = gp(d.cls)[c + 1];
    // FP32: a column that is not the recursion of the one stored before it
    bool cut = false;
    if (sizeof(Real) == 4) cut = gp(d.cut)[(c + 1) >> 5] >> ((c + 1) & 31) & 1;
    // emission of state position p in column c + 1
    auto emission = [&](int p) -> double {
        double e = 1.0;
        if (cls == -1) e = pl[CE * RW + p];
        if (cls >= 0) e = gp(d.vemit)[(size_t)cls * RW + p];
        return e;
    };
    pv = k;
    int pos = 0;
    while (pos < n) {
        const Target<Real> t = tb_target<Real, R>(d, b, k);
        const int pk = lane_pos(k, R);
        const double a0 = alpha[(size_t)c * RW + pk], a1 = alpha[(size_t)(c + 1) * RW + pk];
        const bool stay = !cut && tb_certain<Real>(a0, readlane_r(t.tab, 32 + t.time), a1 * norm,
                                                   emission(pk), uw);
        unsigned long long odd = __ballot(lane >= pos && lane < n && !stay);
        pos = n;
        while (odd) {
            const int x = (int)__ffsll((long long)odd) - 1;
            Real rv[R], tr[R];
            int ti[R];
            row_load<Real, R>(alpha, ce - 1 - x, rv);
            slots_load<R>((const AW_GLOBAL int *)gp(d.linfo) + (size_t)b * RW, lane, ti);
            tb_weights<Real, R>(d, ti, t, tr);
            const int kn = sample_state<Real, R>(rv, tr, S, readlane_d(uw, x));
            if (kn != k) {
                k = kn;
                pv = lane >= x ? k : pv;
                pos = x + 1;
                break;
            }
            odd &= odd - 1;
        }
    }
    if (sw) {
        // the switch into block b (TransMatrixSwitch::get, trans.h:201-209)
        const int rs = cp(d.srcs)[2 * b], cs = cp(d.srcs)[2 * b + 1];
        const AW_GLOBAL int *detn = (const AW_GLOBAL int *)gp(d.ldet) + (size_t)b * RW;
        const int pk = lane_pos(k, R);
        const Real rrk = pl[CRR * RW + pk], crk = pl[CCR * RW + pk];
        // (-1 stays no state)
        auto weight = [&](int s, int dt, Real dp) {
            return (s == cs) ? crk : (s == rs) ? rrk : ((dt & ~DET_SHARED) == k ? dp : Real(0));
        };
        const double u = readlane_d(uw, n);
        const int j = gp(d.pred)[(size_t)b * RW + k];
        bool sure = false;
        if (j != (int)TB_NONE) {
            // (in every lane, lane n has the column's values)
            const int pj = lane_pos(j, R);
            const double a0 = alpha[(size_t)c * RW + pj], a1 = alpha[(size_t)(c + 1) * RW + pk];
            sure = !cut && tb_certain<Real>(a0, weight(j, detn[pj], pl[CDP * RW + pj]), a1 * norm,
                                            emission(pk), u);
        }
        if (__ballot(sure) >> n & 1) {
            k = j;
        } else {
            Real rv[R], tr[R], dp[R];
            int dt[R];
            row_load<Real, R>(alpha, ce - n - 1, rv);
            slots_load<R>(detn, lane, dt);
            slots_load<R>(pl + CDP * RW, lane, dp);
#pragma unroll
            for (int r = 0; r < R; r++) tr[r] = weight(lane * R + r, dt[r], dp[r]);
            k = sample_state<Real, R>(rv, tr, cp(d.soff)[b] - cp(d.soff)[b - 1], u);
        }
        pv = lane >= n ? k : pv;
    }
    return k;
}

// Sample columns hi, hi-1, .., lo given the state k at column hi+1 (block
// blk), storing the samples in dst (nothing when dst is null).  With cmp the
// walk stops at the first column whose sample is the
// one already stored in dst (the chains have met: the rest is that path) and
// returns it; else it returns -1, k being the state of column lo.  The
// uniform of column col is u[L-1-col].  Called by the whole workgroup with
// the same arguments.
template <class Real, int R, int NW>
__device__ __forceinline__ int tb_walk(const DevInst &d, int *lds, int hi, int lo, int &k, int blk,
                                       AW_GLOBAL int *dst, bool cmp)
{
    constexpr int RW = 64 * R;
    const int lane = lane_id(), L = d.L;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int *res = lds;
    unsigned *pred = (unsigned *)(lds + TB_RES * NW);   // NW tables of RW 16-bit states
    const AW_GLOBAL double *ug = gp(d.u);
    const AW_GLOBAL int *bstart = gp(d.bstart);
    int cur = hi + 1, kc = k, bc = blk;
    // lane i holds the first column of block bw - i
    int bw = bc, bsv = bstart[max(bw - lane, 0)];
    while (cur > lo) {
        if (bw - bc > 63 - NW) {
            bw = bc;
            bsv = bstart[max(bw - lane, 0)];
        }
        // this wave's unit: the wave-th run of columns to the left of cur,
        // each within one block and at most TB_SEG long
        int ce = cur, b = bc, ct = 0, nce = 0, nb = 0;
        bool sw = false, live = false;
        unsigned swm = 0;   // units before this one that end in a switch
        for (int i = 0;; i++) {
            const int bs = __builtin_amdgcn_readlane(bsv, bw - b);
            ct = max(max(bs, lo), ce - TB_SEG);
            sw = ct == bs && ct > lo;
            nce = sw ? ct - 1 : ct;
            nb = sw ? b - 1 : b;
            if (i == wave) {
                live = true;
                break;
            }
            if (nce <= lo) break;
            if (sw) swm |= 1u << i;
            ce = nce;
            b = nb;
        }
        const int n = ce - ct;
        double uw = 0.0;
        int old = -1;
        if (live) {
            const int c = max(ce - 1 - lane, 0);
            uw = ug[L - 1 - c];
            if (cmp) old = dst[max(c, lo)];
            if (sw && wave < NW - 1) {
                const AW_GLOBAL unsigned *src =
                    (const AW_GLOBAL unsigned *)gp(d.pred) + (size_t)b * (RW / 2);
                for (int x = lane; x < RW / 2; x += 64) pred[wave * (RW / 2) + x] = src[x];
            }
        }
        __syncthreads();
        // the predicted entry state
        unsigned h = (unsigned)kc;
        for (int i = 0; i < wave && live; i++) {
            if (!(swm >> i & 1)) continue;
            h = __builtin_amdgcn_readfirstlane(
                (int)((const unsigned short *)pred)[i * RW + h]);
            if (h == TB_NONE) live = false;
        }
        int pv = -1, out = -1, match = -1;
        const int nl = sw ? n : n - 1;   // last lane holding a sample
        if (live) {
            out = tb_unit<Real, R>(d, b, ce, n, sw, (int)h, uw, pv);
            if (cmp) {
                const unsigned long long m = __ballot(lane <= nl && old == pv);
                if (m) match = ce - (int)__ffsll((long long)m);
            }
        }
        if (lane == 0) {
            res[RES_OUT * NW + wave] = out;
            res[RES_HYP * NW + wave] = (int)h;
            res[RES_FLAG * NW + wave] = (live ? UNIT_LIVE : 0) | (nce <= lo ? UNIT_FINAL : 0);
            res[RES_NEXT * NW + wave] = nce;
            res[RES_BLK * NW + wave] = nb;
            res[RES_MATCH * NW + wave] = match;
        }
        __syncthreads();
        // the units up to the first whose outcome the next did not assume
        const int i0 = min(lane, NW - 1), i1 = min(lane + 1, NW - 1);
        const int o0 = res[RES_OUT * NW + i0], h1 = res[RES_HYP * NW + i1];
        const int f0 = res[RES_FLAG * NW + i0], f1 = res[RES_FLAG * NW + i1];
        const int m0 = res[RES_MATCH * NW + i0];
        const bool ok = lane < NW - 1 && !(f0 & UNIT_FINAL) && (f1 & UNIT_LIVE) && o0 == h1;
        const int last = (int)__ffsll((long long)~__ballot(ok)) - 1;
        int stop = -1;
        if (cmp) {
            const unsigned long long m = __ballot(lane <= last && m0 >= 0);
            if (m) stop = __builtin_amdgcn_readlane(m0, (int)__ffsll((long long)m) - 1);
        }
        if (wave <= last && dst) {
            const int c = ce - 1 - lane;
            if (lane <= nl && c > stop) dst[c] = pv;
        }
        cur = __builtin_amdgcn_readfirstlane(res[RES_NEXT * NW + last]);
        kc = __builtin_amdgcn_readfirstlane(res[RES_OUT * NW + last]);
        bc = __builtin_amdgcn_readfirstlane(res[RES_BLK * NW + last]);
        if (stop >= 0) return stop;
    }
    k = kc;
    return -1;
}

template <class Real, int R, int NW>
__device__ __forceinline__ void tb_spec(const DevInst d, const Chunk &ch, int *start, int *end, int *lds)
{
    const int L = d.L;
    AW_GLOBAL int *path = gp(d.path);
    // the chain's first state: from the last column (or the state it is
    // conditioned on), or from column cw alone
    int b = ch.last ? d.B - 1 : find_owner(cp(d.bstart), d.B, ch.cw);
    int k = d.last_state;
    if (!ch.last || k < 0) k = sample_alone<Real, R>(d, ch.cw, b, cp(d.u)[L - 1 - ch.cw]);
    int k1 = -1;
    if (ch.last && threadIdx.x == 0) path[L - 1] = k;
    // the warm-up (no columns in the last tile), then the tile
#pragma unroll 1
    for (int ph = ch.last ? 1 : 0; ph < 2; ph++) {
        const int top = ph ? (ch.last ? L - 1 : ch.c1) : ch.cw;
        if (ph && !ch.last) {
            k1 = k;
            b = find_owner(cp(d.bstart), d.B, ch.c1);
        }
        tb_walk<Real, R, NW>(d, lds, top - 1, ph ? ch.c0 : ch.c1, k, b, ph ? path : nullptr, false);
    }
    if (threadIdx.x == 0) {
        *start = k1;
        *end = k;
    }
}

template <class Real, int R, int NW>
__device__ __forceinline__ void tb_rerun(const DevInst d, const Chunk &ch, int k, int *res, int *lds)
{
    AW_GLOBAL int *path = gp(d.path);
    const int b = find_owner(cp(d.bstart), d.B, ch.c1);
    const int col = tb_walk<Real, R, NW>(d, lds, ch.c1 - 1, ch.c0, k, b, path, true);
    if (threadIdx.x == 0) {
        res[0] = col;
        res[1] = col >= 0 ? path[ch.c0] : k;
    }
}

// calls f<R>() for the instance's states per lane
#define TB_FOR_R(R_, CALL)                          \
    switch (R_) {                                   \
    case 1: { constexpr int R = 1; CALL; break; }   \
    case 2: { constexpr int R = 2; CALL; break; }   \
    case 4: { constexpr int R = 4; CALL; break; }   \
    case 6: { constexpr int R = 6; CALL; break; }   \
    case 8: { constexpr int R = 8; CALL; break; }   \
    case 12: { constexpr int R = 12; CALL; break; } \
    default: { constexpr int R = 16; CALL; break; } \
    }

template <class Real, bool BIG>
__global__ __launch_bounds__(64 * tb_waves<BIG>()) void k_tb_spec(const DevInst *__restrict__ D,
                                                                  const Chunk *__restrict__ chunks,
                                                                  const int *__restrict__ list,
                                                                  int *__restrict__ start,
                                                                  int *__restrict__ end)
{
    extern __shared__ int tb_dyn[];
    constexpr int NW = tb_waves<BIG>();
    const int j = list[blockIdx.x];
    const Chunk ch = chunks[j];
    const DevInst &d = D[ch.inst];
    if ((d.R > 16) != BIG) return;   // the other symbol's tile
    if constexpr (BIG) tb_spec<Real, 32, NW>(d, ch, start + j, end + j, tb_dyn);
    else TB_FOR_R(d.R, (tb_spec<Real, R, NW>(d, ch, start + j, end + j, tb_dyn)))
}

template <class Real, bool BIG>
__global__ __launch_bounds__(64 * tb_waves<BIG>()) void k_tb_rerun(const DevInst *__restrict__ D,
                                                                   const Chunk *__restrict__ chunks,
                                                                   const int *__restrict__ idx,
                                                                   const int *__restrict__ k1,
                                                                   int *__restrict__ res)
{
    extern __shared__ int tb_dyn[];
    constexpr int NW = tb_waves<BIG>();
    const Chunk ch = chunks[idx[blockIdx.x]];
    const DevInst &d = D[ch.inst];
    const int k = k1[blockIdx.x];
    int *rs = res + 2 * blockIdx.x;
    if ((d.R > 16) != BIG) return;   // the other symbol's tile
    if constexpr (BIG) tb_rerun<Real, 32, NW>(d, ch, k, rs, tb_dyn);
    else TB_FOR_R(d.R, (tb_rerun<Real, R, NW>(d, ch, k, rs, tb_dyn)))
}

// Tables of the switch into a block b.  Predicted sources: for every state k
// of block b the state j of block b-1 with the largest switch probability
// P(j -> k) (ties: the larger index), TB_NONE where no state leads to k.
// Deterministic targets in ldet: marked where they have several sources, and -1
// for the states that the dense rows take.  One workgroup per block; the candidates (deterministic targets,
// then the two dense rows) meet in LDS.
__global__ __launch_bounds__(256) void k_tb_pred(const DevInst *__restrict__ D,
                                                 const int *__restrict__ blkoff, int ninst)
{
    extern __shared__ unsigned long long best[];   // RW keys, then RW counts
    const int inst = find_owner(blkoff, ninst, (int)blockIdx.x);
    const DevInst &d = D[inst];
    const int b = blockIdx.x - blkoff[inst];
    if (b == 0) return;
    const int R = d.R, RW = 64 * R;
    int *count = (int *)(best + RW);
    const int S1 = cp(d.soff)[b] - cp(d.soff)[b - 1], S2 = cp(d.soff)[b + 1] - cp(d.soff)[b];
    const int rs = cp(d.srcs)[2 * b], cs = cp(d.srcs)[2 * b + 1];
    auto weight = [&](int plane, int p) -> float {
        const size_t x = ((size_t)b * NCOEF + plane) * RW + p;
        return d.fp32 ? gp(d.lcoef32)[x] : (float)gp(d.lcoef)[x];
    };
    auto key = [](float w, int j) {
        return (unsigned long long)__float_as_uint(w) << 32 | (unsigned)(j + 1);
    };
    auto det = gp(d.ldet) + (size_t)b * RW;
    for (int x = threadIdx.x; x < RW; x += 256) {
        best[x] = 0;
        count[x] = 0;
    }
    __syncthreads();
    auto source = [&](int p, int t) {   // a deterministic transition into t
        const int j = pos_state(p, R);
        return j < S1 && t >= 0 && t < S2 && j != rs && j != cs;
    };
    for (int p = threadIdx.x; p < RW; p += 256) {
        const int t = det[p];
        if (source(p, t)) {
            atomicMax(&best[t], key(weight(CDP, p), pos_state(p, R)));
            atomicAdd(&count[t], 1);
        }
    }
    __syncthreads();
    for (int p = threadIdx.x; p < RW; p += 256) {
        const int t = det[p];
        if (!source(p, t)) det[p] = -1;
        else if (count[t] > 1) det[p] = t | DET_SHARED;
    }
    auto out = gp(d.pred) + (size_t)b * RW;
    for (int p = threadIdx.x; p < RW; p += 256) {
        const int k = pos_state(p, R);
        unsigned long long m = best[k];
        if (rs >= 0) {
            const float w = weight(CRR, p);
            if (w > 0.f) m = max(m, key(w, rs));
        }
        if (cs >= 0) {
            const float w = weight(CCR, p);
            if (w > 0.f) m = max(m, key(w, cs));
        }
        out[k] = m ? (unsigned short)((unsigned)m - 1) : (unsigned short)TB_NONE;
    }
}

template <class Kern, class... Args>
int launch(Kern kern, int grid, int block, size_t sh, hipStream_t st, Args... args)
{
    if (set_lds_limit((const void *)kern, sh)) return 1;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(block), sh, st, args...);
    HIP_OK(hipGetLastError());
    return 0;
}

}  // namespace

size_t tb_lds_bytes(int R)
{
    const int NW = R > 16 ? tb_waves<true>() : tb_waves<false>();
    return (size_t)NW * (TB_RES * sizeof(int) + 64 * R * sizeof(short));
}

int launch_tb_pred(const DevInst *D, const int *blkoff, int ninst, int nblk, int Rmax, hipStream_t s)
{
    return launch(k_tb_pred, nblk, 256, (sizeof(unsigned long long) + sizeof(int)) * 64 * Rmax, s, D,
                  blkoff, ninst);
}

int launch_tb_spec(bool fp32, bool big, const DevInst *D, const Chunk *chunks, const int *list,
                   int n, size_t sh, int *start, int *end, hipStream_t s)
{
    const int wg = 64 * (big ? tb_waves<true>() : tb_waves<false>());
    auto kern = fp32 ? (big ? k_tb_spec<float, true> : k_tb_spec<float, false>)
                     : (big ? k_tb_spec<double, true> : k_tb_spec<double, false>);
    return launch(kern, n, wg, sh, s, D, chunks, list, start, end);
}

int launch_tb_rerun(bool fp32, bool big, const DevInst *D, const Chunk *chunks, const int *idx,
                    const int *k1, int n, size_t sh, int *res, hipStream_t s)
{
    const int wg = 64 * (big ? tb_waves<true>() : tb_waves<false>());
    auto kern = fp32 ? (big ? k_tb_rerun<float, true> : k_tb_rerun<float, false>)
                     : (big ? k_tb_rerun<double, true> : k_tb_rerun<double, false>);
    return launch(kern, n, wg, sh, s, D, chunks, idx, k1, res);
}

}  // namespace aw
