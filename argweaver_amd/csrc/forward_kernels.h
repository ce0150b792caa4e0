// forward_kernels.h -- the forward recursion's kernels, instantiated by
// forward_f32.hip and forward_f64.hip.
#pragma once

#include "forward.h"
#include "kernel_util.h"

namespace aw {

//===========================================================================
// forward recursion, one wave per instance (arghmm_forward_alg,
// sample_thread.cpp:394-460; arghmm_forward_block :186-296;
// arghmm_forward_switch :345-389)

// NT1 is a compile-time bound on the T-1 time bins (19 for the usual 20
// time points), so the per-time loops are fully unrolled without padding.
//
// Per block, each lane keeps in registers the factor planes of its R
// states, two 0/1 factors per state (not the first / not the last state of
// its branch: they cut the prefix and suffix sums), and whether the lane
// holds a branch start / end (the carry stops there).  Per state it also
// keeps its time, which gives both the lane holding the other-branch term
// of its time and where its value goes in the per-time partial sums;
// padding states use time bin 31, whose term is 0, so they come out 0 with
// no mask.  The 0/1 factors are floats in both precisions: FP64 runs apply
// them as selects, which keeps their registers at one per state.
template <class Real, int R, int NT1>
struct FwLane {
    Real cf[R], cd[R], cg[R], ck[R], cj[R], ce[R];
    float nf[R], nl[R];
    int boff[R];     // 4 * time: ds_bpermute address of the lane holding TF[time]
    Real m1, m2;
    Real tmc[NT1];   // lane b < T-1: column b of the (a,b) table (FP32)
};

// x times a 0/1 factor m (a select in FP64: the same value)
template <class Real>
__device__ __forceinline__ Real keep(Real x, float m)
{
    if constexpr (sizeof(Real) == 4) return x * m;
    else return (m != 0.f) ? x : Real(0);
}

// The (a,b) table lives in registers (lane b holds column b) for FP32 and
// in LDS for FP64, where registers are short.
template <class Real>
constexpr bool tm_in_lds()
{
    return sizeof(Real) == 8;
}

// Per-time sums are accumulated in GCOPY copies of the 32 time bins, one
// copy per group of 64 / GCOPY consecutive lanes, so that the LDS atomics of
// one instruction seldom meet at one address (colliding atomics are
// serialised).  Bin a, copy c sits at GP[a * GCOPY + c].  The sums are FP64
// in both precisions: ds_add_f64 is much faster than ds_add_f32 here.
constexpr int GCOPY = 16;

template <class Real, int R, int NT1>
__device__ __forceinline__ void fw_load_block(const DevInst &d, int b, FwLane<Real, R, NT1> &fl,
                                              Real *TMS)
{
    constexpr int RW = 64 * R;
    const int lane = threadIdx.x, T1 = d.T - 1;
    // uniform bases, per-lane index: loads use the scalar-base address form
    const AW_GLOBAL Real *coef = planes<Real>(d, b, RW);
    const AW_GLOBAL int *info = gp(d.linfo) + (size_t)b * RW;
    int ti[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int x = r * 64 + lane;
        fl.cf[r] = coef[CF * RW + x];
        fl.cd[r] = coef[CD * RW + x];
        fl.cg[r] = coef[CG * RW + x];
        fl.ck[r] = coef[CK * RW + x];
        fl.cj[r] = coef[CJ * RW + x];
        fl.ce[r] = coef[CE * RW + x];
        ti[r] = info[x];
    }
    bool first = false, last = false;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int t = ti[r] & INFO_TIME;
        fl.nf[r] = (ti[r] & INFO_FIRST) ? 0.f : 1.f;
        fl.nl[r] = (ti[r] & INFO_LAST) ? 0.f : 1.f;
        fl.boff[r] = t * 4;
        first |= (ti[r] & INFO_FIRST) != 0;
        last |= (ti[r] & INFO_LAST) != 0;
    }
    fl.m1 = first ? Real(0) : Real(1);
    fl.m2 = last ? Real(0) : Real(1);
    // Loaded values go straight into their registers: selecting or copying
    // a value whose load is still in flight makes the compiler wait for it
    // at once.  Indices are clamped instead; entries a >= T-1 meet a zero
    // per-time sum and lanes >= T-1 compute terms nobody uses.
    const AW_GLOBAL double *tmb = gp(d.tm) + (size_t)b * T1 * T1;
    const int lc = min(lane, T1 - 1);
    if (tm_in_lds<Real>()) {
        // TMS[a * 32 + b] = P(a -> b); lanes 32..63 duplicate lanes 0..31
        double t[NT1];
#pragma unroll
        for (int a = 0; a < NT1; a++) t[a] = tmb[min(a, T1 - 1) * T1 + lc];
#pragma unroll
        for (int a = 0; a < NT1; a++)
            if (lane < 32) TMS[a * 32 + lane] = (Real)t[a];
    } else {
#pragma unroll
        for (int a = 0; a < NT1; a++) fl.tmc[a] = (Real)tmb[min(a, T1 - 1) * T1 + lc];
    }
}

// variant row v, clamped to the last row (an instance without variant
// columns has one allocated row that is never used)
template <int R>
__device__ __forceinline__ void vrow_load(const DevInst &d, int v, double (&ev)[R])
{
    constexpr int RW = 64 * R;
    const AW_GLOBAL double *row = gp(d.vemit) + (size_t)max(min(v, d.nvar - 1), 0) * RW;
#pragma unroll
    for (int r = 0; r < R; r++) ev[r] = row[r * 64 + threadIdx.x];
}

// 1 / x: FP32 tables use the hardware reciprocal (within 1 ulp; the
// normaliser itself, and so the log-likelihood, is kept exactly), FP64
// tables the correctly rounded division
__device__ __forceinline__ float recip(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double recip(double x) { return 1.0 / x; }

template <class Real>
__device__ __forceinline__ void lds_add(Real *p, Real v)
{
    (void)atomicAdd(p, v);
}

// variant rows staged per LDS refill (at most 16 KB of them), and rows per
// load batch of a refill (bounded by the registers they take)
template <class Real, int R>
constexpr int fw_vst()
{
    return (16384 / (64 * R * (int)sizeof(Real))) < 8 ? (16384 / (64 * R * (int)sizeof(Real))) : 8;
}
template <class Real, int R>
constexpr int fw_vch()
{
    return (32 / R) < 2 ? 2 : (32 / R) > fw_vst<Real, R>() ? fw_vst<Real, R>() : (32 / R);
}

// LDS of the forward kernel, in Reals: partial sums, the previous column in
// state order, the switch targets (plus one dummy slot per lane), staged
// variant rows, the (a,b) table
template <class Real, int R>
constexpr int fw_lds_reals()
{
    return 32 * GCOPY * (int)(sizeof(double) / sizeof(Real)) + 64 * R + (64 * R + 64) +
           fw_vst<Real, R>() * 64 * R + 31 * 32;
}

// wave-wide maximum
__device__ __forceinline__ double wave_max(double x)
{
    for (int off = 32; off > 0; off >>= 1) x = fmax(x, __shfl_xor(x, off));
    return x;
}

// columns between the checks of a re-run tile against its stored columns
constexpr int FW_RECHECK = 128;

template <class Real, int R, int NT1>
__device__ __forceinline__ void fw_instance(const DevInst d, Real *sm, const FwTile tile,
                                            AW_GLOBAL Real *bnd, AW_GLOBAL double *bnorm,
                                            double tol, AW_GLOBAL int *early)
{
    constexpr int RW = 64 * R;
    constexpr int VST = fw_vst<Real, R>();
    constexpr int VCH = fw_vch<Real, R>();
    const int lane = threadIdx.x;
    const int T1 = d.T - 1, L = d.L;
    // carry steps: a branch has at most T-1 states, so it reaches back at
    // most ceil((T-2)/R) lanes from the lane holding its last state
    const int K = (T1 - 1 + R - 1) / R;
    double *GP = (double *)sm;       // 32 x GCOPY: per-time partial sums
    // byte offset of this lane's copy within a time bin's GCOPY copies
    const int gslot = (lane / (64 / GCOPY)) * (int)sizeof(double);
    // the half of bin lane>>1 that this lane reduces, and its read rotation
    double *gq = GP + (lane >> 1) * GCOPY + (lane & 1) * (GCOPY / 2);
    const int grot = (lane >> 1) & (GCOPY / 2 - 1);
    Real *XS = (Real *)(GP + 32 * GCOPY);   // RW: previous column in state order (switch)
    Real *NW = XS + RW;              // RW + 64: switch targets, then a dummy slot per lane
    Real *VS = NW + RW + 64;         // VST rows: staged variant-column emissions
    Real *TMS = VS + VST * RW;       // 31 x 32: the (a,b) table (FP64)
    AW_GLOBAL Real *alpha = (AW_GLOBAL Real *)d.alpha;
    auto norms = gp(d.norms);

    const int c0 = tile.c0, cs = tile.cs;
    // the last column computed: c1 - 1, or c1 into the boundary slot
    const int clast = tile.bout >= 0 ? tile.c1 : tile.c1 - 1;
    FwLane<Real, R, NT1> fl;
    int b = find_owner(cp(d.bstart), d.B, c0);
    int bend = cp(d.bstart)[b] + cp(d.blen)[b];
    fw_load_block<Real, R, NT1>(d, b, fl, TMS);
#pragma unroll
    for (int k = 0; k < 32 * GCOPY / 64; k++) GP[k * 64 + lane] = 0.0;
    // Column classes of a window of 64 columns, one per lane, read with
    // readlane; the next window's are loaded a window ahead.  vmcnt counts
    // the table stores too, so any wait on a load inside the column loop
    // would also wait for the stores of the column before: the windows are
    // an outer loop, and the one wait per window is taken there.
    const AW_GLOBAL int *clsg = gp(d.cls);
    int wb = c0 & ~63;
    int clsv = clsg[min(wb + lane, L - 1)];
    int clsn = clsg[min(wb + 64 + lane, L - 1)];
    // Variant rows (row index = the column's class) are consumed in order
    // and staged in LDS, VST at a time, so that a refill costs a few waits
    // and the columns read their row from LDS.
    int vbase = 0, vend = 0;

    Real x[R], tfs[R], v[R];
    Real sc = Real(1);   // the previous column is x * sc

    // A re-run tile (mode 2) stops once a column it computes agrees with
    // the column stored by its speculative run (relative tolerance tol):
    // the filter is contractive, so the stored columns after it, the
    // normalisers and the boundary column stay within tolerance.
    bool rejoined = false;

    // per-time sums, normaliser, stored row, other-branch term of the next
    // column
    auto finish = [&](int col, bool first) {
#pragma unroll
        for (int r = 0; r < R; r++)
            lds_add((double *)((char *)GP + fl.boff[r] * (2 * GCOPY) + gslot), (double)v[r]);
        // lane l takes the copies of bin l>>1 in its half (l&1), leaving 0
        // (one exchange each; the LDS operations of one wave run in order).
        // Step k reads copy (k + l/2) mod 8 of the half: the lanes of one
        // step then spread over the banks (copy k of every bin would sit in
        // two banks), which also fixes each lane's summation order
        double q[GCOPY / 2];
#pragma unroll
        for (int k = 0; k < GCOPY / 2; k++)
            q[k] = __longlong_as_double((long long)__hip_atomic_exchange(
                (unsigned long long *)(gq + ((k + grot) & (GCOPY / 2 - 1))), 0ull,
                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
#pragma unroll
        for (int w = 1; w < GCOPY / 2; w *= 2)
#pragma unroll
            for (int k = 0; k < GCOPY / 2; k += 2 * w) q[k] += q[k + w];
        const Real g = (Real)(q[0] + dpp_r<DPP_QUAD_SWAP1>(q[0]));   // lanes 2a, 2a+1: G[a]
        // four interleaved partial sums keep the dependency chains short
        Real nq[4] = {Real(0), Real(0), Real(0), Real(0)};
        Real tq[4] = {Real(0), Real(0), Real(0), Real(0)};
#pragma unroll
        for (int a = 0; a < NT1; a++) {
            const Real ga = readlane_r(g, 2 * a);
            nq[a & 3] += ga;
            tq[a & 3] += ga * (tm_in_lds<Real>() ? TMS[a * 32 + (lane & 31)] : fl.tmc[a]);
        }
        const Real norm = (nq[0] + nq[1]) + (nq[2] + nq[3]);
        const Real t = (tq[0] + tq[1]) + (tq[2] + tq[3]);
        // column 0 is stored unnormalised (scale 1); a restarted tile's first
        // column is the boundary column as stored by the tile before
        const Real nsc = (col == 0 || (first && tile.mode == 2)) ? Real(1) : recip(norm);
        if (col >= cs && col < tile.c1) {
            AW_GLOBAL Real *row = alpha + (size_t)col * RW;
            if (tile.mode == 2 && !first && (col - tile.c0) % FW_RECHECK == 0) {
                double dmax = 0.0, amax = 0.0;
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const double nv = (double)(v[r] * nsc), ov = (double)row[r * 64 + lane];
                    dmax = fmax(dmax, fabs(nv - ov));
                    amax = fmax(amax, fabs(nv));
                }
                dmax = wave_max(dmax);
                amax = wave_max(amax);
                rejoined = dmax <= tol * amax;
            }
#pragma unroll
            for (int r = 0; r < R; r++) row[r * 64 + lane] = v[r] * nsc;
            if (lane == 0) {
                double nv = (col == 0) ? ((L == 1) ? (double)norm : 1.0) : (double)norm;
                if (first && tile.mode == 2) nv = bnorm[tile.bin];
                norms[col] = nv;
            }
        } else if (col == tile.c1) {
            AW_GLOBAL Real *row = bnd + (size_t)tile.bout * BND_STRIDE;
#pragma unroll
            for (int r = 0; r < R; r++) row[r * 64 + lane] = v[r] * nsc;
            if (lane == 0) bnorm[tile.bout] = (double)norm;
        }
        // TF[b] lives in lane b; lanes >= T-1 (padding bin 31) hold 0
        const Real tv = (lane < T1) ? t * nsc : Real(0);
#pragma unroll
        for (int r = 0; r < R; r++) {
            tfs[r] = bperm_r(tv, fl.boff[r]);
            x[r] = v[r];
        }
        sc = nsc;
    };

    // first column.  mode 0: the unnormalised prior, not multiplied by the
    // emission (calc_state_priors, trans.cpp:785-831); padding positions
    // hold 0.  mode 1: 1 on every state.  mode 2: the boundary column.
    if (tile.mode == 0) {
        const AW_GLOBAL double *pr = gp(d.lprior);
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = (Real)pr[r * 64 + lane];
    } else if (tile.mode == 1) {
        const int S = cp(d.soff)[b + 1] - cp(d.soff)[b];
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = (lane * R + r < S) ? Real(1) : Real(0);
    } else {
        const AW_GLOBAL Real *src = bnd + (size_t)tile.bin * BND_STRIDE;
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = src[r * 64 + lane];
    }
    finish(c0, true);

    // an empty asm reading the register makes the compiler complete its
    // load here rather than at a use inside the column loop
    asm volatile("" : "+v"(clsv));
    int col = c0 + 1;
    while (col <= clast && !rejoined) {
        if (col >= wb + 64) {
            wb += 64;
            clsv = clsn;
            asm volatile("" : "+v"(clsv));
            clsn = clsg[min(wb + 64 + lane, L - 1)];
        }
        const int wend = min(wb + 63, clast);
    for (; col <= wend; col++) {
        const int cls = __builtin_amdgcn_readlane(clsv, col & 63);
        const bool var = cls >= 0;
        Real ev[R];
        if (var) {
            if (cls >= vend) {
                vbase = cls;
                vend = min(cls + VST, d.nvar);
#pragma unroll
                for (int k0 = 0; k0 < VST; k0 += VCH) {
                    // VST need not be a multiple of VCH
                    double buf[VCH][R];
#pragma unroll
                    for (int k = 0; k < VCH; k++)
                        if (k0 + k < VST) vrow_load<R>(d, vbase + k0 + k, buf[k]);
#pragma unroll
                    for (int k = 0; k < VCH; k++)
#pragma unroll
                        for (int r = 0; r < R; r++)
                            if (k0 + k < VST) VS[(k0 + k) * RW + r * 64 + lane] = (Real)buf[k][r];
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) ev[r] = VS[(cls - vbase) * RW + r * 64 + lane];
        }

        if (col == bend) {
            // switch column: deterministic transitions scattered into NW
            // (the recombination and recoalescence sources excluded), then
            // the two dense rows.  Every load of the column is issued before
            // the first use, branch-free, so the column waits once.
            const int nb = b + 1;
            const int so0 = cp(d.soff)[b], so1 = cp(d.soff)[nb];
            const int S1 = so1 - so0, S2 = cp(d.soff)[nb + 1] - so1;
            const int rs = cp(d.srcs)[2 * nb], cs = cp(d.srcs)[2 * nb + 1];
            const AW_GLOBAL Real *swn = planes<Real>(d, nb, RW);
            const AW_GLOBAL int *detn = gp(d.ldet) + (size_t)nb * RW;
            int dt[R];
            Real dpv[R], rr[R], cr[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int x = r * 64 + lane;
                dt[r] = detn[x];
                dpv[r] = swn[CDP * RW + x];
                rr[r] = swn[CRR * RW + x];
                cr[r] = swn[CCR * RW + x];
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                XS[lane * R + r] = x[r];   // padding slots (s >= S1) are never read
                NW[r * 64 + lane] = Real(0);
            }
            b = nb;
            bend += cp(d.blen)[nb];
            fw_load_block<Real, R, NT1>(d, b, fl, TMS);
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int s = lane * R + r;
                const bool ok = s < S1 && dt[r] >= 0 && s != rs && s != cs;
                lds_add(&NW[ok ? dt[r] : RW + lane], ok ? x[r] * dpv[r] : Real(0));
            }
            const Real prs = (rs != -1) ? XS[max(rs, 0)] * sc : Real(0);
            const Real pcs = (cs != -1) ? XS[max(cs, 0)] * sc : Real(0);
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int s = lane * R + r;
                const Real e = var ? ev[r] : (cls == -1) ? fl.ce[r] : Real(1);
                Real acc = (s < S2) ? NW[s] * sc : Real(0);
                if (rs != -1 && rr[r] > Real(0)) acc += prs * rr[r];
                if (cs != -1 && cr[r] > Real(0)) acc += pcs * cr[r];
                v[r] = (s < S2) ? acc * e : Real(0);
            }
        } else {
            // same-branch prefix sums (younger states) with the carry from
            // the lanes before, suffix sums (older states) with the carry
            // from the lanes after
            Real P[R], Q[R];
            Real p = Real(0);
#pragma unroll
            for (int r = 0; r < R; r++) {
                P[r] = keep(p, fl.nf[r]);
                p = fl.cf[r] * x[r] + P[r];
            }
            Real q = Real(0);
#pragma unroll
            for (int r = R - 1; r >= 0; r--) {
                Q[r] = keep(q, fl.nl[r]);
                q = fl.cd[r] * x[r] + Q[r];
            }
            Real c1 = Real(0), c2 = Real(0);
            for (int k = 0; k < K; k++) {
                c1 = dpp_r<DPP_WAVE_SHR1>(fl.m1 * c1 + p);
                c2 = dpp_r<DPP_WAVE_SHL1>(fl.m2 * c2 + q);
            }
            // the carry reaches the slots before the lane's first branch
            // start (prefix) / after its last branch end (suffix)
            Real f1 = Real(1);
#pragma unroll
            for (int r = 0; r < R; r++) {
                f1 = keep(f1, fl.nf[r]);
                P[r] += c1 * f1;
            }
            Real f2 = Real(1);
#pragma unroll
            for (int r = R - 1; r >= 0; r--) {
                f2 = keep(f2, fl.nl[r]);
                Q[r] += c2 * f2;
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                const Real e = var ? ev[r] : (cls == -1) ? fl.ce[r] : Real(1);
                const Real same = (fl.cg[r] * P[r] + fl.ck[r] * Q[r]) + fl.cj[r] * x[r];
                v[r] = e * (tfs[r] + sc * same);
            }
        }
        finish(col, false);
        if (rejoined) break;
    }
    }
    // the column after the one that rejoined (never 0), else 0
    if (early && lane == 0) *early = rejoined ? col + 1 : 0;
}

// One launch covers every instance of a batch, whatever its states-per-lane
// count: waves of different R run side by side from the start, with no
// dependence on how streams map to hardware queues.
// REDO marks the launches of re-run tiles (a separate symbol, so that
// profiles report the main forward launch on its own).  BIG: the instances
// with 32 states per lane (blocks of 1025-2048 states) run in a symbol of
// their own, launched over the same tiles, so that their register demand
// (spilled to AGPRs and scratch) does not weigh on the others.
template <class Real, int NT1, bool REDO, bool BIG>
__global__ __launch_bounds__(64) void k_fw_all(const DevInst *__restrict__ D,
                                               const FwTile *__restrict__ tiles,
                                               Real *__restrict__ bnd, double *__restrict__ bnorm,
                                               double tol, int *__restrict__ early)
{
    extern __shared__ __align__(16) double fw_dyn[];
    const FwTile t = tiles[blockIdx.x];
    const DevInst &d = D[t.inst];
    Real *sm = (Real *)fw_dyn;
    AW_GLOBAL Real *bg = (AW_GLOBAL Real *)bnd;
    AW_GLOBAL double *ng = (AW_GLOBAL double *)bnorm;
    AW_GLOBAL int *eg = early ? (AW_GLOBAL int *)(early + blockIdx.x) : nullptr;
    if ((d.R > 16) != BIG) return;   // the other symbol's tile
    if constexpr (BIG) {
        fw_instance<Real, 32, NT1>(d, sm, t, bg, ng, tol, eg);
    } else {
        switch (d.R) {
        case 1: fw_instance<Real, 1, NT1>(d, sm, t, bg, ng, tol, eg); break;
        case 2: fw_instance<Real, 2, NT1>(d, sm, t, bg, ng, tol, eg); break;
        case 4: fw_instance<Real, 4, NT1>(d, sm, t, bg, ng, tol, eg); break;
        case 6: fw_instance<Real, 6, NT1>(d, sm, t, bg, ng, tol, eg); break;
        case 8: fw_instance<Real, 8, NT1>(d, sm, t, bg, ng, tol, eg); break;
        case 12: fw_instance<Real, 12, NT1>(d, sm, t, bg, ng, tol, eg); break;
        default: fw_instance<Real, 16, NT1>(d, sm, t, bg, ng, tol, eg); break;
        }
    }
}

// Check of a speculative forward tile's start: the boundary column computed
// by the tile before (slot bin) against the tile's own stored column c0,
// both normalised.  flag = 1 when they differ by more than tol relative to
// the column's largest entry, or the normalisers by more than tol.
template <class Real>
__global__ __launch_bounds__(64) void k_fw_check(const DevInst *__restrict__ D,
                                                 const FwTile *__restrict__ tiles,
                                                 const int *__restrict__ idx,
                                                 const Real *__restrict__ bnd,
                                                 const double *__restrict__ bnorm, double tol,
                                                 int *__restrict__ flags)
{
    const FwTile t = tiles[idx[blockIdx.x]];
    const DevInst &d = D[t.inst];
    const int RW = 64 * d.R, lane = threadIdx.x;
    const Real *a = (const Real *)d.alpha + (size_t)t.cs * RW;
    const Real *q = bnd + (size_t)t.bin * BND_STRIDE;
    double dmax = 0.0, amax = 0.0;
    for (int x = lane; x < RW; x += 64) {
        dmax = fmax(dmax, fabs((double)a[x] - (double)q[x]));
        amax = fmax(amax, fabs((double)q[x]));
    }
    for (int off = 32; off > 0; off >>= 1) {
        dmax = fmax(dmax, __shfl_xor(dmax, off));
        amax = fmax(amax, __shfl_xor(amax, off));
    }
    if (lane == 0) {
        const double n0 = gp(d.norms)[t.cs], n1 = bnorm[t.bin];
        const bool bad = !(dmax <= tol * amax) || !(fabs(n0 - n1) <= tol * fabs(n1));
        flags[blockIdx.x] = bad ? 1 : 0;
    }
}

template <class Real, bool BIG>
int launch_fw(const DevInst *dD, const FwTile *tiles, int cnt, void *bnd, double *bnorm, size_t sh,
              hipStream_t st, int T1max, double tol, int *early)
{
    auto kern = (T1max <= 19) ? k_fw_all<Real, 19, false, BIG> : k_fw_all<Real, MAXT - 1, false, BIG>;
    if constexpr (sizeof(Real) == 4)
        if (early) kern = (T1max <= 19) ? k_fw_all<Real, 19, true, BIG> : k_fw_all<Real, MAXT - 1, true, BIG>;
    if (set_lds_limit((const void *)kern, sh)) return 1;
    hipLaunchKernelGGL(kern, dim3(cnt), dim3(64), sh, st, dD, tiles, (Real *)bnd, bnorm, tol, early);
    HIP_OK(hipGetLastError());
    return 0;
}

}  // namespace aw
