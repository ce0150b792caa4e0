// forward_kernels.h -- the forward recursion's kernels, instantiated by
// forward_f32.hip and forward_f64.hip.
#pragma once

#include <type_traits>

#include "forward.h"
#include "kernel_util.h"

namespace aw {

//===========================================================================
// forward recursion, two waves per tile (arghmm_forward_alg,
// sample_thread.cpp:394-460; arghmm_forward_block :186-296;
// arghmm_forward_switch :345-389)

// NT1 is a compile-time bound on the T-1 time bins (19 for the usual 20
// time points), so the per-time loops are fully unrolled without padding.
//
// A tile's workgroup has two waves, and a column passes between them twice:
//
//   lanes wave   lane l holds the R states l*R .. l*R+R-1 of the lane-run
//                layout: the scan along the branches, the emission, the new
//                column, which it hands over in LDS
//   sums wave    the per-time sums of that column, their product with the
//                (a,b) table, the normaliser, which it hands back; then it
//                stores the row
//
// The lanes wave runs its scan while the sums wave works.  The kernel is bound
// by the latency of that chain: hand over, atomics, their sums, the product,
// hand back, about 990 cycles at 8 FP32 states per lane.  One wave doing both
// is bound by its instruction issue (a dependent instruction every 8 cycles, an
// independent one every 5); four waves sharing the slots out lost more to
// atomics from several waves meeting in LDS than they gained.
//
// us per column at R = 1 / 2 / 4 / 6 / 8 / 12 / 16 states per lane, one
// instance on MI355X, switches included: FP32 0.30 0.31 0.35 0.40 0.45 0.53
// 0.74 (one wave, 16-lane-group copies, readlane product: 0.93 0.82 0.79 0.88
// 0.99 1.24 1.82); FP64 0.36 0.35 0.37 0.42 0.46 0.62 1.5 (1.15 0.95 1.05
// 1.12 1.30 1.67 2.74).  Both waves run the columns between two events (block
// ends, variant columns, windows of 64) in a loop of their own: with the tests
// for events in every column it was 0.44 0.41 0.39 0.45 0.52 0.59 0.83.
constexpr int FW_THREADS = 128;

// The 0/1 factors of a lane's R states: keep(x, r) is x times factor r, add(acc,
// x, r) is acc plus that.  A product where the factor has the table's type, a
// select (the same value) where it is a float beside doubles, and where even
// those would spill, one bit a state, spread over a mask for every use (open():
// once a scan, or the compiler would keep the spread masks in registers).
template <class Real, int R>
struct FwFactors {
    using Fac = std::conditional_t<(sizeof(Real) * R <= 64), Real, float>;
    Fac f[R];
    __device__ __forceinline__ void set(int r, bool on) { f[r] = on ? Fac(1) : Fac(0); }
    __device__ __forceinline__ const FwFactors &open() const { return *this; }
    __device__ __forceinline__ Real keep(Real x, int r) const
    {
        if constexpr (sizeof(Real) == sizeof(Fac)) return x * f[r];
        else return (f[r] != Fac(0)) ? x : Real(0);
    }
    __device__ __forceinline__ Real add(Real acc, Real x, int r) const
    {
        if constexpr (sizeof(Real) == sizeof(Fac)) return fma(x, f[r], acc);
        else return acc + ((f[r] != Fac(0)) ? x : Real(0));
    }
};
template <class Real, int R>
struct FwBits {
    unsigned m = 0;
    __device__ __forceinline__ void set(int r, bool on) { m |= on ? 1u << r : 0u; }
    __device__ __forceinline__ FwBits open() const
    {
        FwBits x = *this;
        asm volatile("" : "+v"(x.m));
        return x;
    }
    __device__ __forceinline__ Real keep(Real x, int r) const
    {
        const int k = (int)(m << (31 - r)) >> 31;
        if constexpr (sizeof(Real) == 4) return __int_as_float(__float_as_int(x) & k);
        else return __hiloint2double(__double2hiint(x) & k, __double2loint(x) & k);
    }
    __device__ __forceinline__ Real add(Real acc, Real x, int r) const { return acc + keep(x, r); }
};

// Per block, each lane of the lanes wave keeps in registers the factor planes
// of its R states, two 0/1 factors per state (not the first / not the last
// state of its branch: they cut the prefix and suffix sums) with their running
// products from the lane's start / end (whether the carry reaches the state),
// and whether the lane holds a branch start / end (the carry stops there), and
// the state's time; padding states use time bin 31, whose term is 0, so they
// come out 0 with no mask.  The 0/1 factors (FwFactors, FwBits) take a register
// or two a state, or a bit: with 16 states per lane in FP64 the products take 2.1
// us per column and the bits 1.5, with 32 in FP32 3.9 (spilled) and 2.2; with 12 in
// FP64 the bits cost 5 %.
template <class Real, int R>
struct FwLane {
    Real cf[R], cd[R], cg[R], ck[R], cj[R], ce[R];
    std::conditional_t<(sizeof(Real) * R >= 128), FwBits<Real, R>, FwFactors<Real, R>> nf, nl, ff, fl;
    const AW_LDS Real *tf[R];   // the handed-back term of the state's time
    Real m1, m2;
    int K;           // carry steps: lanes a branch of the block spans
};

// Per-time sums are accumulated in GCOPY copies of the 32 time bins, copy
// lane % 16 at GP[a * GCOPY + copy].  LDS takes sixteen consecutive lanes of
// an atomic at a time, 3 cycles and 3 more for every further lane at one
// address, 2 for every further lane in one bank: with a copy a lane and
// sixteen copies to a bin neither happens (12.6 cycles an atomic; 44 where
// four lanes share a copy and their states a time).  The sums are FP64 in
// both precisions: ds_add_f32 takes 192 cycles.
constexpr int GCOPY = 16;

// The time bin a lane reduces and multiplies: the wave's 16-lane rows 0 and 1
// take the bins a with a % 4 < 2, rows 2 and 3 the others, position j of a
// row the j-th of them.  Rows of a pair each read half of the copies.  A row
// then holds all the sums its lanes need for their half of the product with
// the (a,b) table (lane b and lane 32 + b: column b), and takes them by a row
// broadcast inside the multiply-add instead of a readlane per bin.
__device__ __forceinline__ int bin_of(int row, int j) { return 4 * (j >> 1) + (j & 1) + 2 * (row >> 1); }

// acc0 / acc1 += g[j] * tm[j] over the even / odd positions j of the lane's
// row.  The compiler does not fuse these broadcasts into the multiply-adds;
// the waits cover the register hazards it cannot see inside.
#define FW_BC(op, acc, src, j) op " " acc ", %2, " src " row_newbcast:" #j " row_mask:0xf bank_mask:0xf\n"
#define FW_BC10(op)                                                                         \
    "s_nop 1\n" FW_BC(op, "%0", "%3", 0) FW_BC(op, "%1", "%4", 1) FW_BC(op, "%0", "%5", 2)   \
    FW_BC(op, "%1", "%6", 3) FW_BC(op, "%0", "%7", 4) FW_BC(op, "%1", "%8", 5)              \
    FW_BC(op, "%0", "%9", 6) FW_BC(op, "%1", "%10", 7) FW_BC(op, "%0", "%11", 8)            \
    FW_BC(op, "%1", "%12", 9)
#define FW_BC16(op)                                                                         \
    FW_BC10(op) FW_BC(op, "%0", "%13", 10) FW_BC(op, "%1", "%14", 11)                       \
    FW_BC(op, "%0", "%15", 12) FW_BC(op, "%1", "%16", 13) FW_BC(op, "%0", "%17", 14)        \
    FW_BC(op, "%1", "%18", 15)
#define FW_T10(t) "v"(t[0]), "v"(t[1]), "v"(t[2]), "v"(t[3]), "v"(t[4]), "v"(t[5]), "v"(t[6]), "v"(t[7]), "v"(t[8]), "v"(t[9])
#define FW_T16(t) FW_T10(t), "v"(t[10]), "v"(t[11]), "v"(t[12]), "v"(t[13]), "v"(t[14]), "v"(t[15])
__device__ __forceinline__ void bin_product(float g, const float (&t)[10], float &a0, float &a1)
{
    asm(FW_BC10("v_fmac_f32_dpp") "s_nop 1" : "+v"(a0), "+v"(a1) : "v"(g), FW_T10(t));
}
__device__ __forceinline__ void bin_product(float g, const float (&t)[16], float &a0, float &a1)
{
    asm(FW_BC16("v_fmac_f32_dpp") "s_nop 1" : "+v"(a0), "+v"(a1) : "v"(g), FW_T16(t));
}
__device__ __forceinline__ void bin_product(double g, const double (&t)[10], double &a0, double &a1)
{
    asm(FW_BC10("v_fmac_f64_dpp") "s_nop 1" : "+v"(a0), "+v"(a1) : "v"(g), FW_T10(t));
}
__device__ __forceinline__ void bin_product(double g, const double (&t)[16], double &a0, double &a1)
{
    asm(FW_BC16("v_fmac_f64_dpp") "s_nop 1" : "+v"(a0), "+v"(a1) : "v"(g), FW_T16(t));
}

// carry chains of at most this many steps run in full; longer ones (few states
// per lane) stop at the block's longest branch
constexpr int FW_KFIX = 8;

// N steps of the carry of the same-branch sums across lanes: y1 = p1 + m1 *
// (y1 of the lane before), y2 = p2 + m2 * (y2 of the lane after).  In FP32 the
// shift is part of the multiply-add; two instructions of the other chain lie
// between a register's write and its shifted read.
template <int N>
__device__ __forceinline__ void carry_steps(float p1, float p2, float m1, float m2, float &y1, float &y2)
{
#pragma unroll
    for (int k = 0; k < N; k++) {
        float z1, z2;
        asm("v_mov_b32 %0, %2\n"
            "v_mov_b32 %1, %3\n"
            "v_fmac_f32_dpp %0, %4, %6 wave_shr:1 row_mask:0xf bank_mask:0xf\n"
            "v_fmac_f32_dpp %1, %5, %7 wave_shl:1 row_mask:0xf bank_mask:0xf"
            : "=&v"(z1), "=&v"(z2)
            : "v"(p1), "v"(p2), "v"(y1), "v"(y2), "v"(m1), "v"(m2));
        y1 = z1;
        y2 = z2;
    }
}
template <int N>
__device__ __forceinline__ void carry_steps(double p1, double p2, double m1, double m2, double &y1, double &y2)
{
#pragma unroll
    for (int k = 0; k < N; k++) {
        y1 = fma(m1, dpp_r<DPP_WAVE_SHR1>(y1), p1);
        y2 = fma(m2, dpp_r<DPP_WAVE_SHL1>(y2), p2);
    }
}

// x of the lane and of its partner in the other 16-lane row of the pair, or
// in the other half of the wave, added (the same sum in both)
__device__ __forceinline__ double add_rows(double x)
{
    const long long v = __double_as_longlong(x);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(v >> 32), (unsigned)(v >> 32), false, false);
    return __longlong_as_double((long long)((unsigned long long)hi[0] << 32 | lo[0])) +
           __longlong_as_double((long long)((unsigned long long)hi[1] << 32 | lo[1]));
}
__device__ __forceinline__ float add_halves(float x)
{
    const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(v[0]) + __uint_as_float(v[1]);
}
__device__ __forceinline__ double add_halves(double x)
{
    const long long v = __double_as_longlong(x);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(v >> 32), (unsigned)(v >> 32), false, false);
    return __longlong_as_double((long long)((unsigned long long)hi[0] << 32 | lo[0])) +
           __longlong_as_double((long long)((unsigned long long)hi[1] << 32 | lo[1]));
}

// the barrier of a tile's workgroup, ordering its LDS accesses
__device__ __forceinline__ void fw_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// plane `which` of block b, one value per slot.  Loaded values go straight into
// their registers: selecting or copying a value whose load is still in flight
// makes the compiler wait for it at once.
template <class Real, int R>
__device__ __forceinline__ void fw_plane(const DevInst &d, int b, int which, Real (&x)[R])
{
    slots_load<R>(planes<Real>(d, b, 64 * R) + which * (64 * R), threadIdx.x & 63, x);
}
template <int R>
__device__ __forceinline__ void fw_row(const int *rows, int b, int (&x)[R])
{
    slots_load<R>((const AW_GLOBAL int *)gp(rows) + (size_t)b * (64 * R), threadIdx.x & 63, x);
}

// Block b in the lanes wave; tv: the handed-back terms
template <class Real, int R, int NT1>
__device__ __forceinline__ void fw_block(const DevInst &d, int b, const Real *tv, FwLane<Real, R> &fl)
{
    int info[R];
    fw_row<R>(d.linfo, b, info);
    fw_plane<Real, R>(d, b, CF, fl.cf);
    fw_plane<Real, R>(d, b, CD, fl.cd);
    fw_plane<Real, R>(d, b, CG, fl.cg);
    fw_plane<Real, R>(d, b, CK, fl.ck);
    fw_plane<Real, R>(d, b, CJ, fl.cj);
    fw_plane<Real, R>(d, b, CE, fl.ce);
    bool first = false, last = false;
    bool f1 = true, f2 = true;
    fl.nf = fl.nl = fl.ff = fl.fl = {};
#pragma unroll
    for (int r = 0; r < R; r++) {
        f1 &= !(info[r] & INFO_FIRST);
        fl.nf.set(r, !(info[r] & INFO_FIRST));
        fl.nl.set(r, !(info[r] & INFO_LAST));
        fl.ff.set(r, f1);
        fl.tf[r] = (const AW_LDS Real *)tv + (info[r] & INFO_TIME);
        first |= (info[r] & INFO_FIRST) != 0;
        last |= (info[r] & INFO_LAST) != 0;
    }
#pragma unroll
    for (int r = R - 1; r >= 0; r--) fl.fl.set(r, f2 &= !(info[r] & INFO_LAST));
    fl.m1 = first ? Real(0) : Real(1);
    fl.m2 = last ? Real(0) : Real(1);
    // the carry crosses lanes without a branch start (end): more steps than
    // the longest run of them, plus one, change nothing
    fl.K = 1;
    if ((NT1 - 1 + R - 1) / R > FW_KFIX) {
        for (unsigned long long m = __ballot(!first); m; m &= m << 1) fl.K++;
        int k2 = 1;
        for (unsigned long long m = __ballot(!last); m; m &= m << 1) k2++;
        fl.K = max(fl.K, k2);
    }
}

// variant row v, clamped to the last row (an instance without variant
// columns has one allocated row that is never used)
template <int R>
__device__ __forceinline__ void vrow_load(const DevInst &d, int v, double (&ev)[R])
{
    constexpr int RW = 64 * R;
    const AW_GLOBAL double *row = gp(d.vemit) + (size_t)max(min(v, d.nvar - 1), 0) * RW;
    slots_load<R>(row, threadIdx.x & 63, ev);
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

// The column handed over: lane l's R values in one run, runs an odd number of
// 16-byte pieces apart (the pieces sixteen lanes access are in distinct banks)
template <class Real, int R>
constexpr int xc_stride()
{
    return ((R * (int)sizeof(Real) + 15) / 16 | 1) * 16 / (int)sizeof(Real);
}

// LDS of the forward kernel: partial sums, the column handed over, the terms
// handed back, the switch targets (plus one dummy slot per lane), staged
// variant rows
template <class Real, int R>
struct FwShared {
    alignas(16) double gp[32 * GCOPY];
    alignas(16) Real xc[64 * xc_stride<Real, R>()];
    alignas(16) Real tv[64];       // the other-branch term of each time bin; [32] the scale, [33] rejoined
    alignas(16) Real nw[64 * R + 64];
    alignas(16) Real vs[fw_vst<Real, R>() * 64 * R];
};

// wave-wide maximum
__device__ __forceinline__ double wave_max(double x)
{
    for (int off = 32; off > 0; off >>= 1) x = fmax(x, __shfl_xor(x, off));
    return x;
}

// columns between the checks of a re-run tile against its stored columns
constexpr int FW_RECHECK = 128;

// The two waves of a tile walk its columns together, two barriers a column:
// after the first the column is in sh.xc, after the second its terms are in
// sh.tv.
//
// REDO: a re-run tile (mode 2).  It stops once a column it computes agrees
// with the column stored by its speculative run (relative tolerance tol): the
// filter is contractive, so the stored columns after it, the normalisers and
// the boundary column stay within tolerance.  early receives the column after
// that one, or 0.
struct FwSpan {
    int c0, cs, c1, mode, bout, bin;
    int clast;   // the last column computed: c1 - 1, or c1 into the boundary slot
    // the first column from col on that is checked against the stored one
    __device__ __forceinline__ int recheck(int col) const
    {
        return c0 + (col - c0 + FW_RECHECK - 1) / FW_RECHECK * FW_RECHECK;
    }
};

// The ends and switch sources of 64 blocks from b0 on, one block per lane,
// read with readlane: scalar loads at a switch would be waited for with the
// next LDS access.
struct FwBlocks {
    int b0, last, rs, rc;
    __device__ __forceinline__ FwBlocks(const DevInst &d, int b) { load(d, b); }
    __device__ __forceinline__ void load(const DevInst &d, int b)
    {
        b0 = b;
        const int x = min(b + (int)(threadIdx.x & 63), d.B - 1);
        last = gp(d.bstart)[x] + gp(d.blen)[x];
        rs = gp(d.srcs)[2 * x];
        rc = gp(d.srcs)[2 * x + 1];
    }
    // block b follows the one before in the window, or opens the next window
    __device__ __forceinline__ void next(const DevInst &d, int b)
    {
        if (b >= b0 + 64) load(d, b);
    }
    __device__ __forceinline__ int end(int b) const { return __builtin_amdgcn_readlane(last, b - b0); }
    __device__ __forceinline__ int recomb(int b) const { return __builtin_amdgcn_readlane(rs, b - b0); }
    __device__ __forceinline__ int recoal(int b) const { return __builtin_amdgcn_readlane(rc, b - b0); }
};

template <class Real, int R, int NT1, bool REDO>
__device__ __forceinline__ void fw_sums(const DevInst &d, FwShared<Real, R> &sh, const FwSpan &sp,
                                        AW_GLOBAL Real *bnd, AW_GLOBAL double *bnorm, double tol,
                                        AW_GLOBAL int *early)
{
    constexpr int RW = 64 * R, NJ = (NT1 + 2) / 4 * 2, XC = xc_stride<Real, R>();
    const int lane = threadIdx.x & 63, T1 = d.T - 1, L = d.L;
    AW_GLOBAL Real *alpha = (AW_GLOBAL Real *)d.alpha;
    auto norms = gp(d.norms);
    // this lane's half of the copies of the bin it reduces (the other half is
    // the lane's of the other row), in four pieces from the (lane / 4)-th on:
    // the pieces that a row reads in one step lie in distinct banks
    double2 *gq = (double2 *)(sh.gp + bin_of(lane >> 4, lane & 15) * GCOPY +
                              (((lane >> 4) ^ (lane >> 1)) & 1) * (GCOPY / 2));
    const int rot = lane >> 2;
    // Of a block: the addresses of the states' bins and copies in the sums,
    // and the lane's part of the (a,b) table.  Indices are clamped: entries
    // a >= T-1 meet a zero sum, and lanes >= T-1 compute terms nobody uses,
    // but for lanes 31 and 63, whose entries of 1 give the normaliser.  The
    // next block's are loaded a block ahead.
    AW_LDS double *gadd[R];
    Real tmc[NJ];
    int ni[R];
    double nt[NJ];
    // The lanes wave loads all of a block at its switch and waits for it; a
    // word of each 128-byte line of it, read here a block ahead, has the lines
    // in cache by then (2 % of a column in FP32, nothing in FP64).
    constexpr bool WARM = sizeof(Real) == 4;
    constexpr int PB = NCOEF * RW * (int)sizeof(Real), NP = WARM ? (PB + 8191) / 8192 : 0;
    unsigned warm[NP + 1];
    auto load = [&](int b) {
        const AW_GLOBAL char *pl = (const AW_GLOBAL char *)planes<Real>(d, b, RW);
        const AW_GLOBAL char *dt = (const AW_GLOBAL char *)(gp(d.ldet) + (size_t)b * RW);
#pragma unroll
        for (int x = 0; x < NP; x++)
            warm[x] = *(const AW_GLOBAL unsigned *)(pl + min((x * 64 + lane) * 128, PB - 4));
        if (WARM) warm[NP] = *(const AW_GLOBAL unsigned *)(dt + min(lane * 128, RW * 4 - 4));
        const AW_GLOBAL int *info = gp(d.linfo) + (size_t)b * RW;
        const AW_GLOBAL double *tm = gp(d.tm) + (size_t)b * T1 * T1 + min(lane & 31, T1 - 1);
        slots_load<R>(info, lane, ni);
#pragma unroll
        for (int j = 0; j < NJ; j++) nt[j] = tm[min(bin_of(lane >> 4, j), T1 - 1) * T1];
    };
    auto unpack = [&] {
#pragma unroll
        for (int x = 0; x <= NP; x++)
            if (WARM) asm volatile("" ::"v"(warm[x]));
#pragma unroll
        for (int r = 0; r < R; r++) {
            gadd[r] = (AW_LDS double *)sh.gp + (ni[r] & INFO_TIME) * GCOPY + (lane & (GCOPY - 1));
        }
#pragma unroll
        for (int j = 0; j < NJ; j++) tmc[j] = (lane & 31) == 31 ? Real(1) : (Real)nt[j];
    };
    int b = find_owner(cp(d.bstart), d.B, sp.c0);
    FwBlocks bl(d, b);
    int bend = bl.end(b);
    load(b);
    for (int k = lane; k < 32 * GCOPY; k += 64) sh.gp[k] = 0.0;
    unpack();
    load(min(b + 1, d.B - 1));
    Real nw = Real(0);   // lane i: the normaliser of the column with col % 64 == i
    bool rejoined = false;
    int col = sp.c0;
    // Columns run in stretches without an event: the first column by itself
    // (its scale), then up to the block's end, the end of a window of 64
    // (normalisers stored), the end of the warm-up, a check against the stored
    // columns, the tile's last column, and the boundary column by itself.
    for (bool done = false; !done;) {
        int ev = min(min(bend - 1, col | 63), sp.clast);
        if (col < sp.c1) ev = min(ev, sp.c1 - 1);
        const bool store = col >= sp.cs;
        if (!store) ev = min(ev, sp.cs - 1);
        // column 0 is stored unnormalised (scale 1); a restarted tile's first
        // column is the boundary column as stored by the tile before
        const bool asis = col == sp.c0 && (col == 0 || (REDO && sp.mode == 2));
        const int chk = REDO ? sp.recheck(col) : 0;
        if (REDO) ev = min(ev, chk);
        if (col == sp.c0) ev = col;
        AW_GLOBAL Real *row = col < sp.c1 ? alpha + (size_t)col * RW
                                           : bnd + (size_t)sp.bout * BND_UNIT;
        for (;; col++, row += RW) {
            fw_barrier();
            Real x[R];
#pragma unroll
            for (int r = 0; r < R; r++) x[r] = sh.xc[lane * XC + r];
#pragma unroll
            for (int r = 0; r < R; r++) (void)__builtin_amdgcn_ds_atomic_fadd_f64(gadd[r], (double)x[r]);
            // the LDS operations of one wave run in order: the sums are
            // complete when they are read, and cleared before the next column's
            double2 q[GCOPY / 4];
#pragma unroll
            for (int k = 0; k < GCOPY / 4; k++) q[k] = gq[(k + rot) & 3];
#pragma unroll
            for (int k = 0; k < GCOPY / 4; k++) gq[(k + rot) & 3] = double2{0.0, 0.0};
            const Real g = (Real)add_rows(((q[0].x + q[0].y) + (q[1].x + q[1].y)) +
                                          ((q[2].x + q[2].y) + (q[3].x + q[3].y)));
            Real a0 = Real(0), a1 = Real(0);
            bin_product(g, tmc, a0, a1);
            const Real t = add_halves(a0 + a1);
            const Real norm = readlane_r(t, 31);
            const Real nsc = asis ? Real(1) : recip(norm);
            // the terms of the time bins, 0 for the padding's, and the scale
            Real tv = (lane < T1) ? t * nsc : Real(0);
            tv = lane == 32 ? nsc : tv;
            if (REDO) {
                if (col == chk && col > sp.c0 && col < sp.c1) {
                    double dmax = 0.0, amax = 0.0;
                    Real old[R];
                    slots_load<R>((const AW_GLOBAL Real *)row, lane, old);
#pragma unroll
                    for (int r = 0; r < R; r++) {
                        const double nv = (double)(x[r] * nsc), ov = (double)old[r];
                        dmax = fmax(dmax, fabs(nv - ov));
                        amax = fmax(amax, fabs(nv));
                    }
                    rejoined = wave_max(dmax) <= tol * wave_max(amax);
                    tv = (lane == 33 && rejoined) ? Real(1) : tv;
                }
            }
            sh.tv[lane] = tv;
            fw_barrier();
            if (store) {
#pragma unroll
                for (int r = 0; r < R; r++) x[r] *= nsc;
                slots_store<R>(row, lane, x);
            }
            nw = (lane == (col & 63)) ? norm : nw;
            if (col == ev) break;
        }
        done = col == sp.clast || (REDO && rejoined);
        if ((col & 63) == 63 || done) {
            const int c = (col & ~63) + lane;
            if (c >= sp.cs && c <= min(col, sp.c1 - 1)) norms[c] = (double)nw;
        }
        if (done) break;
        if (++col == bend) {
            bl.next(d, ++b);
            bend = bl.end(b);
            unpack();
            load(min(b + 1, d.B - 1));
        }
    }
    if (sp.bout >= 0 && !rejoined && lane == (col & 63)) bnorm[sp.bout] = (double)nw;
    // the first column's own normaliser (bnorm's slot: no tile of this launch
    // writes it, see FwPlan)
    if (sp.c0 >= sp.cs && sp.c0 < sp.c1 && lane == 0) {
        if (sp.c0 == 0 && L > 1) norms[0] = 1.0;
        if (REDO && sp.mode == 2) norms[sp.c0] = bnorm[sp.bin];
    }
    // the columns that do not follow from the one stored before them
    auto mark = [&](int c) { atomicOr(&d.cut[c >> 5], 1u << (c & 31)); };
    if (sizeof(Real) == 4 && lane == 0) {
        if (sp.cs > 0) mark(sp.cs);
        if (rejoined && col + 1 < sp.c1) mark(col + 1);
    }
    if (REDO && early && lane == 0) *early = rejoined ? col + 1 : 0;
}

template <class Real, int R, int NT1, bool REDO>
__device__ __forceinline__ void fw_lanes(const DevInst &d, FwShared<Real, R> &sh, const FwSpan &sp,
                                         const AW_GLOBAL Real *bnd)
{
    constexpr int RW = 64 * R, XC = xc_stride<Real, R>();
    constexpr int VST = fw_vst<Real, R>(), VCH = fw_vch<Real, R>();
    // registers allow a loop of its own for plain columns, and a switch's loads
    // all at once
    constexpr bool TWICE = R * sizeof(Real) <= 96;
    const int lane = threadIdx.x & 63, L = d.L;
    int b = find_owner(cp(d.bstart), d.B, sp.c0);
    FwBlocks bl(d, b);
    int bend = bl.end(b);
    FwLane<Real, R> fl;
    fw_block<Real, R, NT1>(d, b, sh.tv, fl);
    for (int k = lane; k < RW; k += 64) sh.nw[k] = Real(0);
    // Column classes of a window of 64 columns, one per lane, read with
    // readlane; the next window's are loaded a window ahead.
    const AW_GLOBAL int *clsg = gp(d.cls);
    int wb = sp.c0 & ~63;
    int clsv = clsg[min(wb + lane, L - 1)];
    int clsn = clsg[min(wb + 64 + lane, L - 1)];
    // Variant rows (row index = the column's class) are consumed in order
    // and staged in LDS, VST at a time, so that a refill costs a few waits
    // and the columns read their row from LDS.
    int vbase = 0, vend = 0;

    // first column.  mode 0: the unnormalised prior, not multiplied by the
    // emission (calc_state_priors, trans.cpp:785-831); padding positions
    // hold 0.  mode 1: 1 on every state.  mode 2: the boundary column.
    Real v[R];
    if (sp.mode == 0) {
        const AW_GLOBAL double *pr = gp(d.lprior);
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = (Real)pr[slot_pos(r, lane, R)];
    } else if (sp.mode == 1) {
        const int S = cp(d.soff)[b + 1] - cp(d.soff)[b];
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = (lane * R + r < S) ? Real(1) : Real(0);
    } else {
        const AW_GLOBAL Real *src = bnd + (size_t)sp.bin * BND_UNIT;
        slots_load<R>(src, lane, v);
    }

    // the column goes to the sums wave
    auto publish = [&] {
#pragma unroll
        for (int r = 0; r < R; r++) sh.xc[lane * XC + r] = v[r];
        fw_barrier();
        // What follows until the second barrier runs beside the sums wave:
        // empty asms keep the compiler from moving it before the first barrier
        // or behind the second.
#pragma unroll
        for (int r = 0; r < R; r++) asm volatile("" : "+v"(v[r]));
    };
    // same-branch prefix sums (younger states) with the carry from the lanes
    // before, suffix sums (older states) with the carry from the lanes after
    auto scan = [&](Real (&same)[R]) {
        Real P[R], Q[R];
        Real p = Real(0), q = Real(0);
        const auto &nf = fl.nf.open(), &nl = fl.nl.open(), &ff = fl.ff.open(), &fe = fl.fl.open();
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int t = R - 1 - r;
            P[r] = nf.keep(p, r);
            Q[t] = nl.keep(q, t);
            p = fma(fl.cf[r], v[r], P[r]);
            q = fma(fl.cd[t], v[t], Q[t]);
        }
        Real y1 = p, y2 = q;
        constexpr int KMAX = (NT1 - 1 + R - 1) / R, KB = KMAX <= FW_KFIX ? KMAX - 1 : 4;
        if constexpr (KB > 0)
            for (int k = 1; k < (KMAX <= FW_KFIX ? 2 : fl.K); k += KB)
                carry_steps<KB>(p, q, fl.m1, fl.m2, y1, y2);
        // the wait covers the chains' last registers, which the compiler does
        // not know to be fresh
        asm("s_nop 1" : "+v"(y1), "+v"(y2));
        y1 = dpp_r<DPP_WAVE_SHR1>(y1);
        y2 = dpp_r<DPP_WAVE_SHL1>(y2);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const Real pr = ff.add(P[r], y1, r), qr = fe.add(Q[r], y2, r);
            // the last slot of a lane adds its two products in the other order
            // in FP32
            const Real two = (sizeof(Real) == 8 || r < R - 1) ? fma(fl.cg[r], pr, fl.ck[r] * qr)
                                                              : fma(fl.ck[r], qr, fl.cg[r] * pr);
            same[r] = fma(fl.cj[r], v[r], two);
            if (TWICE) asm volatile("" : "+v"(same[r]));
        }
    };
    // whether the walk ends at column col
    auto ends = [&](int col) {
        return col == sp.clast || (REDO && (col - sp.c0) % FW_RECHECK == 0 && sh.tv[33] != Real(0));
    };
    // invariant columns without a switch: the columns before `plain`
    auto plain_to = [&](int next) {
        const unsigned long long m = __ballot(clsv != -1) >> (next & 63);
        int n = m ? next + (int)__ffsll((long long)m) - 1 : wb + 64;
        n = min(min(n, bend), sp.clast + 1);
        return REDO ? min(n, sp.recheck(next - 1) + 1) : n;
    };

    for (int col = sp.c0;;) {
        // Every column goes from here to the next one, in this loop while that
        // is a plain one (not where a second copy of the scan would spill).
        int plain = 0;
        if (TWICE && col + 1 < wb + 64) plain = plain_to(col + 1);
        for (; col + 1 < plain; col++) {
            publish();
            Real same[R];
            scan(same);
            fw_barrier();
            const Real sc = sh.tv[32];
            Real tf[R];
#pragma unroll
            for (int r = 0; r < R; r++) tf[r] = *fl.tf[r];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = fl.ce[r] * fma(sc, same[r], tf[r]);
        }
        publish();
        // the next column's class (past the last column: a repeat, unused),
        // emission, and same-branch terms or switch
        const int next = col + 1;
        if (next >= wb + 64) {
            wb += 64;
            clsv = clsn;
            clsn = clsg[min(wb + 64 + lane, L - 1)];
        }
        const int cls = __builtin_amdgcn_readlane(clsv, next & 63);
        const bool sw = next == bend && next < L;
        Real e[R], same[R], rr[R], cr[R];
        Real prs = Real(0), pcs = Real(0);
        if (sw) {
            // switch column: deterministic transitions scattered into nw
            // (the recombination and recoalescence sources excluded); the two
            // dense rows follow below
            bl.next(d, ++b);
            bend = bl.end(b);
            const int rs = bl.recomb(b), rc = bl.recoal(b);
            // (loading the block's data a block ahead gains nothing measurable)
            int dt[R];
            Real dp[R];
            fw_row<R>(d.ldet, b, dt);
            fw_plane<Real, R>(d, b, CDP, dp);
            if (TWICE) {
                fw_plane<Real, R>(d, b, CRR, rr);
                fw_plane<Real, R>(d, b, CCR, cr);
                fw_block<Real, R, NT1>(d, b, sh.tv, fl);
            }
            if (rs != -1) prs = sh.xc[(rs / R) * XC + rs % R];
            if (rc != -1) pcs = sh.xc[(rc / R) * XC + rc % R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const Real x = v[r] * dp[r];
                // atomics (192 cycles over a full wave in FP32) only where
                // several sources meet
                const bool shared = dt[r] >= DET_SHARED;
                sh.nw[dt[r] < 0 || shared ? RW + lane : dt[r]] = x;
                if (shared) lds_add(&sh.nw[dt[r] & ~DET_SHARED], x);
            }
#pragma unroll
            for (int r = 0; r < R; r++) {
                same[r] = sh.nw[lane * R + r];
                sh.nw[lane * R + r] = Real(0);   // for the next switch
            }
            if (!TWICE) fw_block<Real, R, NT1>(d, b, sh.tv, fl);
        } else {
            scan(same);
        }
        if (cls >= 0) {
            if (cls >= vend) {
                vbase = cls;
                vend = min(cls + VST, d.nvar);
#pragma unroll
                for (int k0 = 0; k0 < VST; k0 += VCH) {
                    // VST need not be a multiple of VCH
                    double rows[VCH][R];
#pragma unroll
                    for (int k = 0; k < VCH; k++)
                        if (k0 + k < VST) vrow_load<R>(d, vbase + k0 + k, rows[k]);
#pragma unroll
                    for (int k = 0; k < VCH; k++)
#pragma unroll
                        for (int r = 0; r < R; r++)
                            if (k0 + k < VST) sh.vs[(k0 + k) * RW + slot_pos(r, lane, R)] = (Real)rows[k][r];
                }
            }
#pragma unroll
            for (int r = 0; r < R; r++) e[r] = sh.vs[(cls - vbase) * RW + slot_pos(r, lane, R)];
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) e[r] = cls == -1 ? fl.ce[r] : Real(1);
        }
#pragma unroll
        for (int r = 0; r < R; r++) asm volatile("" : "+v"(same[r]), "+v"(e[r]));
        fw_barrier();
        if (ends(col)) return;
        const Real sc = sh.tv[32];
        if (sw) {
            // the recombination and recoalescence rows; padding slots hold 0 in
            // every row
            if (!TWICE) {
                fw_plane<Real, R>(d, b, CRR, rr);
                fw_plane<Real, R>(d, b, CCR, cr);
            }
#pragma unroll
            for (int r = 0; r < R; r++)
                v[r] = fma(pcs * sc, cr[r], fma(prs * sc, rr[r], same[r] * sc)) * e[r];
        } else {
            Real tf[R];
#pragma unroll
            for (int r = 0; r < R; r++) tf[r] = *fl.tf[r];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = e[r] * fma(sc, same[r], tf[r]);
        }
        col++;
    }
}

template <class Real, int R, int NT1, bool REDO>
__device__ __forceinline__ void fw_instance(const DevInst d, void *lds, const FwTile &t,
                                            AW_GLOBAL Real *bnd, AW_GLOBAL double *bnorm,
                                            double tol, AW_GLOBAL int *early)
{
    FwShared<Real, R> &sh = *(FwShared<Real, R> *)lds;
    auto uni = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
    FwSpan sp{uni(t.c0), uni(t.cs), uni(t.c1), uni(t.mode), uni(t.bout), uni(t.bin), 0};
    sp.clast = sp.bout >= 0 ? sp.c1 : sp.c1 - 1;
    // a re-run's columns are waited for while other instances' tracebacks fill
    // the device
    __builtin_amdgcn_s_setprio(3);
    if (uni((int)threadIdx.x >> 6)) fw_sums<Real, R, NT1, REDO>(d, sh, sp, bnd, bnorm, tol, early);
    else fw_lanes<Real, R, NT1, REDO>(d, sh, sp, bnd);
}

// One launch covers every instance of a batch, whatever its states-per-lane
// count: waves of different R run side by side from the start, with no
// dependence on how streams map to hardware queues.
// REDO marks the launches of re-run tiles (a separate symbol, so that
// profiles report the main forward launch on its own).  BIG: the instances
// with 32 states per lane (blocks of 1025-2048 states) run in a symbol of
// their own, launched over the same tiles, so that their register demand
// (AGPRs, in FP64 scratch) does not weigh on the others.
template <class Real, int NT1, bool REDO, bool BIG>
__global__ __launch_bounds__(FW_THREADS)
void k_fw_all(const DevInst *__restrict__ D, const FwTile *__restrict__ tiles,
              Real *__restrict__ bnd, double *__restrict__ bnorm, double tol, int *__restrict__ early)
{
    extern __shared__ __align__(16) double fw_dyn[];
    const FwTile t = tiles[blockIdx.x];
    const DevInst &d = D[t.inst];
    AW_GLOBAL Real *bg = (AW_GLOBAL Real *)bnd;
    AW_GLOBAL double *ng = (AW_GLOBAL double *)bnorm;
    AW_GLOBAL int *eg = early ? (AW_GLOBAL int *)(early + blockIdx.x) : nullptr;
    if ((d.R > 16) != BIG) return;   // the other symbol's tile
    if constexpr (BIG) {
        fw_instance<Real, 32, NT1, REDO>(d, fw_dyn, t, bg, ng, tol, eg);
    } else {
        switch (d.R) {
        case 1: fw_instance<Real, 1, NT1, REDO>(d, fw_dyn, t, bg, ng, tol, eg); break;
        case 2: fw_instance<Real, 2, NT1, REDO>(d, fw_dyn, t, bg, ng, tol, eg); break;
        case 4: fw_instance<Real, 4, NT1, REDO>(d, fw_dyn, t, bg, ng, tol, eg); break;
        case 6: fw_instance<Real, 6, NT1, REDO>(d, fw_dyn, t, bg, ng, tol, eg); break;
        case 8: fw_instance<Real, 8, NT1, REDO>(d, fw_dyn, t, bg, ng, tol, eg); break;
        case 12: fw_instance<Real, 12, NT1, REDO>(d, fw_dyn, t, bg, ng, tol, eg); break;
        default: fw_instance<Real, 16, NT1, REDO>(d, fw_dyn, t, bg, ng, tol, eg); break;
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
    const Real *q = bnd + (size_t)t.bin * BND_UNIT;
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
    hipLaunchKernelGGL(kern, dim3(cnt), dim3(FW_THREADS), sh, st, dD, tiles,
                       (Real *)bnd, bnorm, tol, early);
    HIP_OK(hipGetLastError());
    return 0;
}

}  // namespace aw
