// Determinants of (ξ, m) blocks from their wave-number factor on gfx950.
//
// Every element of the round-trip matrix is an integral over x = cosh θ in
// [1, ∞) of products of two one-degree functions (the A, B, C, D of the
// reference, src/integration.c:762-888, with I_{l1 l2} = ∫ r_p e^{-αx}
// P_l1^m P_l2^m/(x²-1) dx written under one integral sign):
//   p_l = m P_l^m/√(x²-1),  t_l = √(x²-1) dP_l^m/dx  (m = 0: p_l = 0, t_l = P_l^1),
//   EE = √(a a') Λ Σ_x w (r_TM t t' + |r_TE| p p'),
//   MM = √(b b') Λ Σ_x w (r_TM p p' + |r_TE| t t'),
//   EM = √(a b') Λ Σ_x w (r_TM t p' + |r_TE| p t'),
// all terms positive.  On the nodes of one quadrature grid that is M = FᵀF,
// one row of F per node and polarization, and det(1 - FᵀF) = det(1 - F Fᵀ):
// the determinant of the smaller Gram matrix G = F Fᵀ, whose dimension is
// twice the number of nodes that matter (some 2.2 √(2 lmax) + 30) instead of
// 2 ldim.  A row of F is a ridge of a few standard deviations around the
// degree whose saddle point is the node, so rows of distant nodes do not
// overlap: G is banded, and each of its tiles needs a fraction of the degrees.
// R/L = 200, ldim = 1200: 2400 rows become about 460 with a half-bandwidth
// of 96; R/L = 2000, ldim = 12000: 24000 become about 1400.
//
// Kernels (blockIdx.y, or .x of the last, selects the block):
//   k_upload       the descriptors;
//   k_wave_start   the Mie coefficients of each (object, ξ), and beside them
//                  the nodes and, per run of 64 degrees, the matrix of the
//                  recurrence of P_l^m in l;
//   k_wave_prefix  the states at the runs' starts (where the runs are many);
//   k_wave_norms   the states every 8 degrees and the squared norms of F's rows
//                  per 16;
//   k_wave_window  trace, trace shortcut, the nodes that matter;
//   k_gram         the band of -G on FP64 MFMA, F's rows made on the spot;
//   k_band_ldl     log det(1 - G): banded LDLᵀ, one workgroup per block;
//   k_band_dense   -G as a dense matrix (schedules fixed by the caller, the
//                  pivoted LU);
//   k_wave_rows, k_wave_matrix  F, and M = FᵀF itself (caps_M_init, CHOLESKY mode).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include "blocks.h"
#include "device_math.h"
#include "wave.h"

namespace capsd {

template <typename T>
__device__ __forceinline__ T* at(char* base, int64_t off) { return reinterpret_cast<T*>(base + off); }

typedef double double4_t __attribute__((ext_vector_type(4)));

// F's rows are ordered 2 k + p for node k and polarization p (0 TM, 1 TE): a
// tile of 8 nodes is 16 rows, the unit of the band.

// Exponent of what is zero whatever it is added to: 2^NO_EXP 2^E = 0.
constexpr int NO_EXP = -(1 << 28);

// One step of S_l = √((l-m)!/(l+m)!) P_l^m upward in the degree (DLMF
// 14.10.3), c1 = (2l+1)/√((l+1)²-m²), c2 = √(l²-m²)/√((l+1)²-m²).
__device__ __forceinline__ void degree_step(double c1, double c2, double x, double& p, double& pp)
{
    const double pn = fma(c1 * x, p, -(c2 * pp));
    pp = p;
    p = pn;
}

// log(C(2m, m)/4^m): a product for small m, else the asymptotic series of
// log Γ(m+½)/Γ(m+1) (DLMF 5.11.13), whose first neglected term is below 1e-16
// from m = 16.
__device__ __forceinline__ double log_central_binomial(int m)
{
    if (m < 16) {
        double r = 1;
        for (int k = 1; k <= m; k++) r *= (2 * k - 1) / (2.0 * k);
        return log(r);
    }
    const double i = 1.0 / m, i2 = i * i;
    return -0.5 * log(M_PI * m)
         + i * (-1. / 8 + i2 * (1. / 192 + i2 * (-1. / 640 + i2 * (17. / 14336 - i2 * (31. / 18432)))));
}

__device__ void mie_entry(const MieDesc& t, char* __restrict__ arena, int l)
{
    if (l > t.L) return;
    double lna, lnb;
    mie(t.xi_, t.LbyR, t.epsm1, l, lna, lnb);
    double* a = at<double>(arena, t.off) + (l - 1);
    a[0] = lna;
    a[t.L] = lnb;
    // √a_l and √b_l times √((2l+1)/(l(l+1))) as mantissas of one power of two
    const double g = log((2.0 * l + 1) / ((double)l * (l + 1.0)));
    const double xa = (lna + g) / 2 * (1 / LOG2), xb = (lnb + g) / 2 * (1 / LOG2);
    const double fa = floor(xa);
    a[2 * t.L] = exp2(xa - fa);
    a[3 * t.L] = exp2(xb - fa);
    at<int>(arena, t.off + 32 * (int64_t)t.L)[l - 1] = (int)fa;
}

// The block whose units (workgroups or wavefronts of a launch over all
// blocks) u is one of: first holds the sums of the counts before each block.
__device__ __forceinline__ int block_of(const BlockDesc* __restrict__ desc, int n, int u, int BlockDesc::*first)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (desc[mid].*first <= u) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// A run's matrix (columns a, b, times 2^e) applied to the state (p, dp) 2^E at
// its start; p in [1, 2)
__device__ __forceinline__ void next_run(double2 a, double2 b, int e, double& p, double& dp, int& E)
{
    const double t = fma(a.x, p, b.x * dp), dt = fma(a.y, p, b.y * dp);
    const int f = __builtin_amdgcn_frexp_exp(t) - 1;
    p = ldexp(t, -f);
    dp = ldexp(dt, -f);
    E += e + f;
}

// A batch's descriptors from pinned host memory.  A batch of one block is some
// 80 us of kernels; a copy command before them, one for the results behind them
// (stores of k_band_ldl to pinned memory instead) and a timed event between every
// two stages (stores of the time by their first workgroups instead) took another
// 27 us (116 and 89; an energy at T = 0, five batches: 2.20 and 1.93 ms; measured at
// a step of 0.5 of the grid, 91 us and 2.03 ms at the present 0.45).
__global__ void __launch_bounds__(256) k_upload(const uint4* __restrict__ host, uint4* __restrict__ dev, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dev[i] = host[i];
}

// The time at which a stage began (clock: pinned host memory, or none).
__device__ __forceinline__ void stage_begins(int64_t* clock)
{
    if (clock && threadIdx.x == 0 && blockIdx.x == 0 && blockIdx.y == 0) *clock = wall_clock64();
}

// The first ntab mie_units workgroups: Mie coefficients, one lane per l.  Then
// per block, 64 nodes per wavefront, one lane each: the degrees' recurrence as
// a chain over all of them takes 45 cycles a step (R/L = 2000: 224 us; 14 us
// and k_wave_prefix's 16 so).  Instead each run of 64
// degrees, from d.n_below runs below the window on (the first one shorter),
// gives the 2 x 2 matrix that takes the state at its start to the next run's,
// and k_wave_prefix or k_wave_norms multiply them.
// The state is (S_l, D_l = S_l - S_{l-1}), in which all of the recurrence is
// positive, and with it the matrices and their products lose nothing:
// D_{l+1} = κ S_l + c2 D_l, S_{l+1} = S_l + D_{l+1}, κ = c1 x - c2 - 1 =
// c1 (x-1) + c3.
__global__ void __launch_bounds__(64) k_wave_start(const MieDesc* __restrict__ tabs, int ntab, int mie_units,
                                                   const BlockDesc* __restrict__ desc, int n,
                                                   char* __restrict__ arena, int* __restrict__ status,
                                                   int64_t* __restrict__ clock)
{
    stage_begins(clock);
    const int lane = threadIdx.x;
    int u = blockIdx.x;
    if (u < ntab * mie_units) {
        mie_entry(tabs[u / mie_units], arena, (u % mie_units) * 64 + lane + 1);
        return;
    }
    u -= ntab * mie_units;
    const BlockDesc& d = desc[block_of(desc, n, u, &BlockDesc::unit_start)];
    u -= d.unit_start;
    const int run = u / d.n_waves, k = (u % d.n_waves) * 64 + lane, nP = d.n_waves * 64;
    const int runs = d.n_below + d.n_segs - 1;   // the last one leads nowhere
    if (run >= max(runs, 1)) return;
    const int mm = d.m > 0 ? d.m : 1;
    double x = 1;
    const bool on = k < d.n_nodes;
    const double v = d.v0 + k * d.h, L = v > 40 ? v : log1p(exp(v)), xm1 = d.A * d.A * L * L;
    if (on) x = 1 + xm1;
    if (run == 0) {
        double p = 0, stm = 0, ste = 0;
        int E = NO_EXP;   // lanes without a node: 0 times a power of two that is 0
        if (on) {
            const double sg = 1 / (1 + exp(-v));
            const double x2m1 = xm1 * (x + 1);
            const double dx = 2 * d.A * d.A * L * sg;
            // S_mm = √(C(2mm,mm)/4^mm) (x²-1)^{mm/2}, times e^{-ξx} √(h dx) and, for
            // m > 0, the 1/√(x²-1) of p_l and t_l
            const double lb = 0.5 * (log_central_binomial(mm) + (d.m > 0 ? mm - 1 : mm) * log(x2m1) + log(d.h * dx))
                            - d.xi_ * x;
            const double lb2 = lb * (1 / LOG2), fl = floor(lb2);
            E = (int)fl;
            p = exp((lb2 - fl) * LOG2);
            double rte, rtm;
            fresnel(d.epsm1_plate, d.xi_, d.xi_ * sqrt(x2m1), rte, rtm);
            stm = sqrt(fabs(rtm));
            ste = sqrt(fabs(rte));
            if (!(stm > 0 && ste > 0 && isfinite(stm) && isfinite(ste) && isfinite(lb))) atomicOr(status, 1);
        }
        double* nd = at<double>(arena, d.off_node);
        nd[k] = x;
        nd[nP + k] = stm;
        nd[2 * nP + k] = ste;
        nd[3 * nP + k] = p;
        at<int>(arena, d.off_node + 32 * (int64_t)nP)[k] = E;
    }
    if (runs == 0) return;
    const int l1 = d.lmin + 64 * (run - d.n_below + 1), l0 = max(l1 - 64, mm), n4 = (l1 - l0) & ~3;
    __shared__ double2 cs[64];
    __shared__ double c3s[64];
    {
        const double l = l0 + lane, m2 = (double)mm * mm;
        const double r0 = sqrt((l - mm) * (l + mm)), r1 = sqrt((l + 1 - mm) * (l + 1 + mm)), den = 1 / r1;
        cs[lane] = make_double2((2 * l + 1) * den, r0 * den);
        c3s[lane] = (m2 / (l + r0) + m2 / (l + 1 + r1)) * den;   // c1 - c2 - 1
    }
    __syncthreads();
    const double y = on ? xm1 : 0;
    double p = 1, dp = 0, q = 0, dq = 1;   // the two solutions
    int E = 0, j = 0;
    auto step = [&](int i) {
        const double2 c = cs[i];
        const double kap = fma(c.x, y, c3s[i]);
        dp = fma(kap, p, c.y * dp);
        dq = fma(kap, q, c.y * dq);
        p += dp;
        q += dq;
    };
    for (; j < n4; j += 4) {
#pragma unroll
        for (int t = 0; t < 4; t++) step(j + t);
        if (p > 0x1p300) {   // q < 64 p
            p *= 0x1p-300;
            dp *= 0x1p-300;
            q *= 0x1p-300;
            dq *= 0x1p-300;
            E += 300;
        }
    }
    for (; j < l1 - l0; j++) step(j);
    const int e = __builtin_amdgcn_frexp_exp(p) - 1;
    double2* T = at<double2>(arena, d.off_run) + (int64_t)run * 2 * nP;
    T[k] = make_double2(ldexp(p, -e), ldexp(dp, -e));
    T[nP + k] = make_double2(ldexp(q, -e), ldexp(dq, -e));
    at<int>(arena, d.off_run + 32 * (int64_t)runs * nP)[run * nP + k] = E + e;
}

// What one degree needs, the same for all nodes of a block: c1, c2 of
// degree_step; t_l = l x S_l - rt S_{l-1} (m = 0: l S_l with l = √(l(l+1)), t_l =
// P_l^1); the Mie factors (zero past the window) over 2^e, e the exponent of the
// first of each four degrees, and sh = e less that of the four before.  The
// state (S_l, S_{l-1}) is kept times 2^e: numbers of the size of F over a
// factor near 1, so that no degree needs an exponent of its own.
__device__ __forceinline__ Deg degree(const BlockDesc& d, char* arena, int l)
{
    const int mm = d.m > 0 ? d.m : 1, last = d.lmin + d.ldim - 1;
    const double den = 1 / sqrt((l + 1.0 - mm) * (l + 1.0 + mm));
    const double rt = sqrt(((double)l - mm) * ((double)l + mm));
    const int l4 = l - ((l - d.lmin) & 3);
    const double* a = at<double>(arena, d.off_mie) + (l - 1);
    const int* ea = at<int>(arena, d.off_mie + 32 * (int64_t)d.mie_L);
    Deg g;
    g.c1 = (2.0 * l + 1) * den;
    g.c2 = rt * den;
    g.l = d.m > 0 ? l : sqrt((double)l * (l + 1.0));
    g.rt = d.m > 0 ? rt : 0.0;
    g.e = ea[min(l4, last) - 1];
    g.sh = l4 > d.lmin ? g.e - ea[min(l4 - 4, last) - 1] : 0;
    g.ma = g.mb = g.pad_ = 0;
    if (l <= last) {
        const int e = ea[l - 1] - g.e;
        g.ma = ldexp(a[2 * (int64_t)d.mie_L], e);
        g.mb = ldexp(a[3 * (int64_t)d.mie_L], e);
    }
    return g;
}

__device__ __forceinline__ void shift(double& p, double& pp, int e)
{
    p = ldexp(p, e);
    pp = ldexp(pp, e);
}

// One degree at one node, up to the node's √r: the four products of (t_l, p_l)
// and the Mie factors (a_l, b_l), and the step to the next degree.  xt: x, 1 for m = 0.
__device__ __forceinline__ void degree_rows(const Deg& g, double m, double x, double xt, double& p, double& pp,
                                            double& ta, double& pb, double& pa, double& tb)
{
    const double t = fma(g.l * xt, p, -(g.rt * pp)), q = m * p;
    ta = t * g.ma;
    pb = q * g.mb;
    pa = q * g.ma;
    tb = t * g.mb;
    degree_step(g.c1, g.c2, x, p, pp);
}

// The states at the runs' starts, in place of the matrices that lead to them
// (what k_wave_norms does by itself where the runs are few).
__global__ void __launch_bounds__(64) k_wave_prefix(const BlockDesc* __restrict__ desc, char* __restrict__ arena,
                                                    int64_t* __restrict__ clock)
{
    stage_begins(clock);
    const BlockDesc& d = desc[blockIdx.y];
    if ((int)blockIdx.x >= d.n_waves) return;
    const int nP = d.n_waves * 64, k = blockIdx.x * 64 + threadIdx.x, runs = d.n_below + d.n_segs - 1;
    const double* nd = at<double>(arena, d.off_node);
    double2* T = at<double2>(arena, d.off_run) + k;
    int* TE = at<int>(arena, d.off_run + 32 * (int64_t)runs * nP) + k;
    double p = nd[3 * nP + k], dp = p;   // S_{m-1} = 0
    int E = at<int>(arena, d.off_node + 32 * (int64_t)nP)[k];
    constexpr int AHEAD = 8;
    double2 a[2][AHEAD], b[2][AHEAD];
    int e[2][AHEAD];
    auto fetch = [&](int g, int h) {
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            const int r = min(g + i, runs - 1);
            a[h][i] = T[(int64_t)r * 2 * nP];
            b[h][i] = T[((int64_t)r * 2 + 1) * nP];
            e[h][i] = TE[r * nP];
        }
    };
    auto steps = [&](int g, int h) {
#pragma unroll
        for (int i = 0; i < AHEAD; i++)
            if (g + i < runs) {
                next_run(a[h][i], b[h][i], e[h][i], p, dp, E);
                T[(int64_t)(g + i) * 2 * nP] = make_double2(p, dp);
                TE[(g + i) * nP] = E;
            }
    };
    if (runs == 0) return;
    fetch(0, 0);
    for (int g = 0; g < runs; g += 2 * AHEAD) {
        fetch(g + AHEAD, 1);
        steps(g, 0);
        fetch(g + 2 * AHEAD, 0);
        steps(g + AHEAD, 1);
    }
}

// Runs of 64 degrees at 64 nodes: the state at the run's start from
// k_wave_start's matrices, the states every 8 degrees (for k_gram), the
// squared norms of F's rows over the run, and per chunk and tile of 8 nodes
// the exponent of the largest chunk norm (c_k < 2^e); the degrees' constants
// for k_gram.  Bound by FP64 instructions, 15 per degree and node.
// SPLIT: a workgroup per run and 64 nodes, a chunk per wavefront, which gets
// to its chunk with the bare recurrence; else a run of 128 nodes per wavefront
// (two per lane: half the reads of the degrees' constants), which a batch
// takes that has enough of them.  Both make the same sums.
template <bool SPLIT>
__global__ void __launch_bounds__(256) k_wave_norms(const BlockDesc* __restrict__ desc, int n, char* __restrict__ arena,
                                                    int prefixed, int64_t* __restrict__ clock)
{
    if (!prefixed) stage_begins(clock);
    constexpr int NH = SPLIT ? 1 : 2;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int u = SPLIT ? blockIdx.x : 4 * blockIdx.x + wv;
    const int BlockDesc::*first = SPLIT ? &BlockDesc::unit_split : &BlockDesc::unit_pair;
    const BlockDesc& d = desc[block_of(desc, n, u, const_cast<int BlockDesc::*>(first))];
    u -= SPLIT ? d.unit_split : d.unit_pair;
    const int nw = SPLIT ? d.n_waves : (d.n_waves + 1) / 2, wave = u % nw, s = u / nw, nP = d.n_waves * 64;
    const double m = d.m;
    __shared__ Deg degs_[SPLIT ? 64 : 256];
    __shared__ double part[SPLIT ? 4 : 1][64];
    Deg* degs = degs_ + (SPLIT ? 0 : 64 * wv);
    const int nc = s < d.n_segs ? min(4, d.n_chunks - 4 * s) : 0;
    if ((!SPLIT || wv == 0) && lane < 16 * nc) {
        const Deg g = degree(d, arena, d.lmin + 64 * s + lane);
        degs[lane] = g;
        if (wave == 0) at<Deg>(arena, d.off_deg)[64 * s + lane] = g;
    }
    __syncthreads();
    const double* nd = at<double>(arena, d.off_node);
    double x[NH], p[NH], pp[NH], sum[NH];
    int E[NH], k[NH];
    if (SPLIT ? wv < nc : nc > 0) {
#pragma unroll
        for (int h = 0; h < NH; h++) {
            k[h] = min(wave * 64 * NH + 64 * h + lane, nP - 1);   // (an odd last wave: not stored)
            x[h] = nd[k[h]];
            p[h] = nd[3 * nP + k[h]];
            pp[h] = p[h];   // S - S_{l-1}, until the run's start
            E[h] = at<int>(arena, d.off_node + 32 * (int64_t)nP)[k[h]];
            sum[h] = 0;
        }
        const int runs = d.n_below + d.n_segs - 1;
        const double2* T = at<double2>(arena, d.off_run);
        const int* TE = at<int>(arena, d.off_run + 32 * (int64_t)runs * nP);
        const int to = d.n_below + s;
#pragma unroll 4
        for (int g = prefixed ? max(to - 1, 0) : 0; g < to; g++)
#pragma unroll
            for (int h = 0; h < NH; h++) {
                const double2 a = T[(int64_t)g * 2 * nP + k[h]], b = T[(int64_t)(g * 2 + 1) * nP + k[h]];
                const int e = TE[g * nP + k[h]];
                if (prefixed) {
                    p[h] = a.x;
                    pp[h] = a.y;
                    E[h] = e;
                } else {
                    next_run(a, b, e, p[h], pp[h], E[h]);
                }
            }
#pragma unroll
        for (int h = 0; h < NH; h++) {
            pp[h] = p[h] - pp[h];
            shift(p[h], pp[h], E[h] + degs[0].e);
        }
    }
    for (int c = 0; c < nc; c++) {
        if (SPLIT && c < wv) {
#pragma unroll 4
            for (int j = 0; j < 16; j++) {
                const Deg& g = degs[16 * c + j];
                if ((j & 3) == 0 && c + j > 0) shift(p[0], pp[0], g.sh);
                degree_step(g.c1, g.c2, x[0], p[0], pp[0]);
            }
            continue;
        }
        if (SPLIT && c > wv) break;
        const int ch = 4 * s + c;
        double ntm[NH], nte[NH];
#pragma unroll
        for (int h = 0; h < NH; h++) {
            ntm[h] = nte[h] = 0;
            if (c > 0) shift(p[h], pp[h], degs[16 * c].sh);
        }
#pragma unroll 8
        for (int j = 0; j < 16; j++) {
            const Deg& g = degs[16 * c + j];
#pragma unroll
            for (int h = 0; h < NH; h++) {
                double ta, pb, pa, tb;
                if ((j & 3) == 0 && j > 0) shift(p[h], pp[h], g.sh);
                if ((j & 7) == 0 && wave * 64 * NH + 64 * h < nP)
                    at<double2>(arena, d.off_ck)[(int64_t)(2 * ch + (j >> 3)) * nP + k[h]] = make_double2(p[h], pp[h]);
                degree_rows(g, m, x[h], m > 0 ? x[h] : 1.0, p[h], pp[h], ta, pb, pa, tb);
                ntm[h] = fma(ta, ta, fma(pb, pb, ntm[h]));
                nte[h] = fma(pa, pa, fma(tb, tb, nte[h]));
            }
        }
#pragma unroll
        for (int h = 0; h < NH; h++) {
            const double stm = nd[nP + k[h]], ste = nd[2 * nP + k[h]];
            const double norm = stm * stm * ntm[h] + ste * ste * nte[h];
            sum[h] += norm;
            int e = norm > 0 ? ilogb(norm) + 1 : NO_EXP;   // a NaN norm: the trace is NaN
            e = max(e, dpp_i<DPP_QUAD_X1>(e));
            e = max(e, dpp_i<DPP_QUAD_X2>(e));
            e = max(e, dpp_i<DPP_HALF_MIRROR>(e));
            if ((lane & 7) == 0 && wave * 64 * NH + 64 * h < nP)
                at<int>(arena, d.off_act)[(int64_t)ch * (nP >> 3) + (k[h] >> 3)] = e;
        }
    }
    double* norm = at<double>(arena, d.off_norm) + (int64_t)s * nP;
    if (SPLIT) {
        part[wv][lane] = wv < nc ? sum[0] : 0;
        __syncthreads();
        if (wv > 0 || nc == 0) return;
        double v = part[0][lane];
        for (int c = 1; c < nc; c++) v += part[c][lane];
        norm[wave * 64 + lane] = v;
    } else if (nc > 0) {
#pragma unroll
        for (int h = 0; h < NH; h++)
            if (wave * 64 * NH + 64 * h < nP) norm[k[h]] = sum[h];
    }
}

// F itself, F[2(l-lmin) + (0: a_l, 1: b_l)][row], over 16 degrees and 64 nodes per
// wavefront (k_wave_matrix; k_gram makes its own).
__global__ void __launch_bounds__(256) k_wave_rows(const BlockDesc* __restrict__ desc, char* __restrict__ arena)
{
    const BlockDesc& d = desc[blockIdx.y];
    const int nq = (d.n_chunks + 3) / 4;
    if ((int)blockIdx.x >= d.n_waves * nq) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int wave = blockIdx.x % d.n_waves, c = (blockIdx.x / d.n_waves) * 4 + wv;
    const int nP = d.n_waves * 64, k = wave * 64 + lane;
    const double m = d.m;
    __shared__ Deg degs[4][16];
    const bool in = c < d.n_chunks;
    if (in && lane < 16) degs[wv][lane] = degree(d, arena, d.lmin + 16 * c + lane);
    __syncthreads();
    if (!in) return;
    const int64_t ci = 2 * (int64_t)c * nP + k, ldf = 2 * (int64_t)nP;
    const double* nd = at<double>(arena, d.off_node);
    const double x = nd[k], stm = nd[nP + k], ste = nd[2 * nP + k];
    const double2 s = at<double2>(arena, d.off_ck)[ci];
    double p = s.x, pp = s.y;
    double* F = at<double>(arena, d.off_rows) + 32 * (int64_t)c * ldf + 2 * k;
#pragma unroll 4
    for (int j = 0; j < 16; j++) {
        double ta, pb, pa, tb;
        if ((j & 3) == 0 && j > 0) shift(p, pp, degs[wv][j].sh);
        degree_rows(degs[wv][j], m, x, m > 0 ? x : 1.0, p, pp, ta, pb, pa, tb);
        *reinterpret_cast<double2*>(F) = make_double2(stm * ta, ste * pa);
        *reinterpret_cast<double2*>(F + ldf) = make_double2(stm * pb, ste * tb);
        F += 2 * ldf;
    }
}

// Trace of M = the sum of all rows' squared norms (per node over the runs of 64
// degrees, in quarters, then over the nodes with compensated sums in a fixed
// order), the trace shortcut |tr M| < 1e-8 (src/matrix.c:78-82), and the window: tiles of 8
// nodes from the first to the last node whose rows carry more than 2^-60 of
// the trace (together the others change the determinant by less than a few
// 1e-17 of it; R/L = 20 .. 2000: 10-60 % of the nodes of large m).  dense:
// the matrix dimension for the LU's kernels goes to desc[b].N.
// NT: 1024 threads, one quarter of the runs each (block of R/L = 2000: 118 us with
// 256 threads over its chunks of 16 degrees, 29 so), or 256 for batches of many
// blocks: norms and window of 4000 blocks of R/L = 20 158 us with 1024 and 118
// with 256, of 1000 46 and 40, of 1168 of R/L = 200 400 and 394; of 300 123 and
// 133, of 512 of R/L = 100 100 and 104.
template <int NT>
__global__ void __launch_bounds__(NT) k_wave_window(BlockDesc* __restrict__ desc, char* __restrict__ arena,
                                                    BlockOut* __restrict__ out, const int* __restrict__ status,
                                                    int allow, int dense)
{
    const int b = blockIdx.x, tid = threadIdx.x;
    const BlockDesc& d = desc[b];
    const int nP = d.n_waves * 64;
    const double* cn = at<double>(arena, d.off_norm);
    double* dn = at<double>(arena, d.off_dn);
    constexpr int NQ = 1024 / NT;   // quarters per thread
    __shared__ double part[4][NT == 1024 ? 256 : 1];
    double s = 0, comp = 0;
    for (int k0 = 0; k0 < nP; k0 += 256) {
        const int k = k0 + (tid & 255);
        double v[NQ];
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const int quarter = NQ == 1 ? tid >> 8 : i;
            const int r0 = quarter * d.n_segs / 4, r1 = (quarter + 1) * d.n_segs / 4;
            v[i] = 0;
            if (k < nP) {
#pragma unroll 8
                for (int r = r0; r < r1; r++) v[i] += cn[(int64_t)r * nP + k];
            }
        }
        double q[4];
        if constexpr (NQ == 1) {
            part[tid >> 8][tid & 255] = v[0];
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = part[i][tid & 255];
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = v[i];
        }
        if (tid < 256 && k < nP) {
            const double w = (q[0] + q[1]) + (q[2] + q[3]);
            dn[k] = w;
            double t, e;
            two_sum(s, w, t, e);
            s = t;
            comp += e;
        }
        __syncthreads();
    }
    __shared__ double hs[256], cs[256];
    __shared__ int lo_s, hi_s;
    if (tid < 256) {
        hs[tid] = s;
        cs[tid] = comp;
    }
    if (tid == 0) {
        lo_s = nP;
        hi_s = -1;
    }
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (tid < o) {
            double t, e;
            two_sum(hs[tid], hs[tid + o], t, e);
            hs[tid] = t;
            cs[tid] = (cs[tid] + cs[tid + o]) + e;
        }
        __syncthreads();
    }
    const double trace = hs[0] + cs[0], thr = trace * 0x1p-60;
    for (int k = tid; k < nP; k += NT)
        if (dn[k] > thr) {
            atomicMin(&lo_s, k);
            atomicMax(&hi_s, k);
        }
    __syncthreads();
    if (tid != 0) return;
    BlockOut& o = out[b];
    const bool fin = isfinite(trace);
    o.trace = trace;
    // skip 1: trace shortcut; 3: non-finite trace (no LU, NaN result)
    o.skip = fabs(trace) < 1e-8 ? 1 : (fin ? 0 : 3);
    o.logdet = NAN;
    o.frob2 = o.tr2 = 0;
    o.status = *status;   // of the whole batch: it comes back with the results
    o.delta = allow;
    o.tile0 = lo_s >> 3;
    o.tiles = o.skip || hi_s < 0 ? 0 : (hi_s >> 3) - (lo_s >> 3) + 1;
    o.etr = fin && trace > 0 ? ilogb(trace) : 0;
    if (dense) desc[b].N = 16 * o.tiles;
}

// The band of -G = -F Fᵀ on FP64 MFMA (v_mfma_f64_16x16x4f64): a workgroup of four
// wavefronts takes NC column tiles and for each its BAND_TILES tiles on and
// below the diagonal (the column's own tile is both operands of the diagonal
// one).  The rows of these tiles are made on the spot, a chunk of 16 degrees
// at a time, from the states that k_wave_norms kept (32 bytes instead of 512
// per node and chunk): eight tiles are the 64 lanes of a wavefront, which
// makes degrees 4 w .. 4 w + 3; then the pairs are multiplied.  (Making the next
// chunk in four more wavefronts beside the products gains nothing: FP64
// instructions and FP64 MFMA do not overlap.  Bound by the two together:
// at a grid of step 0.5 99 of 271 us without the products, 223 without the rows.)
// A row's ridge covers a few chunks: a pair of tiles is multiplied over a
// chunk only if the product of their largest chunk norms is at least 2^-60
// tr (by Cauchy-Schwarz what is left out is smaller, below the last bit of
// the trace; R/L = 200, NC = 4: 24 of 75 chunks per strip, 12 of 28 pairs).
// The pairs that count in a chunk lie next to each other, so NC = 4 deals them
// out along the diagonals: wavefront w has tile j + r of column j = (w + r) % 4, for r = 0
// .. 6; the busiest one then has 3.4 on average of 2.9 (whole columns: 4.8).
// The three pairs with the strip's ninth and tenth tile are a step of their
// own over tiles 2 .. 9, where they count at all.
// NC = 1 for batches that would leave CUs idle: two chunks per step in twice
// the wavefronts, a pair each (one block of R/L = 200: 28 us).
// An element sums the same products in the same order for either NC, so its
// bits do not depend on the batch.
// 222 blocks of R/L = 200: 271 to 293 us.  (At a step of 0.5, a tenth fewer
// nodes, 245 to 271, and 309 with an exponent and a power of two per degree and the
// states every 16 degrees, 478 + 124 with F's rows stored by a kernel of their own
// and read back, bound by the loads' latency.)
template <int NC>
__global__ void __launch_bounds__(NC == 4 ? 256 : 512, NC == 4 ? 3 : 2)
    k_gram(const BlockDesc* __restrict__ desc, char* __restrict__ arena, const BlockOut* __restrict__ out, int delta_only,
           int64_t* __restrict__ clock)
{
    stage_begins(clock);
    static_assert(NC == 1 || NC == 4, "columns per workgroup");
    constexpr int NR = NC + BAND_TILES - 1, NS = 8, PITCH = 16 * NS + 16, KS = 32;
    constexpr int NG = NC == 4 ? 1 : 2, NW = 4 * NG;   // chunks per step, wavefronts
    constexpr int PS = NC == 4 ? BAND_TILES : 1;       // pairs per wavefront
    static_assert(NW * PS <= 32 && (NC == 4 || NW >= BAND_TILES), "a bit and a place for every pair");
    static_assert(NR <= NS + 2, "tiles 0 .. 7 and 2 .. 9");
    constexpr int LATE = 1 << 30;
    __shared__ double W[NG][KS][PITCH];   // [2 (l - l0) + (0: a_l, 1: b_l)][row of eight tiles]
    alignas(16) __shared__ Deg degs[NG][16];
    __shared__ int nlist;
    extern __shared__ int2 list[];    // chunk, LATE if from tile 2 on; pairs (bit PS w + i)
    const int b = blockIdx.y;
    const BlockDesc& d = desc[b];
    const BlockOut& o = out[b];
    const int T = o.tiles, J0 = NC * (int)blockIdx.x;
    if (o.skip || J0 >= T || (delta_only && !o.delta)) return;
    const int nP = d.n_waves * 64, nT = nP >> 3, nt = min(NR, T - J0);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, lk = lane >> 4;
    // pair i of wavefront w: column col_of(w, i), tile col_of + row_of
    auto col_of = [](int w, int i) { return NC == 4 ? (w + i) & 3 : 0; };
    auto row_of = [](int w, int i) { return NC == 4 ? i : w; };
    if (wv == 0) {
        const int* act = at<int>(arena, d.off_act) + o.tile0 + J0;
        const int lim = 2 * o.etr - 120;
        int n = 0;
        for (int c0 = 0; c0 < d.n_chunks; c0 += 64) {
            const int c = c0 + lane;
            int e[NR];
            unsigned pa = 0, pb = 0;
#pragma unroll
            for (int t = 0; t < NR; t++) e[t] = c < d.n_chunks && t < nt ? act[(int64_t)c * nT + t] : NO_EXP;
#pragma unroll
            for (int w = 0; w < NW; w++)
#pragma unroll
                for (int i = 0; i < PS; i++) {
                    const int j = col_of(w, i), r = row_of(w, i);
                    if (r >= BAND_TILES) continue;
                    const unsigned on = e[j] + e[j + r] >= lim;
                    (j + r < NS ? pa : pb) |= on << (PS * w + i);
                }
            const unsigned long long ba = __ballot(pa != 0), bb = __ballot(pb != 0), below = (1ull << lane) - 1;
            const int i = n + __popcll(ba & below) + __popcll(bb & below);
            if (pa) list[i] = make_int2(c, (int)pa);
            if (pb) list[i + (pa != 0)] = make_int2(c | LATE, (int)pb);
            n += __popcll(ba) + __popcll(bb);
        }
        if (lane == 0) nlist = n;
    }
    __syncthreads();
    const int ns = nlist;
    const int k0 = 8 * (o.tile0 + J0);
    const double* nd = at<double>(arena, d.off_node);
    const double2* ck = at<double2>(arena, d.off_ck);
    const int* dg = at<int>(arena, d.off_deg) + (tid & 255);   // 4 bytes of a chunk's constants per lane
    // this lane's node: in the (lane/8)-th of the step's eight tiles, from
    // tile 0 or tile 2 on (nodes past the block's are loaded as its last one
    // and not used)
    const int slot = lane >> 3, ka = min(k0 + lane, nP - 1), kb = min(k0 + lane + 16, nP - 1);
    const double xa = nd[ka], xb = nd[kb], m = d.m;
    const int grp = wv >> 2, sub = wv & 3;   // its chunk of the step and four degrees
    // states and constants of a step, loaded two steps ahead
    struct State {
        double2 s;
        int dg, en, pm[NG];
    };
    auto load = [&](int s, State& v) {
        v.en = __builtin_amdgcn_readfirstlane(list[min(NG * s + grp, ns - 1)].x);
#pragma unroll
        for (int g = 0; g < NG; g++) {
            const unsigned pm = list[min(NG * s + g, ns - 1)].y;
            v.pm[g] = NG * s + g < ns ? __builtin_amdgcn_readfirstlane((pm >> (PS * wv)) & ((1u << PS) - 1)) : 0;
        }
        const int c = v.en & ~LATE;
        v.s = ck[(int64_t)(2 * c + (sub >> 1)) * nP + (v.en & LATE ? kb : ka)];
        v.dg = dg[256 * c];
    };
    double4_t acc[PS];
#pragma unroll
    for (int i = 0; i < PS; i++) acc[i] = (double4_t){0, 0, 0, 0};
    auto step = [&](int s, State& v) {
        const int en = v.en;
        unsigned pm[NG];
#pragma unroll
        for (int g = 0; g < NG; g++) pm[g] = v.pm[g];
        // (every wavefront is past the constants of the step before)
        reinterpret_cast<int*>(degs)[tid] = v.dg;
        double p = v.s.x, pp = v.s.y;
        load(s + 2, v);
        __syncthreads();   // and past its products
        {
            // (lanes of tiles that no pair needs run along: numbers, never read)
            const double x = en & LATE ? xb : xa, xt = m > 0 ? x : 1.0;
            if (sub & 1) {   // the state is kept every 8 degrees
                const int j = 4 * (sub - 1);
                double2 cc[4];
#pragma unroll
                for (int q = 0; q < 4; q++) cc[q] = *reinterpret_cast<const double2*>(&degs[grp][j + q].c1);
                const int e = degs[grp][j + 4].sh;
#pragma unroll
                for (int q = 0; q < 4; q++) degree_step(cc[q].x, cc[q].y, x, p, pp);
                shift(p, pp, e);
            }
            Deg g[4];
#pragma unroll
            for (int j = 0; j < 4; j++) g[j] = degs[grp][4 * sub + j];
            double2* w = reinterpret_cast<double2*>(&W[grp][8 * sub][2 * lane]);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                double ta, pb, pa, tb;
                degree_rows(g[j], m, x, xt, p, pp, ta, pb, pa, tb);
                w[j * PITCH] = make_double2(ta, pa);
                w[j * PITCH + PITCH / 2] = make_double2(pb, tb);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NG * PS; i++)
            if (pm[i / PS] >> (i % PS) & 1) {
                const double* wc = &W[i / PS][lk][li - (NC == 4 && en & LATE ? 32 : 0)] + 16 * col_of(wv, i % PS);
                const double* wr = wc + 16 * row_of(wv, i % PS);
                double cv[KS / 4], rv[KS / 4];
#pragma unroll
                for (int q = 0; q < KS / 4; q++) {
                    cv[q] = wc[4 * q * PITCH];
                    rv[q] = NC == 4 && i == 0 ? cv[q] : wr[4 * q * PITCH];
                }
#pragma unroll
                for (int q = 0; q < KS / 4; q++)
                    acc[i % PS] = __builtin_amdgcn_mfma_f64_16x16x4f64(cv[q], rv[q], acc[i % PS], 0, 0, 0);
            }
    };
    if (ns > 0) {
        State v0, v1;
        load(0, v0);
        load(1, v1);
        for (int s = 0; NG * s < ns; s += 2) {
            step(s, v0);
            if (NG * (s + 1) < ns) step(s + 1, v1);
        }
    }
    // lane l, register q: column l/16 + 4q of the column tile, row l%16; tiles
    // are kept column by column; -√r √r' of the two rows at the end
    const double* sr = nd + k0 + nP + (li & 1) * nP + (li >> 1);   // row l%16 of tile 0
    const double* sc = nd + k0 + nP + (lk & 1) * nP + (lk >> 1);   // column l/16 (+ 4q: node + 2q) of tile 0
#pragma unroll
    for (int i = 0; i < PS; i++) {
        const int j = col_of(wv, i), r = row_of(wv, i);
        if (r >= BAND_TILES || J0 + j + r >= T) continue;
        double* B = at<double>(arena, d.off_band) + ((int64_t)(J0 + j) * BAND_TILES + r) * 256 + lane;
        const double s = -sr[8 * (j + r)];
#pragma unroll
        for (int q = 0; q < 4; q++) B[64 * q] = acc[i][q] * (s * sc[8 * j + 2 * q]);
    }
}

// Broadcasts within 16 lanes as DPP operands of the FMAs: v_fmac_f64 takes
// row_newbcast, but the compiler makes a move and an FMA of them, and puts off
// the rows x, which costs 128 spilled registers.  Two wait states have to lie
// between a VALU write and a DPP read of it: the instructions between, or
// s_nop.
#define FMAC_ROW(x, a, l) "v_fmac_f64_dpp %" #x ", %" #a ", %[" #l "] row_newbcast:%[t] row_mask:0xf bank_mask:0xf\n"
#define MOV_ROW(d, a) "v_mov_b64_dpp %" #d ", %" #a " row_newbcast:%[u] row_mask:0xf bank_mask:0xf\n"

// x += a(lane T) lx, a += a(lane T) la for column T + 1 (and x of the two
// behind it); returns the next pivot, a(lane T + 1) of column T + 1
template <int T>
__device__ __forceinline__ double column_next(double (&x)[16], double (&a)[16], double lx, double la)
{
    double d;
    if constexpr (T < 13)
        asm volatile("s_nop 1\n" FMAC_ROW(0, 4, lx) FMAC_ROW(4, 4, la) FMAC_ROW(1, 5, lx) FMAC_ROW(2, 6, lx) MOV_ROW(3, 4)
                     : "+v"(x[T + 1]), "+v"(x[T + 2]), "+v"(x[T + 3]), "=&v"(d), "+v"(a[T + 1])
                     : "v"(a[T + 2]), "v"(a[T + 3]), [lx] "v"(lx), [la] "v"(la), [t] "n"(T), [u] "n"(T + 1));
    else
        asm volatile("s_nop 1\n" FMAC_ROW(0, 2, lx) FMAC_ROW(2, 2, la) "s_nop 1\n" MOV_ROW(1, 2)
                     : "+v"(x[T + 1]), "=&v"(d), "+v"(a[T + 1])
                     : [lx] "v"(lx), [la] "v"(la), [t] "n"(T), [u] "n"(T + 1));
    return d;
}

// ... for a of columns T + 2 .. 15 and x of those that column_next left, from
// column J on; up to four columns per statement (and the two whose x is done), each
// with the wait states before its first read: what the compiler may have moved
// to an operand's register just before it does not see the DPP.
#define COLUMN(x, a) FMAC_ROW(x, a, lx) FMAC_ROW(a, a, la)
template <int T, int J = T < 13 ? T + 4 : T + 2>
__device__ __forceinline__ void columns_rest(double (&x)[16], double (&a)[16], double lx, double la)
{
#define LANES [lx] "v"(lx), [la] "v"(la), [t] "n"(T)
    constexpr int N = J < 16 ? (16 - J < 4 ? 16 - J : 4) : 0;
    if constexpr (T < 13 && J == T + 4) {   // a of T + 2 and T + 3 with it
#define FIRST "s_nop 1\n" FMAC_ROW(0, 0, la) FMAC_ROW(1, 1, la)
#define OPS "+v"(a[T + 2]), "+v"(a[T + 3])
        if constexpr (N == 4)
            asm volatile(FIRST COLUMN(2, 6) COLUMN(3, 7) COLUMN(4, 8) COLUMN(5, 9)
                         : OPS, "+v"(x[J]), "+v"(x[J + 1]), "+v"(x[J + 2]), "+v"(x[J + 3]), "+v"(a[J]),
                           "+v"(a[J + 1]), "+v"(a[J + 2]), "+v"(a[J + 3]) : LANES);
        else if constexpr (N == 3)
            asm volatile(FIRST COLUMN(2, 5) COLUMN(3, 6) COLUMN(4, 7)
                         : OPS, "+v"(x[J]), "+v"(x[J + 1]), "+v"(x[J + 2]), "+v"(a[J]), "+v"(a[J + 1]),
                           "+v"(a[J + 2]) : LANES);
        else if constexpr (N == 2)
            asm volatile(FIRST COLUMN(2, 4) COLUMN(3, 5)
                         : OPS, "+v"(x[J]), "+v"(x[J + 1]), "+v"(a[J]), "+v"(a[J + 1]) : LANES);
        else if constexpr (N == 1)
            asm volatile(FIRST COLUMN(2, 3) : OPS, "+v"(x[J]), "+v"(a[J]) : LANES);
        else
            asm volatile(FIRST : OPS : LANES);
#undef FIRST
#undef OPS
    } else if constexpr (N == 4) {
        asm volatile("s_nop 1\n" COLUMN(0, 4) COLUMN(1, 5) COLUMN(2, 6) COLUMN(3, 7)
                     : "+v"(x[J]), "+v"(x[J + 1]), "+v"(x[J + 2]), "+v"(x[J + 3]), "+v"(a[J]), "+v"(a[J + 1]),
                       "+v"(a[J + 2]), "+v"(a[J + 3]) : LANES);
    } else if constexpr (N == 3) {
        asm volatile("s_nop 1\n" COLUMN(0, 3) COLUMN(1, 4) COLUMN(2, 5)
                     : "+v"(x[J]), "+v"(x[J + 1]), "+v"(x[J + 2]), "+v"(a[J]), "+v"(a[J + 1]), "+v"(a[J + 2])
                     : LANES);
    } else if constexpr (N == 2) {
        asm volatile("s_nop 1\n" COLUMN(0, 2) COLUMN(1, 3)
                     : "+v"(x[J]), "+v"(x[J + 1]), "+v"(a[J]), "+v"(a[J + 1]) : LANES);
    } else if constexpr (N == 1) {
        asm volatile("s_nop 1\n" COLUMN(0, 1) : "+v"(x[J]), "+v"(a[J]) : LANES);
    }
#undef LANES
    if constexpr (J + N < 16) columns_rest<T, J + N>(x, a, lx, la);
}
#undef COLUMN
#undef FMAC_ROW
#undef MOV_ROW

// value of lane N of the lane's 16
template <int N>
__device__ __forceinline__ double row_d(double x)
{
    return __longlong_as_double(
        __builtin_amdgcn_update_dpp(0ll, __double_as_longlong(x), 0x150 + N, 0xf, 0xf, true));
}

// log det(1 - G) of one block by LDLᵀ without pivoting (1 - G is symmetric
// positive definite, so the elimination is stable in any order), in the
// delta form: the matrix holds -G, pivots are u = 1 + d with d the stored
// diagonal, and log u = log1p(d) keeps the accuracy of small blocks.  One
// workgroup of sixteen wavefronts.
// What bounds it is the chain of pivots, 16 per tile column, so
//  - the band is eliminated from both ends at once towards the six tile columns
//    in its middle (half 1 has the order of the tiles reversed; what it
//    subtracts from the middle is added to half 0's before these follow);
//  - a column's pivots run beside the update of the column before: wavefronts
//    0 .. 3 factor, two per half, the others update the tiles behind on MFMA,
//    the next column's first;
//  - the tiles behind stay in registers from the load to their own column:
//    a wavefront has one diagonal of tiles, and only the column in work and
//    the next one are in LDS.
// The pivots' FMAs and the MFMAs share the SIMDs' FP64 units, 1900 and 2800
// cycles of the 7200 that a step takes.  16, 29 and 89 tile columns: 40, 62 and
// 153 us; 15, 26 and 79: 39, 55 and 136 us, and column after column from one end,
// through LDS, 55, 94 and 282 us.
// mercator: the LU-mode rule of src/matrix.c:489-505 first (||M||_F² = tr M² =
// Σ G_ij²; skip = 2: the host returns the two-term series).
// host: pinned host memory for the results of all blocks, also of those that are
// not factored here.
__global__ void __launch_bounds__(1024) k_band_ldl(const BlockDesc* __restrict__ desc, char* __restrict__ arena,
                                                   BlockOut* __restrict__ out, BlockOut* __restrict__ host, int mercator,
                                                   int64_t* __restrict__ clock)
{
    stage_begins(clock);
    constexpr int NTH = 1024, BT = BAND_TILES, COL = BT * 256, MID = BT - 1;
    static_assert(BT == 7, "six diagonals of tiles, dealt to twelve wavefronts");
    __shared__ double S[2][2][COL];
    const int b = blockIdx.x;
    const BlockDesc& d = desc[b];
    BlockOut& o = out[b];
    const int T = o.tiles;
    auto result = [&] {   // (by thread 0, which wrote what is new in it)
        o.t_end = wall_clock64();
        host[b] = o;
    };
    if (o.skip || !o.delta || T <= 0) {
        if (threadIdx.x == 0) result();
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    double* B = at<double>(arena, d.off_band);
    if (mercator) {
        // ||G||_F >= tr G / √N: most blocks are past the rule without a look at G
        const double tr = o.trace, low = fabs(tr) / sqrt(16.0 * T);
        bool may = low < 1;
        if (may) may = low * low / 2 + low + log1p(-low) >= -2e-8 * (fabs(tr) + tr * tr / 2);
        if (may) {
            double* red = &S[0][0][0];
            double f = 0;
            for (int64_t i = tid; i < (int64_t)T * COL; i += NTH) {
                const int r = (int)(i % COL) >> 8, J = (int)(i / COL);
                if (J + r < T) f += (r ? 2.0 : 1.0) * (B[i] * B[i]);
            }
            red[tid] = f;
            __syncthreads();
            for (int s = NTH / 2; s > 0; s >>= 1) {
                if (tid < s) red[tid] += red[tid + s];
                __syncthreads();
            }
            const double f2 = red[0], norm = sqrt(f2);
            bool take = false;
            if (norm < 1) {
                const double merc = -o.trace - f2 / 2, err = fabs(norm * norm / 2 + norm + log1p(-norm));
                take = fabs(err / merc) < 1e-8;
            }
            __syncthreads();
            if (tid == 0) {
                o.frob2 = o.tr2 = f2;
                if (take) {
                    o.skip = 2;
                    result();
                }
            }
            if (take) return;
        }
    }
    const int mid = T < MID ? T : MID, n0 = (T - mid + 1) / 2, n1 = (T - mid) / 2;   // columns of the halves
    // N elements of tile (I, K) of half h from the band: e, e + 64, ..; 0 for
    // what is not there and half 1's middle (both without a use of what is
    // loaded: the wait comes a step later)
    auto load = [&](int h, int I, int K, int e, auto& v) {
        const bool on = I < (h ? n1 : n0) + mid && K >= 0 && !(h && K >= n1);
        const int src = on ? ((h ? T - 1 - I : K) * BT + I - K) * 256 : 0;
#pragma unroll
        for (double& w : v) {
            w = B[src + (h ? (e & 15) << 4 | e >> 4 : e)];
            e += 64;
        }
        return on ? 1.0 : 0.0;
    };
    // pivots of tile column J of half h and the nb tiles below, -L in place of
    // these: a lane has a row of the tiles below (wavefront part 0 the first 64)
    // and a row of the diagonal tile, which every 16 lanes hold, so that a
    // pivot's row comes as a broadcast within 16 lanes (a done row's lane goes
    // on with what nobody reads)
    auto factor = [&](int h, int J, int nb, int part) {
        double* dp = &S[h][J & 1][li];
        double* tp = dp + (1 + min(4 * part + lk, MID - 1)) * 256;
        double a[16], x[16];
#pragma unroll
        for (int t = 0; t < 16; t++) a[t] = dp[16 * t];
#pragma unroll
        for (int t = 0; t < 16; t++) x[t] = tp[16 * t];
        double dt = row_d<0>(a[0]);
        static_for<16>([&](auto tc) {
            constexpr int t = tc;
            // -1/u from the hardware's estimate r: -r (1 + e + e²), e = 1 - u r
            const double u = 1.0 + dt, r = __builtin_amdgcn_rcp(u);
            const double e = fma(-u, r, 1.0), n = fma(-r, fma(e, e, e), -r);
            x[t] *= n;
            if constexpr (t < 15) {
                const double la = a[t] * n;
                dt = column_next<t>(x, a, x[t], la);
                columns_rest<t>(x, a, x[t], la);
            }
        });
        if (4 * part + lk < nb) {
#pragma unroll
            for (int t = 0; t < 16; t++) tp[16 * t] = x[t];
        }
        if (part == 0 && lane < 16) {
#pragma unroll
            for (int t = 0; t < 16; t++) dp[16 * t] = a[t];   // its diagonal: the d
        }
    };
    {
        const int h = wv >> 3;   // column 0: 512 threads
        for (int i = tid & 511; i < COL; i += 512) {
            double v[1];
            const double f = load(h, i >> 8, 0, i & 255, v);
            S[h][0][i] = f != 0 ? v[0] : 0.0;
        }
    }
    // Two programs with the same barriers, so that the registers of one are not
    // held in the other.
    if (wv < 4) {
        const int h = wv >> 1, part = wv & 1, nh = h ? n1 : n0, end = h ? n1 : n0 + mid;
        double pf[2], on = load(h, 7, 1, part * 128 + lane, pf);   // half of the next column's last tile
        __syncthreads();
        for (int J = 0; J < n0 + mid; J++) {
            if (J == n0 && J > 0) {
                if (n1 > 0) {
                    __syncthreads();
                    __syncthreads();
                }
                __syncthreads();
            }
            const int nb = min(MID, n0 + mid - 1 - J);
            if (J == 0 || J == n0) {
                if (J < end) factor(h, J, nb, part);
                __syncthreads();
            }
            if (J + 1 < nh) {
                double* t = &S[h][(J + 1) & 1][MID * 256 + part * 128 + lane];
#pragma unroll
                for (int s = 0; s < 2; s++) t[64 * s] = on != 0 ? pf[s] : 0.0;
                on = load(h, J + 8, J + 2, part * 128 + lane, pf);
            }
            if (J < end && part == 0 && lane < 16)
                B[(h ? T - 1 - J : J) * COL + lane] = S[h][J & 1][17 * lane];   // d, for the logs
            __syncthreads();
            if (J + 1 != nh && J + 1 < end) factor(h, J + 1, min(MID, nb - (J + 1 > n0)), part);
            __syncthreads();
        }
    } else {
        // half and diagonal I - K = fd of the tiles (J + 1 + i + fd, J + 1 + i) in
        // acc[i]; the wavefronts of a SIMD (modulo 4) have 11 or 10 of a step's 42
        const int h = (wv >> 1) & 1, fd = (wv & 1 ? 0x431 : 0x520) >> (4 * ((wv >> 2) - 1)) & 7, nh = h ? n1 : n0;
        double4_t acc[MID];
        double pf[4], on;
#pragma unroll
        for (int i = 0; i < MID; i++) {
            const double f = load(h, 1 + i + fd, 1 + i, lane, pf);
#pragma unroll
            for (int q = 0; q < 4; q++) acc[i][q] = f != 0 ? pf[q] : 0.0;
        }
        on = load(h, 7, 7 - fd, lane, pf);   // the tile that comes in after this step
        __syncthreads();
        for (int J = 0; J < n0 + mid; J++) {
            auto put = [&](double* col) {   // acc[0] to LDS and to the end
                const double4_t t = acc[0];
#pragma unroll
                for (int q = 0; q < 4; q++) col[256 * fd + 64 * q + lane] = t[q];
#pragma unroll
                for (int i = 0; i + 1 < MID; i++) acc[i] = acc[i + 1];
                acc[MID - 1] = t;
            };
            if (J == n0 && J > 0) {   // the middle: the halves' sum
                double* M = &S[0][0][0] + fd * (2 * MID + 1 - fd) / 2 * 256;
                if (n1 > 0) {
#pragma unroll
                    for (int i = 0; i < MID; i++)
                        if (h && i + fd < MID) {
#pragma unroll
                            for (int q = 0; q < 4; q++)
                                M[(MID - 1 - fd - i) * 256 + 16 * li + 4 * q + lk] = acc[i][q];
                        }
                    __syncthreads();
#pragma unroll
                    for (int i = 0; i < MID; i++)
                        if (!h && i + fd < MID) {
#pragma unroll
                            for (int q = 0; q < 4; q++) acc[i][q] += M[i * 256 + 64 * q + lane];
                        }
                    __syncthreads();
                }
                if (!h) put(S[0][J & 1]);
                __syncthreads();
            }
            if (J == 0 || J == n0) __syncthreads();
            const int nb = J < n1 || h == 0 ? min(MID, n0 + mid - 1 - J) : 0;
            const double* const L = S[h][J & 1];
            const bool last = J + 1 == nh;
            double u[4];
            auto update = [&](int i, int k) {   // acc[i], K = J + 1 + k: -= L_I u L_Kᵀ (-L is stored, and d on the diagonal)
                const double *LK = L + 256 * (1 + k) + lane, *LI = LK + 256 * fd;
                double x[4], y[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    x[q] = LK[64 * q];
                    y[q] = LI[64 * q];
                }
#pragma unroll
                for (int q = 0; q < 4; q++)
                    acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[q] * u[q], y[q], acc[i], 0, 0, 0);
            };
            if (fd < nb) {   // the next column
#pragma unroll
                for (int q = 0; q < 4; q++) u[q] = -1.0 - L[17 * (4 * q + lk)];
                update(0, 0);
                put(S[h][(J + 1) & 1]);
            }
            __syncthreads();
            if (fd < nb) {   // the others
#pragma unroll
                for (int i = 0; i + 1 < MID; i++)
                    if (i + 1 + fd < nb) update(i, i + 1);
                if (last) {   // back for the sum
                    const double4_t t = acc[MID - 1];
#pragma unroll
                    for (int i = MID - 1; i > 0; i--) acc[i] = acc[i - 1];
                    acc[0] = t;
                } else {
#pragma unroll
                    for (int i = 0; i < MID; i++)
                        if (i + fd + 1 == MID) {
#pragma unroll
                            for (int q = 0; q < 4; q++) acc[i][q] = on != 0 ? pf[q] : 0.0;
                        }
                    on = load(h, J + 8, J + 8 - fd, lane, pf);
                }
            }
            __syncthreads();
        }
    }
    // Σ log u in double-double
    double ls = 0, lc = 0;
    auto add = [&](double v, double c) {
        double t, e;
        two_sum(ls, v, t, e);
        ls = t;
        lc = (lc + c) + e;
    };
    for (int i = tid; i < 16 * T; i += NTH) {
        const double dv = B[(int64_t)(i >> 4) * COL + (i & 15)];
        add(dv > -0.5 ? log1p(dv) : log(fabs(1.0 + dv)), 0.0);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const double so = __shfl_xor(ls, off), co = __shfl_xor(lc, off);
        add(so, co);
    }
    double* red = &S[0][0][0];
    if (lane == 0) {
        red[2 * wv] = ls;
        red[2 * wv + 1] = lc;
    }
    __syncthreads();
    if (tid != 0) return;
    for (int w = 1; w < NTH / 64; w++) add(red[2 * w], red[2 * w + 1]);
    o.logdet = ls + lc;
    result();
}

// -G dense, column-major (zero outside the band), for the LU's kernels:
// 1 - G (the unit diagonal on it) for blocks of the pivoted LU; full = 0:
// rows from the column's 64-row diagonal block on.  The diagonal of G goes
// to off_diag.
__global__ void __launch_bounds__(256) k_band_dense(const BlockDesc* __restrict__ desc, char* __restrict__ arena,
                                                    const BlockOut* __restrict__ out, int full)
{
    const int b = blockIdx.z;
    const BlockDesc& d = desc[b];
    const int N = d.N, j = blockIdx.y;
    if (out[b].skip || j >= N) return;
    const double* B = at<double>(arena, d.off_band);
    double* A = at<double>(arena, d.off_mat) + (int64_t)j * d.lda;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= N || (!full && i < (j & ~63))) return;
    const int I = i >> 4, J = j >> 4, r = I - J;
    double v = 0;
    if (r >= 0 && r < BAND_TILES) v = B[((int64_t)J * BAND_TILES + r) * 256 + (j & 15) * 16 + (i & 15)];
    else if (r < 0 && -r < BAND_TILES) v = B[((int64_t)I * BAND_TILES - r) * 256 + (i & 15) * 16 + (j & 15)];
    if (i == j) {
        at<double>(arena, d.off_diag)[i] = -v;
        if (!out[b].delta) v += 1.0;
    }
    A[i] = v;
}

// M = FᵀF (mode 1) or -M (mode 0), column-major, on FP64 MFMA: 64 x 64 tiles of
// four wavefronts of 32 x 32, over all nodes; the operands are rows of F's
// storage (a degree's values at consecutive nodes), turned in LDS.  Each
// element sums the same products in the same order as its mirror.  lower:
// tiles above the diagonal are not written.
__global__ void __launch_bounds__(256) k_wave_matrix(const BlockDesc* __restrict__ desc, char* __restrict__ arena,
                                                     const BlockOut* __restrict__ out, int mode, int lower)
{
    constexpr int KS = 16, PITCH = 64 + 16;
    __shared__ double SA[KS][PITCH], SB[KS][PITCH];
    const int b = blockIdx.z;
    const BlockDesc& d = desc[b];
    const int N = 2 * d.ldim, m0 = 64 * blockIdx.x, n0 = 64 * blockIdx.y;
    if (m0 >= N || n0 >= N || (lower && m0 < n0) || (mode == 0 && out[b].skip)) return;
    const int64_t ldf = 2 * (int64_t)d.n_waves * 64;
    const double* F = at<double>(arena, d.off_rows);
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, li = lane & 15, lk = lane >> 4;
    const int wr = 32 * (wv & 1), wc = 32 * (wv >> 1);
    double4_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = (double4_t){0, 0, 0, 0};
    // F's storage holds 32 ceil(ldim/16) rows, so a row tile's last rows may
    // lie past it: they are taken as zero
    const int nrow = 32 * d.n_chunks;
    for (int64_t s = 0; s < ldf; s += KS) {
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int i = tid + 256 * t, r = i >> 3, q = 2 * (i & 7);
            const double2 z = make_double2(0, 0);
            const double2 va = m0 + r < nrow ? *reinterpret_cast<const double2*>(F + (m0 + r) * ldf + s + q) : z;
            const double2 vb = n0 + r < nrow ? *reinterpret_cast<const double2*>(F + (n0 + r) * ldf + s + q) : z;
            SA[q][r] = va.x;
            SA[q + 1][r] = va.y;
            SB[q][r] = vb.x;
            SB[q + 1][r] = vb.y;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < KS; kk += 4) {
            double av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; i++) av[i] = SA[kk + lk][wr + 16 * i + li];
#pragma unroll
            for (int j = 0; j < 2; j++) bv[j] = SB[kk + lk][wc + 16 * j + li];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[j], av[i], acc[i][j], 0, 0, 0);
        }
    }
    // swapped operands: lane l, register q: row wr + 16i + l%16, column wc + 16j + l/16 + 4q
    double* A = at<double>(arena, d.off_mat);
    double* dg = at<double>(arena, d.off_diag);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int row = m0 + wr + 16 * i + li, col = n0 + wc + 16 * j + lk + 4 * q;
                if (row >= N || col >= N) continue;
                double v = acc[i][j][q];
                if (row == col) dg[row] = v;
                if (mode == 0) v = row == col && !out[b].delta ? 1.0 - v : -v;
                A[row + (int64_t)col * d.lda] = v;
            }
}

}  // namespace capsd

using namespace capsd;

extern "C" {

// bytes: rounded up to 16, within both buffers
void capsd_launch_upload(const void* host, void* dev, size_t bytes, hipStream_t s)
{
    const int n = (int)((bytes + 15) / 16);
    hipLaunchKernelGGL(k_upload, dim3((n + 255) / 256), dim3(256), 0, s, (const uint4*)host, (uint4*)dev, n);
}

// units: of all blocks together (BlockDesc::unit_*), or more; clock: where the time at
// which the stage begins goes, or null (here and below)
void capsd_launch_wave_start(const void* tabs, int ntab, int max_mie, const BlockDesc* desc, char* arena, int nblocks,
                             int units, int* status, int64_t* clock, hipStream_t s)
{
    const int mu = (max_mie + 63) / 64;
    hipLaunchKernelGGL(k_wave_start, dim3(ntab * mu + units), dim3(64), 0, s, (const MieDesc*)tabs, ntab, mu, desc,
                       nblocks, arena, status, clock);
}

// split, pairs: the units of k_wave_norms' two forms.  Whole runs in one
// wavefront need one of them per SIMD (16 blocks of R/L = 200, norms and
// window: 33 us whole and 30 split; 8: 30 and 26; 64: 47 and 51).
// max_runs: with more than 8 runs k_wave_prefix pays for its launch (norms and
// window, 2 runs: 16 us with it and 14 without; 222 blocks of 19: 104 and 116;
// 188: 62 and 172).
void capsd_launch_wave_norms(const BlockDesc* desc, char* arena, int nblocks, int split, int pairs, int max_runs,
                             int max_waves, int64_t* clock, hipStream_t s)
{
    const int prefixed = max_runs > 8;
    if (prefixed) hipLaunchKernelGGL(k_wave_prefix, dim3(max_waves, nblocks), dim3(64), 0, s, desc, arena, clock);
    if (pairs < 1024)
        hipLaunchKernelGGL(k_wave_norms<true>, dim3(split), dim3(256), 0, s, desc, nblocks, arena, prefixed, clock);
    else
        hipLaunchKernelGGL(k_wave_norms<false>, dim3((pairs + 3) / 4), dim3(256), 0, s, desc, nblocks, arena, prefixed,
                           clock);
}

void capsd_launch_wave_rows(const BlockDesc* desc, char* arena, int nblocks, int max_wq, hipStream_t s)
{
    hipLaunchKernelGGL(k_wave_rows, dim3(max_wq, nblocks), dim3(256), 0, s, desc, arena);
}

void capsd_launch_wave_window(BlockDesc* desc, char* arena, BlockOut* out, const int* status, int nblocks, int allow,
                              int dense, hipStream_t s)
{
    if (nblocks < 256)
        hipLaunchKernelGGL(k_wave_window<1024>, dim3(nblocks), dim3(1024), 0, s, desc, arena, out, status, allow, dense);
    else
        hipLaunchKernelGGL(k_wave_window<256>, dim3(nblocks), dim3(256), 0, s, desc, arena, out, status, allow, dense);
}

// The band of -G, ncol (1 or 4) column tiles per workgroup; max_chunks: the
// blocks' largest n_chunks
void capsd_launch_gram(const BlockDesc* desc, char* arena, const BlockOut* out, int nblocks, int max_waves,
                       int max_chunks, int ncol, int delta_only, int64_t* clock, hipStream_t s)
{
    const int T = max_waves * 8;
    const size_t lds = 2 * (size_t)max_chunks * sizeof(int2);   // two steps per chunk at most
    if (ncol == 1)
        hipLaunchKernelGGL(k_gram<1>, dim3(T, nblocks), dim3(512), lds, s, desc, arena, out, delta_only, clock);
    else
        hipLaunchKernelGGL(k_gram<4>, dim3((T + 3) / 4, nblocks), dim3(256), lds, s, desc, arena, out, delta_only, clock);
}

void capsd_launch_band_ldl(const BlockDesc* desc, char* arena, BlockOut* out, BlockOut* host, int nblocks, int mercator,
                           int64_t* clock, hipStream_t s)
{
    hipLaunchKernelGGL(k_band_ldl, dim3(nblocks), dim3(1024), 0, s, desc, arena, out, host, mercator, clock);
}

void capsd_launch_band_dense(const BlockDesc* desc, char* arena, const BlockOut* out, int nblocks, int max_waves,
                             int full, hipStream_t s)
{
    const int N = max_waves * 128;
    hipLaunchKernelGGL(k_band_dense, dim3((N + 255) / 256, N, nblocks), dim3(256), 0, s, desc, arena, out, full);
}

void capsd_launch_wave_matrix(const BlockDesc* desc, char* arena, const BlockOut* out, int nblocks, int max_ldim,
                              int mode, int lower, hipStream_t s)
{
    const int t = (2 * max_ldim + 63) / 64;
    hipLaunchKernelGGL(k_wave_matrix, dim3(t, t, nblocks), dim3(256), 0, s, desc, arena, out, mode, lower);
}

}  // extern "C"
