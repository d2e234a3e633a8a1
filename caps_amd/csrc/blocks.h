// Layout of one batch of (ξ, m) round-trip-matrix blocks in HBM.
//
// A batch is a set of blocks (of one or several caps objects).  The host
// fills one BlockDesc per block; every kernel takes the descriptor array and
// the arena base pointer and finds its block through blockIdx (the batch
// dimension).
// All per-block tables live in one device arena, at the offsets recorded in
// the descriptor (in bytes, 256-byte aligned).
#pragma once
#include <stdint.h>

namespace capsd {

struct BlockDesc {
    // physics of the block
    double xi_;          // ξ(L+R)/c
    double alpha;        // 2 ξ(L+R)/c
    double epsm1_plate;  // ε(iξ)-1 of the plate (+inf: perfect reflector)
    double LbyR;
    int m, lmin, ldim;      // window l in [lmin, lmin+ldim)
    int N;                  // dimension of the matrix to factor (k_wave_window
                            // sets it for the dense form of a Gram matrix)
    int is_pr;              // plate is a perfect reflector: I_TE = -|I_TM|
    // quadrature grid: v_k = v0 + k h, k < n_nodes, x(v) = 1 + A² softplus(v)²
    // (of the wave-number factor, or of the K integrals of the tables)
    double v0, h, A;
    int n_nodes, n_waves;   // n_waves: wavefronts of 64 nodes
    int n_chunks;           // runs of 16 degrees of the window
    int mie_L;              // degrees 1 .. mie_L of the block's Mie table
    // K and I tables (caps_integrate_init): ν in [mu, nu_max], l in [lo, lo+nl)
    int mu, nu_max, nK;
    int lo, nl;
    int lda;                // leading dimension of the matrix, if there is one
    // byte offsets into the arena; nP = 64 n_waves
    int64_t off_mie;    // the block's MieDesc table
    int64_t off_node;   // 4 nP doubles: x, √r_TM, √|r_TE|, S_m; nP ints: its exponent
    int64_t off_run;    // per run of 64 degrees but the last: 2 nP double2 (k_wave_start's
                        // matrices by columns), then nP ints of each: their exponents
    int64_t off_ck;     // 2 n_chunks nP double2: S_l, S_{l-1} every 8 degrees (degree())
    int64_t off_norm;   // n_segs nP doubles: squared norms of the rows' runs of 64 degrees
    int64_t off_act;    // n_chunks nP/8 ints: exponent of a tile's largest chunk norm
    int64_t off_dn;     // nP doubles: squared norms of the rows
    int64_t off_deg;    // 16 n_chunks Deg: the degrees' constants
    int64_t off_rows;   // F: 32 n_chunks rows (degree; a_l, b_l) of 2 nP doubles
    int64_t off_band;   // nP/8 columns of BAND_TILES tiles of 16 x 16: -G
    int64_t off_a0;     // nl + (2 nl - 1) doubles: parts of log a0 of I
    int64_t off_kpart;  // n_waves * nK * KPart
    int64_t off_k;      // 2 pols * nK * KEnt (K = m * 2^e), then 2 pols * nK
                        // doubles log|K|
    int64_t off_i;      // I = mant * 2^exp: 2 pols * nl*nl signed double mantissas,
                        // then 2 pols * nl*nl int exponents
    int64_t off_mat;    // lda * N doubles (column-major)
    int64_t off_diag;   // N doubles: diagonal of M (or G)
    int64_t off_cpart;  // n_rtiles x N doubles: per row tile, the column sums
                        // of |M_ij| over i != j (written with the matrix)
    int n_rtiles;       // row tiles of off_cpart (0: none)
    int n_below, n_segs;    // runs of 64 degrees below the window and in it
    // units of the blocks before this one: k_wave_start's workgroups, and
    // k_wave_norms' workgroups (split) or wavefronts
    int unit_start, unit_split, unit_pair;
};

// The band of G: tiles on and below the diagonal per column of 16 x 16 tiles
// (8 nodes each).  Rows of F fall off like e^{-δ²/16} in the distance δ = h
// times the node distance, and G_ij enters the determinant squared: what lies
// more than 48 nodes (δ = 21.6) apart changes it by less than 1e-16 of its
// value, the tail of x -> 1 of the smallest m included (scanned over R/L
// 0.1 .. 300, ξ 1e-4 .. 100, ε-1 from 0.1 to perfect reflectors, m up to 20: no
// difference to the full matrix above the 2e-15 of the eigenvalues compared).
constexpr int BAND_TILES = 7;

// Constants of one degree of a block's window (see degree() in waves.hip).
struct Deg {
    double c1, c2, l, rt, ma, mb, pad_;
    int e, sh;
};

// One Mie table: degrees 1 .. L at one ξ of one object; at off: L doubles each
// of log|a_l|, log|b_l| and the mantissas of √(a_l g_l), √(b_l g_l), g_l =
// (2l+1)/(l(l+1)), over a common power of two, then L ints: its exponent.
struct MieDesc {
    double xi_, LbyR, epsm1;
    int64_t off;
    int L, pad_;
};

// Partial K sums of one wave of quadrature nodes for one ν.
struct KPart {
    double s_te, s_tm;
    int e;
    int pad_;
};

// One K_ν value as signed mantissa times 2^e, read by the I recurrence with
// a single 16-byte load.
struct KEnt {
    double m;
    int e;
    int pad_;
};
// zeroed KEnt entries in front of every block's K table (BlockDesc::off_k
// is at least this far into the arena; 256 bytes are reserved)
constexpr int K_GUARD = 16;

// Per-block scalar results.
struct BlockOut {
    double trace;       // tr M (Kahan)
    double logdet;      // log|det(1-M)| from the LU (NAN if skipped)
    double frob2;       // ||M||_F^2 (LU mode only)
    double tr2;         // tr M^2 (LU mode only)
    int skip;           // LU skipped (trace shortcut)
    int status;         // 0 ok; nonzero: numerical failure flag
    int delta;          // 1: the matrix holds -M (1 - M without its unit
                        // diagonal; 1 - M is column diagonally dominant, so
                        // partial pivoting exchanges no rows) and the LU
                        // runs without pivot search on u = 1 + d, summing
                        // log1p(d); 0: the matrix holds 1 - M (or a user
                        // matrix), LU with partial pivoting
    int tile0, tiles;   // the nodes that matter: tiles of 8 nodes (G has
                        // 16 tiles rows)
    int etr;            // exponent of the trace
    int64_t t_end;      // wall_clock64 at the end of k_band_ldl
};

}  // namespace capsd
