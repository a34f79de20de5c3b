// blfid_dev.h -- device-side plan tables shared by the host planner and the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>

#define DEV_TERM_STRIDE 10 /* Cxx Cyy Czz Cxy Cxz Cyz  fdiag  fflip  i  j(-1 for CSA) */
#define DEV_MAX_TERMS 128
#define DEV_MAX_SPINS 12
#define DEV_MAX_BLOCK 256 /* largest Hilbert-space block (k_eig pair tables) */
// Scratch of one block beyond DEV_LDS_BLOCK in the eigen-solver, besides its b x b iterate: the
// rotations of up to 16 index pairs (16 x 16 each), then its sweep flags
#define EIGB_V 4096
#define EIGB_EXTRA (EIGB_V + 16)
#define DEV_LDS_BLOCK 80  /* blocks up to this size keep k_eig's matrix in LDS */
// Row padding (floats) of the LDS-resident product planes (chain_mfma, SymTile): rows of
// 16 M + LDS_PAD floats, a multiple of four so that every row starts on 16 bytes (8, 12 and 20
// measured no faster on the batched clusters).
#ifndef LDS_PAD
#define LDS_PAD 4
#endif
// The FP64 planes (k_expdyson_d): rows of 16 M + 2 doubles put the 32 eight-byte operands that
// half a wave reads (16 rows, two columns) into distinct banks; with a padding of four, rows r and
// r + 8 met in the same ones (41% of the kernel's cycles were bank conflicts).
#define LDS_PAD_D 2

struct DevPlan {
    int S, N;      // spins, Hilbert dimension
    int n;         // steps per rotor period (1 for the static path)
    int npts;      // FID points
    int nterms;    // anisotropic interaction terms
    int nblocks;   // Hilbert-space blocks
    int npairs;    // coupled (I,J) block pairs of det / rho_eff
    long Lsum;     // sum of b^2 over blocks: per-(crystallite,step) matrix storage
    long Etot;     // sum of b_I*b_J over pairs: correlation elements per crystallite
    double theta;  // 2*pi*tau
    const double *terms;   // nterms x DEV_TERM_STRIDE
    const double *dconst;  // N: isotropic diagonal of H (-iso_csa m_i + J m_i m_j)
    const double *ffconst; // S x S: constant flip-flop coefficients (strong J / 2)
    const int *ff_off;     // S x S + 1: per ordered spin pair, its run in ff_term
    const int *ff_term;    // terms with a flip-flop part, listed under both orders of their pair
    const double *xd_cst;  // N x 7: diagonal of each basis state as (1, w) . xd_cst, w the six
                           // quadratic products of v = R_P^T u (fused kernel's H build)
    const double *xd_fpr;  // S x S x 7: flip-flop coefficient of each ordered pair, likewise
    const double *u3;      // n x 3: row 2 of cartSpin at each step midpoint
    const double *RP;      // K x 9: cartPowder of each crystallite (row-major)
    const int *blk_dim;    // nblocks
    const int *blk_soff;   // nblocks: offset of the block in the state list (sum of b)
    const long *blk_uoff;  // nblocks: offset of the block in Lsum storage
    const int *blk_states; // N: basis-state index of each block-local row
    const int *pair_I, *pair_J;
    const long *pair_eoff; // element offset of each pair (sum of bI*bJ)
    const int *pair_doff;  // start of each pair's det CSR row pointer (bI+1 entries)
    const int *pair_roff;  // start of each pair's rho_eff CSR row pointer (bJ+1 entries)
    const int *d_rowptr, *d_col;
    const double *d_val;   // complex, interleaved
    const int *r_rowptr, *r_col;
    const double *r_val;   // complex, interleaved
    // point-to-point propagation with rf
    int usign;             // step propagator exp(usign * i theta H): -1 gamma-COMPUTE, +1 ptop
    int akeep;             // Dyson products kept per crystallite (n, or 2 when only A_n is used)
    int nrfiso;            // pulsed isotopes
    const int *spin_rf;    // S: pulsed-isotope slot of each spin or -1
    const double *rf;      // n x nrfiso x 3: amp/2, phase, offset of each step
    const double *thetak;  // n: 2 pi tau_k of steps of unequal length, or NULL (all theta)
    int rt_from_q;         // 1: R(s,r) = Q_rev + conj(Q(r,s)), R is neither formed nor stored
    // correlation elements (Ecorr <= Etot): position in a step's Q row, state-list positions of
    // column (block I) and row (block J), position of the reverse element (s,r) of pair (J,I) or -1
    long Ecorr;
    const int *corr_pos, *corr_r, *corr_s, *corr_rev;
    double *expflops;      // 16: executed flops per tile variant of the propagator [0..7] and
                           // the fused propagator + Dyson chain [8..15] (profiling), or NULL
    int bf16x3;            // complex64 products as three bf16 matrix-core products (BLFID_C64_BF16X3)
    long Estr;             // Q / R row stride per step: Etot padded to a multiple of 16 elements
    int nparts;            // FID partial sums per crystallite (correlation segments or block pairs)
    int rt_rev;            // rt_from_q and some element has a reverse element (corr_rev >= 0)
    const int *xd_off;     // nblocks + 1: start of each block's flip-flop positions in xd_list
    const int *xd_list;    // per block of <= DEV_LDS_BLOCK states: (r LDK + q) << 8 | (i S + j),
                           // LDK the plane rows of the plan's precision
    const int *elem_r;     // Etot: state-list position of each pair element's column (block I)
    const int *elem_s;     // Etot: state-list position of each pair element's row (block J)
    const void *rho_c;     // prepared rho per crystallite of the batch on the block pairs (storage
                           // precision, conj(rho_JI) at element r + s b_I), or NULL
    int corr_auto_chunks;  // leading correlation chunks whose elements have no reverse element
                           // (rt_from_q plans): they take the autocorrelation kernel
    // launch choices of the autotuner (0 everywhere: the defaults)
    int tn_cap[9];         // persistent-grid cap (workgroups) per kernel family, indexed like the
                           // profiling phases: exp 0, dyson 1, eig 2, bmul 3, qr 4, corr 5,
                           // reduce 6, static 7, expdyson 8
    int tn_corr;           // k_corr variant: 0 four FID points per thread up to 1024 points
                           // (eight above) at the default occupancy, 1 the same at two waves
                           // per SIMD (no register spill), 2 eight points per thread
    int eig_sweeps;        // sweeps of k_eigb_* over the whole device (0: EIGB_SWEEPS)
    int tn_qr;             // k_qr form per complex64 tile class: bit M-1 set takes the other form
                           // (per-step for classes 1-2, step-walking for 3-4; class 1 by k_bq1)
};

// Persistent-grid cap of a kernel family: the tuned value or 4096 workgroups; single-wave
// workgroups (tile class 1) take four times as many.
#define GRID_CAP 4096
inline long tuned_cap(const DevPlan *P, int fam, int M) {
    const long c = P->tn_cap[fam] > 0 ? P->tn_cap[fam] : GRID_CAP;
    return M == 1 ? 4 * c : c;
}

// Correlation work split (k_corr), shared by the host planner and the kernel: a crystallite's
// Ecorr elements are cut into chunks of CH elements (corr_chunk: CORR_SPAN / L with transforms of L
// points, min(CORR_SPAN / n, 256 / ceil(n / 8)) with the direct sum) and the chunks into segments of up to CORR_SEG_CHUNKS; each segment writes one FID partial sum.
#define CORR_TW 256
#define CORR_SPAN 2048
#define CORR_VTAB 1024 /* complex128 entries of the period table, within the second buffer */
#define CORR_PPT 8
#define CORR_SEG_CHUNKS 64
#define CORR_SEG_MIN 8
// log2 of the transform length of the FFT variant, or 0 where the direct sum is taken.  A power of
// two from 16 to 512 is transformed at its own length; any other n from CORR_PAD_MIN to 256 is
// zero-padded to the power of two L >= 2 n, whose cyclic correlation holds the linear one, folded
// back to period n (two or three transforms of at most 4 n points against 8 n^2 flops).  Direct sum
// and padded transforms, k_corr in us, 1154 crystallites (4 spins FP64, 512 points | 6 spins FP64
// and complex64, 1000 points):
//   n    5: 105 133 | 1350 1539, 1252 1274      n  65: 217 180 | 2820 1869, 2574 1705
//   n    8: 110 109 | 1375 1402, 1289 1276      n 100: 333 194 | 3796 2032, 3250 1932
//   n    9: 109  57 | 1687 1005, 1555  844      n 127: 448 200 | 5429 1970, 4566 1871
//   n   31: 130  62 | 1952  655, 1841  592      n 129: 469 542 | 5544 5603, 4575 3250
//   n   33: 162 101 | 1693 1149, 1569 1038      n 160: 923 566 | 7868 5700, 6247 3273
//   n   45: 184 104 | 1861 1144, 1730 1032      n 255: 1251 624 | 14801 6140, 11111 3563
// so the direct sum is kept below 9, where the padded chunks would hold mostly zeros, and above 256,
// which would need transforms beyond 512 points; just above 128 the two are even.  Both are as far from
// extended-precision FIDs.
#define CORR_PAD_MIN 9
__host__ __device__ inline int corr_fft_ln(int n) {
    const bool p2 = (n & (n - 1)) == 0;
    if (p2 ? (n < 16 || n > 2 * CORR_TW) : (n < CORR_PAD_MIN || n > CORR_TW)) return 0;
    int ln = 0;
    while ((1 << ln) < (p2 ? n : 2 * n)) ln++;
    return ln;
}
__host__ __device__ inline bool corr_use_fft(int n) { return corr_fft_ln(n) > 0; }
// elements per chunk of the direct sum
__device__ __host__ inline int corr_direct_chunk(int n) {
    int npg = (n + CORR_PPT - 1) / CORR_PPT;
    int a = CORR_SPAN / n, b = 256 / npg;
    int ch = a < b ? a : b;
    return ch < 1 ? 1 : ch;
}
// elements per chunk: the FFT variant fills CORR_SPAN points
__device__ __host__ inline int corr_chunk(int n) {
    const int ln = corr_fft_ln(n);
    return ln > 0 ? CORR_SPAN >> ln : corr_direct_chunk(n);
}
// Chunks per segment: about CORR_SEG_MIN segments (a few crystallites fill the device), of up to
// CORR_SEG_CHUNKS chunks.  A crystallite's partial sums of npts points take CORR_PART_BYTES at
// most (FIDs beyond 30000 points) as long as a segment then stays within CORR_SEG_CHUNKS chunks of
// the direct sum's elements: longer segments would hold a batch to fewer, longer tasks, and a
// million-point FID took eight times the storage of its results per crystallite.
#define CORR_PART_BYTES (4 << 20)
__device__ __host__ inline int corr_seg_chunks(int n, int npts, int nchunk) {
    int c = (nchunk + CORR_SEG_MIN - 1) / CORR_SEG_MIN;
    c = c < 4 ? 4 : c > CORR_SEG_CHUNKS ? CORR_SEG_CHUNKS : c;
    const int most = CORR_SEG_CHUNKS * corr_direct_chunk(n) / corr_chunk(n);
    while (c < most && (double)((nchunk + c - 1) / c) * npts * 16.0 > CORR_PART_BYTES) c = c < most / 2 ? 2 * c : most;
    return c;
}
__device__ __host__ inline int corr_range_segments(int n, int npts, int nchunk) {
    if (nchunk <= 0) return 0;
    const int spc = corr_seg_chunks(n, npts, nchunk);
    return (nchunk + spc - 1) / spc;
}
// FID partial sums of a correlation: the segments of the autocorrelation chunks [0, A) and of
// the general chunks [A, nchunk), each range segmented on its own
__device__ __host__ inline int corr_segments(int n, int npts, long Ecorr, int auto_chunks = 0) {
    const int CH = corr_chunk(n);
    const int nchunk = (int)((Ecorr + CH - 1) / CH);
    return corr_range_segments(n, npts, auto_chunks) + corr_range_segments(n, npts, nchunk - auto_chunks);
}
