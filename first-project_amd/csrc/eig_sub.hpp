// eig_sub.hpp -- the r <= 32 largest eigenpairs of a symmetric n x n FP64 matrix (n <= 128)
// by subspace iteration with a Rayleigh-Ritz step, in one 256-thread workgroup, for matrices
// whose top-r eigenvalues stand clear of the rest (the Grams of a Tucker fit: signal
// eigenvalues over a noise floor).  HOOI passes the previous iteration's factor as the start,
// HOSVD a fixed pseudo-random block.
//
// Method (Golub & Van Loan, 4th ed., 8.2.4 orthogonal iteration, 8.1.2 Rayleigh-Ritz, 8.5.2
// parallel cyclic Jacobi):
//   V = orth(V0); repeat { Z = A V; H = V^T Z; rho = ||Z - V H||_F;
//                          stop when rho <= 1e-12 ||H||_F; V = orth(Z) }
//   (H + H^T)/2 = W diag(theta) W^T by cyclic Jacobi in round-robin order; eigenvectors V W.
// orth() is Cholesky QR of the column-normalised block, done twice when the first pass finds
// nearly dependent columns.  Every product (A V, V^T Z, V S, X^T X, X M, V W) runs on FP64
// MFMA (v_mfma_f64_16x16x4f64: exact products, FP64 accumulation), with A held in registers
// for the whole call; the Cholesky factorisation and triangular inverse run in one wave's
// registers; the Jacobi rounds take one barrier each.
//
// The result is accepted only under a certificate that the theta are the r LARGEST
// eigenvalues, valid for any symmetric A: with orthonormal V and residual bound e = rho +
// ||offdiag(H after Jacobi)||_F, r distinct eigenvalues lie within e of the theta (Kahan), so
// every other eigenvalue lambda obeys lambda^2 <= ||A||_F^2 - sum (theta_k - e)^2; the theta are
// the top r when theta_min - e exceeds the square root of that bound (plus 1e-12 ||A||_F^2 for
// rounding).  Otherwise -- slow convergence, rank loss, no certificate -- the caller runs the
// full tridiagonal solver.  Output conventions match it: ascending eigenvalue order, entry of
// largest magnitude (lowest index on ties) positive.
#pragma once
#include "eig.hpp"

namespace tdx {

static constexpr int kSubMaxR = 32;
static constexpr int kSubRows = kEigMaxN;     // V and Z always hold 128 rows (zero past n)
// row stride of the n x r blocks V, Z: 16 rows read down a column (sub_xm) hit distinct LDS banks
static constexpr int kSubLd = kSubMaxR + 4;
static constexpr int kSubHld = kSubMaxR + 1;  // row stride of the r x r blocks H, W, S, M
static constexpr int kSubMaxIt = 12;

// dynamic LDS doubles of the subspace path (any n <= 128): V, Z (128 x kSubLd), H, W, S, M
// (kSubMaxR x kSubHld), 64 reduction slots, signs (32), positions (32 ints) and a flag
__host__ __device__ constexpr long eig_sub_doubles(int) {
    return 2L * kSubRows * kSubLd + 4L * kSubMaxR * kSubHld + 64 + 32 + 16 + 8;
}

typedef double sub_d4 __attribute__((ext_vector_type(4)));
// D += A B on a 16 x 16 tile: lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16] of the
// 4-deep slice; register v of lane l holds D[l / 16 + 4 v][l % 16]
__device__ __forceinline__ sub_d4 sub_mfma(double a, double b, sub_d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
// x of lane j (j wave-uniform)
__device__ __forceinline__ double sub_rl(double x, int j) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, j), hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), j);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// 1/sqrt(a) to full double precision: the hardware estimate refined by two Newton steps
// (y <- y (3 - a y^2) / 2); a is finite and positive wherever it is used here
__device__ __forceinline__ double rsq_f64(double a) {
    double y = __builtin_amdgcn_rsq(a);
    y = y * fma(-0.5 * a * y, y, 1.5);
    y = y * fma(-0.5 * a * y, y, 1.5);
    return y;
}

// sum over the workgroup; every thread gets the total (red: 4 doubles, reused after a barrier)
__device__ inline double sub_blk_sum(double v, double *red) {
    v = wave_sum_f64(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// sums of two values at once (red: 8 doubles)
__device__ inline void sub_blk_sum2(double &u, double &v, double *red) {
    u = wave_sum_f64(u);
    v = wave_sum_f64(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = u;
        red[4 + (threadIdx.x >> 6)] = v;
    }
    __syncthreads();
    u = (red[0] + red[1]) + (red[2] + red[3]);
    v = (red[4] + red[5]) + (red[6] + red[7]);
}

// The Jacobi rotation of the symmetric 2 x 2 block (app, apq; apq, aqq): t = sign(tau) / (|tau| +
// sqrt(tau^2 + 1)), c = 1 / sqrt(t^2 + 1), s = t c, with the hardware reciprocal / reciprocal-root
// estimates refined by two Newton steps (full FP64 precision; c^2 + s^2 = 1 to rounding).  The
// identity for apq = 0 (or too small for 1 / apq); |tau| is held at 1e150, where the angle is far
// below any rounding.
struct SubRot {
    double c, s, t;
};
__device__ __forceinline__ SubRot sub_rot(double app, double aqq, double apq) {
    const bool on = fabs(apq) > 1e-300;
    const double b = on ? apq : 1.0, d = on ? aqq - app : 1e300;
    const double tau = d * rcp_f64(b + b), at = fmin(fabs(tau), 1e150);
    const double a2 = fma(at, at, 1.0);
    const double t = rcp_f64(fma(a2, rsq_f64(a2), at));
    SubRot q;
    q.c = rsq_f64(fma(t, t, 1.0));
    q.t = on ? copysign(t, tau) : 0.0;
    q.s = q.t * q.c;
    return q;
}

// Out (32 x 32, stride kSubHld) = X^T Y over the 128 rows of X, Y (stride kSubLd); wave w
// computes tile (w / 2, w % 2)
__device__ inline void sub_gram(const double *X, const double *Y, double *Out) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
    const int tr = wv >> 1, tc = wv & 1;
    sub_d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
    for (int ks = 0; ks < kSubRows / 4; ++ks) {
        const int k = 4 * ks + lk;
        acc = sub_mfma(X[k * kSubLd + 16 * tr + lr], Y[k * kSubLd + 16 * tc + lr], acc);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) Out[(16 * tr + lk + 4 * v) * kSubHld + 16 * tc + lr] = acc[v];
}

// acc = rows 32 w .. 32 w + 31 of X (128 x 32, stride kSubLd) times M (32 x 32, stride kSubHld)
__device__ inline void sub_xm(const double *X, const double *M, sub_d4 (&acc)[2][2]) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) acc[rt][ct] = sub_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int ks = 0; ks < kSubMaxR / 4; ++ks) {
        const int k = 4 * ks + lk;
        const double a0 = X[(32 * wv + lr) * kSubLd + k], a1 = X[(32 * wv + 16 + lr) * kSubLd + k];
        const double b0 = M[k * kSubHld + lr], b1 = M[k * kSubHld + 16 + lr];
        acc[0][0] = sub_mfma(a0, b0, acc[0][0]);
        acc[0][1] = sub_mfma(a0, b1, acc[0][1]);
        acc[1][0] = sub_mfma(a1, b0, acc[1][0]);
        acc[1][1] = sub_mfma(a1, b1, acc[1][1]);
    }
}

// stores the rows < n of a sub_xm / product result into Y (stride kSubLd)
__device__ inline void sub_store_rows(const sub_d4 (&acc)[2][2], double *Y, int n) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 32 * wv + 16 * rt + lk + 4 * v;
            if (i < n) {
                Y[i * kSubLd + lr] = acc[rt][0][v];
                Y[i * kSubLd + 16 + lr] = acc[rt][1][v];
            }
        }
}

// X (rows < n, columns < r; zero elsewhere) <- orthonormal basis of its column span by
// Cholesky QR of the column-normalised block: S = X^T X, its normalised Cholesky factor L and
// L^{-1} in wave 0's registers, X <- X diag(1/sqrt(S_jj)) L^{-T}.
// Returns the smallest Cholesky pivot (1 for orthonormal input; 0 when a column is zero or
// numerically dependent: the call then leaves X unchanged).
// Lanes 0 .. 31 hold the rows of the normalised S, lanes 32 .. 63 the columns of the identity:
// step j of the right-looking factorisation (scale entry j by 1 / L_jj, subtract L_mj times it
// from entry m) is the same instruction for both and turns the identity into L^{-1}, so L_mj is
// broadcast once.  The factorisation of 32 columns takes 8.6 us of a pass's 13 us (all of it one
// wave's work; with a substitution of its own, square roots and divisions the pass took 20 us).
// Not inlined: one copy of the unrolled code, and its registers are not added to the caller's.
__device__ __noinline__ double sub_orth_pass(double *X, int n, int r_, double *S, double *M, double *flag) {
    const int r = __builtin_amdgcn_readfirstlane(r_);  // (uniform also where this is a call)
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    sub_gram(X, X, S);
    __syncthreads();
    if (wv == 0) {
        const int l = lane & 31;
        const bool unit = lane >= 32;
        double a[kSubMaxR];
#pragma unroll
        for (int j = 0; j < kSubMaxR; ++j) a[j] = S[l * kSubHld + j];
        const double dg = (l < r) ? S[l * kSubHld + l] : 1.0;
        const double cl = (dg > 0.0) ? 1.0 / sqrt(dg) : 0.0;
        bool bad = __any(l < r && !(cl > 0.0));
#pragma unroll
        for (int j = 0; j < kSubMaxR; ++j)
            a[j] = unit ? ((j == l) ? 1.0 : 0.0) : (l < r && j < r) ? a[j] * (cl * sub_rl(cl, j)) : 0.0;
        double pmin = 1.0;
#pragma unroll
        for (int j = 0; j < kSubMaxR; ++j) {
            if (j < r) {
                const double d = sub_rl(a[j], j);
                pmin = fmin(pmin, d);
                bad |= !(d > 1e-10);
                const double lj = a[j] * rsq_f64(bad ? 1.0 : d);  // L[l][j] (for l == j: sqrt(d)); L^{-1}[j][l]
                a[j] = lj;
#pragma unroll
                for (int b = (j + 1) / 8; b < kSubMaxR / 8; ++b)
                    if (8 * b < r) {
                        // (all broadcasts before the first use: a scalar register written by a
                        // vector instruction is not ready at once)
                        double t[8];
#pragma unroll
                        for (int m = 0; m < 8; ++m)
                            if (8 * b + m > j) t[m] = sub_rl(lj, 8 * b + m);
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int m = 0; m < 8; ++m)
                            if (8 * b + m > j) a[8 * b + m] = fma(-lj, t[m], a[8 * b + m]);
                    }
            }
        }
        // row c of M = diag(cl) L^{-T}: M[c][i] = cl_c * Linv[i][c]
        if (!bad && unit)
#pragma unroll
            for (int i = 0; i < kSubMaxR; ++i) M[l * kSubHld + i] = (l < r && i < r) ? cl * a[i] : 0.0;
        if (lane == 0) flag[0] = bad ? 0.0 : pmin;
    }
    __syncthreads();
    const double pm = flag[0];
    if (!(pm > 0.0)) return 0.0;  // uniform
    sub_d4 acc[2][2];
    sub_xm(X, M, acc);
    __syncthreads();  // every wave has read X
    sub_store_rows(acc, X, n);
    __syncthreads();
    return pm;
}

__device__ inline bool sub_orth(double *X, int n, int r, double *S, double *M, double *flag) {
    double p = 0.0;
    for (int pass = 0; pass < 2; ++pass) {
        p = sub_orth_pass(X, n, r, S, M, flag);
        if (!(p > 0.0) || p >= 1e-2) break;  // (below: CholQR2)
    }
    return p > 0.0;
}

// Ag: n x n symmetric (column-major) in global memory.  U0: n x r FP32 start block
// (column-major) or null for the built-in one.  On success writes U (n x r FP32, may alias U0)
// and w (optional) like sym_top_eigvecs_block and returns true; returns false having written
// nothing.  Launch with kEigThreads threads and eig_sub_doubles(n) * 8 bytes of dynamic LDS.
// rotate = false (HOOI before its last iteration, where only the span of U matters: every
// later product contracts U U^T): when the span is certified cheaply (below) U is the
// orthonormal basis V itself, in no particular order and without the Rayleigh-Ritz rotation;
// otherwise the full path runs.
__device__ inline bool sym_top_eigvecs_subspace(const double *Ag, int n, int r, const float *U0, float *U,
                                                double *w, double *smem, bool rotate = true) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, lr = lane & 15, lk = lane >> 4;
    double *V = smem;
    double *Z = V + kSubRows * kSubLd;
    double *H = Z + kSubRows * kSubLd;
    double *Wm = H + kSubMaxR * kSubHld;
    double *S = Wm + kSubMaxR * kSubHld;
    double *M = S + kSubMaxR * kSubHld;
    double *red = M + kSubMaxR * kSubHld;  // 64 slots
    double *sg = red + 64;                 // 32 signs
    int *pos = reinterpret_cast<int *>(sg + 32);  // 32 ints
    double *flag = sg + 48;

    // start block; rows n.. and columns r.. stay zero throughout
    for (int e = tid; e < kSubRows * kSubLd; e += kEigThreads) {
        const int i = e / kSubLd, c = e % kSubLd;
        double v = 0.0;
        if (c < r && i < n) {
            if (U0) {
                v = (double)U0[(long)c * n + i];
            } else {
                // integer mix of (i, c) to a uniform value in [-1, 1); the blocks it gives for
                // n <= 128, r <= 32 have column-normalised condition numbers below 600
                unsigned x = ((unsigned)i * 0x9E3779B1u) ^ ((unsigned)(c + 1) * 0x85EBCA77u);
                x ^= x >> 16;
                x *= 0x7FEB352Du;
                x ^= x >> 15;
                x *= 0x846CA68Bu;
                x ^= x >> 16;
                v = (double)(x >> 8) * (2.0 / 16777216.0) - 1.0;
            }
        }
        V[e] = v;
        Z[e] = 0.0;
    }
    // A in registers as MFMA A operands: rows 32 wv + 16 rt + lr, columns 4 ks + lk
    double gA[2][kSubRows / 4];
    double f2 = 0.0;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int ks = 0; ks < kSubRows / 4; ++ks) {
            const int i = 32 * wv + 16 * rt + lr, k = 4 * ks + lk;
            const double g = (i < n && k < n) ? Ag[i + (long)k * n] : 0.0;
            gA[rt][ks] = g;
            f2 = fma(g, g, f2);
        }
    f2 = sub_blk_sum(f2, red);  // (its barriers also publish the start block)
    if (!sub_orth(V, n, r, S, M, flag)) return false;

    double rho = 0.0, hf = 0.0, rho_prev = 0.0;
    bool conv = false;
    for (int it = 0; it < kSubMaxIt; ++it) {
        // Z = A V
        {
            sub_d4 acc[2][2];
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct) acc[rt][ct] = sub_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int kb = 0; kb < kSubRows / 16; ++kb)
                if (16 * kb < n)
#pragma unroll
                    for (int ks = 4 * kb; ks < 4 * kb + 4; ++ks) {
                        const double *vr = V + (4 * ks + lk) * kSubLd + lr;
                        const double b0 = vr[0], b1 = vr[16];
#pragma unroll
                        for (int rt = 0; rt < 2; ++rt) {
                            acc[rt][0] = sub_mfma(gA[rt][ks], b0, acc[rt][0]);
                            acc[rt][1] = sub_mfma(gA[rt][ks], b1, acc[rt][1]);
                        }
                    }
            sub_store_rows(acc, Z, n);
        }
        __syncthreads();
        // S = V^T Z
        sub_gram(V, Z, S);
        __syncthreads();
        // rho = ||Z - V S||_F, H = (S + S^T) / 2, ||H||_F
        double rr = 0.0, hh = 0.0;
        {
            sub_d4 acc[2][2];
            sub_xm(V, S, acc);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int i = 32 * wv + 16 * rt + lk + 4 * v, c = 16 * ct + lr;
                        if (i < n && c < r) {
                            const double d = Z[i * kSubLd + c] - acc[rt][ct][v];
                            rr = fma(d, d, rr);
                        }
                    }
        }
        // (S, and so H, is zero past r)
        for (int e = tid; e < kSubMaxR * kSubMaxR; e += kEigThreads) {
            const int a = e / kSubMaxR, b = e % kSubMaxR;
            const double h = 0.5 * (S[a * kSubHld + b] + S[b * kSubHld + a]);
            H[a * kSubHld + b] = h;
            hh = fma(h, h, hh);
        }
        sub_blk_sum2(rr, hh, red);
        rho = sqrt(rr);
        hf = sqrt(hh);
        if (rho <= 1e-12 * hf) {
            conv = true;
            break;
        }
        if (it >= 2 && rho > 0.25 * rho_prev) return false;  // too slow for this path
        rho_prev = rho;
        if (!sub_orth(Z, n, r, S, M, flag)) return false;
        double *t = V;
        V = Z;
        Z = t;
    }
    if (!conv || !(hf > 0.0)) return false;

    if (!rotate) {
        // Span certificate without the eigenvalues of H: with orthonormal V and residual rho,
        // r eigenvalues lambda_k of A lie within rho of the eigenvalues theta_k of H (Kahan).  If
        // every theta_k > t = rho + b with b^2 = ||A||_F^2 - sum (theta_k - rho)^2 (+ rounding),
        // then lambda_k > b, and every other eigenvalue has lambda^2 <= ||A||_F^2 -
        // sum lambda_k^2 <= b^2: the span of V is the top-r invariant subspace.  sum (theta_k -
        // rho)^2 = ||H||_F^2 - 2 rho tr(H) + r rho^2, and theta_min > t holds exactly when
        // H - t I has a Cholesky factorisation with positive pivots.
        double tr = 0.0;
        for (int c = 0; c < r; ++c) tr += H[c * kSubHld + c];
        const double ss = hf * hf - 2.0 * rho * tr + (double)r * rho * rho;
        const double b2 = fmax(f2 - ss, 0.0) + 1e-12 * f2;
        const double t = rho + sqrt(b2);
        for (int e = tid; e < r * r; e += kEigThreads) {
            const int a = e / r, bb = e % r;
            S[a * kSubHld + bb] = H[a * kSubHld + bb] - ((a == bb) ? t : 0.0);
        }
        if (tid == 0) *flag = 1.0;
        __syncthreads();
        // right-looking Cholesky of the r x r block, one barrier per pivot
        for (int k = 0; k < r; ++k) {
            const double d = S[k * kSubHld + k];
            if (!(d > 0.0)) {
                if (tid == 0) *flag = 0.0;
                break;  // uniform: every thread read the same pivot
            }
            const double dinv = 1.0 / d;
            const int m2 = r - k - 1;
            for (int e = tid; e < m2 * m2; e += kEigThreads) {
                const int i = k + 1 + e / m2, j = k + 1 + e % m2;
                S[i * kSubHld + j] = fma(-S[i * kSubHld + k] * dinv, S[k * kSubHld + j], S[i * kSubHld + j]);
            }
            __syncthreads();
        }
        __syncthreads();
        if (*flag > 0.0) {
            for (int e = tid; e < n * r; e += kEigThreads) {
                const int i = e % n, c = e / n;
                U[(long)c * n + i] = (float)V[i * kSubLd + c];
            }
            return true;
        }
        __syncthreads();
    }

    // ---- Rayleigh-Ritz: H = W diag(theta) W^T by cyclic Jacobi, round-robin pairs ----
    // The pairs of a round partition the indices, so H falls into 2 x 2 blocks (pair i, pair j), one
    // for each thread, which turns its block from both sides and writes it to the other of two
    // buffers: a round has one barrier.  A thread computes the rotation of its pair j and takes that
    // of pair i from the lane of its wave that has it.  It also turns columns p, q of pair i of W in
    // rows j, j + 16.  A round is one chain of latencies (0.50 us at r = 32; 1.15 us with a barrier
    // between the rows' and the columns' half, two pairs a thread one after the other and branches in
    // the rotation: the 186 rounds of r = 32 took 213 us, 93 us this way).  An odd r has index r as the partner without entries (row and column r of H are
    // zero).  The buffers lie in Z; their stride spreads the rows of a wave over the LDS banks.
    constexpr int ld = 48;
    double *Hc = Z, *Hn = Z + kSubMaxR * ld;
    for (int e = tid; e < kSubMaxR * kSubMaxR; e += kEigThreads) {
        const int a = e / kSubMaxR, b = e % kSubMaxR;
        Hc[a * ld + b] = H[a * kSubHld + b];
        Wm[a * kSubHld + b] = a == b ? 1.0 : 0.0;
    }
    __syncthreads();
    const int re = r + (r & 1), npair = re >> 1, m = re - 1;
    const int i0 = tid >> 4, j0 = tid & 15;
    // Round k's pair g: (re - 1, k) for g = 0, (k + g, k - g) modulo m otherwise.  Threads past the
    // last pair repeat pair 0 (H: the same values twice; W: on a copy in M that nobody reads), so a
    // round has no branch and its loads stand first.
    const int gi = i0 < npair ? i0 : 0, gj = j0 < npair ? j0 : 0;
    const bool dg = gi == gj;
    double *w0 = (i0 < npair ? Wm : M) + j0 * kSubHld, *w1 = w0 + 16 * kSubHld;
    auto next = [&](int &p, int &row) {  // p + 1 modulo m and its row's offset
        const bool wrap = p + 1 == m;
        p = wrap ? 0 : p + 1;
        row = wrap ? 0 : row + ld;
    };
    double off = 0.0;
    bool jconv = (m <= 0);
    for (int sw = 0; sw < 16 && !jconv; ++sw) {
        int pi = gi ? gi : m, qi = gi ? m - gi : 0, pj = gj ? gj : m, qj = gj ? m - gj : 0;
        int rpi = pi * ld, rqi = qi * ld, rpj = pj * ld, rqj = qj * ld;
        for (int k = 0; k < m; ++k) {
            const double ajp = Hc[rpj + pj], ajq = Hc[rqj + qj], ajo = Hc[rpj + qj];
            __builtin_amdgcn_sched_barrier(0);  // (first: the rotation waits for them alone)
            const double b00 = Hc[rpi + pj], b01 = Hc[rpi + qj], b10 = Hc[rqi + pj], b11 = Hc[rqi + qj];
            const double w0p = w0[pi], w0q = w0[qi], w1p = w1[pi], w1q = w1[qi];
            __builtin_amdgcn_sched_barrier(0);
            const SubRot rj = sub_rot(ajp, ajq, ajo);
            const double ic = __shfl(rj.c, i0, 64), is = __shfl(rj.s, i0, 64);
            const double t00 = ic * b00 - is * b10, t01 = ic * b01 - is * b11;
            const double t10 = is * b00 + ic * b10, t11 = is * b01 + ic * b11;
            // (the diagonal block is set exactly)
            Hn[rpi + pj] = dg ? ajp - rj.t * ajo : rj.c * t00 - rj.s * t01;
            Hn[rpi + qj] = dg ? 0.0 : rj.s * t00 + rj.c * t01;
            Hn[rqi + pj] = dg ? 0.0 : rj.c * t10 - rj.s * t11;
            Hn[rqi + qj] = dg ? ajq + rj.t * ajo : rj.s * t10 + rj.c * t11;
            w0[pi] = ic * w0p - is * w0q;
            w0[qi] = is * w0p + ic * w0q;
            w1[pi] = ic * w1p - is * w1q;
            w1[qi] = is * w1p + ic * w1q;
            if (gi) next(pi, rpi);
            next(qi, rqi);
            if (gj) next(pj, rpj);
            next(qj, rqj);
            __syncthreads();
            double *t = Hc;
            Hc = Hn;
            Hn = t;
        }
        double o = 0.0;
#pragma unroll
        for (int u = 0; u < kSubMaxR * kSubMaxR / kEigThreads; ++u) {
            const int a = (tid + u * kEigThreads) / kSubMaxR, b = (tid + u * kEigThreads) % kSubMaxR;
            const double h = Hc[a * ld + b];
            o = fma(h, (a != b && a < r && b < r) ? h : 0.0, o);
        }
        off = sqrt(sub_blk_sum(o, red));
        jconv = off <= 1e-14 * hf;
    }
    if (!jconv) return false;
    if (tid < r) H[tid * kSubHld + tid] = Hc[tid * ld + tid];
    __syncthreads();

    // ---- certificate that the theta are the r largest eigenvalues ----
    const double eb = rho + off;
    double tmin = 1e300, ssq = 0.0;
    for (int c = 0; c < r; ++c) {
        const double th = H[c * kSubHld + c];
        tmin = fmin(tmin, th);
        const double d = fmax(th - eb, 0.0);
        ssq = fma(d, d, ssq);
    }
    const double rest = fmax(f2 - ssq, 0.0) + 1e-12 * f2;
    if (!(tmin - eb > sqrt(rest))) return false;

    // ---- eigenvectors Y = V W (into Z), ascending order, sign, FP32 ----
    {
        sub_d4 acc[2][2];
        sub_xm(V, Wm, acc);
        sub_store_rows(acc, Z, n);
    }
    if (tid < r) {
        const double th = H[tid * kSubHld + tid];
        int rank = 0;
        for (int k = 0; k < r; ++k) {
            const double tk = H[k * kSubHld + k];
            rank += (tk < th) || (tk == th && k < tid);
        }
        pos[tid] = rank;
        if (w) w[rank] = th;
    }
    __syncthreads();
    {
        const int c = tid >> 3, part8 = tid & 7;  // 8 lanes of one wave per column
        double best = -1.0;
        int bi = n;
        if (c < r)
            for (int i = part8; i < n; i += 8) {
                const double a = fabs(Z[i * kSubLd + c]);
                if (a > best) {
                    best = a;
                    bi = i;
                }
            }
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
            const double ob = __shfl_xor(best, o, 64);
            const int oi = __shfl_xor(bi, o, 64);
            if (ob > best || (ob == best && oi < bi)) {
                best = ob;
                bi = oi;
            }
        }
        if (c < r && part8 == 0) sg[c] = (Z[bi * kSubLd + c] < 0.0) ? -1.0 : 1.0;
    }
    __syncthreads();
    for (int e = tid; e < n * r; e += kEigThreads) {
        const int i = e % n, c = e / n;
        U[(long)pos[c] * n + i] = (float)(sg[c] * Z[i * kSubLd + c]);
    }
    return true;
}

}  // namespace tdx
