// tucker.hip -- Tucker HOSVD and HOOI for gfx950.
//
// HOSVD (src/tucker_hosvd.cu:3-81, src/tucker4_hosvd.cu:3-121): per mode the Gram of the
// unfolding X(n) X(n)^T, a symmetric eigensolve, and the eigenvectors of the r_n largest
// eigenvalues in ascending order (the reference copies the last r columns of the
// ascending syevdx output, src/tucker_hosvd.cu:68-70); core = X x_1 U_1^T ... x_d U_d^T.
// HOOI (decomposition/GPU/normal/tucker/tucker_hooi.cu:103-168, generalised to order 4):
// per mode, Y = X x_{m != n} U_m^T, then the same Gram + eigensolve on Y(n).
//
// The Gram never forms an unfolded copy (the reference materialises X2 with t2m and, for
// order 4, X2 and X3 by identity-matrix GEMMs, src/tucker4_hosvd.cu:23-37): a workgroup
// accumulates an In x In FP32 tile over a range of the (P, In, Q) view's fibres (gram_f32.hip,
// gram_any.hip, gram.hip), partial tiles are summed in FP64 in a fixed order.  The eigensolve is the FP64
// tridiagonal solver in one workgroup (subspace iteration first where the top eigenvalues
// stand clear of the rest, warm-started from the previous factor in HOOI); eigenvector signs
// are fixed so that the entry of largest magnitude is positive (syevdx leaves the sign
// unspecified).
#include "common.hpp"
#include "eig.hpp"
#include "eig_sub.hpp"
#include "linalg.hpp"
#include <algorithm>
#include <vector>

namespace tdx {

int ttm_generic(const float *X, int order, const long *dims, int mode, const float *U, long lda, long ldi, long Ra,
                float *Y, hipStream_t s);
int gram_mfma_launch(const void *X, int xtype, long P, long In, long Q, float *part, int max_parts, hipStream_t s);
int gram_any_launch(const void *X, int xtype, long P, long In, long Q, float *part, int max_parts, hipStream_t s);
int ttm_generic_t(const void *X, int xtype, int order, const long *dims, int mode, const float *U, long lda, long ldi,
                  long Ra, float *Y, hipStream_t s);
int ttm_bf16_hooi(const void *X, int xtype, int order, const long *dims, int mode, const float *U, long lda, long ldi,
                  long Ra, float *Y, hipStream_t s);

static constexpr int kGramMaxN = 128;
static constexpr int kGramChunk = 64;  // fibres a step of k_gram_partial

// Partial Grams of the (P, In, Q) view, FP32 FMAs over a range of fibres k = p + P q in order: HOOI on
// BF16 storage only (see bf16_hooi in unfold_gram; k_gram_any sums in another order).  A workgroup
// takes a 32 x 32 block bi <= bj (blockIdx.y) of the tile, a thread 2 x 2 entries; 64 fibres of the two
// row blocks are staged a step, the next 64 in flight.  The order of an entry's sum is that of a
// workgroup owning the whole tile (8 x 8 entries a
// thread, 500-730 us a mode of 125 x 101 x 77; HOOI of 60 x 97 x 65 3.16 ms with it, 1.43 this way).
__device__ __forceinline__ float ldx(const float *p, long i) { return p[i]; }
__device__ __forceinline__ float ldx(const uint16_t *p, long i) { return __uint_as_float((uint32_t)p[i] << 16); }

template <typename T>
__global__ __launch_bounds__(256) void k_gram_partial(const T *__restrict__ X, long P, long In, long Q,
                                                      long kper, float *__restrict__ part) {
    __shared__ float xs[64][kGramChunk + 1];  // rows: 32 of block bi, 32 of block bj
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    int bi = 0, bj = blockIdx.y;
    for (const int nb = (int)((In + 31) / 32); bj >= nb - bi; ++bi) bj -= nb - bi;
    bj += bi;
    const long K = P * Q;
    const long k0 = blockIdx.x * kper, k1 = min(k0 + kper, K);
    float acc[2][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}};
    // element u of a thread: row and fibre of the step, lanes along what is contiguous
    constexpr int NL = 64 * kGramChunk / 256;
    float v[NL];
    auto at = [&](int u, int &r, int &kk) {
        const int e = tid + 256 * u;
        if (P == 1) r = e % 64, kk = e / 64;
        else kk = e % kGramChunk, r = e / kGramChunk;
    };
    auto load = [&](long kb) {
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            int r, kk;
            at(u, r, kk);
            const long a = r < 32 ? 32 * bi + r : 32 * bj + r - 32, k = kb + kk;
            const bool on = k < k1 && a < In;
            const long kc = on ? k : k0, q = kc / P;
            v[u] = ldx(X, (kc - q * P) + (on ? a : 0) * P + q * P * In);
            if (!on) v[u] = 0.0f;
        }
    };
    load(k0);
    for (long kb = k0; kb < k1; kb += kGramChunk) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            int r, kk;
            at(u, r, kk);
            xs[r][kk] = v[u];
        }
        __syncthreads();
        load(kb + kGramChunk);
#pragma unroll 8
        for (int kk = 0; kk < kGramChunk; ++kk) {
            const float a0 = xs[2 * ty][kk], a1 = xs[2 * ty + 1][kk];
            const float b0 = xs[32 + 2 * tx][kk], b1 = xs[32 + 2 * tx + 1][kk];
            acc[0][0] = fmaf(a0, b0, acc[0][0]);
            acc[0][1] = fmaf(a0, b1, acc[0][1]);
            acc[1][0] = fmaf(a1, b0, acc[1][0]);
            acc[1][1] = fmaf(a1, b1, acc[1][1]);
        }
    }
    float *dst = part + (long)blockIdx.x * kGramMaxN * kGramMaxN + (32L * bi + 2 * ty) * kGramMaxN + 32 * bj + 2 * tx;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) dst[i * kGramMaxN + j] = acc[i][j];
}

// G = the sum of the nblk FP32 partial Grams (pitch kGramMaxN), in FP64: a workgroup takes 64
// consecutive entries (a, b) of the upper triangle (b fastest: contiguous reads) and its four
// waves the four quarters of the block range (each summed in block order, 8 loads in
// flight); the quarters are added in order and the sum written to both triangles, so G is
// symmetric bit for bit.  Grid: ceil(In^2 / 64).
__global__ __launch_bounds__(256) void k_gram_sum(const float *__restrict__ part, int nblk, long In,
                                                  double *__restrict__ G) {
    __shared__ double sh[4][64];
    const int lane = threadIdx.x & 63, rg = threadIdx.x >> 6;
    const long f = blockIdx.x * 64L + lane;
    const long a = f / In, b = f - a * In;
    const bool on = f < In * In && a <= b;
    double s = 0.0;
    if (on) {
        const int k0 = (int)((long)rg * nblk / 4), k1 = (int)((long)(rg + 1) * nblk / 4);
        const float *p = part + a * kGramMaxN + b;
        constexpr long kStride = (long)kGramMaxN * kGramMaxN;
        for (int k = k0; k < k1; k += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = p[(long)(k + u < k1 ? k + u : k1 - 1) * kStride];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (k + u < k1) s += (double)v[u];
        }
    }
    sh[rg][lane] = s;
    __syncthreads();
    if (rg == 0 && on) {
        const double t = ((sh[0][lane] + sh[1][lane]) + sh[2][lane]) + sh[3][lane];
        G[a + b * In] = t;
        G[b + a * In] = t;
    }
}

// Top-r eigenvectors of a symmetric n x n G (FP64), one workgroup each: U (n x r, col-major
// FP32) receives the eigenvectors of the r largest eigenvalues in ascending order.  With
// try_sub the subspace-iteration path runs first (start block U0, or a built-in one when U0
// is null; U0 may alias U) and the tridiagonal solver only when it declines.  method (optional,
// device) receives 1 for the subspace path, 0 for the tridiagonal one.
// A solve is one workgroup's chain of 110 to 160 us whatever the size of the tensor, so the independent
// ones of an HOSVD (a mode each) share one launch: three modes of 125 x 101 x 77 take 115 + 130 +
// 155 us one after the other.
struct EigJob {
    const double *G;
    int n, r;
    const float *U0;
    float *U;
    double *w, *scratch;
    int *method;
};
struct EigJobs {
    EigJob j[4];
};
__global__ __launch_bounds__(kEigThreads) void k_top_eigvecs(EigJobs jobs, int try_sub, int rotate) {
    extern __shared__ double smem[];
    const EigJob q = jobs.j[blockIdx.x];
    if (try_sub && q.r <= kSubMaxR) {
        if (sym_top_eigvecs_subspace(q.G, q.n, q.r, q.U0, q.U, q.w, smem, rotate != 0)) {
            if (q.method && threadIdx.x == 0) *q.method = 1;
            return;
        }
        __syncthreads();  // the LDS is reused below
    }
    sym_top_eigvecs_block(q.G, q.n, q.r, q.U, q.w, q.scratch, q.scratch + (long)q.n * q.n, smem);
    if (q.method && threadIdx.x == 0) *q.method = 0;
}

// ||X||^2 in FP64 (Kahan per thread), block partials.  Eight loads in flight: with one, 128^4
// took 500 us (2.1 TB/s).
__global__ __launch_bounds__(256) void k_norm2_blocks(const float *__restrict__ X, long n, double *__restrict__ part) {
    __shared__ double sh[256];
    double s = 0.0, c = 0.0;
    const long st = (long)gridDim.x * 256;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < n; e += 8 * st) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = X[e + u * st < n ? e + u * st : e];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double x = e + u * st < n ? (double)v[u] : 0.0;
            const double y = x * x - c, t = s + y;
            c = (t - s) - y;
            s = t;
        }
    }
    s = block_sum(s, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ void k_sum_to(const double *__restrict__ part, int n, double *__restrict__ out) {
    __shared__ double sh[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += part[i];
    s = block_sum(s, sh);
    if (threadIdx.x == 0) *out = s;
}

// ---------------------------------------------------------------------------
struct TuckerWs {
    float *gram_part = nullptr;
    int gram_blocks = 0;
    double *G = nullptr;
    double *Q = nullptr;
    float *y0 = nullptr, *y1 = nullptr, *y2 = nullptr;
    double *scal = nullptr;
    uint16_t *xb = nullptr;
    DeviceLease mem;  // all of it
};

// bf16_hooi: HOOI iterations on BF16 storage round the factors to BF16, so an entry next to the middle
// of two BF16 values turns the last bits of a sum into differences of 1e-4 in the results.  Their Grams
// and products keep the summation order (and so the bits) they have always had: the register kernels
// of gram.hip and ttm.hip and the per-entry ones.
static int unfold_gram(const void *X, int xtype, int order, const long *dims, int mode, TuckerWs &W, double *G,
                       hipStream_t s, bool bf16_hooi = false) {
    long P = 1, Q = 1;
    for (int m = 0; m < mode; ++m) P *= dims[m];
    for (int m = mode + 1; m < order; ++m) Q *= dims[m];
    const long In = dims[mode];
    if (In > kGramMaxN) return record(TDX_ERR_UNSUPPORTED);
    // the BF16 kernel for whole vectors (gram.hip), the LDS kernels otherwise
    int nb = 0;
    if (xtype == TDX_BF16 || bf16_hooi)
        nb = gram_mfma_launch(X, xtype, P, In, Q, W.gram_part, W.gram_blocks < 512 ? W.gram_blocks : 512, s);
    if (nb == 0 && bf16_hooi) {
        const long K = P * Q, want = std::max(1L, std::min((long)W.gram_blocks, ceil_div(K, 2048L)));
        const long kper = ceil_div(ceil_div(K, want), 32L) * 32;
        nb = (int)ceil_div(K, kper);
        const int n32 = (int)ceil_div(In, 32L);
        const dim3 g((unsigned)nb, (unsigned)(n32 * (n32 + 1) / 2));
        if (xtype == TDX_BF16)
            k_gram_partial<uint16_t><<<g, 256, 0, s>>>((const uint16_t *)X, P, In, Q, kper, W.gram_part);
        else
            k_gram_partial<float><<<g, 256, 0, s>>>((const float *)X, P, In, Q, kper, W.gram_part);
        TDX_LAUNCH_CHECK();
    }
    if (nb == 0) nb = gram_any_launch(X, xtype, P, In, Q, W.gram_part, W.gram_blocks, s);
    if (nb < 0) return record(TDX_ERR_HIP);
    k_gram_sum<<<(int)ceil_div(In * In, 64L), 256, 0, s>>>(W.gram_part, nb, In, G);
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

// TDX_EIG_SUBSPACE=0 keeps every eigensolve on the tridiagonal path (A/B comparisons)
static bool subspace_enabled() {
    static int on = -1;
    if (on < 0) {
        const char *e = getenv("TDX_EIG_SUBSPACE");
        on = (e && e[0] == '0') ? 0 : 1;
    }
    return on != 0;
}

static long eig_kernel_lds_doubles(int n) {
    const long a = eig_lds_doubles(n), b = eig_sub_doubles(n);
    return a > b ? a : b;
}

// njobs <= 4 independent eigensolves in one launch; scratch: 2 n^2 doubles each.  try_sub: try the
// subspace path first, starting from U0 (or the built-in block when U0 is null).  rotate = 0: an
// orthonormal basis of the top-r subspace is enough (the subspace path may then skip its
// Rayleigh-Ritz rotation; w is not written then).
static int top_eigvecs(const EigJob *jobs, int njobs, int try_sub, hipStream_t s, int rotate = 1) {
    EigJobs a{};
    int nmax = 1;
    for (int k = 0; k < njobs; ++k) {
        const EigJob &q = jobs[k];
        if (q.n < 1 || q.n > kEigMaxN || q.r < 1 || q.r > q.n) return record(TDX_ERR_ARG);
        a.j[k] = q;
        nmax = q.n > nmax ? q.n : nmax;
    }
    static bool attr_set = false;
    if (!attr_set) {
        TDX_HIP(hipFuncSetAttribute((const void *)k_top_eigvecs, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)(sizeof(double) * eig_kernel_lds_doubles(kEigMaxN))));
        attr_set = true;
    }
    const int sub = (try_sub && subspace_enabled()) ? 1 : 0;
    k_top_eigvecs<<<njobs, kEigThreads, sizeof(double) * eig_kernel_lds_doubles(nmax), s>>>(a, sub, rotate);
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

static int ws_setup(TuckerWs &W, int order, const long *dims, const long *ranks, bool bf16) {
    W.gram_blocks = 1024;
    // largest intermediate of a TTM chain: the first contraction of the biggest mode
    long N = 1;
    for (int m = 0; m < order; ++m) N *= dims[m];
    long maxsz = 0;
    for (int m = 0; m < order; ++m) {
        long sz = N / dims[m] * ranks[m];
        if (sz > maxsz) maxsz = sz;
    }
    Parts p;
    const size_t gp = p.add(sizeof(float) * (size_t)W.gram_blocks * kGramMaxN * kGramMaxN);
    const size_t g = p.add(sizeof(double) * 4 * kGramMaxN * kGramMaxN);
    const size_t q = p.add(sizeof(double) * 8 * kGramMaxN * kGramMaxN);
    const size_t sc = p.add(sizeof(double) * 2048);
    const size_t y0 = p.add(sizeof(float) * maxsz), y1 = p.add(sizeof(float) * maxsz), y2 = p.add(sizeof(float) * maxsz);
    const size_t xb = p.add(bf16 ? sizeof(uint16_t) * N : 0);
    const int st = W.mem.take(p.bytes);
    if (st) return st;
    char *b = W.mem.ptr();
    W.gram_part = (float *)(b + gp);
    W.G = (double *)(b + g);
    W.Q = (double *)(b + q);
    W.scal = (double *)(b + sc);
    W.y0 = (float *)(b + y0);
    W.y1 = (float *)(b + y1);
    W.y2 = (float *)(b + y2);
    W.xb = (uint16_t *)(b + xb);
    return TDX_OK;
}

// Y = X x_{m in modes} U_m^T applied in the listed order, results alternating between the
// buffers a and b (X itself when nmodes == 0); cur: the dims of X in, of the result out
static int ttm_seq(const void *X, int xtype, int order, long *cur, const long *ranks, float *const *U,
                   const int *modes, int nmodes, float *a, float *b, const float **out, hipStream_t s,
                   bool bf16_hooi = false) {
    const void *src = X;
    for (int t = 0; t < nmodes; ++t) {
        const int m = modes[t];
        float *dst = (t & 1) ? b : a;
        auto *ttm = bf16_hooi ? ttm_bf16_hooi : ttm_generic_t;
        int st = ttm(src, t == 0 ? xtype : TDX_F32, order, cur, m, U[m], cur[m], 1, ranks[m], dst, s);
        if (st) return st;
        cur[m] = ranks[m];
        src = dst;
    }
    *out = (const float *)src;
    return TDX_OK;
}

// core = X x_1 U_1^T ... x_d U_d^T from the FP32 tensor, slowest mode first
static int core_from(const float *X, int order, const long *dims, const long *ranks, float *const *U, TuckerWs &W,
                     float *core, hipStream_t s) {
    int modes[4], nm = 0;
    for (int m = order - 1; m >= 1; --m) modes[nm++] = m;
    long cur[4];
    for (int m = 0; m < order; ++m) cur[m] = dims[m];
    const float *Y = nullptr;
    int st = ttm_seq(X, TDX_F32, order, cur, ranks, U, modes, nm, W.y0, W.y1, &Y, s);
    if (st) return st;
    return ttm_generic(Y, order, cur, 0, U[0], dims[0], 1, ranks[0], core, s);
}

static int tucker_run(const float *X, int order, const long *dims, const long *ranks, int iters, float *core,
                      float *const *U, double *relerr_hist, int bf16) {
    if (!X || !core || !U || order < 2 || order > 4) return record(TDX_ERR_ARG);
    for (int m = 0; m < order; ++m) {
        if (dims[m] <= 0 || ranks[m] <= 0 || ranks[m] > dims[m] || !U[m]) return record(TDX_ERR_ARG);
        if (dims[m] > kGramMaxN) return record(TDX_ERR_UNSUPPORTED);
    }
    hipStream_t s = stream();
    TuckerWs W;
    int st = ws_setup(W, order, dims, ranks, bf16 != 0);
    if (st) return st;
    long N = 1;
    for (int m = 0; m < order; ++m) N *= dims[m];
    // BF16 storage: the Grams of X and the first TTM of every chain stream a BF16 copy
    const void *Xs = X;
    int xtype = TDX_F32;
    if (bf16) {
        st = tdx_quantize_bf16(X, W.xb, N);
        if (st) return st;
        Xs = W.xb;
        xtype = TDX_BF16;
    }
    // HOSVD init.  Only the spans matter when HOOI iterations follow (every later product contracts
    // U U^T), but from eigenvectors the last iteration's solves start with a nearly diagonal H and
    // take fewer Jacobi sweeps, one after the other, where the HOSVD's run side by side (128^4, ranks
    // 32, one iteration: 2.89 ms without this rotation, 2.70 with it).  Not with BF16 storage, whose
    // products round U's entries and so depend on the basis.
    const bool bf16_hooi = bf16 && iters > 0;  // (see unfold_gram)
    EigJob jobs[4];
    for (int m = 0; m < order; ++m) {
        double *G = W.G + (long)m * kGramMaxN * kGramMaxN;
        st = unfold_gram(Xs, xtype, order, dims, m, W, G, s, bf16_hooi);
        if (st) return st;
        jobs[m] = EigJob{G, (int)dims[m], (int)ranks[m], nullptr, U[m], nullptr, W.Q + 2L * m * kGramMaxN * kGramMaxN,
                         nullptr};
    }
    st = top_eigvecs(jobs, order, 1, s, !bf16_hooi);
    if (st) return st;
    // ||X||^2 serves the error history only: a pass over X that a call without one does not make
    if (relerr_hist) {
        k_norm2_blocks<<<1024, 256, 0, s>>>(X, N, W.scal);
        k_sum_to<<<1, 256, 0, s>>>(W.scal, 1024, W.scal + 1024);
        TDX_LAUNCH_CHECK();
    }
    double nx2 = 0.0;
    long nc = 1;
    for (int m = 0; m < order; ++m) nc *= ranks[m];
    // HOOI with a dimension tree: the modes split into L = {0..h-1} and R = {h..d-1};
    // T = X x_{R} U^T serves every n in L, then T = X x_{L} U^T (with the new U_L) every n in
    // R, so X is streamed twice per iteration rather than d times.  Each T contracts its
    // slowest mode first.
    const int h = order / 2;
    const float *Y = nullptr;  // the last product: all modes but d-1 contracted
    long ydims[4];
    for (int it = 0; it < iters; ++it) {
        for (int half = 0; half < 2; ++half) {
            const int n0 = half ? h : 0, n1 = half ? order : h;
            int tm[4], nt = 0;
            for (int m = order - 1; m >= 0; --m)
                if (m < n0 || m >= n1) tm[nt++] = m;
            long tdims[4];
            for (int m = 0; m < order; ++m) tdims[m] = dims[m];
            const float *T = nullptr;
            st = ttm_seq(Xs, xtype, order, tdims, ranks, U, tm, nt, W.y0, W.y1, &T, s, bf16_hooi);
            if (st) return st;
            float *fa = (T == W.y0) ? W.y1 : W.y0;
            for (int n = n0; n < n1; ++n) {
                int sm[4], ns = 0;
                for (int m = n1 - 1; m >= n0; --m)
                    if (m != n) sm[ns++] = m;
                for (int m = 0; m < order; ++m) ydims[m] = tdims[m];
                st = ttm_seq(T, TDX_F32, order, ydims, ranks, U, sm, ns, W.y2, fa, &Y, s, bf16_hooi);
                if (!st) st = unfold_gram(Y, TDX_F32, order, ydims, n, W, W.G, s, bf16_hooi);
                // warm start: the factor of the previous iteration spans nearly the same subspace;
                // eigenvectors (ascending, sign convention) only in the last iteration
                const EigJob job{W.G, (int)dims[n], (int)ranks[n], U[n], U[n], nullptr, W.Q, nullptr};
                if (!st) st = top_eigvecs(&job, 1, 1, s, it == iters - 1);
                if (st) return st;
            }
        }
        if (relerr_hist) {
            // relerr^2 = 1 - ||core||^2/||X||^2.  The core comes from the last Y (all modes
            // but d-1 contracted); with BF16 storage it is recomputed from the FP32 tensor.
            if (bf16) st = core_from(X, order, dims, ranks, U, W, core, s);
            else st = ttm_generic(Y, order, ydims, order - 1, U[order - 1], dims[order - 1], 1, ranks[order - 1],
                                  core, s);
            if (st) return st;
            {
                // ||core||^2: block partials (the first 1024 slots are free once ||X||^2 is summed)
                const int nb = (int)(ceil_div(nc, 1024L) < 1024 ? ceil_div(nc, 1024L) : 1024);
                k_norm2_blocks<<<nb, 256, 0, s>>>(core, nc, W.scal);
                k_sum_to<<<1, 256, 0, s>>>(W.scal, nb, W.scal + 1025);
            }
            double hv[2];
            TDX_HIP(hipMemcpyAsync(hv, W.scal + 1024, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
            TDX_HIP(hipStreamSynchronize(s));
            nx2 = hv[0];
            relerr_hist[it] = sqrt(fmax(nx2 - hv[1], 0.0) / nx2);
        }
    }
    // The final core, always from the FP32 tensor.  After an iteration on FP32 storage the last Y
    // holds all modes but d-1 contracted with the final factors, so one small TTM is left (a chain
    // over X took 0.36 ms of the 4.62 ms of HOSVD and one iteration of 128^4, ranks 32); with an error
    // history the last iteration has already made the core.
    if (iters == 0 || (bf16 && !relerr_hist)) st = core_from(X, order, dims, ranks, U, W, core, s);
    else if (!relerr_hist)
        st = ttm_generic(Y, order, ydims, order - 1, U[order - 1], dims[order - 1], 1, ranks[order - 1], core, s);
    if (st) return st;
    TDX_HIP(hipStreamSynchronize(s));
    W.mem.done();
    return TDX_OK;
}

}  // namespace tdx

using namespace tdx;

extern "C" {

int tdx_unfold_gram_ex(const void *X, int dtype, int order, const long *dims, int mode, double *G) {
    TDX_CHECK_ARG(X && dims && G && order >= 2 && order <= 4 && mode >= 0 && mode < order);
    TDX_CHECK_ARG(dtype == TDX_F32 || dtype == TDX_BF16);
    for (int m = 0; m < order; ++m) TDX_CHECK_ARG(dims[m] > 0);
    TuckerWs W;
    W.gram_blocks = 1024;
    int st = W.mem.take(sizeof(float) * (size_t)W.gram_blocks * kGramMaxN * kGramMaxN);
    if (st) return st;
    W.gram_part = (float *)W.mem.ptr();
    st = unfold_gram(X, dtype, order, dims, mode, W, G, stream());
    if (!st) {
        TDX_HIP(hipStreamSynchronize(stream()));
        W.mem.done();
    }
    return record(st);
}

int tdx_unfold_gram(const float *X, int order, const long *dims, int mode, double *G) {
    return tdx_unfold_gram_ex(X, TDX_F32, order, dims, mode, G);
}

int tdx_sym_eig_topr_ex(const double *G, long n, long r, const float *U0, int flags, float *U, double *w,
                        int *method) {
    TDX_CHECK_ARG(G && U && n >= 1 && n <= kEigMaxN && r >= 1 && r <= n);
    void *scr = nullptr;
    int st = workspace(WS_MISC2, sizeof(double) * 2 * n * n + 256, &scr);
    if (st) return st;
    int *dmethod = (int *)((char *)scr + sizeof(double) * 2 * n * n);
    const EigJob job{G, (int)n, (int)r, U0, U, w, (double *)scr, dmethod};
    st = top_eigvecs(&job, 1, (flags & TDX_EIG_TRY_SUBSPACE) ? 1 : 0, stream());
    int hm = 0;
    if (!st) TDX_HIP(hipMemcpyAsync(&hm, dmethod, sizeof(int), hipMemcpyDeviceToHost, stream()));
    if (!st) TDX_HIP(hipStreamSynchronize(stream()));
    if (!st && method) *method = hm;
    return record(st);
}

int tdx_sym_eig_topr(const double *G, long n, long r, float *U, double *w) {
    return tdx_sym_eig_topr_ex(G, n, r, nullptr, 0, U, w, nullptr);
}

int tdx_tucker_hooi(const float *X, int order, const long *dims, const long *ranks, int iters, int bf16_ttm,
                    float *core, float *const *U, double *relerr_hist) {
    if (!dims || !ranks || iters < 0) return record(TDX_ERR_ARG);
    return record(tucker_run(X, order, dims, ranks, iters, core, U, relerr_hist, bf16_ttm));
}

int tdx_tucker_hosvd(const float *X, float *core, float *U1, float *U2, float *U3, long a, long b, long c, long r1,
                     long r2, long r3) {
    const long dims[3] = {a, b, c}, ranks[3] = {r1, r2, r3};
    float *U[3] = {U1, U2, U3};
    return record(tucker_run(X, 3, dims, ranks, 0, core, U, nullptr, 0));
}

int tdx_tucker_hosvd4(const float *X, float *core, float *U1, float *U2, float *U3, float *U4, long a, long b, long c,
                      long d, long r1, long r2, long r3, long r4) {
    const long dims[4] = {a, b, c, d}, ranks[4] = {r1, r2, r3, r4};
    float *U[4] = {U1, U2, U3, U4};
    return record(tucker_run(X, 4, dims, ranks, 0, core, U, nullptr, 0));
}

// reference tucker_tensorcore (src/tucker_tensorcore.cu): reduced-precision Grams and TTM
// chain; here the Grams and the first TTM stream a BF16 copy, everything accumulates in FP32
int tdx_tucker_tensorcore(const float *X, float *core, float *U1, float *U2, float *U3, long a, long b, long c,
                          long r1, long r2, long r3) {
    const long dims[3] = {a, b, c}, ranks[3] = {r1, r2, r3};
    float *U[3] = {U1, U2, U3};
    return record(tucker_run(X, 3, dims, ranks, 0, core, U, nullptr, 1));
}

}  // extern "C"
