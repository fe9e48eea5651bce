// recon.hip -- reconstruction, residual norms, synthetic CP tensors and the generic
// mode-n product used by the Tucker path.
#include "common.hpp"
#include <algorithm>
#include <math.h>

namespace tdx {

__device__ double block_sum_d(double v, double *sh) {
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] += sh[t + s];
        __syncthreads();
    }
    double r = sh[0];
    __syncthreads();
    return r;
}

struct FacArgs {
    const float *U[4];
    long dims[4];
    int order;
    int R;
};

// The CP model and its residual, x_hat[i, c] = sum_r U_0[i, r] w[c, r] over the fibres c =
// (i_1, .., i_{d-1}) with w[c, r] = U_1[i_1, r] (U_2[i_2, r] U_3[i_3, r]), on FP32 MFMA.
//  RES = false: writes x_hat (gencp / gencp4, src/rse.cu:17-30,53-73)
//  RES = true: sums (x - x_hat)^2 and x^2 in FP64 (compensated CP residual)
// A workgroup walks a range of fibres 64 at a time: its threads form w for them in LDS (a lane a
// fibre, whose digits advance by a mixed-radix addition; the next 64's factor entries are in
// flight meanwhile), RW of its waves take a block of 64 rows each and the other 4 / RW share the
// four blocks of 16 fibres.  A wave's U_0 rows stay in registers as the A operand (KS k-steps of 4
// columns; BIG, ranks above 64, reloads them per block of 64 columns).  Lane (lm, lg) holds rows
// 16 t + 4 lg .. + 3 of fibre lm: 16-byte loads and stores of whole 64-byte runs, 4-byte aligned.
// Bound by HBM (512 x 384 x 320: 252 MB, 55 us at the 4.6 TB/s of a large copy).  One thread per
// entry, with a load of U_0 for every multiply-add, took 496 us (model) and 828 us (residual) at
// rank 32; these take 68 and 90 us (each wave loading its own w: 157 and 215).
typedef float rc_f4 __attribute__((ext_vector_type(4)));
typedef float rc_f4u __attribute__((ext_vector_type(4), aligned(4)));
static constexpr int kModelLd = 80;  // W row pitch: 4 rows of 16 fibres in distinct banks

template <bool RES, int KS, int RW, bool BIG>
__global__ __launch_bounds__(256, 2) void k_cp_model(FacArgs f, float *__restrict__ out, const float *__restrict__ X,
                                                     long ntile, long tper, int nrg, double *__restrict__ part) {
    extern __shared__ float W[];  // [max(4 KS, R rounded up to 64)][kModelLd]
    __shared__ double sh[RES ? 256 : 1];
    constexpr int FW = 4 / RW;
    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), rw = wave % RW, fw = wave / RW;
    const long I = f.dims[0], D1 = f.dims[1], D2 = f.dims[2], D3 = f.dims[3];
    const long nfib = D1 * D2 * D3;
    const int R = f.R;
    const long row0 = ((long)(blockIdx.x % nrg) * RW + rw) * 64;
    const long t0 = (blockIdx.x / nrg) * tper, t1 = min(t0 + tper, ntile);
    const float *U0 = f.U[0], *U1 = f.U[1], *U2 = f.order > 2 ? f.U[2] : nullptr,
                *U3 = f.order > 3 ? f.U[3] : nullptr;
    double s1 = 0.0, c1 = 0.0, s2 = 0.0, c2 = 0.0;

    float aop[4][KS];
    auto load_a = [&](int r0) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float *p = U0 + min(row0 + 16 * t + lm, I - 1);
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const int r = r0 + 4 * k + lg;
                aop[t][k] = p[(r < R ? r : 0) * I];
            }
#pragma unroll
            for (int k = 0; k < KS; ++k)
                if (r0 + 4 * k + lg >= R) aop[t][k] = 0.0f;
        }
    };
    // this lane's fibre of the 64 and its digits
    long c = 64 * t0 + lane;
    long i1 = c % D1, i2 = (c / D1) % D2, i3 = c / D1 / D2;
    const long A1 = 64 % D1, A2 = (64 / D1) % D2, A3 = 64 / D1 / D2;
    float w1[KS], w2[KS], w3[KS];  // columns r0 + wave + 4 k of the fibre's factor rows
    auto load_w = [&](int r0) {
        const bool on = c < nfib;
        const float *p1 = U1 + (on ? i1 : 0), *p2 = U2 ? U2 + (on ? i2 : 0) : U1, *p3 = U3 ? U3 + (on ? i3 : 0) : U1;
        int rb = r0 + wave;
        asm volatile("" : "+s"(rb));  // (hoisted out of the loop the column offsets fill the scalar registers)
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const long r = rb + 4 * k < R ? rb + 4 * k : 0;
            w1[k] = p1[r * D1];
            if (U2) w2[k] = p2[r * D2];
            if (U3) w3[k] = p3[r * D3];
        }
    };
    auto store_w = [&](int r0) {
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            // reference order: the KR of the later modes is formed first (src/rse.cu:65-66)
            float q = 1.0f, v = w1[k];
            if (U2) q = w2[k];
            if (U3) q *= w3[k];
            if (U2) v *= q;
            W[(r0 + wave + 4 * k) * kModelLd + lane] = r0 + wave + 4 * k < R ? v : 0.0f;
        }
    };
    auto advance = [&]() {
        c += 64;
        i1 += A1;
        i2 += A2;
        i3 += A3;
        if (i1 >= D1) {
            i1 -= D1;
            ++i2;
        }
        if (i2 >= D2) {
            i2 -= D2;
            ++i3;
        }
    };
    const bool rows = row0 + 64 <= I;  // uniform
    if (!BIG && t0 < t1) {
        load_w(0);
        load_a(0);
    }
    for (long tl = t0; tl < t1; ++tl) {
        __syncthreads();  // every wave is done with the previous W
        if constexpr (BIG) {
            for (int r0 = 0; r0 < R; r0 += 4 * KS) {
                load_w(r0);
                store_w(r0);
            }
            advance();
        } else {
            store_w(0);
        }
        __syncthreads();
        if constexpr (!BIG) {
            advance();
            load_w(0);  // past the last tile: valid addresses, never consumed
        }
        if (row0 >= I) continue;  // (a row block past the extent: this wave only forms w)
        for (int fb = fw; fb < 4; fb += FW) {
            const long cf = 64 * tl + 16 * fb + lm;  // this lane's fibre of the block
            const bool on = cf < nfib, full = rows && 64 * tl + 16 * fb + 16 <= nfib;
            rc_f4 x[4];
            if constexpr (RES) {
                const float *p = X + (on ? cf : 0) * I + row0 + 4 * lg;
                if (full) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) x[t] = *reinterpret_cast<const rc_f4u *>(p + 16 * t);
                } else {
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int v = 0; v < 4; ++v) x[t][v] = p[min(16L * t + v, I - 1 - row0 - 4 * lg)];
                }
            }
            rc_f4 acc[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] = rc_f4{0.f, 0.f, 0.f, 0.f};
            for (int r0 = 0; r0 < (BIG ? R : 1); r0 += 4 * KS) {
                if (BIG) load_a(r0);
                const float *wp = W + (r0 + lg) * kModelLd + 16 * fb + lm;
#pragma unroll
                for (int k = 0; k < KS; ++k) {
                    const float w = wp[4 * k * kModelLd];
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        if (row0 + 16 * t < I)
                            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(aop[t][k], w, acc[t], 0, 0, 0);
                }
            }
            // (the wait states between a matrix result and its first read: hipcc counted one too few on
            // the way past the skipped row blocks)
            asm volatile("s_nop 9" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const long i = row0 + 16 * t + 4 * lg;
                if constexpr (RES) {
                    // four squares added, then compensated
                    double d2 = 0.0, x2 = 0.0;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        double xv = (double)x[t][v], d = xv - (double)acc[t][v];
                        if (!full && !(on && i + v < I)) xv = d = 0.0;
                        d2 = fma(d, d, d2);
                        x2 = fma(xv, xv, x2);
                    }
                    double y = d2 - c1, s = s1 + y;
                    c1 = (s - s1) - y;
                    s1 = s;
                    y = x2 - c2;
                    s = s2 + y;
                    c2 = (s - s2) - y;
                    s2 = s;
                } else {
                    float *p = out + (on ? cf : 0) * I + i;
                    if (full) {
                        *reinterpret_cast<rc_f4u *>(p) = acc[t];
                    } else if (on) {
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            if (i + v < I) p[v] = acc[t][v];
                    }
                }
            }
        }
    }
    if constexpr (RES) {
        s1 = block_sum_d(s1, sh);
        s2 = block_sum_d(s2, sh);
        if (tid == 0) {
            part[2 * blockIdx.x] = s1;
            part[2 * blockIdx.x + 1] = s2;
        }
    }
}

// Synthetic tensors: for each fibre along mode 0 (fixed i_1..i_{d-1}) w[r] = prod_{m>=1}
// U_m[i_m, r] in LDS, then x_hat[i] = sum_r U_0[i, r] w[r]; writes x_hat and accumulates x_hat^2
// and e^2 for E ~ N(0,1).
__global__ __launch_bounds__(256) void k_cp_fibres(FacArgs f, float *__restrict__ out, double *__restrict__ part,
                                                   uint64_t seed, uint32_t strm) {
    __shared__ float w[64 * 4];
    __shared__ double sh[256];
    const long I0 = f.dims[0];
    long nfib = 1;
    for (int m = 1; m < f.order; ++m) nfib *= f.dims[m];
    double s1 = 0.0, c1 = 0.0, s2 = 0.0, c2 = 0.0;
    for (long fib = blockIdx.x; fib < nfib; fib += gridDim.x) {
        __syncthreads();
        for (int r = threadIdx.x; r < f.R; r += blockDim.x) {
            long rem = fib;
            float p = 1.0f;
            // reference order: the KR of the later modes is formed first (src/rse.cu:65-66)
            float q = 1.0f;
            for (int m = 1; m < f.order; ++m) {
                long idx = rem % f.dims[m];
                rem /= f.dims[m];
                if (m == 1) p = f.U[1][idx + r * f.dims[1]];
                else q = (m == 2) ? f.U[2][idx + r * f.dims[2]] : q * f.U[m][idx + r * f.dims[m]];
            }
            w[r] = (f.order > 2) ? p * q : p;
        }
        __syncthreads();
        for (long i = threadIdx.x; i < I0; i += blockDim.x) {
            float acc = 0.0f;
            for (int r = 0; r < f.R; ++r) acc = fmaf(f.U[0][i + r * I0], w[r], acc);
            const long e = fib * I0 + i;
            out[e] = acc;
            uint64_t n = (uint64_t)e;
            uint64_t blk = (2 * n) >> 2;
            uint32_t c[4] = {(uint32_t)blk, (uint32_t)(blk >> 32), strm, 0u};
            philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
            int wd = (int)((2 * n) & 3);
            double u1 = (double)word_to_uniform(c[wd]), u2 = (double)word_to_uniform(c[wd + 1]);
            double g = (double)(float)(sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2));
            double y = (double)acc * (double)acc - c1, t = s1 + y;
            c1 = (t - s1) - y; s1 = t;
            y = g * g - c2; t = s2 + y;
            c2 = (t - s2) - y; s2 = t;
        }
    }
    s1 = block_sum_d(s1, sh);
    s2 = block_sum_d(s2, sh);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = s1;
        part[2 * blockIdx.x + 1] = s2;
    }
}

// X += scale * E with scale = eta * sqrt(sum1 / sum2) computed from the partials
__global__ void k_add_noise(float *__restrict__ X, long n, const double *__restrict__ part, int nparts, double eta,
                            uint64_t seed, uint32_t strm) {
    __shared__ double sh[256];
    __shared__ float scale;
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) {
        a += part[2 * i];
        b += part[2 * i + 1];
    }
    a = block_sum_d(a, sh);
    b = block_sum_d(b, sh);
    if (threadIdx.x == 0) scale = (b > 0.0) ? (float)(eta * sqrt(a / b)) : 0.0f;
    __syncthreads();
    const float sc = scale;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
        uint64_t nn = (uint64_t)e;
        uint64_t blk = (2 * nn) >> 2;
        uint32_t c[4] = {(uint32_t)blk, (uint32_t)(blk >> 32), strm, 0u};
        philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
        int wd = (int)((2 * nn) & 3);
        double u1 = (double)word_to_uniform(c[wd]), u2 = (double)word_to_uniform(c[wd + 1]);
        float g = (float)(sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2));
        X[e] = X[e] + sc * g;
    }
}

// ||X - X1||^2 and ||X||^2 (FP64, compensated) partials (src/rse.cu:4-15 without clobbering X1).
// Bound by HBM: 4 elements of each per load (VEC) and four loads in flight; the squares of a
// load are added before the compensated sum.  63 M elements (512 x 384 x 320): 151 us with one
// element a load and one load in flight, 80 us here.
template <bool VEC>
__global__ __launch_bounds__(256) void k_rse_partial(const float *__restrict__ X, const float *__restrict__ X1, long n,
                                                     double *__restrict__ part) {
    __shared__ double sh[256];
    constexpr int W = VEC ? 4 : 1;
    typedef float vec __attribute__((ext_vector_type(4)));
    double s1 = 0.0, c1 = 0.0, s2 = 0.0, c2 = 0.0;
    const long n4 = n / W, st = (long)gridDim.x * 256;
    auto take = [&](double d2, double x2) {
        double y = d2 - c1, t = s1 + y;
        c1 = (t - s1) - y; s1 = t;
        y = x2 - c2; t = s2 + y;
        c2 = (t - s2) - y; s2 = t;
    };
    for (long e = blockIdx.x * 256L + threadIdx.x; e < n4; e += 4 * st) {
        float a[4][W], b[4][W];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const long i = e + u * st < n4 ? e + u * st : e;
            if constexpr (VEC) {
                const vec va = __builtin_nontemporal_load(reinterpret_cast<const vec *>(X) + i);
                const vec vb = __builtin_nontemporal_load(reinterpret_cast<const vec *>(X1) + i);
#pragma unroll
                for (int q = 0; q < 4; ++q) a[u][q] = va[q], b[u][q] = vb[q];
            } else {
                a[u][0] = X[i];
                b[u][0] = X1[i];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            double d2 = 0.0, x2 = 0.0;
#pragma unroll
            for (int q = 0; q < W; ++q) {
                const double x = a[u][q], d = x - (double)b[u][q];
                d2 = fma(d, d, d2);
                x2 = fma(x, x, x2);
            }
            if (e + u * st < n4) take(d2, x2);
        }
    }
    if (VEC && blockIdx.x == 0 && threadIdx.x < n - 4 * n4) {
        const double x = X[4 * n4 + threadIdx.x], d = x - (double)X1[4 * n4 + threadIdx.x];
        take(d * d, x * x);
    }
    s1 = block_sum_d(s1, sh);
    s2 = block_sum_d(s2, sh);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = s1;
        part[2 * blockIdx.x + 1] = s2;
    }
}

__global__ void k_ratio(const double *__restrict__ part, int nparts, double *__restrict__ out) {
    __shared__ double sh[256];
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) {
        a += part[2 * i];
        b += part[2 * i + 1];
    }
    a = block_sum_d(a, sh);
    b = block_sum_d(b, sh);
    if (threadIdx.x == 0) out[0] = (b > 0.0) ? sqrt(a / b) : 0.0;
}

// Mode-n product on a (P, In, Q) view:
//   Y[p + a*P + q*P*Ra] = sum_{i < In} U[a*lda + i*ldi] * X[p + i*P + q*P*In]
// (reference ttm, src/ttm.cu:21,29,37, with lda = 1, ldi = d; transposed factor with
//  lda = In, ldi = 1; Tucker expansion core -> tensor with lda = 1, ldi = I).
int ttm_mfma_launch(const void *X, int xtype, long P, long In, long Q, const float *U, long lda, long ldi, long Ra,
                    float *Y, hipStream_t s);
// X is FP32 (xtype TDX_F32) or BF16 bit patterns (TDX_BF16)
int ttm_any_launch(const void *X, int xtype, long P, long In, long Q, const float *U, long lda, long ldi, long Ra,
                   float *Y, hipStream_t s);

int ttm_generic_t(const void *X, int xtype, int order, const long *dims, int mode, const float *U, long lda, long ldi,
                  long Ra, float *Y, hipStream_t s) {
    long P = 1, Q = 1;
    for (int m = 0; m < mode; ++m) P *= dims[m];
    for (int m = mode + 1; m < order; ++m) Q *= dims[m];
    // BF16: the register kernel for the shapes it covers (ttm.hip); the general one otherwise
    const int mf = xtype != TDX_BF16 ? 0 : ttm_mfma_launch(X, xtype, P, dims[mode], Q, U, lda, ldi, Ra, Y, s);
    if (mf < 0) return record(TDX_ERR_HIP);
    if (mf > 0) return TDX_OK;
    return ttm_any_launch(X, xtype, P, dims[mode], Q, U, lda, ldi, Ra, Y, s);
}

__device__ __forceinline__ float ld_elem(const float *p, long i) { return p[i]; }
__device__ __forceinline__ float ld_elem(const uint16_t *p, long i) { return __uint_as_float((uint32_t)p[i] << 16); }
// the factor entry as it enters the product: unchanged for FP32 storage, rounded to BF16
// (nearest-even) for BF16 storage, as on the MFMA path
__device__ __forceinline__ float coef(float u, const float *) { return u; }
__device__ __forceinline__ float coef(float u, const uint16_t *) {
    return __uint_as_float(f32_to_bf16_bits(u) << 16);
}

// one output a thread (of the shapes that ttm.hip does not cover, in HOOI on BF16 storage)
template <typename T>
__global__ __launch_bounds__(256) void k_ttm_generic(const T *__restrict__ X, long P, long In, long Q,
                                                     const float *__restrict__ U, long lda, long ldi, long Ra,
                                                     float *__restrict__ Y) {
    const long n = P * Ra * Q;
    for (long e = blockIdx.x * 256L + threadIdx.x; e < n; e += (long)gridDim.x * 256) {
        const long p = e % P;
        const long a = (e / P) % Ra;
        const long q = e / (P * Ra);
        const T *x = X + p + q * P * In;
        const float *u = U + a * lda;
        float acc = 0.0f;
        for (long i = 0; i < In; ++i) acc = fmaf(coef(u[i * ldi], x), ld_elem(x, i * P), acc);
        Y[e] = acc;
    }
}

// the product of HOOI on BF16 storage, whose summation order stays as it is (tucker.hip, unfold_gram)
int ttm_bf16_hooi(const void *X, int xtype, int order, const long *dims, int mode, const float *U, long lda, long ldi,
                  long Ra, float *Y, hipStream_t s) {
    long P = 1, Q = 1;
    for (int m = 0; m < mode; ++m) P *= dims[m];
    for (int m = mode + 1; m < order; ++m) Q *= dims[m];
    const int mf = ttm_mfma_launch(X, xtype, P, dims[mode], Q, U, lda, ldi, Ra, Y, s);
    if (mf < 0) return record(TDX_ERR_HIP);
    if (mf > 0) return TDX_OK;
    const int g = (int)std::max(1L, std::min(ceil_div(P * Ra * Q, 256L), 65536L));
    if (xtype == TDX_BF16)
        k_ttm_generic<uint16_t><<<g, 256, 0, s>>>((const uint16_t *)X, P, dims[mode], Q, U, lda, ldi, Ra, Y);
    else
        k_ttm_generic<float><<<g, 256, 0, s>>>((const float *)X, P, dims[mode], Q, U, lda, ldi, Ra, Y);
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

int ttm_generic(const float *X, int order, const long *dims, int mode, const float *U, long lda, long ldi, long Ra,
                float *Y, hipStream_t s) {
    return ttm_generic_t(X, TDX_F32, order, dims, mode, U, lda, ldi, Ra, Y, s);
}

static constexpr long kModelBlocks = 2048;
// row groups of a k_cp_model launch: the most row blocks a workgroup can take (4, 2 or 1) with at
// most a sixth of them past the extent
static long model_row_waves(long I0) {
    const long nrc = ceil_div(I0, 64L);
    for (long rw = 4; rw > 1; rw /= 2)
        if (6 * (ceil_div(nrc, rw) * rw - nrc) <= nrc) return rw;
    return 1;
}
// the most workgroups such a launch has (a small one has at most 1024)
static long model_blocks(long I0) { return kModelBlocks + ceil_div(I0, 64L); }

static int fac_args(FacArgs &f, int order, const long *dims, const float *const *U, long R) {
    if (R > 256) return record(TDX_ERR_UNSUPPORTED);
    f.order = order;
    f.R = (int)R;
    for (int m = 0; m < 4; ++m) {
        f.U[m] = m < order ? U[m] : nullptr;
        f.dims[m] = m < order ? dims[m] : 1;
    }
    return TDX_OK;
}

// the model into out, or (X) its residual partials into part, one pair per block of *blocks
static int cp_model_launch(int order, const long *dims, const float *const *U, long R, float *out, const float *X,
                           double *part, int *blocks, hipStream_t s) {
    FacArgs f{};
    int st = fac_args(f, order, dims, U, R);
    if (st) return st;
    // about kModelBlocks workgroups; one row block each where that leaves compute units idle
    // (512 x 16 x 8: 9.3 us in 4 workgroups of four row blocks, 6.1 in 16 of one)
    const long ntile = ceil_div(f.dims[1] * f.dims[2] * f.dims[3], 64L), nrc = ceil_div(dims[0], 64L);
    const long rw = nrc * ntile <= device_cus() ? 1 : model_row_waves(dims[0]), nrg = ceil_div(nrc, rw);
    const long tper = std::max(1L, ceil_div(nrg * ntile, kModelBlocks));
    const int grid = (int)(nrg * ceil_div(ntile, tper));
    if (blocks) *blocks = grid;
    const int ks = R <= 16 ? 4 : R <= 32 ? 8 : R <= 48 ? 12 : 16;
    const size_t lds = sizeof(float) * kModelLd * (size_t)std::max(4L * ks, ceil_div(R, 64L) * 64L * (R > 64));
#define TDX_MODEL2(KS_, RW_, BIG_)                                                                                  \
    do {                                                                                                            \
        if (BIG_ && lds > 65536)                                                                                    \
            TDX_HIP(hipFuncSetAttribute(X ? (const void *)k_cp_model<true, KS_, RW_, BIG_>                          \
                                          : (const void *)k_cp_model<false, KS_, RW_, BIG_>,                        \
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                     \
        if (X) k_cp_model<true, KS_, RW_, BIG_><<<grid, 256, lds, s>>>(f, out, X, ntile, tper, (int)nrg, part);     \
        else k_cp_model<false, KS_, RW_, BIG_><<<grid, 256, lds, s>>>(f, out, X, ntile, tper, (int)nrg, part);      \
    } while (0)
#define TDX_MODEL(KS_, BIG_)                         \
    do {                                             \
        if (rw == 4) TDX_MODEL2(KS_, 4, BIG_);       \
        else if (rw == 2) TDX_MODEL2(KS_, 2, BIG_);  \
        else TDX_MODEL2(KS_, 1, BIG_);               \
    } while (0)
    if (R > 64) TDX_MODEL(16, true);
    else if (ks == 4) TDX_MODEL(4, false);
    else if (ks == 8) TDX_MODEL(8, false);
    else if (ks == 12) TDX_MODEL(12, false);
    else TDX_MODEL(16, false);
#undef TDX_MODEL
#undef TDX_MODEL2
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

}  // namespace tdx

using namespace tdx;

extern "C" {

int tdx_gencp(float *rec, const float *A, const float *B, const float *C, long a, long b, long c, long r) {
    TDX_CHECK_ARG(rec && A && B && C && a > 0 && b > 0 && c > 0 && r > 0);
    const long dims[3] = {a, b, c};
    const float *U[3] = {A, B, C};
    return record(cp_model_launch(3, dims, U, r, rec, nullptr, nullptr, nullptr, stream()));
}

int tdx_gencp4(float *rec, const float *A, const float *B, const float *C, const float *D, long a, long b, long c,
               long d, long r) {
    TDX_CHECK_ARG(rec && A && B && C && D && a > 0 && b > 0 && c > 0 && d > 0 && r > 0);
    const long dims[4] = {a, b, c, d};
    const float *U[4] = {A, B, C, D};
    return record(cp_model_launch(4, dims, U, r, rec, nullptr, nullptr, nullptr, stream()));
}

int tdx_cp_relerr(const void *X, int dtype, const float *scales, int order, const long *dims,
                  const float *const *factors, long rank, double *relerr) {
    TDX_CHECK_ARG(X && dims && factors && relerr && order >= 2 && order <= 4 && rank > 0);
    if (dtype != TDX_F32) return record(TDX_ERR_UNSUPPORTED);
    (void)scales;
    const long blocks = model_blocks(dims[0]);
    void *ws = nullptr;
    int st = workspace(WS_MISC0, sizeof(double) * (2 * blocks + 1), &ws);
    if (st) return st;
    double *part = (double *)ws;
    hipStream_t s = stream();
    int used = 0;
    st = cp_model_launch(order, dims, factors, rank, nullptr, (const float *)X, part, &used, s);
    if (st) return record(st);
    k_ratio<<<1, 256, 0, s>>>(part, used, part + 2 * blocks);
    TDX_LAUNCH_CHECK();
    TDX_HIP(hipMemcpyAsync(relerr, part + 2 * blocks, sizeof(double), hipMemcpyDeviceToHost, s));
    TDX_HIP(hipStreamSynchronize(s));
    return record(TDX_OK);
}

int tdx_gen_cp_tensor(float *X, int order, const long *dims, const float *const *factors, long rank, double eta,
                      uint64_t seed, uint32_t strm) {
    TDX_CHECK_ARG(X && dims && factors && order >= 2 && order <= 4 && rank > 0 && eta >= 0.0);
    const int blocks = 2048;
    void *ws = nullptr;
    int st = workspace(WS_MISC1, sizeof(double) * 2 * blocks, &ws);
    if (st) return st;
    double *part = (double *)ws;
    hipStream_t s = stream();
    long N = 1;
    for (int m = 0; m < order; ++m) N *= dims[m];
    FacArgs f{};
    st = fac_args(f, order, dims, factors, rank);
    if (st) return st;
    k_cp_fibres<<<blocks, 256, 0, s>>>(f, X, part, seed, strm);
    TDX_LAUNCH_CHECK();
    long g = ceil_div(N, 256);
    if (g > 65536) g = 65536;
    k_add_noise<<<(int)g, 256, 0, s>>>(X, N, part, blocks, eta, seed, strm);
    TDX_LAUNCH_CHECK();
    return record(TDX_OK);
}

int tdx_rse(const float *X, const float *X1, long m, float *error) {
    TDX_CHECK_ARG(X && X1 && error && m > 0);
    const int blocks = (int)std::min(2048L, ceil_div(m, 1024L));
    void *ws = nullptr;
    int st = workspace(WS_MISC0, sizeof(double) * (2 * blocks + 1), &ws);
    if (st) return st;
    double *part = (double *)ws;
    hipStream_t s = stream();
    if (((((uintptr_t)X) | ((uintptr_t)X1)) & 15) == 0) k_rse_partial<true><<<blocks, 256, 0, s>>>(X, X1, m, part);
    else k_rse_partial<false><<<blocks, 256, 0, s>>>(X, X1, m, part);
    k_ratio<<<1, 256, 0, s>>>(part, blocks, part + 2 * blocks);
    TDX_LAUNCH_CHECK();
    double r = 0.0;
    TDX_HIP(hipMemcpyAsync(&r, part + 2 * blocks, sizeof(double), hipMemcpyDeviceToHost, s));
    TDX_HIP(hipStreamSynchronize(s));
    *error = (float)r;
    return record(TDX_OK);
}

int tdx_ttm(const float *X, const float *U, float *XU, long flag, long a, long b, long c, long d) {
    TDX_CHECK_ARG(X && U && XU && a > 0 && b > 0 && c > 0 && d > 0);
    TDX_CHECK_ARG(flag >= 1 && flag <= 3);
    const long dims[3] = {a, b, c};
    // U is d x (mode size), col-major: U[p + i*d]
    return record(ttm_generic(X, 3, dims, (int)flag - 1, U, 1, d, d, XU, stream()));
}

int tdx_ttm_t(const float *X, int order, const long *dims, int mode, const float *U, long r, float *Y) {
    TDX_CHECK_ARG(X && dims && U && Y && order >= 2 && order <= 4 && mode >= 0 && mode < order && r > 0);
    return record(ttm_generic(X, order, dims, mode, U, dims[mode], 1, r, Y, stream()));
}

int tdx_ttm_ex(const void *X, int dtype, int order, const long *dims, int mode, const float *U, long r, float *Y) {
    TDX_CHECK_ARG(X && dims && U && Y && order >= 2 && order <= 4 && mode >= 0 && mode < order && r > 0);
    TDX_CHECK_ARG(dtype == TDX_F32 || dtype == TDX_BF16);
    for (int m = 0; m < order; ++m) TDX_CHECK_ARG(dims[m] > 0);
    return record(ttm_generic_t(X, dtype, order, dims, mode, U, dims[mode], 1, r, Y, stream()));
}

// Tucker reconstruction core x_1 U_1 ... x_d U_d by successive expansions
static int gentucker_n(float *rec, const float *core, const float *const *U, int order, const long *dims,
                       const long *ranks) {
    hipStream_t s = stream();
    long cur[4];
    for (int m = 0; m < order; ++m) cur[m] = ranks[m];
    // the intermediates of steps 0 .. order-2 ping-pong between two workspaces; the last
    // step writes into rec, so it does not size them
    long maxsz = 1;
    {
        long sz = 1;
        for (int m = 0; m < order; ++m) sz *= ranks[m];
        for (int m = 0; m < order - 1; ++m) {
            sz = sz / ranks[m] * dims[m];
            if (sz > maxsz) maxsz = sz;
        }
    }
    void *w0 = nullptr, *w1 = nullptr;
    int st = workspace(WS_MISC2, sizeof(float) * maxsz, &w0);
    if (st) return st;
    st = workspace(WS_MISC3, sizeof(float) * maxsz, &w1);
    if (st) return st;
    const float *src = core;
    for (int m = 0; m < order; ++m) {
        float *dst = (m == order - 1) ? rec : ((m & 1) ? (float *)w1 : (float *)w0);
        // Y[p, i, q] = sum_c U_m[i + c*I_m] * src[p, c, q]
        st = ttm_generic(src, order, cur, m, U[m], 1, dims[m], dims[m], dst, s);
        if (st) return st;
        cur[m] = dims[m];
        src = dst;
    }
    return TDX_OK;
}

int tdx_gentucker(float *rec, const float *core, const float *A, const float *B, const float *C, long a, long b,
                  long c, long r1, long r2, long r3) {
    TDX_CHECK_ARG(rec && core && A && B && C && a > 0 && b > 0 && c > 0 && r1 > 0 && r2 > 0 && r3 > 0);
    const long dims[3] = {a, b, c}, ranks[3] = {r1, r2, r3};
    const float *U[3] = {A, B, C};
    return record(gentucker_n(rec, core, U, 3, dims, ranks));
}

int tdx_gentucker4(float *rec, const float *core, const float *A, const float *B, const float *C, const float *D,
                   long a, long b, long c, long d, long r1, long r2, long r3, long r4) {
    TDX_CHECK_ARG(rec && core && A && B && C && D && a > 0 && b > 0 && c > 0 && d > 0);
    TDX_CHECK_ARG(r1 > 0 && r2 > 0 && r3 > 0 && r4 > 0);
    const long dims[4] = {a, b, c, d}, ranks[4] = {r1, r2, r3, r4};
    const float *U[4] = {A, B, C, D};
    return record(gentucker_n(rec, core, U, 4, dims, ranks));
}

}  // extern "C"
