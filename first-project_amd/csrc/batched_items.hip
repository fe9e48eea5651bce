// batched_items.hip -- batched CP-ALS with the work cut into items of equal size instead of
// tensors: an item is a run of slices X(:, :, k0 .. k1) of one tensor (8K to 48K floats), so a
// batch of uneven tensors fills the chip to the end of each pass.  Where a workgroup walked a
// whole tensor (1024 tensors on 768 workgroups, slab phases between barriers) the two passes
// over X took 620 and 865 us and the reduction of T 261 us a sweep (0.74 GB of X); these take
// 190, 200 and 54 us, the passes over X at 3.9 TB/s of it.  Bound by HBM (160 us at the 4.6 TB/s
// of a large copy) with the start and end of an item (factor blocks, the waves' sum) on top.
//
// A sweep: mode 0 partials (one pass over X), solve 0, T = X x_0 A^T with the mode-1 partials
// (the other pass), solve 1, mode 2 from T, solve 2.  A solve adds the partials of its tensor's
// items in FP64 in item order, so results do not depend on the schedule.
//
// No tile goes through LDS: a wave's MFMA operands are 16-byte loads of X along i (4 bytes
// aligned suffices), two steps in flight, and the waves of a workgroup meet only at the end.
#include "batched.hpp"
#include "linalg.hpp"
#include <algorithm>

namespace tdx {

typedef float it_f4 __attribute__((ext_vector_type(4)));
template <int N> struct ItVec;
template <> struct ItVec<1> { typedef float T; };
template <> struct ItVec<2> { typedef float T __attribute__((ext_vector_type(2), aligned(4))); };
template <> struct ItVec<4> { typedef float T __attribute__((ext_vector_type(4), aligned(4))); };
__device__ __forceinline__ float it_get(float v, int) { return v; }
template <typename V> __device__ __forceinline__ float it_get(const V &v, int i) { return v[i]; }

// ||X||^2 of an item's run, FP64 with Kahan compensation per thread (184 M floats of 1024
// tensors: 1280 us with one workgroup per tensor and one load in flight, 140 us here)
__global__ __launch_bounds__(256) void k_bi_norm2(const float *__restrict__ X, const IDesc *__restrict__ desc,
                                                  const IItem *__restrict__ items, double *__restrict__ npart) {
    __shared__ double red[4];
    const IItem it = items[blockIdx.x];
    const IDesc *d = desc + it.t;
    const long IJ = (long)d->I * d->J;
    const float *x = X + d->xoff + it.k0 * IJ;
    const int n = (int)((it.k1 - it.k0) * IJ);
    double s = 0.0, c = 0.0;
    for (int e0 = threadIdx.x; e0 < n; e0 += 8 * 256) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = x[e0 + 256 * u < n ? e0 + 256 * u : e0];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double q = e0 + 256 * u < n ? (double)v[u] : 0.0;
            const double y = q * q - c, t = s + y;
            c = (t - s) - y;
            s = t;
        }
    }
    s = bsum<256>(s, red);
    if (threadIdx.x == 0) npart[it.id] = s;
}

__global__ __launch_bounds__(256) void k_bi_norm_sum(const IDesc *__restrict__ desc, int n,
                                                     const double *__restrict__ npart, double *__restrict__ normx2) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    double s = 0.0;
    for (int k = 0; k < desc[t].nit; ++k) s += npart[desc[t].item0 + k];
    normx2[t] = s;
}

// Mode 0: M[i, r] = sum over the item's columns c = j + k J of X[i, c] B[j, r] C[k, r].  A wave
// takes every fourth step of 16 columns; lane (lm, lg) loads VEC consecutive rows from row
// 16 VEC g + VEC lm (moved back to fit the column at its end: the rows it then holds twice are
// written twice with the same value) of columns 4 u + lg, so register t of the load is the A
// operand of row tile t, rows start(m) + t.  VEC (1, 2, 4) and NG follow the extent I.
template <int VEC, int NG>
__device__ __forceinline__ void it_mode0(const float *__restrict__ x, int I, int J, int R, int k0, int k1,
                                         const float *Bs, const float *Cs, float *red, float *__restrict__ part) {
    typedef typename ItVec<VEC>::T V;
    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = k0 * J, c1 = k1 * J;
    const int mJ = (1 << 21) / J + 1;  // c / J = (c mJ) >> 21 for c < 128 J, J <= 128
    const int nstep = (c1 - c0 + 15) / 16;
    int rs[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) rs[g] = min(16 * VEC * g + VEC * lm, I - VEC);
    it_f4 acc[NG][VEC];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int t = 0; t < VEC; ++t) acc[g][t] = it_f4{0.f, 0.f, 0.f, 0.f};
    auto load = [&](V (&v)[4][NG], int st) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = min(c0 + 16 * st + 4 * u + lg, c1 - 1);
#pragma unroll
            for (int g = 0; g < NG; ++g) v[u][g] = *reinterpret_cast<const V *>(x + c * I + rs[g]);
        }
    };
    auto mul = [&](V (&v)[4][NG], int st) {
        const bool tail = c0 + 16 * st + 16 > c1;  // uniform: columns past the run count as zero
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = c0 + 16 * st + 4 * u + lg, cc = min(c, c1 - 1);
            const int k = (int)(((unsigned)cc * (unsigned)mJ) >> 21), j = cc - k * J;
            float b = Bs[j * kBMaxR + lm] * Cs[(k - k0) * kBMaxR + lm];
            if (tail) b = c < c1 ? b : 0.0f;
#pragma unroll
            for (int g = 0; g < NG; ++g)
#pragma unroll
                for (int t = 0; t < VEC; ++t) {
                    float a = it_get(v[u][g], t);
                    if (tail) a = c < c1 ? a : 0.0f;
                    acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc[g][t], 0, 0, 0);
                }
        }
    };
    V va[4][NG], vb[4][NG];
    if (wave < nstep) load(va, wave);
    for (int st = wave; st < nstep; st += 8) {
        load(vb, min(st + 4, nstep - 1));  // (every load unconditional: see next in it_mode1)
        mul(va, st);
        load(va, min(st + 8, nstep - 1));
        if (st + 4 < nstep) mul(vb, st + 4);
    }
    __syncthreads();  // the factor blocks are done with: red shares their LDS
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int t = 0; t < VEC; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = min(16 * VEC * g + VEC * (4 * lg + v), I - VEC) + t;
                red[(wave * kBMaxDim + row) * kBMaxR + lm] = acc[g][t][v];
            }
    __syncthreads();
    for (int e = tid; e < I * R; e += 256) {
        const int i = e % I, r = e / I;
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) s += red[(w * kBMaxDim + i) * kBMaxR + r];
        part[e] = s;
    }
}

__global__ __launch_bounds__(256, 3) void k_bi_mode0(const float *__restrict__ X, const float *__restrict__ U,
                                                     const IDesc *__restrict__ desc, const IItem *__restrict__ items,
                                                     float *__restrict__ part, int *__restrict__ sweep_ctr) {
    __shared__ __attribute__((aligned(16))) float lds[4 * kBMaxDim * kBMaxR];
    float *Bs = lds, *Cs = lds + kBMaxDim * kBMaxR;
    if (blockIdx.x == 0 && threadIdx.x == 0) *sweep_ctr += 1;
    const IItem it = items[blockIdx.x];
    const IDesc *d = desc + it.t;
    const int I = d->I, J = d->J, K = d->K, R = d->R;
    const float *B = U + d->uoff[1], *C = U + d->uoff[2];
    for (int e = threadIdx.x; e < J * kBMaxR; e += 256) {
        const int r = e / J, j = e % J;
        Bs[j * kBMaxR + r] = r < R ? B[j + r * J] : 0.0f;
    }
    const int nk = it.k1 - it.k0;
    for (int e = threadIdx.x; e < nk * kBMaxR; e += 256) {
        const int r = e / nk, k = e % nk;
        Cs[k * kBMaxR + r] = r < R ? C[it.k0 + k + r * K] : 0.0f;
    }
    __syncthreads();
    const float *x = X + d->xoff;
    float *p = part + it.poff;
    if (I <= 16) it_mode0<1, 1>(x, I, J, R, it.k0, it.k1, Bs, Cs, lds, p);
    else if (I <= 32) it_mode0<2, 1>(x, I, J, R, it.k0, it.k1, Bs, Cs, lds, p);
    else if (I <= 64) it_mode0<4, 1>(x, I, J, R, it.k0, it.k1, Bs, Cs, lds, p);
    else it_mode0<4, 2>(x, I, J, R, it.k0, it.k1, Bs, Cs, lds, p);
}

// Mode 1 and T: T[c, r] = sum_i X[i, c] A[i, r] (c = j + k J), M[j, r] += T[c, r] C[k, r].  A wave
// takes every fourth slice k, 16 columns j a tile; lane (lm, lg) loads 4 consecutive i of column
// lm from i = 16 q + 4 lg (moved back to fit the column; an i already counted by another lane
// has weight zero), and A's rows for them stay in registers for the whole item.  The finished
// tile goes to T and, times C[k], into the wave's part of M in LDS.
template <int NQ>
__device__ __forceinline__ void it_mode1(const float *__restrict__ x, const float *__restrict__ A, int I, int J,
                                         int R, int Rq, int k0, int k1, const float *Cs, float *Mw,
                                         float *__restrict__ T, float *__restrict__ part) {
    typedef typename ItVec<4>::T V;
    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int NJ = (J + 15) / 16;
    int is[NQ];
    uint32_t counted = 0;
    it_f4 aop[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        is[q] = max(min(16 * q + 4 * lg, I - 4), 0);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int i = is[q] + s;
            const bool on = i >= 16 * q + 4 * lg && i < I;
            counted |= (uint32_t)on << (4 * q + s);
            aop[q][s] = on && lm < R ? A[i + lm * I] : 0.0f;
        }
    }
    it_f4 *mw = reinterpret_cast<it_f4 *>(Mw) + wave * (kBMaxDim / 16) * 64 + lane;
    for (int jt = 0; jt < NJ; ++jt) mw[jt * 64] = it_f4{0.f, 0.f, 0.f, 0.f};
    const int ntile = (k1 - k0 - wave + 3) / 4 * NJ;  // of this wave (k1 - k0 >= 1)
    auto load = [&](V (&v)[NQ], int k, int jt) {
        const float *p = x + (k * J + min(16 * jt + lm, J - 1)) * I;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            if (NQ == 2 && I < 4) {
#pragma unroll
                for (int s = 0; s < 4; ++s) v[q][s] = p[min(s, I - 1)];
            } else {
                v[q] = *reinterpret_cast<const V *>(p + is[q]);
            }
        }
    };
    auto mul = [&](V (&v)[NQ], int k, int jt) {
        it_f4 t0 = {0.f, 0.f, 0.f, 0.f}, t1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const float a = (counted >> (4 * q + s)) & 1u ? v[q][s] : 0.0f;
                if (s & 1) t1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, aop[q][s], t1, 0, 0, 0);
                else t0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a, aop[q][s], t0, 0, 0, 0);
            }
        t0 += t1;
        const float cv = Cs[(k - k0) * kBMaxR + lm];
        mw[jt * 64] += t0 * cv;
        if (lm < Rq) {
            float *tp = T + ((long)k * J + 16 * jt + 4 * lg) * Rq + lm;
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (16 * jt + 4 * lg + u < J) tp[u * Rq] = t0[u];
        }
    };
    // tiles in order (k, jt), two register buffers; past the last tile the last one is reloaded
    // (a load issued on some paths only makes the compiler's wait counting drain the queue)
    int kf = k0 + wave, jf = 0, left = ntile;
    auto next = [&](V (&v)[NQ]) {
        load(v, kf, jf);
        if (left > 1) {
            --left;
            if (++jf == NJ) {
                jf = 0;
                kf += 4;
            }
        }
    };
    V va[NQ], vb[NQ];
    if (ntile > 0) {
        int k = k0 + wave, jt = 0;
        auto step = [&]() {
            if (++jt == NJ) {
                jt = 0;
                k += 4;
            }
        };
        next(va);
        for (int p = 0; p < ntile; p += 2) {
            next(vb);
            mul(va, k, jt);
            step();
            next(va);
            if (p + 1 < ntile) mul(vb, k, jt);
            step();
        }
    }
    __syncthreads();
    // register v of lane (lm, lg) of tile jt: row 16 jt + 4 lg + v, column lm
    for (int e = tid; e < J * R; e += 256) {
        const int j = e % J, r = e / J;
        const int at = ((j >> 4) * 64 + ((j >> 2) & 3) * 16 + r) * 4 + (j & 3);
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) s += Mw[w * (kBMaxDim / 16) * 256 + at];
        part[e] = s;
    }
}

__global__ __launch_bounds__(256, 3) void k_bi_mode1(const float *__restrict__ X, const float *__restrict__ U,
                                                     const IDesc *__restrict__ desc, const IItem *__restrict__ items,
                                                     float *__restrict__ part, float *__restrict__ T) {
    __shared__ __attribute__((aligned(16))) float Mw[4 * kBMaxDim * kBMaxR];
    __shared__ float Cs[kBMaxDim * kBMaxR];
    const IItem it = items[blockIdx.x];
    const IDesc *d = desc + it.t;
    const int I = d->I, J = d->J, K = d->K, R = d->R, Rq = d->Rq;
    const float *A = U + d->uoff[0], *C = U + d->uoff[2];
    const int nk = it.k1 - it.k0;
    for (int e = threadIdx.x; e < nk * kBMaxR; e += 256) {
        const int r = e / nk, k = e % nk;
        Cs[k * kBMaxR + r] = r < R ? C[it.k0 + k + r * K] : 0.0f;
    }
    __syncthreads();
    const float *x = X + d->xoff;
    float *p = part + it.poff, *t = T + d->toff;
    if (I <= 32) it_mode1<2>(x, A, I, J, R, Rq, it.k0, it.k1, Cs, Mw, t, p);
    else if (I <= 64) it_mode1<4>(x, A, I, J, R, Rq, it.k0, it.k1, Cs, Mw, t, p);
    else if (I <= 96) it_mode1<6>(x, A, I, J, R, Rq, it.k0, it.k1, Cs, Mw, t, p);
    else it_mode1<8>(x, A, I, J, R, Rq, it.k0, it.k1, Cs, Mw, t, p);
}

// Mode 2 from T: M[k, r] = sum_j T[j + k J, r] B[j, r] for the item's k, complete (no partial):
// a wave per k, a lane per (j, four columns), then the lanes of equal columns are added.
__global__ __launch_bounds__(256) void k_bi_mode2(const float *__restrict__ U, const float *__restrict__ T,
                                                  const IDesc *__restrict__ desc, const IItem *__restrict__ items,
                                                  float *__restrict__ part) {
    __shared__ __attribute__((aligned(16))) float Bs[kBMaxDim * kBMaxR];
    const IItem it = items[blockIdx.x];
    const IDesc *d = desc + it.t;
    const int J = d->J, R = d->R, Rq = d->Rq, nq = Rq / 4, kc = d->kc;
    const float *B = U + d->uoff[1];
    for (int e = threadIdx.x; e < J * kBMaxR; e += 256) {
        const int r = e / J, j = e % J;
        Bs[j * kBMaxR + r] = r < R ? B[j + r * J] : 0.0f;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rq = lane & (nq - 1), n = J * nq, sq = nq >> 1;  // nq = 1, 2, 4: sq its logarithm
    for (int k = it.k0 + wave; k < it.k1; k += 4) {
        const it_f4 *tp = reinterpret_cast<const it_f4 *>(T + d->toff) + (long)k * n;
        it_f4 v[8], s = {0.f, 0.f, 0.f, 0.f};  // n <= 512: eight loads in flight
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (64 * u < n) v[u] = tp[min(lane + 64 * u, n - 1)];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (64 * u < n) {
                const int x = lane + 64 * u;
                if (x < n) s += v[u] * *reinterpret_cast<const it_f4 *>(Bs + (x >> sq) * kBMaxR + 4 * rq);
            }
        for (int o = 32; o >= nq; o >>= 1)
#pragma unroll
            for (int q = 0; q < 4; ++q) s[q] += __shfl_xor(s[q], o, 64);
        if (lane < nq)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (4 * rq + q < R) part[it.poff + (k - it.k0) + (4 * rq + q) * kc] = s[q];
    }
}

// U_n = M V^{-1}, G_n = U_n^T U_n and, after mode 2, the fit: one workgroup per tensor.  M is the
// FP64 sum of the items' partials in item order (mode 2: every item holds its own rows).
template <int MODE>
__global__ __launch_bounds__(256) void k_bi_solve(float *__restrict__ U, const float *__restrict__ part,
                                                  double *__restrict__ G, const IDesc *__restrict__ desc,
                                                  const double *__restrict__ normx2, double *__restrict__ fit_hist,
                                                  int max_sweeps, const int *__restrict__ sweep_ctr,
                                                  int *__restrict__ status) {
    constexpr int BS = 256, RR16 = kBMaxR * kBMaxR;
    __shared__ double Ms[kBMaxDim * kBMaxR];
    __shared__ float Un[kBMaxDim * kBMaxR];
    __shared__ double V[RR16], L[RR16], W[RR16], Vi[RR16];
    __shared__ double sh[BS], cs[4 * (kBMaxR / 2 + 1)];
    __shared__ double red[BS / 64];
    __shared__ int fail;
    const int tid = threadIdx.x, t = blockIdx.x;
    const int sweep = *sweep_ctr;
    const IDesc *d = desc + t;
    const int R = d->R, In = sel3(MODE, d->I, d->J, d->K), nit = d->nit, kc = d->kc, pstep = d->pstep;
    const long uon = d->uoff[MODE];
    const float *p = part + d->pbase;
    double *Gt = G + (long)t * 3 * RR16;
    for (int e = tid; e < In * R; e += BS) {
        if constexpr (MODE == 2) {
            const int k = e % In, b = e / In, q = k / kc;
            Ms[e] = (double)p[(long)q * pstep + (k - q * kc) + b * kc];
        } else {
            double s = 0.0;
            for (int q = 0; q < nit; q += 8) {
                float v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = p[(long)min(q + u, nit - 1) * pstep + e];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (q + u < nit) s += (double)v[u];
            }
            Ms[e] = s;
        }
    }
    for (int e = tid; e < R * R; e += BS) {
        double v = 1.0;
#pragma unroll
        for (int m = 0; m < 3; ++m)
            if (m != MODE) v *= Gt[m * RR16 + e];
        V[e] = v;
    }
    __syncthreads();
    if (block_spd_inverse<1>(V, L, W, Vi, R, cs, sh, &fail) && tid == 0) atomicOr(status, 1);
    double ip = 0.0;
    for (int e = tid; e < In * R; e += BS) {
        const int i = e % In, b = e / In;
        double s = 0.0;
        for (int a = 0; a < R; ++a) s += Ms[i + a * In] * Vi[a + b * R];
        const float u = (float)s;
        Un[e] = u;
        U[uon + e] = u;
        ip += Ms[e] * (double)u;
    }
    __syncthreads();
    double ip_last = 0.0;
    if (MODE == 2) ip_last = bsum<BS>(ip, red);
    double hx = 0.0;
    for (int e = tid; e < R * R; e += BS) {
        const int a = e % R, b = e / R;
        double s = 0.0;
        for (int i = 0; i < In; ++i) s += (double)Un[i + a * In] * (double)Un[i + b * In];
        Gt[MODE * RR16 + e] = s;
        if (MODE == 2) hx += Gt[e] * Gt[RR16 + e] * s;
    }
    if (MODE == 2) {
        hx = bsum<BS>(hx, red);
        if (tid == 0 && sweep < max_sweeps) {
            const double nx2 = normx2[t];
            fit_hist[(long)t * max_sweeps + sweep] = sqrt(fabs(nx2 - 2.0 * ip_last + hx) / nx2);
        }
    }
}

// Grams of the initial factors, a workgroup per (tensor, mode)
__global__ __launch_bounds__(256) void k_bi_gram(const float *__restrict__ U, const IDesc *__restrict__ desc,
                                                 double *__restrict__ G) {
    __shared__ float Us[kBMaxDim * kBMaxR];
    const int t = blockIdx.x, m = blockIdx.y;
    const IDesc *d = desc + t;
    const int R = d->R, Im = sel3(m, d->I, d->J, d->K);
    for (int e = threadIdx.x; e < Im * R; e += 256) Us[e] = U[d->uoff[m] + e];
    __syncthreads();
    for (int e = threadIdx.x; e < R * R; e += 256) {
        const int a = e % R, b = e / R;
        double s = 0.0;
        for (int i = 0; i < Im; ++i) s += (double)Us[i + a * Im] * (double)Us[i + b * Im];
        G[((long)t * 3 + m) * (kBMaxR * kBMaxR) + e] = s;
    }
}

// Items of about total / (16 per CU) floats, 8K to 48K: short enough that the last ones end
// together, long enough that a partial (I R floats) is a few percent of the run it sums.
// Whole slices, a multiple of the workgroup's four waves where a tensor has as many.
void items_plan(ItemPlan &p, const BDesc *d, long n) {
    long total = 0;
    for (long t = 0; t < n; ++t) total += (long)d[t].I * d[t].J * d[t].K;
    const long target = std::max(8192L, std::min(49152L, total / (16L * device_cus())));
    p.desc.resize(n);
    for (long t = 0; t < n; ++t) {
        IDesc &q = p.desc[t];
        q.I = d[t].I, q.J = d[t].J, q.K = d[t].K, q.R = d[t].R;
        q.xoff = d[t].xoff;
        for (int m = 0; m < 3; ++m) q.uoff[m] = d[t].uoff[m];
        q.Rq = q.R <= 4 ? 4 : q.R <= 8 ? 8 : 16;
        const long slice = (long)q.I * q.J;
        q.kc = (int)std::min<long>(q.K, std::max(4L, target / slice / 4 * 4));
        q.nit = (int)ceil_div((long)q.K, (long)q.kc);
        q.pstep = (std::max(std::max(q.I, q.J), q.kc) * q.R + 3) / 4 * 4;
        q.pbase = p.part_floats;
        q.toff = p.t_floats;
        q.item0 = (int)p.items.size();
        for (int k = 0; k < q.nit; ++k) {
            IItem it;
            it.t = (int)t;
            it.k0 = k * q.kc;
            it.k1 = std::min(q.K, it.k0 + q.kc);
            it.id = (int)p.items.size();
            it.poff = p.part_floats + (long)k * q.pstep;
            p.items.push_back(it);
        }
        p.part_floats += (long)q.nit * q.pstep;
        p.t_floats += (long)q.J * q.K * q.Rq;
    }
    // largest first, in 64 classes of size (a comparison sort of the 4-5 thousand items of 1024 tensors
    // took 0.2 ms)
    constexpr int kClasses = 64;
    long most = 1;
    auto size = [&](const IItem &a) { return (long)(a.k1 - a.k0) * p.desc[a.t].I * p.desc[a.t].J; };
    for (const IItem &a : p.items) most = std::max(most, size(a));
    auto cls = [&](const IItem &a) { return kClasses - 1 - (int)(size(a) * (kClasses - 1) / most); };
    size_t at[kClasses + 1] = {0};
    for (const IItem &a : p.items) ++at[cls(a) + 1];
    for (int c = 0; c < kClasses; ++c) at[c + 1] += at[c];
    std::vector<IItem> sorted(p.items.size());
    for (const IItem &a : p.items) sorted[at[cls(a)]++] = a;
    p.items.swap(sorted);
}

int items_prologue(const ItemBuffers &b, const float *X, const float *U, double *normx2, hipStream_t s) {
    k_bi_norm2<<<b.nitems, 256, 0, s>>>(X, b.desc, b.items, b.npart);
    k_bi_norm_sum<<<(int)ceil_div((long)b.ntensors, 256L), 256, 0, s>>>(b.desc, b.ntensors, b.npart, normx2);
    k_bi_gram<<<dim3((unsigned)b.ntensors, 3u), 256, 0, s>>>(U, b.desc, b.G);
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

int items_sweep(const ItemBuffers &b, const float *X, float *U, const double *normx2, double *fit, int max_sweeps,
                int *sweep_ctr, int *status, hipStream_t s) {
    const int n = b.ntensors;
    k_bi_mode0<<<b.nitems, 256, 0, s>>>(X, U, b.desc, b.items, b.part, sweep_ctr);
    k_bi_solve<0><<<n, 256, 0, s>>>(U, b.part, b.G, b.desc, normx2, fit, max_sweeps, sweep_ctr, status);
    k_bi_mode1<<<b.nitems, 256, 0, s>>>(X, U, b.desc, b.items, b.part, b.T);
    k_bi_solve<1><<<n, 256, 0, s>>>(U, b.part, b.G, b.desc, normx2, fit, max_sweeps, sweep_ctr, status);
    k_bi_mode2<<<b.nitems, 256, 0, s>>>(U, b.T, b.desc, b.items, b.part);
    k_bi_solve<2><<<n, 256, 0, s>>>(U, b.part, b.G, b.desc, normx2, fit, max_sweeps, sweep_ctr, status);
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

}  // namespace tdx
