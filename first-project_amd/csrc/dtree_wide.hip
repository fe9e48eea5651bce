// dtree_wide.hip -- the shared pass of an order-3 CP-ALS sweep for the tensors whose products are not
// rounded to one BF16 part: FP32 storage (three parts of X and of A) and the opening sweeps' BF16
// storage with hi + lo coefficients.  As in dtree.hip
//   T[i2][i1][r] = sum_{i0} X[i0, i1, i2] A[i0][r],  M1[i1][r] = sum_{i2} T C,  M2[i2][r] = sum_{i1} T B
// with one pass over X (k_tw_m1) and one over T (k_tw_m2), but T stays FP32.
//
// k_tw_m1: a workgroup of 8 waves owns 256 rows i1, a wave 32 of them, and a range of i2.  A chunk of
// 256 bytes along i0 (64 FP32 or 128 BF16 elements) of two slabs i2 is multiplied with the chunk's
// panel parts, which do not fit in LDS for all of I0 (384 KB at I0 = 1024, 64 columns): they are cut
// once a sweep (k_tw_parts) in operand order and staged chunk by chunk in two buffers, 24 KB for the
// 128 KB of X that share them, one barrier a chunk.  A tile goes from 16-byte loads of whole lines
// through the wave's part of LDS (rows of 272 bytes) into operand order while the next one is in
// flight, as in mttkrp_f32.hip, whose exact three-part FP32 products, whose FP32 way for tiles with
// infinities or values near the largest and whose halves for small entries are used here too.  The 64-term sums enter the FP32
// tile of T once; a finished tile is stored as the lanes hold it (1 KB a store) and, times C, added to
// the mode-1 partial.
// Bound by power and HBM as the MTTKRP kernels it replaces.  1024^3 rank 64: FP32 955 us (4.8 TB/s of X
// and T) and 47 for the pass over T, where modes 1 and 2 took 978 each; split BF16 444 (5.4 TB/s) and
// 47, where they took 409 each.  The parts take 13 us beside the inverse's 26.
//   * A's columns are scaled by a power of two to a largest entry in [1, 2), undone in C and B, so T
//     neither overflows nor loses bits where the factors' magnitudes are uneven.
#include "mttkrp.hpp"
#include "vinv.hpp"
#include <algorithm>

namespace tdx {

typedef float tw_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 tw_b8 __attribute__((ext_vector_type(8)));
typedef uint32_t tw_u4 __attribute__((ext_vector_type(4)));

static constexpr int kTwLd = 68;                 // floats per LDS row of a tile
static constexpr int kTwTile = 32 * kTwLd;       // floats of a wave's tile
static constexpr int kTwWaves = 8, kTwRows = 32 * kTwWaves;

// ST 0: FP32, 1: BF16.  KSN: k-steps of 32 a chunk, NP: parts of a coefficient
template <int ST> struct TwSt;
template <> struct TwSt<0> { static constexpr int KSN = 2, NP = 3; };
template <> struct TwSt<1> { static constexpr int KSN = 4, NP = 2; };

struct TwArgs {
    const void *X;
    const float *panelA, *panelC;
    const uint4 *parts;   // [chunk][k-step][part][column block][lane]
    const float *scale;   // Rp powers of two, then a flag: the panel holds an infinity
    float *T, *partial;
    long I0, I1, I2;
    int blocks_i1, i2per;
};

// 8 values -> NP parts, each what is left rounded to BF16
template <int NP>
__device__ __forceinline__ void tw_split(const tw_f4 &a, const tw_f4 &b, uint4 (&o)[NP]) {
    float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
#pragma unroll
    for (int k = 0; k < NP; ++k) {
        uint32_t w[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            w[h] = bf16_pair(v[2 * h], v[2 * h + 1]);
            v[2 * h] -= __uint_as_float(w[h] << 16);
            v[2 * h + 1] -= __uint_as_float(w[h] & 0xffff0000u);
        }
        o[k] = uint4{w[0], w[1], w[2], w[3]};
    }
}
__device__ __forceinline__ tw_b8 tw_op(const uint4 &v) { return __builtin_bit_cast(tw_b8, v); }

// The parts of the mode-0 panel, a workgroup a chunk of 32 KSN rows, and, as the first workgroup, mode
// 1's inverse (13 and 26 us at 1024 x 64 one after the other).  Every workgroup finds the columns'
// largest magnitudes itself (the panel is 256 KB at I0 = 1024).
template <int KSN, int NP, int NS>
__global__ __launch_bounds__(256) void k_tw_parts(const float *__restrict__ panel, long I0, int Rp,
                                                  uint4 *__restrict__ parts, float *__restrict__ scale, VinvJob j) {
    if (blockIdx.x == 0) {
        vinv_job<NS>(j);
        return;
    }
    __shared__ float mx[256], sc[64];
    const long chunk = (long)blockIdx.x - 1;
    const int tid = threadIdx.x, nb = Rp / 16, ng = 256 / Rp;
    const long nrow8 = (I0 + 7) / 8;
    float m = 0.0f;
    if (tid < ng * Rp) {
        const int c = tid % Rp;
        for (long i = tid / Rp; i < nrow8; i += ng) {
            const tw_f4 *p = reinterpret_cast<const tw_f4 *>(panel + (i * Rp + c) * 8);
            const tw_f4 u = p[0], v = p[1];
#pragma unroll
            for (int q = 0; q < 4; ++q) m = fmaxf(m, fmaxf(fabsf(u[q]), fabsf(v[q])));  // (NaN left out)
        }
    }
    mx[tid] = m;
    const bool inf = __syncthreads_or(m == __uint_as_float(0x7f800000u)) != 0;
    if (tid < Rp) {
        for (int g = 1; g < ng; ++g) m = fmaxf(m, mx[g * Rp + tid]);
        int x = (int)(__float_as_uint(m) >> 23) - 127;
        x = x == 128 ? 0 : x > 126 ? 126 : x < -126 ? -126 : x;  // (2^-x has no normal value at the ends)
        sc[tid] = __uint_as_float((uint32_t)(127 - x) << 23);
        if (chunk == 0) scale[tid] = __uint_as_float((uint32_t)(127 + x) << 23);
        if (chunk == 0 && tid == 0) scale[Rp] = inf ? 1.0f : 0.0f;
    }
    __syncthreads();
    for (int e = tid; e < KSN * nb * 64; e += 256) {
        const int lane = e & 63, b = (e >> 6) % nb, ks = (e >> 6) / nb, c = 16 * b + (lane & 15);
        const long i = chunk * 32 * KSN + 32 * ks + 8 * (lane >> 4);
        tw_f4 u = {0.f, 0.f, 0.f, 0.f}, v = u;
        if (i < I0) {  // (rows past I0 within the panel's groups of 8 are zero)
            const tw_f4 *p = reinterpret_cast<const tw_f4 *>(panel + ((i >> 3) * Rp + c) * 8);
            u = p[0] * sc[c], v = p[1] * sc[c];
        }
        uint4 o[NP];
        tw_split<NP>(u, v, o);
#pragma unroll
        for (int k = 0; k < NP; ++k) parts[((chunk * KSN + ks) * NP + k) * nb * 64 + b * 64 + lane] = o[k];
    }
}

template <int ST, int NB>
__global__ __launch_bounds__(64 * kTwWaves, 1) void k_tw_m1(TwArgs a) {
    constexpr int KSN = TwSt<ST>::KSN, NP = TwSt<ST>::NP, Rp = 16 * NB;
    constexpr int PC = KSN * NP * NB * 64, NPL = (PC + 511) / 512;  // 16-byte operands a chunk, a thread
    constexpr int EV = ST == 0 ? 4 : 8, ES = ST == 0 ? 4 : 2;       // elements a load, bytes an element
    extern __shared__ __align__(16) unsigned char tw_lds[];
    uint4 *ps = reinterpret_cast<uint4 *>(tw_lds);  // two buffers of PC
    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float *xs = reinterpret_cast<float *>(ps + 2 * PC) + wave * kTwTile;
    const int bi = blockIdx.x % a.blocks_i1, split = blockIdx.x / a.blocks_i1;
    const long I0 = a.I0, I1 = a.I1;
    const long i2s = (long)split * a.i2per, i2e = min(i2s + a.i2per, a.I2);
    const long row0 = (long)bi * kTwRows + 32 * wave;
    const int nfc = (int)((I0 + 32 * KSN - 1) / (32 * KSN));
    const bool act = row0 < I1;  // a wave past the rows only helps staging the panel
    const long ntile = (I1 + 31) / 32;

    // this lane's rows (lane / 16) + 4 u; past the extent the last row again (its T rows meet zero
    // coefficients, its partial rows are not read)
    const long rb0 = min(row0, I1 - 1);
    uint32_t ro[8];  // byte offsets from row rb0 (I0 < 2^24)
#pragma unroll
    for (int u = 0; u < 8; ++u) ro[u] = (uint32_t)(min(row0 + (lane >> 4) + 4 * u, I1 - 1) - rb0) * (uint32_t)(I0 * ES);
    float sc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) sc[nb] = a.scale[16 * nb + lm];
    const bool pinf = ST == 0 && a.scale[Rp] != 0.0f;

    // tiles in order (pair of slabs, chunk, slab of the pair); past the last one it is repeated
    long li2 = i2s;
    int lfc = 0, lj = 0;
    uint4 xv[8];
    auto load = [&]() {
        const long i2 = min(li2 + lj, i2e - 1);
        const long f0 = (long)lfc * (32 * KSN);
        const char *p = (const char *)a.X + ((i2 * I1 + rb0) * I0 + f0) * ES;
        const uint32_t fl = (uint32_t)min((long)(EV * (lane & 15)), I0 - EV - f0) * ES;
#pragma unroll
        for (int u = 0; u < 8; ++u) xv[u] = ld_stream(reinterpret_cast<const uint4 *>(p + (ro[u] + fl)));
        if (++lj == 2) {
            lj = 0;
            if (++lfc == nfc) {
                lfc = 0;
                if (li2 + 2 < i2e) li2 += 2;
            }
        }
    };
    tw_u4 pl[NPL];
    auto load_parts = [&](int fc) {
#pragma unroll
        for (int q = 0; q < NPL; ++q) pl[q] = reinterpret_cast<const tw_u4 *>(a.parts)[(long)fc * PC + min(tid + 512 * q, PC - 1)];
    };
    auto store_parts = [&](int buf) {
#pragma unroll
        for (int q = 0; q < NPL; ++q)
            if (PC % 512 == 0 || tid + 512 * q < PC) reinterpret_cast<tw_u4 *>(ps)[buf * PC + tid + 512 * q] = pl[q];
    };

    tw_f4 acc[2][2][NB], m1[2][NB];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) m1[rb][nb] = tw_f4{0.f, 0.f, 0.f, 0.f};

    // one tile: through LDS into operand order, the next one's loads, the products
    auto step = [&](tw_f4 (&ac)[2][NB], const uint4 *pb, int fc) {
        bool fp32 = false, halves = false;  // (as in mttkrp_f32.hip)
        if constexpr (ST == 0) {
            float big = 0.0f, least = __uint_as_float(0x7f800000u);  // magnitudes (NaN left out)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(big) : "v"(xv[u].x), "v"(xv[u].y));
                asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(big) : "v"(xv[u].z), "v"(xv[u].w));
                asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(least) : "v"(xv[u].x), "v"(xv[u].y));
                asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(least) : "v"(xv[u].z), "v"(xv[u].w));
            }
            if (pinf || __any(big > 0x1p119f || least < 0x1p-100f)) {
                fp32 = pinf || __any(big > 0x1p119f);
                uint32_t key = ~0u;
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    key = min(key, min(min(small_key(__uint_as_float(xv[u].x)), small_key(__uint_as_float(xv[u].y))),
                                       min(small_key(__uint_as_float(xv[u].z)), small_key(__uint_as_float(xv[u].w)))));
                halves = __any(key < kSmallKey);
            }
        }
        const bool in = fc * (32 * KSN) + EV * (lane & 15) < I0;
        if ((fc + 1) * (32 * KSN) > I0) {
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (!in) xv[u] = uint4{0u, 0u, 0u, 0u};
        }
        // (a wave's LDS operations complete in order: no barrier between its stores and loads)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < 8; ++u)
            *reinterpret_cast<uint4 *>(xs + ((lane >> 4) + 4 * u) * kTwLd + 4 * (lane & 15)) = xv[u];
        __builtin_amdgcn_wave_barrier();
        load();
        __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the MFMAs
        if constexpr (ST == 0) {
            if (fp32) {
                // FP32 products
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const float si = 1.0f / sc[nb];
#pragma unroll
                    for (int rb = 0; rb < 2; ++rb) {
                        tw_f4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                        for (int q = 0; q < 4; ++q) {
                            const tw_f4 av =
                                *reinterpret_cast<const tw_f4 *>(xs + (16 * rb + lm) * kTwLd + 16 * q + 4 * lg);
                            const long i = 64L * fc + 16 * q + 4 * lg;
                            const tw_f4 bv = *reinterpret_cast<const tw_f4 *>(
                                a.panelA + ((i >> 3) * Rp + 16 * nb + lm) * 8 + (i & 7));
#pragma unroll
                            for (int c = 0; c < 4; ++c)
                                t = __builtin_amdgcn_mfma_f32_16x16x4f32(av[c], si * bv[c], t, 0, 0, 0);
                        }
                        ac[rb][nb] += t;
                        asm volatile("" : "+v"(ac[rb][nb]));  // (added before any branch, as below)
                    }
                }
                return;
            }
            auto split_row = [&](int rb, int ks, uint4 (&x)[3], auto value) {
                const float *p = xs + (16 * rb + lm) * kTwLd + 32 * ks + 8 * lg;
                tw_f4 u = *reinterpret_cast<const tw_f4 *>(p), v = *reinterpret_cast<const tw_f4 *>(p + 4);
#pragma unroll
                for (int c = 0; c < 4; ++c) u[c] = value(u[c]), v[c] = value(v[c]);
                tw_split<3>(u, v, x);
            };
            // s + the products, smallest terms first
            auto products = [&](const uint4 (&x)[3], const uint4 (&p)[3], tw_f4 s) {
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tw_op(x[2]), tw_op(p[0]), s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tw_op(x[0]), tw_op(p[2]), s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tw_op(x[1]), tw_op(p[1]), s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tw_op(x[1]), tw_op(p[0]), s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tw_op(x[0]), tw_op(p[1]), s, 0, 0, 0);
                return __builtin_amdgcn_mfma_f32_16x16x32_bf16(tw_op(x[0]), tw_op(p[0]), s, 0, 0, 0);
            };
            if (halves) {
#pragma unroll 1
                for (int h = 0; h < 4; ++h) {
                    const int ks = h & 1, half = h >> 1;
                    uint4 x[2][3];
#pragma unroll
                    for (int rb = 0; rb < 2; ++rb)
                        split_row(rb, ks, x[rb], [&](float v) { return magnitude_half(v, half); });
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        uint4 p[3];
#pragma unroll
                        for (int k = 0; k < 3; ++k) p[k] = pb[((ks * 3 + k) * NB + nb) * 64 + lane];
#pragma unroll
                        for (int rb = 0; rb < 2; ++rb) {
                            const tw_f4 s = products(x[rb], p, tw_f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                            for (int v = 0; v < 4; ++v) ac[rb][nb][v] = fmaf(s[v], half ? 0x1p-64f : 1.0f, ac[rb][nb][v]);
                            asm volatile("" : "+v"(ac[rb][nb]));
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                return;
            }
            tw_f4 t[2][NB];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                uint4 x[2][3];
#pragma unroll
                for (int rb = 0; rb < 2; ++rb) split_row(rb, ks, x[rb], [](float v) { return v; });
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    uint4 p[3];
#pragma unroll
                    for (int k = 0; k < 3; ++k) p[k] = pb[((ks * 3 + k) * NB + nb) * 64 + lane];
#pragma unroll
                    for (int rb = 0; rb < 2; ++rb)
                        t[rb][nb] = products(x[rb], p, ks == 0 ? tw_f4{0.f, 0.f, 0.f, 0.f} : t[rb][nb]);
                }
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int rb = 0; rb < 2; ++rb) {
                    ac[rb][nb] += t[rb][nb];
                    asm volatile("" : "+v"(ac[rb][nb]));
                }
        } else {
#pragma unroll
            for (int ks = 0; ks < KSN; ++ks) {
                uint4 x[2];
#pragma unroll
                for (int rb = 0; rb < 2; ++rb)
                    x[rb] = *reinterpret_cast<const uint4 *>(xs + (16 * rb + lm) * kTwLd + 16 * ks + 4 * lg);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const uint4 hi = pb[((ks * 2 + 0) * NB + nb) * 64 + lane], lo = pb[((ks * 2 + 1) * NB + nb) * 64 + lane];
#pragma unroll
                    for (int rb = 0; rb < 2; ++rb) {
                        ac[rb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tw_op(x[rb]), tw_op(lo), ac[rb][nb], 0, 0, 0);
                        ac[rb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tw_op(x[rb]), tw_op(hi), ac[rb][nb], 0, 0, 0);
                    }
                }
            }
        }
    };

    load_parts(0);
    load();
    store_parts(0);
    __syncthreads();
    int buf = 0;
    for (long i2 = i2s; i2 < i2e; i2 += 2) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[j][rb][nb] = tw_f4{0.f, 0.f, 0.f, 0.f};
        for (int fc = 0; fc < nfc; ++fc) {
            load_parts(fc + 1 < nfc ? fc + 1 : 0);
            __builtin_amdgcn_sched_barrier(0);
            if (act) {
                step(acc[0], ps + buf * PC, fc);
                step(acc[1], ps + buf * PC, fc);
            }
            buf ^= 1;
            store_parts(buf);  // (read last before the previous barrier)
            __syncthreads();
        }
        // (C's rows only now: held over the chunks, they spilled)
        float cv[2][NB];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const long k = min(i2 + j, i2e - 1);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) cv[j][nb] = a.panelC[((k >> 3) * Rp + 16 * nb + lm) * 8 + (k & 7)];
        }
        // (hipcc has left out wait states before the first read of a matrix result behind a branch)
        asm volatile("s_nop 15");
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) asm volatile("" : "+v"(acc[j][rb][nb]));
        if (act)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                if (i2 + j < i2e) {
                    tw_f4 *tp = reinterpret_cast<tw_f4 *>(a.T) + ((i2 + j) * ntile + row0 / 32) * (2 * NB * 64) + lane;
#pragma unroll
                    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb) {
                            tp[(rb * NB + nb) * 64] = acc[j][rb][nb];
                            const float w = cv[j][nb] * sc[nb];
#pragma unroll
                            for (int v = 0; v < 4; ++v) m1[rb][nb][v] = fmaf(acc[j][rb][nb][v], w, m1[rb][nb][v]);
                        }
                }
    }
    // register v of lane (lm, lg): row 16 rb + 4 lg + v, column 16 nb + lm
    float *dst = a.partial + ((long)split * a.blocks_i1 * kTwRows + row0) * Rp;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) dst[(16 * rb + 4 * lg + v) * Rp + 16 * nb + lm] = m1[rb][nb][v];
}

// Mode 2 from T, with the mode's inverse as the first workgroup (as in dtree.hip): a wave takes two
// slabs i2 and tper tiles of 32 rows i1; lane (lm, lg) multiplies its four rows of a 16 x 16 block by
// B's, read once for both slabs, and the lane groups are added at the end.
template <int NB, int NS>
__global__ __launch_bounds__(256) void k_tw_m2(const float *__restrict__ T, const float *__restrict__ panelB,
                                               const float *__restrict__ scale, float *__restrict__ partial, long I1,
                                               long I2, int tper, int nb2, VinvJob j) {
    if (blockIdx.x == 0) {
        vinv_job<NS>(j);
        return;
    }
    constexpr int Rp = 16 * NB;
    const int blk = (int)blockIdx.x - 1, lane = threadIdx.x & 63, lm = lane & 15, lg = lane >> 4, wave = threadIdx.x >> 6;
    const int split = blk / nb2;
    const long i2 = 2 * (4L * (blk % nb2) + wave);
    if (i2 >= I2) return;
    const long ntile = (I1 + 31) / 32, t0 = (long)split * tper, t1 = min(t0 + tper, ntile);
    const tw_f4 *tp0 = reinterpret_cast<const tw_f4 *>(T) + i2 * ntile * (2 * NB * 64) + lane;
    const tw_f4 *tp1 = i2 + 1 < I2 ? tp0 + ntile * (2 * NB * 64) : tp0;
    float sc[NB], s0[NB], s1[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) sc[nb] = scale[16 * nb + lm], s0[nb] = s1[nb] = 0.0f;
    for (long t = t0; t < t1; ++t)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            tw_f4 u[NB], w[NB], b[NB];
            const long i = 32 * t + 16 * rb + 4 * lg;  // (the panel's rows are padded with zeros)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                u[nb] = tp0[(t * 2 + rb) * NB * 64 + nb * 64];
                w[nb] = tp1[(t * 2 + rb) * NB * 64 + nb * 64];
                b[nb] = *reinterpret_cast<const tw_f4 *>(panelB + ((i >> 3) * Rp + 16 * nb + lm) * 8 + (i & 7));
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float y = b[nb][v] * sc[nb];
                    s0[nb] = fmaf(u[nb][v], y, s0[nb]);
                    s1[nb] = fmaf(w[nb][v], y, s1[nb]);
                }
        }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        s0[nb] += __shfl_xor(s0[nb], 16);
        s1[nb] += __shfl_xor(s1[nb], 16);
        s0[nb] += __shfl_xor(s0[nb], 32);
        s1[nb] += __shfl_xor(s1[nb], 32);
    }
    if (lg == 0) {
        float *dst = partial + ((long)split * I2 + i2) * Rp + lm;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            dst[16 * nb] = s0[nb];
            if (i2 + 1 < I2) dst[Rp + 16 * nb] = s1[nb];
        }
    }
}

// ---------------------------------------------------------------------------
// host side

template <int ST, int NB>
static int tw_kernel(const TwPlan &p, const TwArgs *a, hipStream_t s) {
    if (!a) {
        TDX_HIP(hipFuncSetAttribute((const void *)k_tw_m1<ST, NB>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)p.lds));
        return TDX_OK;
    }
    k_tw_m1<ST, NB><<<p.blocks_i1 * p.nsplit1, 64 * kTwWaves, p.lds, s>>>(*a);
    return TDX_OK;
}
template <int ST>
static int tw_by_nb(const TwPlan &p, const TwArgs *a, hipStream_t s) {
    switch (p.Rp / 16) {
        case 1: return tw_kernel<ST, 1>(p, a, s);
        case 2: return tw_kernel<ST, 2>(p, a, s);
        case 3: return tw_kernel<ST, 3>(p, a, s);
        default: return tw_kernel<ST, 4>(p, a, s);
    }
}

int tw_plan(TwPlan &p, int order, const long *dims, int dtype, long R, const void *X, bool enabled) {
    p = TwPlan();
    if (!enabled || order != 3 || R < 1 || R > 64 || ((uintptr_t)X & 15) != 0) return TDX_OK;
    if (dtype != TDX_F32 && dtype != TDX_BF16) return TDX_OK;
    const bool f32 = dtype == TDX_F32;
    p.st = f32 ? 0 : 1;
    p.Rp = (int)(ceil_div(R, 16L) * 16);
    p.I0 = dims[0], p.I1 = dims[1], p.I2 = dims[2];
    if (p.I0 % (f32 ? 4 : 8) != 0 || p.I0 >= (1L << 24)) return TDX_OK;
    // T is written and read once, 8 Rp bytes a fibre, where the pass over X that it saves reads es I0
    // bytes: worth it from es I0 = 8 Rp on.  Sweeps with the separate passes and with this
    // one, FP32: 1024 x 1024 x 256 rank 64 880 -> 631 us, 256 x 512 x 512 rank 64 382 -> 317, 128 x 512
    // x 1024 rank 64 (es I0 = 8 Rp) 397 -> 352, 64 x 1024 x 1024 rank 64 (4 Rp) 413 -> 415.  Below
    // 2^25 elements a pass is as short as the launches: 512 x 256 x 256 rank 16 130 -> 117, 256^3 rank
    // 16 89 -> 91.
    const long es = f32 ? 4 : 2, N = p.I0 * p.I1 * p.I2;
    if (es * p.I0 < 8L * p.Rp || N < (1L << 25)) return TDX_OK;
    const int ksn = f32 ? 2 : 4, np = f32 ? 3 : 2;
    p.nfc = (int)ceil_div(p.I0, 32L * ksn);
    p.chunk_ops = ksn * np * (p.Rp / 16) * 64;
    p.lds = 2 * sizeof(uint4) * p.chunk_ops + sizeof(float) * kTwTile * kTwWaves;
    p.blocks_i1 = (int)ceil_div(p.I1, (long)kTwRows);
    const long ns = std::min(std::max(1L, (long)device_cus() / p.blocks_i1), ceil_div(p.I2, 2L));
    p.i2per = (int)(ceil_div(ceil_div(p.I2, ns), 2L) * 2);
    p.nsplit1 = (int)ceil_div(p.I2, (long)p.i2per);
    // about 16 waves per CU for the pass over T
    const long ntile = ceil_div(p.I1, 32L);
    const long n2 = std::max(1L, std::min(ceil_div(32L * device_cus(), p.I2), ntile));
    p.tper = (int)ceil_div(ntile, n2);
    p.nsplit2 = (int)ceil_div(ntile, (long)p.tper);
    p.nb2 = (int)ceil_div(p.I2, 8L);
    const int rc = p.st == 0 ? tw_by_nb<0>(p, nullptr, nullptr) : tw_by_nb<1>(p, nullptr, nullptr);
    if (rc) return rc;
    p.on = true;
    return TDX_OK;
}

// ws: p.ws_bytes()
int tw_m1_launch(const TwPlan &p, const void *X, const float *panelA, const float *panelC, void *ws, float *partial,
                 const VinvJob &inverse, hipStream_t s) {
    if (!p.on) return record(TDX_ERR_UNSUPPORTED);
    float *T = (float *)ws;
    uint4 *parts = (uint4 *)((char *)ws + p.t_bytes());
    float *scale = (float *)(parts + (size_t)p.nfc * p.chunk_ops);
#define TDX_TWP(NS_)                                                                                              \
    do {                                                                                                          \
        if (p.st == 0) k_tw_parts<2, 3, NS_><<<1 + p.nfc, 256, 0, s>>>(panelA, p.I0, p.Rp, parts, scale, inverse); \
        else k_tw_parts<4, 2, NS_><<<1 + p.nfc, 256, 0, s>>>(panelA, p.I0, p.Rp, parts, scale, inverse);          \
    } while (0)
    if (p.Rp == 16) TDX_TWP(4);
    else if (p.Rp == 32) TDX_TWP(8);
    else TDX_TWP(16);
#undef TDX_TWP
    TwArgs a{X, panelA, panelC, parts, scale, T, partial, p.I0, p.I1, p.I2, p.blocks_i1, p.i2per};
    const int rc = p.st == 0 ? tw_by_nb<0>(p, &a, s) : tw_by_nb<1>(p, &a, s);
    if (rc) return rc;
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

int tw_m2_launch(const TwPlan &p, const void *ws, const float *panelB, float *partial, const VinvJob &inverse,
                 hipStream_t s) {
    if (!p.on) return record(TDX_ERR_UNSUPPORTED);
    const float *T = (const float *)ws;
    const float *scale = (const float *)((const char *)ws + p.t_bytes() + sizeof(uint4) * p.nfc * p.chunk_ops);
    const int grid = 1 + p.nb2 * p.nsplit2;
#define TDX_TW2(NB_, NS_) \
    k_tw_m2<NB_, NS_><<<grid, 256, 0, s>>>(T, panelB, scale, partial, p.I1, p.I2, p.tper, p.nb2, inverse)
    switch (p.Rp / 16) {
        case 1: TDX_TW2(1, 4); break;
        case 2: TDX_TW2(2, 8); break;
        case 3: TDX_TW2(3, 16); break;
        default: TDX_TW2(4, 16); break;
    }
#undef TDX_TW2
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

}  // namespace tdx
