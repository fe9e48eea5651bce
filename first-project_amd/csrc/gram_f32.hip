// gram_f32.hip -- Gram of a mode-n unfolding, G = X(n) X(n)^T, In <= 128, of an FP32 tensor with
// whole 16-byte vectors, its products formed from three BF16 parts per element.
//
// X is read as the (P, In, Q) view, column k = p + P q of the unfolding a fibre.  A workgroup
// walks its range of columns in steps of 64; every element of the (rows x 64) tile is cut once,
// on its way from registers to LDS, into x = x1 + x2 + x3 exactly, each part what is left rounded
// to BF16.  v_mfma_f32_16x16x32_bf16 multiplies x1 y1, x1 y2, x2 y1, x1 y3, x2 y2 and x3 y1
// exactly and adds them in FP32 (the terms left out are below 2^-25 of |x y|, of either sign); the
// sums of a step enter the FP32 accumulators once, so the chains of roundings stay short.  Every
// workgroup writes the FP32 partial of its range; the caller adds them in FP64.
//   * G needs the block pairs bi <= bj of its 16 x 16 blocks only.  Wave w takes the block rows w
//     and nb - 1 - w: nb + 1 pairs each, whose column operands it reads from LDS once (34 operand blocks
//     a step with 8 block rows; from 113 rows on the waves hold pairs that need 22).
//   * LDS rows are 64 BF16 of a part (128 bytes); chunk c of 8 lies at c ^ (row / 2 ^ row / 16) mod
//     8, so 16 rows of one chunk hit distinct banks, and so do the rows of a transposing store
//     but for their parity.
//   * Loads along the contiguous index: along p, or, for P = 1, 4 rows of 4 columns transposed in
//     registers.  The next step's are in flight meanwhile.
//   * A tile with an entry above 2^60 (its products may overflow, an infinity has no parts) or below
//     2^-100 but not zero (its last part would lose bits) is read again and multiplied in FP32 (every
//     tile of 128^3 x 32: 94 / 90 / 96 -> 264 / 249 / 250 us for modes 0 .. 2).
//
// A step is a chain (wait, cut, barrier, operand reads, products) and two workgroups of 128 rows
// fill a CU: at 128^4 the matrix pipe is busy 44 % and LDS 24 % of the time, at 2.05 GHz.  Modes 0 .. 3 on FP32 matrix instructions before: 128^4 420 /
// 396 / 393 / 395 -> 275 / 272 / 299 / 307 us, 252 / 244 / 249 / 250 with the pairs of 22 blocks (1.07
// GB: 165 us at 6.5 TB/s), 64^4 32 / 25 / 25 / 25 -> 22 / 22 / 22 / 22, 256 x 128 x 128 15 / 13 -> 10 / 10;
// errors against 64 bits 7e-9 -> 5e-9 (64^4), 2.2e-8 -> 1.1e-8 (124 x 100 x 76), 3.7e-8 -> 1.6e-8
// (64 x 48 x 40).  Not faster: eight waves a tile (128 registers spill), the pair counts at compile
// time.
#include "common.hpp"
#include <algorithm>

namespace tdx {

typedef float gf_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 gf_b8 __attribute__((ext_vector_type(8)));

static constexpr int kGfN = 128, kGfK = 64;

// workgroups per CU (and waves per SIMD): registers allow two of 128 rows
constexpr int gf_wgs(int nb) { return nb > 4 ? 2 : 3; }
int gram_f32_wgs(long In) { return gf_wgs((int)ceil_div(In, 16L)); }

// FULL (all 8 row blocks): a wave's nine pairs form blocks of their own, 3 x 3 or a triangle and
// what fits beside it, so that the waves read 22 operand blocks a step instead of 34
struct GfWave {
    int n, blk[6], a[9], b[9];  // row blocks, and the pairs as positions among them
};
constexpr GfWave kGfWaves[4] = {
    {6, {0, 1, 2, 3, 4, 5}, {0, 0, 0, 1, 1, 1, 2, 2, 2}, {3, 4, 5, 3, 4, 5, 3, 4, 5}},
    {5, {0, 1, 2, 6, 7, 7}, {0, 0, 1, 1, 2, 2, 3, 3, 4}, {3, 4, 3, 4, 3, 4, 3, 4, 4}},
    {5, {3, 4, 5, 6, 7, 7}, {0, 0, 1, 1, 2, 2, 0, 1, 2}, {3, 4, 3, 4, 3, 4, 0, 1, 2}},
    {6, {0, 1, 2, 3, 4, 5}, {0, 0, 0, 1, 1, 2, 3, 3, 4}, {0, 1, 2, 1, 2, 2, 4, 5, 5}},
};
template <int W> struct GfIs {
    static constexpr int w = W;
};

// NB: row blocks, at least ceil(In / 16)
template <bool PC, int NB, bool FULL>
__global__ __launch_bounds__(256, gf_wgs(NB)) void k_gram_f32(const float *__restrict__ X, long P, long In, long Q, long kper,
                                                     float *__restrict__ part) {
    constexpr int NR = 16 * NB;
    __shared__ uint4 xs[3 * NR * 8];
    __shared__ int odd[2];
    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long K = P * Q;
    const long kbeg = (long)blockIdx.x * kper, kend = min(kbeg + kper, K);
    const int nb = (int)((In + 15) / 16);
    const int b1 = wave, b2 = nb - 1 - wave;  // this wave's block rows (none: b2 < b1)
    if (tid < 2) odd[tid] = 0;

    // P > 1: row tid / 16 + 16 u, columns k .. k + 3, a vector a load; k = p + P q is stepped without
    // a division.  P = 1: 4 x 4 blocks of rows 4 rq .. and columns k + 4 KQ u .., four vectors a load.
    constexpr int NT = PC ? NR / 16 : NR / 64, RQ = NR / 4, KQ = 4 * (256 / (4 * RQ));
    const int rq = (tid >> 2) & (RQ - 1), kq = PC ? tid & 15 : (tid & 3) + 4 * (tid / (4 * RQ));
    long k = kbeg + 4 * kq;  // of the step to be loaded
    long q = PC ? k / P : 0, p = PC ? k - q * P : 0;
    const long qs = kGfK / P, ps = kGfK - qs * P;
    float4 xq[PC ? NT : 4 * NT];
    auto load = [&](int u) {
        if constexpr (PC) {
            // (P % 4 == 0: a vector lies in one run, and is inside as a whole)
            xq[u] = ld_stream(reinterpret_cast<const float4 *>(X + (k < K ? p + q * P * In : 0) +
                                                               min((long)(tid >> 4) + 16 * u, In - 1) * P));
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                xq[4 * u + c] = ld_stream(reinterpret_cast<const float4 *>(
                    X + min(4L * rq, In - 4) + min(k + 4 * KQ * u + c, K - 1) * In));  // In % 4 == 0
        }
    };
    auto advance = [&]() {
        k += kGfK;
        if constexpr (PC) {
            p += ps;
            q += qs;
            const bool wrap = p >= P;
            p -= wrap ? P : 0;
            q += wrap;
        }
    };
    // four consecutive columns of a row: their parts to LDS
    float m = 0.0f;       // largest magnitude of the step (NaN left out: it stays NaN in its parts)
    uint32_t key = ~0u;   // and least small_key
    auto put = [&](int row, int kq, float4 x) {
        key = min(key, min(min(small_key(x.x), small_key(x.y)), min(small_key(x.z), small_key(x.w))));
        asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(x.x), "v"(x.y));
        asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(x.z), "v"(x.w));
        uint2 *d = reinterpret_cast<uint2 *>(xs + row * 8 + ((kq >> 1) ^ (((row >> 1) ^ (row >> 4)) & 7))) + (kq & 1);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const uint2 w = {bf16_pair(x.x, x.y), bf16_pair(x.z, x.w)};
            d[k * NR * 16] = w;
            x.x -= __uint_as_float(w.x << 16), x.y -= __uint_as_float(w.x & 0xffff0000u);
            x.z -= __uint_as_float(w.y << 16), x.w -= __uint_as_float(w.y & 0xffff0000u);
        }
    };
    auto store = [&](long k0, int u) {
        if constexpr (PC) {
            put((tid >> 4) + 16 * u, kq, k0 + 4 * kq < K ? xq[u] : float4{0.f, 0.f, 0.f, 0.f});
        } else {
            float v[4][4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const bool on = k0 + 4 * (kq + KQ * u) + c < K;
                const float4 w = xq[4 * u + c];
                v[0][c] = on ? w.x : 0.f, v[1][c] = on ? w.y : 0.f, v[2][c] = on ? w.z : 0.f, v[3][c] = on ? w.w : 0.f;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) put(4 * rq + t, kq + KQ * u, float4{v[t][0], v[t][1], v[t][2], v[t][3]});
        }
    };
    auto operand = [&](int b, int ks, int k) {
        const uint4 v = xs[(k * NR + 16 * b + lm) * 8 + ((4 * ks + lg) ^ ((lm >> 1) ^ (b & 7)))];
        return __builtin_bit_cast(gf_b8, v);
    };
    // FULL: the wave's pairs
    gf_f4 accf[9];
    if constexpr (FULL)
#pragma unroll
        for (int p = 0; p < 9; ++p) accf[p] = gf_f4{0.f, 0.f, 0.f, 0.f};
    auto full_step = [&](auto w) {
        constexpr GfWave g = kGfWaves[decltype(w)::w];
        gf_f4 s[9];
        gf_b8 o[6][3];
        // smallest terms first, as in mul below; the first half's leading parts are read again for it
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
            for (int j = 0; j < g.n; ++j)
#pragma unroll
                for (int k = 0; k < 3; ++k) o[j][k] = operand(g.blk[j], ks, k);
#pragma unroll
            for (int p = 0; p < 9; ++p) {
                const gf_b8(&a)[3] = o[g.a[p]], (&b)[3] = o[g.b[p]];
                gf_f4 t = ks == 0 ? gf_f4{0.f, 0.f, 0.f, 0.f} : s[p];
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], b[0], t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[2], t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[1], t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], b[0], t, 0, 0, 0);
                s[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], b[1], t, 0, 0, 0);
            }
        }
#pragma unroll
        for (int ks = 1; ks >= 0; --ks) {
            if (ks == 0)
#pragma unroll
                for (int j = 0; j < g.n; ++j) o[j][0] = operand(g.blk[j], 0, 0);
#pragma unroll
            for (int p = 0; p < 9; ++p)
                s[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o[g.a[p]][0], o[g.b[p]][0], s[p], 0, 0, 0);
        }
#pragma unroll
        for (int p = 0; p < 9; ++p) {
            accf[p] += s[p];
            asm volatile("" : "+v"(accf[p]));  // (before the branch, as below)
        }
    };
    // FP32 products of the tile at k0, from memory: four consecutive columns of a row a lane
    auto odd_run = [&](long k0) {  // of the tile's first column (in scalar registers)
        const long kd = PC ? k0 / P : 0;
        return (long)__builtin_amdgcn_readfirstlane((int)(kd >> 32)) << 32 |
               (uint32_t)__builtin_amdgcn_readfirstlane((int)kd);
    };
    auto odd_values = [&](long k0, long kd, int q, int blk) {
        int lo = lane;
        uint32_t pd = (uint32_t)P;
        asm volatile("" : "+v"(lo), "+s"(pd));  // (hoisted out of the loop over steps the rows' offsets spill)
        const long k = k0 + 16 * q + 4 * (lo >> 4), row = min((long)(16 * blk + (lo & 15)), In - 1);
        gf_f4 v;  // (every load unconditional)
        if constexpr (PC) {
            const long t = k - kd * P;
            const long d = P > 64 ? (long)(t >= P) : (long)((uint32_t)t / pd);
            v = *reinterpret_cast<const gf_f4 *>(X + (k < K ? (t - d * P) + (kd + d) * P * In : 0) + row * P);
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = X[min(k + c, K - 1) * In + row];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) v[c] = k + c < K ? v[c] : 0.0f;
        return v;
    };
    auto full_odd = [&](auto w, long k0) {
        constexpr GfWave g = kGfWaves[decltype(w)::w];
        const long kd = odd_run(k0);
#pragma unroll 1
        for (int q = 0; q < 4; ++q) {
            gf_f4 v[6];
#pragma unroll
            for (int j = 0; j < g.n; ++j) v[j] = odd_values(k0, kd, q, g.blk[j]);
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int j = 0; j < 9; ++j)
                    accf[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[g.a[j]][c], v[g.b[j]][c], accf[j], 0, 0, 0);
        }
        __builtin_amdgcn_s_sleep(1);  // (the last results are in place before any branch)
    };
    auto by_wave = [&](auto f) {
        if (wave == 0) f(GfIs<0>());
        else if (wave == 1) f(GfIs<1>());
        else if (wave == 2) f(GfIs<2>());
        else f(GfIs<3>());
    };
    // acc1[t], acc2[t]: block rows b1, b2 with block column nb - 1 - t
    gf_f4 acc1[NB], acc2[NB / 2];
#pragma unroll
    for (int t = 0; t < NB; ++t) acc1[t] = gf_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NB / 2; ++t) acc2[t] = gf_f4{0.f, 0.f, 0.f, 0.f};
    if (kbeg < kend)
#pragma unroll
        for (int u = 0; u < NT; ++u) load(u);
    advance();
    int par = 0;
    for (long k0 = kbeg; k0 < kend; k0 += kGfK, par ^= 1) {
        __syncthreads();
        if (tid == 0) odd[par ^ 1] = 0;  // (read by every wave before this barrier, set after the next)
        // (a register's next load leaves as soon as it is free; past the range: clamped addresses or
        // the next range's, never consumed)
        m = 0.0f, key = ~0u;
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            store(k0, u);
            load(u);
            __builtin_amdgcn_sched_barrier(0);
        }
        advance();
        if (m > 0x1p60f || key < kSmallKey) odd[par] = 1;  // FP32 products are needed
        __syncthreads();
        if (b2 < b1) continue;
        if constexpr (FULL) {
            if (odd[par]) by_wave([&](auto w) { full_odd(w, k0); });
            else by_wave(full_step);
            continue;
        }
        if (odd[par]) {
            const long kd = odd_run(k0);
#pragma unroll 1
            for (int q = 0; q < 4; ++q) {
                const gf_f4 v1 = odd_values(k0, kd, q, b1), v2 = odd_values(k0, kd, q, b2);
#pragma unroll
                for (int t = 0; t < NB; ++t)
                    if (nb - 1 - t >= b1) {
                        const gf_f4 w = odd_values(k0, kd, q, nb - 1 - t);
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            acc1[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1[c], w[c], acc1[t], 0, 0, 0);
                            if (t < NB / 2 && t <= wave && b2 > b1)
                                acc2[t < NB / 2 ? t : 0] =
                                    __builtin_amdgcn_mfma_f32_16x16x4f32(v2[c], w[c], acc2[t < NB / 2 ? t : 0], 0, 0, 0);
                        }
                    }
            }
            __builtin_amdgcn_s_sleep(1);  // (as below: the last results are in place before any branch)
            continue;
        }
        gf_b8 a1[2][3], a2[2][3];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int k = 0; k < 3; ++k) a1[ks][k] = operand(b1, ks, k), a2[ks][k] = operand(b2, ks, k);
        // the step's sums, smallest terms first (so two roundings at the size of the sum)
        auto mul = [&](const gf_b8 (&a)[2][3], const gf_b8 (&b)[2][3]) {
            gf_f4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][2], b[ks][0], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][0], b[ks][2], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][1], b[ks][1], s, 0, 0, 0);
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][1], b[ks][0], s, 0, 0, 0);
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][0], b[ks][1], s, 0, 0, 0);
            }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
                s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][0], b[ks][0], s, 0, 0, 0);
            return s;
        };
#pragma unroll
        for (int t = 0; t < NB; ++t)
            if (nb - 1 - t >= b1) {
                gf_b8 b[2][3];
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int k = 0; k < 3; ++k) b[ks][k] = operand(nb - 1 - t, ks, k);
                // (the sums are added before the branch: hipcc left out the wait states that a read
                // of a matrix result needs where it had moved the add behind one)
                acc1[t] += mul(a1, b);
                asm volatile("" : "+v"(acc1[t]));
                if (t < NB / 2 && t <= wave && b2 > b1) {
                    acc2[t < NB / 2 ? t : 0] += mul(a2, b);
                    asm volatile("" : "+v"(acc2[t < NB / 2 ? t : 0]));
                }
            }
    }
    // register v of lane (lm, lg): row 4 lg + v, column lm of the pair's block
    float *dst = part + (long)blockIdx.x * kGfN * kGfN;
    if constexpr (FULL) {
        by_wave([&](auto w) {
            constexpr GfWave g = kGfWaves[decltype(w)::w];
#pragma unroll
            for (int p = 0; p < 9; ++p)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    dst[(16 * g.blk[g.a[p]] + 4 * lg + v) * kGfN + 16 * g.blk[g.b[p]] + lm] = accf[p][v];
        });
        return;
    }
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int c = 16 * (nb - 1 - t) + lm;
            if (b2 >= b1 && nb - 1 - t >= b1) dst[(16 * b1 + 4 * lg + v) * kGfN + c] = acc1[t][v];
            if (t < NB / 2 && t <= wave && b2 > b1) dst[(16 * b2 + 4 * lg + v) * kGfN + c] = acc2[t < NB / 2 ? t : 0][v];
        }
}

// Partial Grams (upper triangle of each kGfN^2 block, row-major) in part, of nblk ranges of kper
// columns.  Requires X 16-byte aligned, P % 4 == 0, or P = 1 and In % 4 == 0; In <= kGfN.
void gram_f32_launch(const float *X, long P, long In, long Q, long kper, float *part, unsigned nblk, hipStream_t s) {
    const int nb = (int)ceil_div(In, 16L);
    if (P > 1) {
        if (nb <= 2) k_gram_f32<true, 2, false><<<nblk, 256, 0, s>>>(X, P, In, Q, kper, part);
        else if (nb <= 4) k_gram_f32<true, 4, false><<<nblk, 256, 0, s>>>(X, P, In, Q, kper, part);
        else if (nb < 8) k_gram_f32<true, 8, false><<<nblk, 256, 0, s>>>(X, P, In, Q, kper, part);
        else k_gram_f32<true, 8, true><<<nblk, 256, 0, s>>>(X, P, In, Q, kper, part);
    } else {
        // (at least 64 rows: a 4 x 4 block for every thread)
        if (nb <= 4) k_gram_f32<false, 4, false><<<nblk, 256, 0, s>>>(X, P, In, Q, kper, part);
        else if (nb < 8) k_gram_f32<false, 8, false><<<nblk, 256, 0, s>>>(X, P, In, Q, kper, part);
        else k_gram_f32<false, 8, true><<<nblk, 256, 0, s>>>(X, P, In, Q, kper, part);
    }
}

}  // namespace tdx
