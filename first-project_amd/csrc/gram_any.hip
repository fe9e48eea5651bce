// gram_any.hip -- Gram of a mode-n unfolding, G = X(n) X(n)^T, In <= 128, on FP32 MFMA with the
// tensor tile staged in LDS, element by element: FP32 and BF16 tensors without whole vectors.
//
// X is read as the (P, In, Q) view, column k = p + P q of the unfolding a fibre.  A workgroup
// walks its range of columns in steps of 64: the (rows x 64) tile goes to LDS as [row][k]
// (rows of 68 floats: a lane's 4 consecutive k are one 16-byte operand read, 16 rows in distinct
// banks) while the next step's elements are in flight in registers.  G needs the block pairs
// bi <= bj of its 16 x 16 blocks only (36 of 64 at 128 rows); the four waves take them in turn,
// a pair reading its two operands from LDS.  Each wave keeps two chains of sums (even and odd
// groups of 16 columns).  Every workgroup writes the FP32 partial of its range; the caller adds
// them in FP64.
//
// Latency bound at the sizes that come here, so it wants many workgroups: 125 x 101 x 77 took
// 500-730 us a mode with one workgroup per 2048 columns (7 of them) on vector FMAs and takes 13-17 us.
#include "common.hpp"
#include <algorithm>

namespace tdx {

typedef float ga_f4 __attribute__((ext_vector_type(4)));

static constexpr int kGaN = 128, kGaK = 64, kGaLd = 68;

__device__ __forceinline__ float ga_f32(float v) { return v; }
__device__ __forceinline__ float ga_f32(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }

// NP: pairs per wave, ceil(nb (nb + 1) / 2 / 4) for nb = ceil(In / 16) row blocks, rounded up
template <typename ET, bool PC, int NP>
__global__ __launch_bounds__(256, 2) void k_gram_any(const ET *__restrict__ X, long P, long In, long Q, long kper,
                                                     float *__restrict__ part) {
    constexpr int NL = kGaN * kGaK / 256;  // loads per thread and step
    __shared__ __attribute__((aligned(16))) float xs[kGaN * kGaLd];
    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long K = P * Q;
    const long kbeg = (long)blockIdx.x * kper, kend = min(kbeg + kper, K);
    const int nb = (int)((In + 15) / 16), npair = nb * (nb + 1) / 2;
    const int nrow = 16 * nb;

    // lanes along k (P > 1) or along the rows (P = 1), 32 elements
    ET xe[NL];
    auto load = [&](long k0) {
        if constexpr (PC) {
            const long k = min(k0 + lane, K - 1), q = k / P;
            const ET *p = X + (k - q * P) + q * P * In;
            long r0 = wave;
            asm volatile("" : "+s"(r0));  // (hoisted out of the loop the row offsets fill the scalar registers)
#pragma unroll
            for (int u = 0; u < NL; ++u)
                if (4 * u < nrow) xe[u] = p[min(r0 + 4 * u, In - 1) * P];
        } else {
#pragma unroll
            for (int u = 0; u < NL / 4; ++u)
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    xe[4 * u + c] = X[min((long)(tid & 127), In - 1) + min(k0 + 4 * ((tid >> 7) + 2 * u) + c, K - 1) * In];
        }
    };
    auto store = [&](long k0) {
        if constexpr (PC) {
            const bool on = k0 + lane < K;
#pragma unroll
            for (int u = 0; u < NL; ++u)
                if (4 * u < nrow) xs[(wave + 4 * u) * kGaLd + lane] = on ? ga_f32(xe[u]) : 0.0f;
        } else {
#pragma unroll
            for (int u = 0; u < NL / 4; ++u) {
                const int kq = (tid >> 7) + 2 * u;
                float4 w;
                w.x = k0 + 4 * kq + 0 < K ? ga_f32(xe[4 * u + 0]) : 0.0f;
                w.y = k0 + 4 * kq + 1 < K ? ga_f32(xe[4 * u + 1]) : 0.0f;
                w.z = k0 + 4 * kq + 2 < K ? ga_f32(xe[4 * u + 2]) : 0.0f;
                w.w = k0 + 4 * kq + 3 < K ? ga_f32(xe[4 * u + 3]) : 0.0f;
                *reinterpret_cast<float4 *>(xs + (tid & 127) * kGaLd + 4 * kq) = w;
            }
        }
    };

    // pair p = wave + 4 j of the list (0,0) (0,1) .. (0,nb-1) (1,1) ..: the row blocks' LDS offsets
    int oi[NP], oj[NP];
#pragma unroll
    for (int j = 0; j < NP; ++j) {
        int p = min(wave + 4 * j, npair - 1), bi = 0;
        while (p >= nb - bi) p -= nb - bi++;
        oi[j] = 16 * bi;
        oj[j] = 16 * (bi + p);
    }
    ga_f4 acc[NP][2];
#pragma unroll
    for (int j = 0; j < NP; ++j) acc[j][0] = acc[j][1] = ga_f4{0.f, 0.f, 0.f, 0.f};
    if (kbeg < kend) load(kbeg);
    for (long k0 = kbeg; k0 < kend; k0 += kGaK) {
        __syncthreads();
        store(k0);
        __syncthreads();
        load(k0 + kGaK);  // past the range: clamped addresses or the next range's, never consumed
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float *xp = xs + lm * kGaLd + 16 * q + 4 * lg;
#pragma unroll
            for (int j = 0; j < NP; ++j) {
                const float4 a = *reinterpret_cast<const float4 *>(xp + oi[j] * kGaLd);
                const float4 b = *reinterpret_cast<const float4 *>(xp + oj[j] * kGaLd);
                acc[j][q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc[j][q & 1], 0, 0, 0);
                acc[j][q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc[j][q & 1], 0, 0, 0);
                acc[j][q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc[j][q & 1], 0, 0, 0);
                acc[j][q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc[j][q & 1], 0, 0, 0);
            }
        }
    }
    // register v of lane (lm, lg): row 4 lg + v, column lm of the pair's block
    float *dst = part + (long)blockIdx.x * kGaN * kGaN;
#pragma unroll
    for (int j = 0; j < NP; ++j)
        if (wave + 4 * j < npair)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                dst[(oi[j] + 4 * lg + v) * kGaN + oj[j] + lm] = acc[j][0][v] + acc[j][1][v];
}

int gram_f32_wgs(long In);
void gram_f32_launch(const float *X, long P, long In, long Q, long kper, float *part, unsigned nblk, hipStream_t s);

template <typename ET>
static void ga_launch(const ET *X, long P, long In, long Q, long kper, float *part, unsigned g, hipStream_t s) {
    const int nb = (int)ceil_div(In, 16L), np = (int)ceil_div(nb * (nb + 1) / 2, 4L);
#define TDX_GA(NP_)                                                                                     \
    do {                                                                                                \
        if (P > 1) k_gram_any<ET, true, NP_><<<g, 256, 0, s>>>(X, P, In, Q, kper, part);           \
        else k_gram_any<ET, false, NP_><<<g, 256, 0, s>>>(X, P, In, Q, kper, part);                \
    } while (0)
    if (np <= 1) TDX_GA(1);
    else if (np <= 3) TDX_GA(3);
    else if (np <= 6) TDX_GA(6);
    else TDX_GA(9);
#undef TDX_GA
}

// Partial Grams (upper triangle of each kGaN^2 block, row-major) in part; returns their number,
// at most max_parts, or -1 on a launch error.
int gram_any_launch(const void *X, int xtype, long P, long In, long Q, float *part, int max_parts, hipStream_t s) {
    // whole vectors of an FP32 tensor: gram_f32.hip (element by element 64^4 takes 32-38 us a mode
    // and 128^4 446-487; 21-22 and 277-318 there)
    const bool vec = xtype == TDX_F32 && ((uintptr_t)X & 15) == 0 && (P > 1 ? P % 4 == 0 : In % 4 == 0);
    const long steps = ceil_div(P * Q, (long)kGaK);
    // the workgroups that fill the chip; at least two steps each, whose loads overlap, so that a partial
    // (64 KB) is not written for one tile of 32 KB
    const int wgs = vec ? gram_f32_wgs(In) : 3;
    long nblk = std::min<long>(std::min((long)wgs * device_cus(), (long)max_parts), ceil_div(steps, 2L));
    const long kper = ceil_div(steps, nblk) * kGaK;
    nblk = ceil_div(P * Q, kper);
    if (xtype == TDX_BF16) ga_launch<uint16_t>((const uint16_t *)X, P, In, Q, kper, part, (unsigned)nblk, s);
    else if (vec) gram_f32_launch((const float *)X, P, In, Q, kper, part, (unsigned)nblk, s);
    else ga_launch<float>((const float *)X, P, In, Q, kper, part, (unsigned)nblk, s);
    return hipGetLastError() == hipSuccess ? (int)nblk : -1;
}

}  // namespace tdx
