// ttm_any.hip -- mode-n tensor-times-matrix through LDS on FP32 MFMA, any shape and alignment:
//   Y[p, a, q] = sum_i X[p, i, q] U(i, a),  U(i, a) = U[i * ldi + a * lda],
// X the (P, In, Q) view of an FP32 or BF16 tensor (BF16: U rounded to BF16, as on the other
// path), Y the (P, Ra, Q) FP32 result.  All FP32 tensors come here, and BF16 ones whose mode is
// longer than 128, whose rank is above 64 or whose extents hold no whole vectors
// (src/ttm.cu:21,29,37 takes any of them).
//
// A GEMM of the fibres k = p + P q (rows) with U: a workgroup owns TM fibres x up to 64 columns
// and walks i in steps of 64.  The TM x 64 tile of X and the 64 x 16 NB block of U are staged in
// LDS (rows of 68 floats: a lane's 4 consecutive i are one 16-byte operand read, 16 rows in
// distinct banks) while the next step's elements are in flight in registers; the result leaves
// through LDS in whole lines.  X is read element by element, 64 lanes on 256 contiguous bytes
// (along p, or along i when P = 1), so nothing has to be aligned; with whole vectors (VEC) a
// thread loads 16 bytes, along p four fibres of four i transposed in registers.
// Bound by HBM.  512 x 384 x 256 FP32 with 48 columns (221-252 MB a mode, 48-55 us at the 4.6 TB/s
// of a large copy): 880-1450 us with a thread per output, 81-89 us element by element, 68-75 us
// with vectors.  128^4 to 32 columns (1.34 GB, 291 us): 293-315 us, 382 us with U and four steps
// of X held in one wave's registers; its later, small products 10-84 us against 27-136.
#include "common.hpp"

namespace tdx {

typedef float ta_f4 __attribute__((ext_vector_type(4)));

static constexpr int kTaK = 64, kTaLd = 68, kTaCols = 64;

struct TaArgs {
    const void *X;
    const float *U;
    float *Y;
    long P, In, Q, Ra, lda, ldi, rows;
    int ncb;
};

__device__ __forceinline__ float ta_f32(float v) { return v; }
__device__ __forceinline__ float ta_f32(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }
__device__ __forceinline__ float ta_coef(float u, float) { return u; }
__device__ __forceinline__ float ta_coef(float u, uint16_t) { return __uint_as_float((uint32_t)f32_to_bf16_bits(u) << 16); }

// PC: P > 1 (fibres contiguous along p); NB column blocks of 16; RPW row blocks of 16 per wave;
// VEC (FP32, 16-byte aligned, P % 4 == 0 or, for P = 1, In % 4 == 0): 16-byte loads of X
template <typename ET, bool PC, int NB, int RPW, bool VEC>
__global__ __launch_bounds__(256, 2) void k_ttm_any(TaArgs a) {
    constexpr int TM = 64 * RPW, NU = TM / 16, NL = TM / 4, NC = 4 * NB, CW = 16 * NB;
    __shared__ __attribute__((aligned(16))) float xs[TM * kTaLd];
    __shared__ __attribute__((aligned(16))) float bs[CW * kTaLd];
    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cb = blockIdx.x % a.ncb;
    const long row0 = (long)(blockIdx.x / a.ncb) * TM;
    const int col0 = cb * kTaCols;
    const long P = a.P, In = a.In, rows = a.rows;
    const ET *__restrict__ X = reinterpret_cast<const ET *>(a.X);
    const float *__restrict__ U = a.U;

    // this thread's fibre (PC: row tid % TM of the tile, the same for every load)
    long xrow = 0;
    if constexpr (PC) {
        // (VEC: the first of the thread's four fibres, tid % (TM / 4); rows % 4 == 0, and a quad
        // lies in one run of p)
        const long r = VEC ? min(row0 + 4 * (tid % (TM / 4)), rows - 4) : min(row0 + tid % TM, rows - 1), q = r / P;
        xrow = (r - q * P) + q * P * In;
    }
    // U: lanes along i where it is contiguous there, else along the columns
    const bool ui = a.ldi == 1;
    ET xv[VEC ? 1 : NL];
    float4 xq[VEC ? NL / 4 : 1];
    float uv[NC];
    auto load = [&](long i0) {
#pragma unroll
        for (int u = 0; u < NB; ++u)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int e = tid + 256 * u;
                const long i = ui ? i0 + lane : i0 + 4 * (e / CW) + c;
                const long col = min((long)col0 + (ui ? wave * NC + 4 * u + c : e % CW), a.Ra - 1);
                uv[4 * u + c] = U[min(i, In - 1) * a.ldi + col * a.lda];
            }
        if constexpr (VEC && PC) {
            // 4 fibres x 4 consecutive i a task, RPW tasks a thread
#pragma unroll
            for (int u = 0; u < RPW; ++u) {
                const int kq = (tid + 256 * u) / (TM / 4);
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    xq[4 * u + c] = ld_stream(reinterpret_cast<const float4 *>(X + xrow + min(i0 + 4 * kq + c, In - 1) * P));
            }
        } else if constexpr (VEC) {
            const ET *xp = X + min(i0 + 4 * (tid & 15), In - 4);
#pragma unroll
            for (int u = 0; u < NU; ++u)
                xq[u] = ld_stream(reinterpret_cast<const float4 *>(xp + min(row0 + (tid >> 4) + 16 * u, rows - 1) * In));
        } else if constexpr (PC) {
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int kq = __builtin_amdgcn_readfirstlane((tid + 256 * u) / TM);
#pragma unroll
                for (int c = 0; c < 4; ++c) xv[4 * u + c] = X[xrow + min(i0 + 4 * kq + c, In - 1) * P];
            }
        } else {
            const ET *xp = X + min(i0 + lane, In - 1);
            long r0 = row0 + wave;
            asm volatile("" : "+s"(r0));  // (hoisted out of the loop the row offsets fill the scalar registers)
#pragma unroll
            for (int u = 0; u < NL; ++u) xv[u] = xp[min(r0 + 4 * u, rows - 1) * In];
        }
    };
    ta_f4 acc[RPW][NB];
#pragma unroll
    for (int rp = 0; rp < RPW; ++rp)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[rp][nb] = ta_f4{0.f, 0.f, 0.f, 0.f};

    load(0);
    for (long i0 = 0; i0 < In; i0 += kTaK) {
        __syncthreads();
        if constexpr (VEC && PC) {
#pragma unroll
            for (int u = 0; u < RPW; ++u) {
                const int kq = (tid + 256 * u) / (TM / 4);
                float v[4][4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const bool on = i0 + 4 * kq + c < In;
                    const float4 w = xq[4 * u + c];
                    v[0][c] = on ? w.x : 0.f, v[1][c] = on ? w.y : 0.f, v[2][c] = on ? w.z : 0.f, v[3][c] = on ? w.w : 0.f;
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    *reinterpret_cast<float4 *>(xs + (4 * (tid % (TM / 4)) + t) * kTaLd + 4 * kq) =
                        float4{v[t][0], v[t][1], v[t][2], v[t][3]};
            }
        } else if constexpr (VEC) {
            const bool on = i0 + 4 * (tid & 15) < In;
#pragma unroll
            for (int u = 0; u < NU; ++u)
                *reinterpret_cast<float4 *>(xs + ((tid >> 4) + 16 * u) * kTaLd + 4 * (tid & 15)) =
                    on ? xq[u] : float4{0.f, 0.f, 0.f, 0.f};
        } else if constexpr (PC) {
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int e = tid + 256 * u, kq = e / TM;
                float4 v;
                v.x = (i0 + 4 * kq + 0 < In) ? ta_f32(xv[4 * u + 0]) : 0.0f;
                v.y = (i0 + 4 * kq + 1 < In) ? ta_f32(xv[4 * u + 1]) : 0.0f;
                v.z = (i0 + 4 * kq + 2 < In) ? ta_f32(xv[4 * u + 2]) : 0.0f;
                v.w = (i0 + 4 * kq + 3 < In) ? ta_f32(xv[4 * u + 3]) : 0.0f;
                *reinterpret_cast<float4 *>(xs + (e % TM) * kTaLd + 4 * kq) = v;
            }
        } else {
#pragma unroll
            for (int u = 0; u < NL; ++u)
                xs[(wave + 4 * u) * kTaLd + lane] = (i0 + lane < In) ? ta_f32(xv[u]) : 0.0f;
        }
        if (ui) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
                bs[(wave * NC + c) * kTaLd + lane] = (i0 + lane < In) ? ta_coef(uv[c], ET()) : 0.0f;
        } else {
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int e = tid + 256 * u, kq = e / CW;
                float4 v;
                v.x = (i0 + 4 * kq + 0 < In) ? ta_coef(uv[4 * u + 0], ET()) : 0.0f;
                v.y = (i0 + 4 * kq + 1 < In) ? ta_coef(uv[4 * u + 1], ET()) : 0.0f;
                v.z = (i0 + 4 * kq + 2 < In) ? ta_coef(uv[4 * u + 2], ET()) : 0.0f;
                v.w = (i0 + 4 * kq + 3 < In) ? ta_coef(uv[4 * u + 3], ET()) : 0.0f;
                *reinterpret_cast<float4 *>(bs + (e % CW) * kTaLd + 4 * kq) = v;
            }
        }
        __syncthreads();
        load(i0 + kTaK);  // past the last step: clamped addresses, never consumed
        __builtin_amdgcn_sched_barrier(0);
        const int nsub = (int)min((In - i0 + 15) / 16, 4L);
        for (int q = 0; q < nsub; ++q) {
            float4 av[RPW], bv[NB];
#pragma unroll
            for (int rp = 0; rp < RPW; ++rp)
                av[rp] = *reinterpret_cast<const float4 *>(xs + (16 * (RPW * wave + rp) + lm) * kTaLd + 16 * q + 4 * lg);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                bv[nb] = *reinterpret_cast<const float4 *>(bs + (16 * nb + lm) * kTaLd + 16 * q + 4 * lg);
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int rp = 0; rp < RPW; ++rp) {
                    const float x = c == 0 ? av[rp].x : c == 1 ? av[rp].y : c == 2 ? av[rp].z : av[rp].w;
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        const float y = c == 0 ? bv[nb].x : c == 1 ? bv[nb].y : c == 2 ? bv[nb].z : bv[nb].w;
                        acc[rp][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, acc[rp][nb], 0, 0, 0);
                    }
                }
        }
    }
    // the tile through LDS: [column][row] (PC) or [row][column], then contiguous stores.  Register
    // v of lane (lm, lg) holds row 4 lg + v, column lm of its block.
    __syncthreads();
    const int nc = (int)min((long)CW, a.Ra - col0), nr = (int)min((long)TM, rows - row0);
    if constexpr (PC) {
        constexpr int LD = TM + 4;
        static_assert(CW * LD <= TM * kTaLd, "the result tile fits the tensor tile");
#pragma unroll
        for (int rp = 0; rp < RPW; ++rp)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                *reinterpret_cast<ta_f4 *>(xs + (16 * nb + lm) * LD + 16 * (RPW * wave + rp) + 4 * lg) = acc[rp][nb];
        __syncthreads();
        const int rl = tid % TM;
        if (rl < nr) {
            const long r = row0 + rl, q = r / P;
            float *y = a.Y + (r - q * P) + q * P * a.Ra + (long)col0 * P;
            for (int c = tid / TM; c < nc; c += 256 / TM) y[c * P] = xs[c * LD + rl];
        }
    } else {
#pragma unroll
        for (int rp = 0; rp < RPW; ++rp)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    xs[(16 * (RPW * wave + rp) + 4 * lg + v) * kTaLd + 16 * nb + lm] = acc[rp][nb][v];
        __syncthreads();
        for (int e = tid; e < nr * nc; e += 256) {
            const int r = e / nc, c = e - r * nc;
            a.Y[(row0 + r) * a.Ra + col0 + c] = xs[r * kTaLd + c];
        }
    }
}

template <typename ET, bool PC, int RPW, bool VEC>
static void ta_launch(const TaArgs &a, int nb, unsigned grid, hipStream_t s) {
    switch (nb) {
        case 1: k_ttm_any<ET, PC, 1, RPW, VEC><<<grid, 256, 0, s>>>(a); break;
        case 2: k_ttm_any<ET, PC, 2, RPW, VEC><<<grid, 256, 0, s>>>(a); break;
        case 3: k_ttm_any<ET, PC, 3, RPW, VEC><<<grid, 256, 0, s>>>(a); break;
        default: k_ttm_any<ET, PC, 4, RPW, VEC><<<grid, 256, 0, s>>>(a); break;
    }
}

int ttm_any_launch(const void *X, int xtype, long P, long In, long Q, const float *U, long lda, long ldi, long Ra,
                   float *Y, hipStream_t s) {
    TaArgs a{X, U, Y, P, In, Q, Ra, lda, ldi, P * Q, (int)ceil_div(Ra, (long)kTaCols)};
    const int nb = Ra >= kTaCols ? 4 : (int)ceil_div(Ra, 16L);
    // 128 fibres a workgroup share a U block; 64 where that leaves compute units idle
    const bool wide = ceil_div(a.rows, 128L) * a.ncb >= device_cus();
    const unsigned grid = (unsigned)(ceil_div(a.rows, wide ? 128L : 64L) * a.ncb);
    const bool pc = P > 1, vec = xtype == TDX_F32 && ((uintptr_t)X & 15) == 0 && (pc ? P : In) % 4 == 0;
#define TDX_TA(ET_, VEC_)                                                                                             \
    do {                                                                                                              \
        if (pc) wide ? ta_launch<ET_, true, 2, VEC_>(a, nb, grid, s) : ta_launch<ET_, true, 1, VEC_>(a, nb, grid, s); \
        else wide ? ta_launch<ET_, false, 2, VEC_>(a, nb, grid, s) : ta_launch<ET_, false, 1, VEC_>(a, nb, grid, s);  \
    } while (0)
    if (xtype == TDX_BF16) TDX_TA(uint16_t, false);
    else if (vec) TDX_TA(float, true);
    else TDX_TA(float, false);
#undef TDX_TA
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

}  // namespace tdx
