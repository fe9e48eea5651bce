// mttkrp_any.hip -- fused MTTKRP for every shape and alignment: any leading extent, any rank,
// tensors that do not start on a 16-byte boundary.  FP32, BF16 and FP8 storage.
//
// The tensor is read as the (P, In, Q) view of the output mode (P, Q: the extents before and
// after it) and the contraction index is k = p + P q, whose mixed-radix digits over the
// contracted modes in mode order are the factor rows.  X is addressed element by element
// (p + row P + q P In), so no extent has to be a multiple of anything and no K step is padded
// but the last one.
//
// A workgroup owns TM output rows (128, 64, 32 or 16, by the extent) x up to 64 columns and a
// range of K; per step of 64 k it stages the TM x 64 tensor tile and the Khatri-Rao block
// (FP32, one product per slow factor) in LDS while the next step's tensor elements and factor
// rows are loaded into registers, and multiplies on v_mfma_f64_16x16x4f64: exact FP64 products
// of FP32 operands and FP64 sums.  FP64 keeps the accuracy of a scalar FP64 accumulation; at
// 72 TFLOP/s the matrix work takes 36 us where the tensor's 129 MB take 28 us from HBM
// (401 x 317 x 253, rank 20 in 32 padded columns), so the path is bound by HBM up to rank 16 and
// by the FP64 matrix pipe above about 32.  Measured there: 77 / 69 / 69 us for modes 0 / 1 / 2,
// where one lane per column summing element by element took 10.5 ms (a chain of dependent
// FP64 additions, with the index digits divided out for every element).
//   * output mode 0 (M0): rows are contiguous in memory; lanes run over rows and a thread loads
//     four consecutive k, which leave as one 16-byte LDS store;
//   * other modes: k is contiguous (runs of P); lanes run over the 64 k of the step, and every
//     lane carries its own digits, advanced by a mixed-radix addition (no division in the loop).
// LDS rows have 68 floats: a lane reads 4 consecutive k of a row as one 16-byte operand for four
// MFMAs (k is assigned to the 4 k-slots so that a lane group owns 4 consecutive k), 16 rows
// falling into distinct banks.
#include "mttkrp.hpp"

namespace tdx {

typedef double any_d4 __attribute__((ext_vector_type(4)));
typedef float any_f2 __attribute__((ext_vector_type(2)));

static constexpr int kAnyK = 64;    // k per step
static constexpr int kAnyLd = 68;   // LDS row pitch (floats)
static constexpr int kAnyCols = 64; // columns per workgroup at most

struct AnyArgs {
    const void *X;
    const float *panel[3];   // of the contracted modes, in mode order
    const float *row_scale;  // FP8 storage, mode 0
    float *partial;
    const int *skip;
    long D[3];               // extents of the contracted modes (1 past nm)
    long T[3];               // digits of kAnyK in the radices D
    long P, In, K, kper;
    int nm, Rp, rowtiles, ncb;
};

template <int ST> struct AnyElem;
template <> struct AnyElem<0> { typedef float T; };
template <> struct AnyElem<1> { typedef uint16_t T; };
template <> struct AnyElem<2> { typedef uint8_t T; };
__device__ __forceinline__ float any_f32(float v) { return v; }
__device__ __forceinline__ float any_f32(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }
__device__ __forceinline__ float any_f32(uint8_t v) {
    const any_f2 d = __builtin_amdgcn_cvt_pk_f32_fp8((int)v, false);
    return d.x;
}

// RW waves along the rows, RPW row blocks of 16 per wave; the other 4 / RW waves split each
// step's k and are added at the end in a fixed order
template <int ST, bool M0, int NB, int RW, int RPW>
__global__ __launch_bounds__(256, 2) void k_mttkrp_any(AnyArgs a) {
    typedef typename AnyElem<ST>::T ET;
    constexpr int TM = 16 * RW * RPW, KW = 4 / RW;
    constexpr int NU = TM / 16;       // M0: groups of four k per thread and step
    constexpr int NL = TM / 4;        // loads per thread and step
    constexpr int NC = 4 * NB;        // Khatri-Rao columns per thread
    __shared__ __attribute__((aligned(16))) float xs[TM * kAnyLd];
    __shared__ __attribute__((aligned(16))) float bs[16 * NB * kAnyLd];
    __shared__ double red[KW > 1 ? 4 * 256 * NB : 1];
    if (a.skip && *a.skip) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 15, lg = lane >> 4;
    const int rowtile = blockIdx.x % a.rowtiles;
    const int cb = (blockIdx.x / a.rowtiles) % a.ncb;
    const long split = blockIdx.x / a.rowtiles / a.ncb;
    const long row0 = (long)rowtile * TM;
    const int col0 = cb * kAnyCols;
    const long kbeg = split * a.kper, kend = min(kbeg + a.kper, a.K);
    const ET *__restrict__ X = reinterpret_cast<const ET *>(a.X);
    const long In = a.In, P = a.P, K = a.K;
    const int Rp = a.Rp;

    // the k of this lane (columns of the step): digits, and the tensor offset p + q P In
    const long D0 = a.D[0], D1 = a.D[1];
    long kl = kbeg + lane;
    long i0, i1, i2, pk = 0, xo = 0;
    const long TP = M0 ? 0 : kAnyK % P, TQ = M0 ? 0 : kAnyK / P;
    {
        const long k = kl < K ? kl : K - 1;
        i0 = k % D0;
        i1 = (k / D0) % D1;
        i2 = k / D0 / D1;
        if constexpr (!M0) {
            pk = k % P;
            xo = pk + (k / P) * P * In;
        }
    }
    ET xv[NL];
    float f0[NC], f1[NC], f2[NC];
    bool kok = false, kokx = false;
    long kx = kbeg;  // first k of the step whose loads are issued next
    auto load = [&]() {
        // factor rows first: they are consumed with the tensor elements, and waiting for them
        // must not wait for loads issued later
        kok = kl < K;
        const long j0 = kok ? i0 : 0, j1 = kok ? i1 : 0, j2 = kok ? i2 : 0;
        const float *p0 = a.panel[0] + ((j0 >> 3) * Rp) * 8 + (j0 & 7);
#pragma unroll
        for (int c = 0; c < NC; ++c) f0[c] = p0[min(col0 + wave * NC + c, Rp - 1) * 8];
        if (a.nm > 1) {
            const float *p1 = a.panel[1] + ((j1 >> 3) * Rp) * 8 + (j1 & 7);
#pragma unroll
            for (int c = 0; c < NC; ++c) f1[c] = p1[min(col0 + wave * NC + c, Rp - 1) * 8];
        }
        if (a.nm > 2) {
            const float *p2 = a.panel[2] + ((j2 >> 3) * Rp) * 8 + (j2 & 7);
#pragma unroll
            for (int c = 0; c < NC; ++c) f2[c] = p2[min(col0 + wave * NC + c, Rp - 1) * 8];
        }
        if constexpr (M0) {
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int e = tid + 256 * u;
                int kq = e / TM;
                if constexpr (TM >= 64) kq = __builtin_amdgcn_readfirstlane(kq);
                const long r = min(row0 + e % TM, In - 1);
#pragma unroll
                for (int c = 0; c < 4; ++c) xv[4 * u + c] = X[r + min(kx + 4 * kq + c, K - 1) * In];
            }
        } else {
            kokx = kok;
            const ET *xp = X + (kok ? xo : 0);
            // opaque: hoisted out of the loop, the NL row offsets overflow the scalar registers
            long r0 = row0 + wave;
            asm volatile("" : "+s"(r0));
#pragma unroll
            for (int u = 0; u < NL; ++u) xv[u] = xp[min(r0 + 4 * u, In - 1) * P];
        }
    };
    auto advance = [&]() {
        kx += kAnyK;
        kl += kAnyK;
        i0 += a.T[0];
        i1 += a.T[1];
        i2 += a.T[2];
        if (i0 >= D0) {
            i0 -= D0;
            ++i1;
        }
        if (i1 >= D1) {
            i1 -= D1;
            ++i2;
        }
        if constexpr (!M0) {
            pk += TP;
            xo += TP + TQ * P * In;
            if (pk >= P) {
                pk -= P;
                xo += P * In - P;
            }
        }
    };

    any_d4 acc[RPW][NB];
#pragma unroll
    for (int rp = 0; rp < RPW; ++rp)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[rp][nb] = any_d4{0.0, 0.0, 0.0, 0.0};
    const int wr = wave % RW, wk = wave / RW;

    if (kbeg < kend) load();
    for (long k0 = kbeg; k0 < kend; k0 += kAnyK) {
        __syncthreads();  // every wave is done with the previous step's tiles
        if constexpr (M0) {
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int e = tid + 256 * u, kq = e / TM;
                float4 v;
                v.x = (k0 + 4 * kq + 0 < K) ? any_f32(xv[4 * u + 0]) : 0.0f;
                v.y = (k0 + 4 * kq + 1 < K) ? any_f32(xv[4 * u + 1]) : 0.0f;
                v.z = (k0 + 4 * kq + 2 < K) ? any_f32(xv[4 * u + 2]) : 0.0f;
                v.w = (k0 + 4 * kq + 3 < K) ? any_f32(xv[4 * u + 3]) : 0.0f;
                *reinterpret_cast<float4 *>(xs + (e % TM) * kAnyLd + 4 * kq) = v;
            }
        } else {
#pragma unroll
            for (int u = 0; u < NL; ++u) xs[(wave + 4 * u) * kAnyLd + lane] = kokx ? any_f32(xv[u]) : 0.0f;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            float v = f0[c];
            if (a.nm > 1) v *= f1[c];
            if (a.nm > 2) v *= f2[c];
            bs[(wave * NC + c) * kAnyLd + lane] = kok ? v : 0.0f;
        }
        __syncthreads();
        advance();
        load();  // past the last step: clamped addresses, never consumed
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < 4 / KW; ++q) {
            const int kb = 16 * (q * KW + wk) + 4 * lg;
            float4 av[RPW], bv[NB];
#pragma unroll
            for (int rp = 0; rp < RPW; ++rp)
                av[rp] = *reinterpret_cast<const float4 *>(xs + (16 * (RPW * wr + rp) + lm) * kAnyLd + kb);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                bv[nb] = *reinterpret_cast<const float4 *>(bs + (16 * nb + lm) * kAnyLd + kb);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                double bd[NB];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    bd[nb] = (double)(c == 0 ? bv[nb].x : c == 1 ? bv[nb].y : c == 2 ? bv[nb].z : bv[nb].w);
#pragma unroll
                for (int rp = 0; rp < RPW; ++rp) {
                    const double x = (double)(c == 0 ? av[rp].x : c == 1 ? av[rp].y : c == 2 ? av[rp].z : av[rp].w);
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        acc[rp][nb] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, bd[nb], acc[rp][nb], 0, 0, 0);
                }
            }
        }
    }
    // the waves that share rows, added in wave order
    if constexpr (KW > 1) {
        __syncthreads();
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int v = 0; v < 4; ++v) red[(wave * NB + nb) * 256 + 4 * lane + v] = acc[0][nb][v];
        __syncthreads();
        if (wk != 0) return;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                double s = red[(wr * NB + nb) * 256 + 4 * lane + v];
#pragma unroll
                for (int w = 1; w < KW; ++w) s += red[((wr + RW * w) * NB + nb) * 256 + 4 * lane + v];
                acc[0][nb][v] = s;
            }
    }
    // register v of lane (lm, lg): row lg + 4 v of the block, column lm
#pragma unroll
    for (int rp = 0; rp < RPW; ++rp)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const long r = row0 + 16 * (RPW * wr + rp) + lg + 4 * v;
            if (r >= In) continue;
            float sc = 1.0f;
            if constexpr (M0 && ST == 2) sc = a.row_scale[r];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const int col = col0 + 16 * nb + lm;
                if (col < Rp) a.partial[(split * In + r) * Rp + col] = (float)acc[rp][nb][v] * sc;
            }
        }
}

// rows per workgroup: the widest tile the extent fills (a tile's empty rows cost matrix work,
// not memory traffic)
static int any_tile(long In) { return In > 64 ? 128 : In > 32 ? 64 : In > 16 ? 32 : 16; }

void mttkrp_any_plan(MttkrpPlan &p) {
    const long In = p.dims[p.mode];
    long K = 1;
    size_t panels = 0;  // bytes of the factor panels, as the entry points lay them out
    for (int m = 0; m < p.order; ++m)
        if (m != p.mode) {
            K *= p.dims[m];
            panels += (sizeof(float) * (size_t)panel_floats(p.dims[m], p.Rp) + 255) & ~size_t(255);
        }
    p.rows_per_wg = any_tile(In);
    p.rowtiles = (int)ceil_div(In, (long)p.rows_per_wg);
    p.rows_pad = In;
    p.ksteps = K;
    const long ncb = ceil_div((long)p.Rp, (long)kAnyCols), steps = ceil_div(K, (long)kAnyK);
    // two workgroups per CU; at least four steps per split, so that its partial costs less to
    // sum than the split gains
    long ns = ceil_div(2L * device_cus(), (long)p.rowtiles * ncb);
    ns = std::min(ns, ceil_div(steps, 4L));
    // the partials and panels together stay within the fixed scratch of the no-allocation entry
    // point wherever one split does
    const size_t one = sizeof(float) * (size_t)In * p.Rp;
    if (panels < kNoAllocScratchBytes) ns = std::min(ns, (long)((kNoAllocScratchBytes - panels) / one));
    else ns = 1;
    if (ns < 1) ns = 1;
    p.ksteps_per_split = ceil_div(steps, ns) * kAnyK;
    p.nsplit = (int)ceil_div(K, p.ksteps_per_split);
}

template <int ST, bool M0, int RW, int RPW>
static void any_launch(const AnyArgs &a, int nb, int grid, hipStream_t s) {
    switch (nb) {
        case 1: k_mttkrp_any<ST, M0, 1, RW, RPW><<<grid, 256, 0, s>>>(a); break;
        case 2: k_mttkrp_any<ST, M0, 2, RW, RPW><<<grid, 256, 0, s>>>(a); break;
        case 3: k_mttkrp_any<ST, M0, 3, RW, RPW><<<grid, 256, 0, s>>>(a); break;
        default: k_mttkrp_any<ST, M0, 4, RW, RPW><<<grid, 256, 0, s>>>(a); break;
    }
}

template <int ST, bool M0>
static void any_launch(const AnyArgs &a, int tm, int nb, int grid, hipStream_t s) {
    if (tm == 128) any_launch<ST, M0, 4, 2>(a, nb, grid, s);
    else if (tm == 64) any_launch<ST, M0, 4, 1>(a, nb, grid, s);
    else if (tm == 32) any_launch<ST, M0, 2, 1>(a, nb, grid, s);
    else any_launch<ST, M0, 1, 1>(a, nb, grid, s);
}

int mttkrp_any_launch(const MttkrpPlan &p, const void *X, const float *const *panels, const float *row_scale,
                      float *partial, hipStream_t s, const int *skip) {
    AnyArgs a{};
    a.X = X;
    a.row_scale = row_scale;
    a.partial = partial;
    a.skip = skip;
    a.P = 1;
    a.K = 1;
    a.In = p.dims[p.mode];
    for (int m = 0; m < 3; ++m) a.D[m] = 1;
    for (int m = 0; m < p.order; ++m) {
        if (m == p.mode) continue;
        if (m < p.mode) a.P *= p.dims[m];
        a.K *= p.dims[m];
        a.D[a.nm] = p.dims[m];
        a.panel[a.nm++] = panels[m];
    }
    a.T[0] = kAnyK % a.D[0];
    a.T[1] = (kAnyK / a.D[0]) % a.D[1];
    a.T[2] = kAnyK / a.D[0] / a.D[1];
    a.kper = p.ksteps_per_split;
    a.Rp = p.Rp;
    a.rowtiles = p.rowtiles;
    a.ncb = (int)ceil_div((long)p.Rp, (long)kAnyCols);
    const int nb = p.Rp >= kAnyCols ? 4 : p.Rp / 16, tm = p.rows_per_wg;
    const int grid = a.rowtiles * a.ncb * p.nsplit;
    const bool m0 = p.mode == 0;
    if (p.dtype == TDX_F32) {
        if (m0) any_launch<0, true>(a, tm, nb, grid, s);
        else any_launch<0, false>(a, tm, nb, grid, s);
    } else if (p.dtype == TDX_BF16) {
        if (m0) any_launch<1, true>(a, tm, nb, grid, s);
        else any_launch<1, false>(a, tm, nb, grid, s);
    } else {
        if (m0) any_launch<2, true>(a, tm, nb, grid, s);
        else any_launch<2, false>(a, tm, nb, grid, s);
    }
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

}  // namespace tdx
