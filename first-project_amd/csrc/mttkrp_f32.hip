// mttkrp_f32.hip -- fused MTTKRP of an FP32 tensor (orders 3 and 4, rank <= 64, whole 16-byte
// vectors along mode 0), its products formed from three BF16 parts per operand.
//
//   M[i_n, r] = sum_slow w_slow[r] (sum_f X[i_n, f, slow] P_f[f, r]),
//   w_slow[r] = prod over the other contracted modes of their factor rows:
// the inner sum over a chunk of 64 fast indices is a product with the same 64 x Rp panel block for
// every slow index, so that block is prepared once per chunk and no Khatri-Rao block is formed; w
// scales the finished 64-term sums on their way into the FP32 accumulator, which also keeps the
// chains of FP32 roundings short (64 products, then one term per slow index).
//
// Products: x = x1 + x2 + x3 exactly, each part what is left rounded to BF16, and the same for p;
// v_mfma_f32_16x16x32_bf16 multiplies x1 p1, x1 p2, x2 p1, x1 p3, x2 p2 and x3 p1 exactly and adds
// them in FP32.  The terms left out are below 2^-25 of |x p|, of either sign: less than the
// rounding of an FP32 product.  (Parts cut off instead of rounded leave 2^-22, always of the
// product's sign, which does not average out.)  Six BF16 products take 0.38 of the time of the FP32
// matrix instruction and less power: with that one the kernel ran at 1.8-2.1 GHz.  The parts of X
// are cut in registers as the operands are read (5.5 vector operations an element, once).
//   * A panel column is scaled by a power of two to a largest entry in [1, 2) (undone in w), so
//     that factors of uneven magnitude neither overflow nor lose bits in the 64-term sums.
//   * An infinity has no such parts (inf - inf), and sums of values near the largest would overflow
//     before w scales them: a tile with entries above 2^119 and a chunk whose panel holds an infinity
//     are multiplied in FP32 (v_mfma_f32_16x16x4_f32) by w p instead.  NaN stays NaN.
//   * An entry below 2^-110 would lose bits of its last part, down to 11 of 24 at 2^-120: a tile with
//     any entry below 2^-100 but zero is multiplied in two halves of its magnitudes (magnitude_half).
//     The least magnitude is found with the largest; only tiles where it is below 2^-100 are looked
//     over for what is not zero.  (Panel entries keep 2^-134 of their column's largest in the chunk.)
//     Without such entries 0.2 us of a launch of 7 (64 x 48 x 40) and nothing at 1024^3; with one entry
//     in five such, 512^3 rank 16 92 / 98 / 107 -> 160 / 183 / 183 us, rank 64 129 / 157 / 172 -> 273 /
//     298 / 273.
// Errors against 64 bits, FP32 products with one long chain of sums before: 2.3e-6 -> 3.1e-7
// (1024^3 rank 64), 8.5e-7 -> 1.5e-7 (512^3 rank 33), 4.4e-7 -> 1.1e-7 (128^3 rank 16).
// Bound by power (1.65-1.7 GHz while the tensor streams; matrix pipe 46 %, LDS 27 %) and HBM.  Modes 0 / 1 / 2, FP32 matrix
// instructions before: 1024^3 rank 64 1352 / 1223 / 1212 -> 1104 / 980 / 1009 us (0.66 ms is the
// stream's time at 6.5 TB/s), rank 32 806 / 790 / 790 -> 717 / 694 / 753, rank 16 664 / 669 / 655
// -> 621 / 658 / 669; 256^3 rank 20 20-21 -> 17-19; 640 x 72 x 1024 rank 40 89 / 89 / 55 -> 68 / 59
// / 45.  Two workgroups per CU: three leave 168 registers, which spill from 32 columns on (512^3
// rank 32: 103 / 118 / 123 us, 88 / 90 / 103 with two).
//
// Work of a workgroup (the plan of the LDS kernel): 128 output rows, one chunk of 64 fast indices
// (rarely a group of chunks) and a range of slow indices.  Each of its waves owns 32 rows and
// runs on its own, without a barrier: a 32 x 64 tile goes from 16-byte loads of whole lines into
// the wave's part of LDS (rows of 68 floats) and comes back 8 consecutive f a lane; the next
// tile's loads are in flight meanwhile.
//   n > 0: rows are strided; 16 lanes read the 256 bytes of a row, 4 rows a load.
//   n = 0 (TR): rows are contiguous; 8 lanes read the 128 bytes of a fast index, 8 fast indices a
//     load; lane group g holds f = 8 g .. + 7 of four rows, which leave as 16-byte stores of 4 f
//     each; row 4 j + t goes to LDS row 8 t + j, so a store's lanes hit distinct banks, and the
//     rows are mapped back when the partial is written.
#include "mttkrp.hpp"
#include "vinv.hpp"

namespace tdx {

typedef float mf_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 mf_b8 __attribute__((ext_vector_type(8)));

static constexpr int kMfLd = 68;

struct MfArgs {
    const float *X;
    const float *panel[4];
    const float *fpanel;
    float *partial;
    const int *skip;
    long stride[4];
    long dims[4];
    long In, If, S, sper, rows_pad;
    int mode, nslow, rowtiles;
    int cps, nss, ncg;
    int slow[2];
};

// the three parts of 8 consecutive values, packed as BF16 operands
struct MfParts {
    uint4 p[3];
};
struct MfRows {
    MfParts r[2];
};
__device__ __forceinline__ MfParts mf_split(const mf_f4 &a, const mf_f4 &b) {
    float v[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    MfParts o;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        uint32_t w[4];
#pragma unroll
        for (int h = 0; h < 4; ++h) {
            w[h] = bf16_pair(v[2 * h], v[2 * h + 1]);
            v[2 * h] -= __uint_as_float(w[h] << 16);
            v[2 * h + 1] -= __uint_as_float(w[h] & 0xffff0000u);
        }
        o.p[k] = uint4{w[0], w[1], w[2], w[3]};
    }
    return o;
}
__device__ __forceinline__ mf_b8 mf_op(const uint4 &v) { return __builtin_bit_cast(mf_b8, v); }

template <int NB, bool TR>
__device__ __forceinline__ void mf_block(const MfArgs &a, const int block) {
    constexpr int Rp = 16 * NB;
    __shared__ __attribute__((aligned(16))) float lds[4][32 * kMfLd];
    __shared__ uint4 bs[2 * 3 * NB * 64];  // [k-step][part][column block][lane]
    __shared__ float scl[Rp], mxs[8][Rp];
    __shared__ int inf_s;
    if (a.skip && *a.skip) return;
    const int tid = threadIdx.x, lane = tid & 63, lm = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    float *xs = lds[wave];
    // workgroups that run side by side read whole rows of the tensor between them: adjacent row
    // tiles for TR, adjacent chunk groups otherwise
    int rowtile;
    long cgroup, srange;
    if constexpr (TR) {
        rowtile = block % a.rowtiles;
        const long split = block / a.rowtiles;
        cgroup = split / a.nss;
        srange = split % a.nss;
    } else {
        cgroup = block % a.ncg;
        const long rest = block / a.ncg;
        rowtile = (int)(rest % a.rowtiles);
        srange = rest / a.rowtiles;
    }
    const long split = cgroup * a.nss + srange;
    const long row0 = (long)rowtile * 128 + 32 * wave;
    const long nfc = ceil_div(a.If, 64L);
    const long fc0 = cgroup * a.cps, fc1 = min(fc0 + a.cps, nfc);
    const long sl0 = srange * a.sper, nsl = min(sl0 + a.sper, a.S) - sl0;
    const long sn = a.stride[a.mode], sf = TR ? a.stride[1] : 1;
    float *dst = a.partial + (split * a.rows_pad + row0) * Rp;

    mf_f4 acc[2][NB];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[rb][nb] = mf_f4{0.f, 0.f, 0.f, 0.f};

    const int sm0 = a.slow[0], sm1 = (a.nslow > 1) ? a.slow[1] : a.slow[0];
    const long sd0 = a.dims[sm0], st0 = a.stride[sm0], st1 = (a.nslow > 1) ? a.stride[sm1] : 0;
    if (nsl > 0)
        for (long fc = fc0; fc < fc1; ++fc) {
            const long f0 = fc * 64;
            const bool full = f0 + 64 <= a.If;
            // this lane's loads: n > 0 rows lane / 16 + 4 u at f = 4 (lane % 16); TR rows
            // 4 (lane % 8) .. + 3 at f = 8 (lane / 8) + u.  Past the extents: valid addresses.
            const float *xp[8];
            uint32_t ok = 0;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const long f = f0 + (TR ? 8 * (lane >> 3) + u : 4 * (lane & 15));
                const long r = row0 + (TR ? 4 * (lane & 7) : (lane >> 4) + 4 * u);
                const bool in = f < a.If;
                ok |= (uint32_t)in << u;
                // (TR: the extent is a multiple of 4 rows, so a group of 4 is whole)
                xp[u] = a.X + (in ? f : 0) * sf + min(r, TR ? a.In - 4 : a.In - 1) * (TR ? 1 : sn);
            }
            // the next slow index to load: digits, tensor offset, indices left (the last repeats)
            long i0 = sl0 % sd0, i1 = (a.nslow > 1) ? sl0 / sd0 : 0, off = i0 * st0 + i1 * st1, left = nsl;
            struct Buf {
                float4 x[8];
                float wa[NB], wb[NB];
            };
            auto load = [&](Buf &b) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    b.wa[nb] = a.panel[sm0][((i0 >> 3) * Rp + 16 * nb + lm) * 8 + (i0 & 7)];
                    // (one slow mode: its row 0, unused; a conditional load went through scratch)
                    b.wb[nb] = a.panel[sm1][((i1 >> 3) * Rp + 16 * nb + lm) * 8 + (i1 & 7)];
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) b.x[u] = ld_stream(reinterpret_cast<const float4 *>(xp[u] + off));
                if (left > 1) {
                    --left;
                    ++i0;
                    off += st0;
                    if (i0 == sd0) {
                        i0 = 0;
                        ++i1;
                        off += st1 - sd0 * st0;
                    }
                }
            };
            Buf A;
            load(A);  // the first tile is on its way while the panel chunk is prepared
            // the panel chunk: its scaled parts in operand order (entry (ks, k, nb, lane):
            // P[f0 + 32 ks + 8 lg .. + 7][16 nb + lm]; zero past the extent)
            constexpr int NE = (2 * NB + 3) / 4;
            mf_f4 pv[NE][2];
            __syncthreads();  // (a group of chunks: every wave is done with the previous ones)
            if (tid == 0) inf_s = 0;
#pragma unroll
            for (int j = 0; j < NE; ++j) {
                const int e = min(wave + 4 * j, 2 * NB - 1), ks = e / NB, c = 16 * (e % NB) + lm;
                const float *pp = a.fpanel + (((f0 + 32 * ks + 8 * lg) >> 3) * Rp + c) * 8;
                pv[j][0] = *reinterpret_cast<const mf_f4 *>(pp);
                pv[j][1] = *reinterpret_cast<const mf_f4 *>(pp + 4);
                float m = 0.0f;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(pv[j][h][0]), "v"(pv[j][h][1]));
                    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(pv[j][h][2]), "v"(pv[j][h][3]));
                }
                mxs[4 * ks + lg][c] = m;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < NE; ++j) {
                const int e = min(wave + 4 * j, 2 * NB - 1), ks = e / NB, nb = e % NB, c = 16 * nb + lm;
                float m = mxs[0][c];
#pragma unroll
                for (int g = 1; g < 8; ++g) m = fmaxf(m, mxs[g][c]);
                if (m == __uint_as_float(0x7f800000u)) inf_s = 1;
                // (2^126 and 2^-126 at the ends, where 2^-x has no normal value)
                int x = (int)(__float_as_uint(m) >> 23) - 127;
                x = x > 126 ? 126 : x < -126 ? -126 : x;
                if (ks == 0 && lg == 0) scl[c] = __uint_as_float((uint32_t)(127 + x) << 23);
                const float s = __uint_as_float((uint32_t)(127 - x) << 23);
                const MfParts q = mf_split(pv[j][0] * s, pv[j][1] * s);
#pragma unroll
                for (int k = 0; k < 3; ++k) bs[((ks * 3 + k) * NB + nb) * 64 + lane] = q.p[k];
            }
            __syncthreads();
            if (row0 >= a.In) continue;
            const bool pinf = inf_s != 0;
            float sc[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) sc[nb] = scl[16 * nb + lm];
            auto step = [&](Buf &b) {
                float w[NB];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) w[nb] = (a.nslow > 1) ? b.wa[nb] * b.wb[nb] : b.wa[nb];
                // (before the entries past the extent become zero: they are entries of the tensor still)
                float big = 0.0f, least = __uint_as_float(0x7f800000u);  // magnitudes (NaN left out)
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(big) : "v"(b.x[u].x), "v"(b.x[u].y));
                    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(big) : "v"(b.x[u].z), "v"(b.x[u].w));
                    asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(least) : "v"(b.x[u].x), "v"(b.x[u].y));
                    asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(least) : "v"(b.x[u].z), "v"(b.x[u].w));
                }
                bool fp32 = false, halves = false;
                if (__builtin_expect(pinf || __any(big > 0x1p119f || least < 0x1p-100f), 0)) {
                    fp32 = pinf || __any(big > 0x1p119f);
                    uint32_t key = ~0u;
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        key = min(key, min(min(small_key(b.x[u].x), small_key(b.x[u].y)),
                                           min(small_key(b.x[u].z), small_key(b.x[u].w))));
                    halves = __any(key < kSmallKey);
                }
                if (!full) {
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (!((ok >> u) & 1u)) b.x[u] = float4{0.f, 0.f, 0.f, 0.f};
                }
                // (a wave's LDS operations complete in order: no barrier between its stores and loads)
                __builtin_amdgcn_wave_barrier();
                if constexpr (TR) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        float v[8];
#pragma unroll
                        for (int u = 0; u < 8; ++u)
                            v[u] = t == 0 ? b.x[u].x : t == 1 ? b.x[u].y : t == 2 ? b.x[u].z : b.x[u].w;
                        float *d = xs + (8 * t + (lane & 7)) * kMfLd + 8 * (lane >> 3);
                        *reinterpret_cast<float4 *>(d) = float4{v[0], v[1], v[2], v[3]};
                        *reinterpret_cast<float4 *>(d + 4) = float4{v[4], v[5], v[6], v[7]};
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        *reinterpret_cast<float4 *>(xs + ((lane >> 4) + 4 * u) * kMfLd + 4 * (lane & 15)) = b.x[u];
                }
                __builtin_amdgcn_wave_barrier();
                load(b);
                __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the MFMAs
                if (__builtin_expect(fp32, 0)) {
                    // FP32 products with w times the unscaled panel
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                        for (int rb = 0; rb < 2; ++rb) {
                            mf_f4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
                            for (int q = 0; q < 4; ++q) {
                                const mf_f4 av = *reinterpret_cast<const mf_f4 *>(xs + (16 * rb + lm) * kMfLd + 16 * q + 4 * lg);
                                const long i = f0 + 16 * q + 4 * lg;
                                const mf_f4 bv = *reinterpret_cast<const mf_f4 *>(
                                    a.fpanel + ((i >> 3) * Rp + 16 * nb + lm) * 8 + (i & 7));
#pragma unroll
                                for (int c = 0; c < 4; ++c)
                                    t = __builtin_amdgcn_mfma_f32_16x16x4f32(av[c], w[nb] * bv[c], t, 0, 0, 0);
                            }
                            acc[rb][nb] += t;
                        }
                    return;
                }
                auto split_rows = [&](int ks, auto value) {
                    MfRows x;
#pragma unroll
                    for (int rb = 0; rb < 2; ++rb) {
                        const float *xp = xs + (16 * rb + lm) * kMfLd + 32 * ks + 8 * lg;
                        mf_f4 u = *reinterpret_cast<const mf_f4 *>(xp), v = *reinterpret_cast<const mf_f4 *>(xp + 4);
#pragma unroll
                        for (int c = 0; c < 4; ++c) u[c] = value(u[c]), v[c] = value(v[c]);
                        x.r[rb] = mf_split(u, v);
                    }
                    return x;
                };
                // s + the products of row block rb, smallest terms first
                auto products = [&](const MfParts &x, const uint4 (&p)[3], mf_f4 s) {
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mf_op(x.p[2]), mf_op(p[0]), s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mf_op(x.p[0]), mf_op(p[2]), s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mf_op(x.p[1]), mf_op(p[1]), s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mf_op(x.p[1]), mf_op(p[0]), s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mf_op(x.p[0]), mf_op(p[1]), s, 0, 0, 0);
                    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(mf_op(x.p[0]), mf_op(p[0]), s, 0, 0, 0);
                };
                if (__builtin_expect(halves, 0)) {
                    // (a k-step of a half at a time: arranged as below, registers spill)
#pragma unroll 1
                    for (int h = 0; h < 4; ++h) {
                        const int ks = h & 1, half = h >> 1;
                        const MfRows x = split_rows(ks, [&](float v) { return magnitude_half(v, half); });
                        // (2^-64 is taken out of both factors, so that neither underflows)
                        const float down = half ? 0x1p-32f : 1.0f;
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb) {
                            uint4 p[3];
#pragma unroll
                            for (int k = 0; k < 3; ++k) p[k] = bs[((ks * 3 + k) * NB + nb) * 64 + lane];
                            const float ws = w[nb] * sc[nb] * down;
#pragma unroll
                            for (int rb = 0; rb < 2; ++rb) {
                                const mf_f4 s = products(x.r[rb], p, mf_f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                                for (int v = 0; v < 4; ++v) acc[rb][nb][v] = fmaf(s[v] * down, ws, acc[rb][nb][v]);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                    return;
                }
                mf_f4 t[2][NB];
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    const MfRows x = split_rows(ks, [](float v) { return v; });
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) {
                        uint4 p[3];
#pragma unroll
                        for (int k = 0; k < 3; ++k) p[k] = bs[((ks * 3 + k) * NB + nb) * 64 + lane];
#pragma unroll
                        for (int rb = 0; rb < 2; ++rb)
                            t[rb][nb] = products(x.r[rb], p, ks == 0 ? mf_f4{0.f, 0.f, 0.f, 0.f} : t[rb][nb]);
                    }
                }
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    const float ws = w[nb] * sc[nb];
#pragma unroll
                    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                        for (int v = 0; v < 4; ++v) acc[rb][nb][v] = fmaf(t[rb][nb][v], ws, acc[rb][nb][v]);
                }
            };
            for (long s = 0; s < nsl; ++s) step(A);
        }
    // register v of lane (lm, lg): LDS row 16 rb + 4 lg + v, column lm of each block
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int j = 16 * rb + 4 * lg + v, r = TR ? 4 * (j & 7) + (j >> 3) : j;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) dst[r * Rp + 16 * nb + lm] = acc[rb][nb][v];
        }
}

template <int NB, bool TR>
__global__ __launch_bounds__(256, 2) void k_mttkrp_f32(MfArgs a) {
    mf_block<NB, TR>(a, blockIdx.x);
}

// A CP-ALS sweep at rank <= 16: the first workgroup computes the mode's inverse, which depends on
// what this product depends on, so a mode is two launches instead of three (128^3 rank 16: 7.4 us for
// the product and 5.8 for the inverse in a row, 7.3 to 8.1 with both in one launch; 20 sweeps 1.69 ->
// 1.32 ms).
template <bool TR>
__global__ __launch_bounds__(256, 2) void k_mttkrp_f32_inv(MfArgs a, VinvJob j) {
    if (blockIdx.x == 0) vinv_job<4>(j);
    else mf_block<1, TR>(a, blockIdx.x - 1);
}

int mttkrp_f32_launch(const MttkrpPlan &p, const void *X, const float *const *panels, float *partial, hipStream_t s,
                      const int *skip, const VinvJob *inverse) {
    MfArgs a{};
    a.X = (const float *)X;
    const int fm = (p.mode == 0) ? 1 : 0;
    long st = 1;
    for (int m = 0; m < 4; ++m) {
        a.panel[m] = (m < p.order) ? panels[m] : nullptr;
        a.dims[m] = (m < p.order) ? p.dims[m] : 1;
        a.stride[m] = st;
        st *= a.dims[m];
    }
    a.fpanel = panels[fm];
    a.partial = partial;
    a.skip = skip;
    a.mode = p.mode;
    a.In = p.dims[p.mode];
    a.If = p.dims[fm];
    a.rowtiles = p.rowtiles;
    a.rows_pad = p.rows_pad;
    a.S = p.ksteps;
    a.sper = p.ksteps_per_split;
    a.cps = p.lds_cps;
    a.nss = p.lds_nss;
    a.ncg = p.nsplit / p.lds_nss;
    for (int m = 1; m < p.order; ++m)
        if (m != p.mode && m != fm) a.slow[a.nslow++] = m;
    const int grid = p.rowtiles * p.nsplit;
#define TDX_F32_LAUNCH(NB_)                                                  \
    do {                                                                     \
        if (p.mode == 0) k_mttkrp_f32<NB_, true><<<grid, 256, 0, s>>>(a);    \
        else k_mttkrp_f32<NB_, false><<<grid, 256, 0, s>>>(a);               \
    } while (0)
    if (inverse) {
        if (p.mode == 0) k_mttkrp_f32_inv<true><<<grid + 1, 256, 0, s>>>(a, *inverse);
        else k_mttkrp_f32_inv<false><<<grid + 1, 256, 0, s>>>(a, *inverse);
        TDX_LAUNCH_CHECK();
        return TDX_OK;
    }
    switch (p.Rp / 16) {
        case 1: TDX_F32_LAUNCH(1); break;
        case 2: TDX_F32_LAUNCH(2); break;
        case 3: TDX_F32_LAUNCH(3); break;
        default: TDX_F32_LAUNCH(4); break;
    }
#undef TDX_F32_LAUNCH
    TDX_LAUNCH_CHECK();
    return TDX_OK;
}

}  // namespace tdx
