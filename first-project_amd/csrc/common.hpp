// common.hpp -- shared host/device definitions of libtdx (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>
#include "../../include/tdx.h"

namespace tdx {

// ---- status plumbing -------------------------------------------------------
int record(int status);
int record_hip(hipError_t e, const char *what, const char *file, int line);
hipStream_t stream();
// compute units of the current device (cached per device)
int device_cus();

#define TDX_HIP(call)                                                              \
    do {                                                                           \
        hipError_t e_ = (call);                                                    \
        if (e_ != hipSuccess) return tdx::record_hip(e_, #call, __FILE__, __LINE__); \
    } while (0)

#define TDX_TRY(call)                  \
    do {                               \
        const int st_ = (call);        \
        if (st_ != TDX_OK) return st_; \
    } while (0)

#define TDX_CHECK_ARG(cond)                          \
    do {                                             \
        if (!(cond)) return tdx::record(TDX_ERR_ARG); \
    } while (0)

#define TDX_LAUNCH_CHECK() TDX_HIP(hipGetLastError())

// ---- workspace pool: grow-only named slots, reused across calls --------------
enum WsSlot {
    WS_PARTIAL = 0,  // MTTKRP split-K partial sums
    WS_PANEL0,       // factor panels (one slot per mode)
    WS_PANEL1,
    WS_PANEL2,
    WS_PANEL3,
    WS_MISC0,
    WS_MISC1,
    WS_MISC2,
    WS_MISC3,
    WS_STORE,        // CP-ALS: the BF16 / FP8 copy of the tensor for the main phase
    WS_STORE_SCALES, // CP-ALS: its FP8 slice scales
    WS_STORE_BF16,   // CP-ALS, FP8 storage with split-operand opening sweeps: the BF16 copy
    WS_COUNT
};
int workspace(int slot, size_t bytes, void **ptr);
void release_workspace();

// ---- exclusive leases: device memory and streams a synchronous call holds until it returns ------
// A call used to allocate and free these each time (HOSVD + HOOI of 128^4, 0.9 GB: 1.2 ms of 4.0; the
// batched CP-ALS of 1024 tensors: 0.5 ms of 3.6).  A lease takes an idle block of the current device
// that is large enough (the smallest such) or allocates one; nobody else has it meanwhile, so calls
// from several threads and on several streams do not meet.  done() says that all work on it has
// finished: the destructor then keeps it for a later call, up to 4 idle blocks of 2 GiB together and 4
// idle streams; without it (a call that failed) or past those bounds it is freed.
// tdx_release_workspace frees what is idle, and so does a device_malloc that finds no memory.
class DeviceLease {
  public:
    DeviceLease() = default;
    DeviceLease(const DeviceLease &) = delete;
    DeviceLease &operator=(const DeviceLease &) = delete;
    ~DeviceLease();
    int take(size_t bytes);
    void done() { done_ = true; }
    char *ptr() const { return (char *)p_; }

  private:
    void *p_ = nullptr;
    size_t bytes_ = 0;
    int dev_ = 0;
    bool done_ = false;
};
// a blocking stream of default priority
class StreamLease {
  public:
    StreamLease() = default;
    StreamLease(const StreamLease &) = delete;
    StreamLease &operator=(const StreamLease &) = delete;
    ~StreamLease();  // waits for the stream first
    int take();
    void done() { done_ = true; }
    hipStream_t get() const { return s_; }

  private:
    hipStream_t s_ = nullptr;
    int dev_ = 0;
    bool done_ = false;
};
void release_leases();
// hipMalloc for everything the library allocates: where memory has run out, again after the idle
// leases and the cached CP-ALS plans, which no call is using, have been freed
int device_malloc(void **p, size_t bytes);
template <typename T>
int device_malloc(T **p, size_t bytes) {
    return device_malloc((void **)p, bytes);
}
// consecutive parts of one block, 256-byte aligned
struct Parts {
    size_t bytes = 0;
    size_t add(size_t n) {
        const size_t o = bytes;
        bytes += (n + 255) & ~size_t(255);
        return o;
    }
};
// frees the cached CP-ALS plans (als.hip); tdx_release_workspace calls it
void release_cp_plans();
// the fixed device scratch of tdx_mttkrp_ex_noalloc (64 MiB per GPU): its address on the
// current device, taken once per device by hipGetSymbolAddress (mttkrp.hip)
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
int noalloc_scratch(void **ptr);
// FP8 mode-1 slice quantisation in steps (elementwise.hip): slice_amax zeroes and fills amax[I];
// fp8_from_amax writes the scales (max / 448, 1 for an all-zero slice) and the E4M3 codes
int slice_amax(const float *X, uint32_t *amax, long I, long n_rest, hipStream_t s);
int fp8_from_amax(const float *X, const uint32_t *amax, uint8_t *Xq, float *scales, long I, long n_rest,
                  hipStream_t s);

__host__ __device__ inline long ceil_div(long a, long b) { return (a + b - 1) / b; }

// Streaming (nontemporal) loads for data read exactly once per kernel, such as the tensor in
// MTTKRP: on MI355X a read stream of 16-byte nontemporal loads runs at ~7.1 TB/s against
// ~6.3 TB/s with the default cache policy.
__device__ __forceinline__ uint4 ld_stream(const uint4 *p) {
    typedef unsigned v4 __attribute__((ext_vector_type(4)));
    const v4 t = __builtin_nontemporal_load(reinterpret_cast<const v4 *>(p));
    return uint4{t.x, t.y, t.z, t.w};
}
__device__ __forceinline__ float4 ld_stream(const float4 *p) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    const v4 t = __builtin_nontemporal_load(reinterpret_cast<const v4 *>(p));
    return float4{t.x, t.y, t.z, t.w};
}
__device__ __forceinline__ uint2 ld_stream(const uint2 *p) {
    typedef unsigned v2 __attribute__((ext_vector_type(2)));
    const v2 t = __builtin_nontemporal_load(reinterpret_cast<const v2 *>(p));
    return uint2{t.x, t.y};
}

// ---- FP32 values as three BF16 parts (mttkrp_f32.hip, dtree_wide.hip, gram_f32.hip) -------------
// Two values rounded to nearest even, in one register: a conversion instruction that the compiler knows
// (inside an asm statement it is placed without regard to matrix instructions that still read or write
// its register), opaque so that the halves taken out of it are not converted once more each.
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{lo, hi}), b2));
    asm("" : "+v"(w));
    return w;
}
// A value below 2^-100, unless it is zero, would lose bits of its last part.  small_key orders the
// magnitudes as unsigned integers with zero past every value, so the least key of a tile says whether
// it holds such an entry.
constexpr uint32_t kSmallKey = 2u * 0x0d800000u - 1u;  // of 2^-100
__device__ __forceinline__ uint32_t small_key(float v) { return 2u * __float_as_uint(v) - 1u; }
// Such a tile is multiplied twice, half 0 with the entries from 2^-64 up, half 1 with the others times
// 2^64 (exact; NaN stays in half 0).
__device__ __forceinline__ float magnitude_half(float v, int half) {
    const bool small = fabsf(v) < 0x1p-64f;
    return half ? (small ? v * 0x1p64f : 0.0f) : (small ? 0.0f : v);
}

// ---- device helpers ------------------------------------------------------------
__device__ __forceinline__ uint32_t f2u(float x) { return __float_as_uint(x); }
__device__ __forceinline__ float u2f(uint32_t u) { return __uint_as_float(u); }

// IEEE round-to-nearest-even FP32 -> BF16 (NaN kept quiet); identical to the oracle
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float x) {
    uint32_t u = f2u(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// OCP E4M3FN, RNE, saturating at 448, NaN -> 0x7f (software rounding, bit-exact by construction)
__device__ __forceinline__ uint8_t f32_to_e4m3_bits(float x) {
    uint32_t u = f2u(x);
    uint8_t sign = (uint8_t)((u >> 24) & 0x80u);
    uint32_t au = u & 0x7fffffffu;
    if (au > 0x7f800000u) return (uint8_t)(sign | 0x7f);
    float ax = u2f(au);
    if (ax >= 464.0f) return (uint8_t)(sign | 0x7e);
    if (ax < 0.015625f) {
        // quantum 2^-9: scale exactly into integer+fraction, round half to even
        float v = ax * 512.0f;  // exact (power of two scaling, no underflow for normals >= 2^-126 * 512)
        float fl = floorf(v);
        float rem = v - fl;
        uint32_t m = (uint32_t)fl;
        if (rem > 0.5f || (rem == 0.5f && (m & 1u))) m++;
        return (uint8_t)(sign | m);
    }
    int e = (int)((au >> 23) & 0xff) - 127;
    uint32_t mant = au & 0x7fffffu;
    uint32_t q = ((uint32_t)(e + 7) << 3) | (mant >> 20);
    uint32_t rem = mant & 0xfffffu;
    if (rem > 0x80000u || (rem == 0x80000u && (q & 1u))) q++;
    if (q > 0x7e) q = 0x7e;
    return (uint8_t)(sign | q);
}

// Philox-4x32-10 (Salmon et al., SC'11) -- same stream definition as the oracle
__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        uint32_t lo0 = 0xD2511F53u * c[0];
        uint32_t hi0 = __umulhi(0xD2511F53u, c[0]);
        uint32_t lo1 = 0xCD9E8D57u * c[2];
        uint32_t hi1 = __umulhi(0xCD9E8D57u, c[2]);
        uint32_t n0 = hi1 ^ c[1] ^ k0;
        uint32_t n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0; c[1] = lo1; c[2] = n2; c[3] = lo0;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

__device__ __forceinline__ uint32_t philox_word(uint64_t seed, uint32_t strm, uint64_t n) {
    uint64_t blk = n >> 2;
    uint32_t c[4] = {(uint32_t)blk, (uint32_t)(blk >> 32), strm, 0u};
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    return c[n & 3];
}

__device__ __forceinline__ float word_to_uniform(uint32_t w) {
    return ((float)(w >> 9) + 0.5f) * (1.0f / 8388608.0f);
}

}  // namespace tdx
