// batched.hpp -- shared by the batched CP-ALS designs (batched.hip, batched_items.hip).
#pragma once
#include "common.hpp"
#include <vector>

namespace tdx {

constexpr int kBMaxDim = 128;
constexpr int kBMaxR = 16;
constexpr int kSlabCols = 128;  // columns per slab (per-column scratch Ys)

struct BDesc {
    long xoff;
    long uoff[3];
    int I, J, K, R;
    long toff;  // split design with T: X x_0 A^T of the tensor (J K x R floats) at toff
};

typedef float bf32x4 __attribute__((ext_vector_type(4)));

// sum over the workgroup: wave shuffles, then one value per wave through LDS (sh >= BS/64
// doubles); every thread returns the total
template <int BS>
__device__ inline double bsum(double v, double *sh) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int tid = threadIdx.x;
    __syncthreads();
    if ((tid & 63) == 0) sh[tid >> 6] = v;
    __syncthreads();
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < BS / 64; ++w) r += sh[w];
    return r;
}

__device__ inline int sel3(int m, int a, int b, int c) { return m == 0 ? a : (m == 1 ? b : c); }
__device__ inline long sel3l(int m, long a, long b, long c) { return m == 0 ? a : (m == 1 ? b : c); }


// ---- the item design (batched_items.hip) ----
// A tensor's slices X(:, :, k) in runs of kc; every run is one workgroup's work item
struct IDesc {
    long xoff, toff, pbase;  // floats: the tensor, its T, its first item's partial
    long uoff[3];
    int I, J, K, R;
    int Rq;                  // columns of T (4, 8 or 16)
    int kc, nit, pstep;      // slices per item, items, floats between the items' partials
    int item0;               // first item (index into the norm partials)
};
struct IItem {
    int t, k0, k1, id;
    long poff;
};
struct ItemPlan {
    std::vector<IDesc> desc;
    std::vector<IItem> items;  // largest first
    long part_floats = 0, t_floats = 0;
};
void items_plan(ItemPlan &p, const BDesc *d, long n);
struct ItemBuffers {
    const IDesc *desc;
    const IItem *items;
    int ntensors, nitems;
    float *part, *T;
    double *G, *npart;
};
// ||X||^2 of every tensor and the Grams of the initial factors
int items_prologue(const ItemBuffers &b, const float *X, const float *U, double *normx2, hipStream_t s);
// one sweep; *sweep_ctr counts the sweeps begun (-1 before the first)
int items_sweep(const ItemBuffers &b, const float *X, float *U, const double *normx2, double *fit, int max_sweeps,
                int *sweep_ctr, int *status, hipStream_t s);

}  // namespace tdx
