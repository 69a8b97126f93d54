// mas_tail.h -- the coarse end ("tail") of the MAS apply: the levels whose R
// fits one workgroup's LDS, shared by k_mas_finish (mas.hip) and the
// one-launch PCG (persist.hip).
#pragma once

#include "linsys.h"

namespace sgipc
{

constexpr int BANK = 16;
constexpr int BD   = 48;  // 3 * BANK
constexpr int ZB   = 64;  // Z entries per bank: one per lane, lanes 48..63 padding

constexpr int kMaxLevels = 6;  // compute_num_levels' bound
struct TailPlan
{
    int lt    = 0;  // first tail level (L: no tail)
    int base  = 0;  // global id of the tail's first node (a multiple of 16)
    int span  = 0;  // padded nodes of the tail
    int first = 0;  // padded nodes of level lt
    int count[kMaxLevels] = {};
    int off[kMaxLevels]   = {};
};

// the plan whose tail starts at the first level >= 1 with fits(span, levels)
template <typename F>
inline TailPlan tail_plan(int L, const std::vector<int>& lvl, F&& fits)
{
    TailPlan tp;
    for(int q = 0; q < L; q++)
    {
        tp.count[q] = lvl[2 * q];
        tp.off[q]   = lvl[2 * q + 1];
    }
    for(tp.lt = 1; tp.lt < L; tp.lt++)
    {
        tp.base  = tp.off[tp.lt];
        tp.first = (tp.count[tp.lt] + BANK - 1) / BANK * BANK;
        tp.span  = (tp.off[L - 1] + tp.count[L - 1] - tp.base + BANK - 1) / BANK * BANK;
        if(fits(tp.span, L - tp.lt))
            return tp;
    }
    tp.base = tp.span = tp.first = 0;
    return tp;
}

// Ordering of LDS between the lanes of one wave: the LDS instructions of a
// wave execute in program order, so a compiler-only wave barrier suffices;
// __syncthreads would also make the wave wait for its outstanding global
// stores (workgroup-scope release).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_wave_barrier();
}

// 16 bytes of T
template <typename T>
struct alignas(16) Vec16
{
    T v[16 / sizeof(T)];
};

// row `row` of bank gb's inverse (symmetric: the column the product needs)
template <typename T>
__device__ __forceinline__ void row_load(const T* __restrict__ inv, int gb, int row, T (&pv)[BD])
{
    constexpr int   W = 16 / sizeof(T);
    const Vec16<T>* P = reinterpret_cast<const Vec16<T>*>(inv + (size_t)gb * BD * BD + row * BD);
#pragma unroll
    for(int u = 0; u < BD / W; u++)
    {
        Vec16<T> q = P[u];
#pragma unroll
        for(int k = 0; k < W; k++)
            pv[u * W + k] = q.v[k];
    }
}

template <typename T>
__device__ __forceinline__ T row_product(const T (&pv)[BD], const T* rs)
{
    T z = 0;
#pragma unroll
    for(int u = 0; u < BD; u++)
        z += pv[u] * rs[u];
    return z;
}

// One bank's product z = Binv R with one wave: lane u < 48 holds R_u, lane
// t < 48 produces z_t (lanes 48..63 compute a copy of lane 0's and store it
// into the bank's padding).  The 48 entries a lane needs (column t of the
// stored transpose) are loaded before the products so their latencies
// overlap; every lane stores unconditionally so the compiler keeps the loads
// together instead of sinking them into a guarded block.
template <typename T>
__device__ __forceinline__ void bank_load(const T* __restrict__ inv, int gb, T (&pv)[BD])
{
    const int t  = __lane_id();
    const int tc = t < BD ? t : 0;
    const T*  P  = inv + (size_t)gb * BD * BD + tc;
#pragma unroll
    for(int u = 0; u < BD; u++)
        pv[u] = P[u * BD];
}

// component c of a cluster's sum: the members (mask of lanes of a 16-node
// bank whose R starts at rs) added in node order
template <typename T>
__device__ __forceinline__ T member_sum(const T* rs, unsigned mask, int c)
{
    T m[BANK], s = 0;
#pragma unroll
    for(int u = 0; u < BANK; u++)
        m[u] = rs[3 * u + c];
#pragma unroll
    for(int u = 0; u < BANK; u++)
        s = (mask >> u) & 1u ? s + m[u] : s;
    return s;
}

}  // namespace sgipc
