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

// 16 bytes of T
template <typename T>
struct alignas(16) Vec16
{
    T v[16 / sizeof(T)];
};

// row `row` of the dense inverse of coarse bank gb (banks of levels >= 1 have
// one beside the packed form; gb counts from the first of them)
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

// Bank inverses are symmetric and stored by circulant diagonals: entry
// [d * 48 + t] is S[t][(t + d) mod 48] for d = 0 .. 24, 1,200 values instead of
// 2,304.  Row t is then D_d[t] at column t + d and D_d[t - d] at column t - d
// (d = 1 .. 23), D_0[t] and D_24[t]; for every d the 48 lanes of a bank read
// 48 consecutive values, twice (the second time from the cache).  Reading the
// inverses bounds the level-0 launch of a large system: 173,225 rows, FP32
// inverses, 16.2 us per launch against 23.7 us dense.
constexpr int kDiag = 25;
constexpr int kBankPack = kDiag * BD;

// place of S[t][u] in the packed inverse
__host__ __device__ __forceinline__ int pack_at(int t, int u)
{
    const int d = u >= t ? u - t : u - t + BD;
    return d < kDiag ? d * BD + t : (BD - d) * BD + u;
}

// One bank's product with one wave: lane t < 48 produces z_t (lanes 48..63 a
// copy of lane 0's).  The values a lane needs are loaded before the products so
// their latencies overlap.
template <typename T>
struct BankRow
{
    T a[kDiag], m[kDiag];  // S[t][t + d], S[t][t - d] (m[0], m[24] unused)
    __device__ __forceinline__ void load(const T* __restrict__ inv, int gb)
    {
        const int l = (int)__lane_id(), t = l < BD ? l : 0;
        const T*  P = inv + (size_t)gb * kBankPack;
#pragma unroll
        for(int d = 0; d < kDiag; d++)
        {
            a[d] = P[d * BD + t];
            if(d > 0 && d < kDiag - 1)
                m[d] = P[d * BD + (t >= d ? t - d : t - d + BD)];
        }
    }
    // R: the bank's 48 values, twice in a row (LDS)
    __device__ __forceinline__ T product(const T* R) const
    {
        const int l = (int)__lane_id(), t = l < BD ? l : 0;
        T         z = a[0] * R[t] + a[kDiag - 1] * R[t + kDiag - 1];
#pragma unroll
        for(int d = 1; d < kDiag - 1; d++)
        {
            z += a[d] * R[t + d];
            z += m[d] * R[t - d + BD];
        }
        return z;
    }
};

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
