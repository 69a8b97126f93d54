// persist.hip -- FP64 PCG in one launch.
//
// The iteration is solve_t's (linsys.hip), the reference's (pcg_solver.cu:
// 171-304).  With one launch per operation an iteration of a system that does
// not fill the chip costs four launches, each a chain of dependent memory
// round trips behind a launch boundary.  Here every workgroup keeps its rows'
// x, r, z, A p and p in LDS and most of its matrix blocks in registers for the
// whole solve and meets the others at three grid barriers per iteration: after
// p.Ap, after the level-1 restriction, after r.z (two with block Jacobi), one
// more for every coarse level below the tail and one at a check iteration (x for
// the residual).  A barrier with its exchange is 1.9 us with 2 workgroups, 2.9 us with 32, 4.2 us
// with 256; they bound the small systems.  The level-0 products run between
// arriving at the second one and waiting for it; LDS left over keeps the
// inverse rows of the tail products and level-0 inverses.  Per iteration, a
// launch per operation against this: 24.2 / 13.1 us on 425 rows, 18 / 8.5 us on
// 7,560 (block Jacobi), 25.7 / 13.5 us on 6,480 (FP64 MAS), 38.4 / 21.4 us on
// 46,656 (where the barriers take half, and the level-0 products and the
// tail's R, which every workgroup reads and restricts whole, most of the rest).
//
// Exchange between workgroups: only z (read back by the neighbours' halos),
// the coarse R and Z, and, for contact columns, p; at check iterations x.
// They are stored and loaded with relaxed agent-scope atomics, which go
// through to the memory all XCDs share, so no L2 is written back or
// invalidated; a workgroup's stores are acknowledged (vmcnt(0) in every wave)
// before its barrier word is stored.  Matrix, inverses and indices are
// constant during the launch and stay in the caches.
//
// Barrier words carry the workgroup's partial sum and the barrier's number
// in the same 64-bit store (two halves of the double), so seeing the number
// means having the sum; every workgroup adds the partials in the same order.
// Two sets of words alternate: a workgroup stores into a set again only after
// a barrier that all have left the set's previous use for.  Waits are bounded:
// a workgroup that runs out of polls leaves, the others follow at their next
// wait, and each sets ctl[2]; the caller then solves with a launch per
// operation.
#include "persist.h"

#include <algorithm>
#include <condition_variable>
#include <mutex>
#include <optional>

#include "../../include/sgipc.h"
#include "mas_tail.h"

namespace sgipc
{

namespace
{
typedef unsigned long long u64;

constexpr int kPT        = 512;            // threads of a workgroup
constexpr int kPW        = kPT / 64;       // waves
constexpr int kRowL      = 4;              // lanes per block row
constexpr int kPassRows  = kPT / kRowL;    // rows of one SpMV pass
constexpr int kMaxRows   = 2 * kPassRows;
constexpr int kMaxGroups = 256;
// rows per workgroup while there are workgroups to add.  More workgroups make
// the barriers longer, fewer the work between them: with 32 / 64 / 128 rows an
// iteration takes 13.1 / 13.6 / 17.1 us on 425 rows, 15.1 / 13.5 / 19.6 us on
// 6,480 rows (FP64 MAS), 9.6 / 8.5 / 10.3 us on 7,560 rows (block Jacobi)
constexpr int kGroupRows = 64;
// Rows that a level-0 bank counts for when the rows are shared out: the waves
// take one bank product each at a time, and banks hold 3 .. 16 rows.  By rows
// alone the workgroups of a 46,656-row system get up to 25 banks, 17 on
// average, and wait for the largest; with 8 rows per bank up to 22
constexpr int kBankRows  = 8;
// Contact blocks of a workgroup's rows beyond the first kPT follow in rounds of
// kPT, one after the other, while all other workgroups wait; the four lanes of a
// row sum its part of a round.  A launch per operation instead leaves the
// longest row to four lanes.  ns: of a round, of a round per block of the
// longest row in it, of a launch per operation per block of the longest row,
// and what one launch gains without contact.  us per iteration, one launch / a
// launch per operation, by blocks of a workgroup and of its longest row: 743,
// 162: 18 / 28; 1,317, 88: 20 / 26; 1,831, 444: 34 / 42; 2,803, 690: 56 / 55;
// 4,190, 279: 69 / 38; 4,904, 1,220: 98 / 82; 20,928, 5,184: 461 / 278.
constexpr int kRoundNs = 4500, kRoundRowNs = 13, kRowNs = 50, kGainNs = 10000;
constexpr int kSlotWords = 4;              // two doubles in four words
// R of a 16-node bank in LDS takes 50 entries instead of 48: the members of
// consecutive clusters lie in consecutive banks, and 48 would put their reads
// on the same LDS banks
constexpr int kRB  = 50;
constexpr int kRow = BD + 1;  // cached inverse row
constexpr int kR0  = 2 * BD + 2;  // r of a level-0 bank, twice in a row
constexpr size_t kPLds   = 156 * 1024;     // LDS of a workgroup at most

template <typename T>
__device__ __forceinline__ T ld_agent(const T* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_agent(T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T>
struct PersistArgs
{
    int        groups, nloc, nhalo;  // LDS extents
    int        cache, keep_off;      // LDS for cached inverse rows and banks: T's, byte offset
    const int *rstart, *bstart, *hptr, *hcol;
    const unsigned short* lcol;
    const int*            rowptr;
    const double*         vals;
    const int *           rp2, *cols2;  // contact rows (may be null)
    const double*         vals2;
    const double*         b;
    double *              x, *z, *p0, *p1;
    const double*         dinv;  // block Jacobi
    // MAS
    const int *     vert_of_slot, *bank_first, *bank_ncl, *chain, *child_bank;
    const unsigned* child_mask;
    const T *       inv, *dense;
    T *             R, *Z;
    int             L, nbank, first_dense;
    TailPlan        tp;
    // stop test
    double rel2, abs2, q_ref;
    int    use_rz, maxit, every;
    u64*    slots;
    int*     ctl;
    double*  out;
    int      polls;
    unsigned lds;  // bytes of a workgroup's LDS
};

struct Barrier
{
    u64*     slots;
    int      groups, b;
    unsigned epoch = 0;
    double * part, *tot;  // LDS: 2 kPW each
    int*     fail;        // LDS: a wait ran out, most polls of one

    __device__ __forceinline__ u64* words(int g) const
    {
        return slots + ((size_t)(epoch & 1u) * groups + g) * kSlotWords;
    }

    // N sums (0 .. 2) of this workgroup: stored with the barrier's number once
    // every global store of the workgroup is acknowledged
    template <int N>
    __device__ __forceinline__ void arrive(double v = 0.0, double w = 0.0)
    {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if(N > 0)
            v = wave_sum(v);
        if(N > 1)
            w = wave_sum(w);
        if(N > 0 && __lane_id() == 0)
        {
            part[threadIdx.x >> 6]         = v;
            part[kPW + (threadIdx.x >> 6)] = w;
        }
        __syncthreads();
        epoch++;
        if(N == 0 && threadIdx.x == 0)
            st_agent(words(b), (u64)epoch);
        if((int)threadIdx.x < N)
        {
            double s = 0.0;
            for(int i = 0; i < kPW; i++)
                s += part[kPW * threadIdx.x + i];
            u64*      w8 = words(b) + 2 * threadIdx.x;
            const u64 u  = (u64)__double_as_longlong(s);
            st_agent(w8, (u << 32) | epoch);
            st_agent(w8 + 1, (u & 0xffffffff00000000ull) | epoch);
        }
    }

    // all workgroups have arrived: their N sums; false when a wait ran out
    template <int N>
    __device__ __forceinline__ bool wait(double* v = nullptr, double* w = nullptr)
    {
        double s0 = 0.0, s1 = 0.0;
        if((int)threadIdx.x < groups)
        {
            constexpr int M  = N > 0 ? 2 * N : 1;
            const u64*    w8 = words(threadIdx.x);
            u64           q[M];
            int           n = 0;
            bool          there;
            do
            {
                there = true;
#pragma unroll
                for(int i = 0; i < M; i++)
                    q[i] = ld_agent(w8 + i);
#pragma unroll
                for(int i = 0; i < M; i++)
                    there = there && (unsigned)q[i] == epoch;
            } while(!there && ++n < fail[1]);
            if(!there)
                *fail = 1;
            if(N > 0)
                s0 = __longlong_as_double((long long)((q[0] >> 32)
                                                      | (q[M > 1 ? 1 : 0] & 0xffffffff00000000ull)));
            if(N > 1)
                s1 = __longlong_as_double((long long)((q[M > 2 ? 2 : 0] >> 32)
                                                      | (q[M > 3 ? 3 : 0] & 0xffffffff00000000ull)));
        }
        if(N > 0)
        {
            s0 = wave_sum(s0);
            if(N > 1)
                s1 = wave_sum(s1);
            if(__lane_id() == 0)
            {
                tot[threadIdx.x >> 6]         = s0;
                tot[kPW + (threadIdx.x >> 6)] = s1;
            }
        }
        __syncthreads();
        if(N > 0)
        {
            double t0 = 0.0, t1 = 0.0;
            for(int i = 0; i < kPW; i++)
            {
                t0 += tot[i];
                t1 += tot[kPW + i];
            }
            *v = t0;
            if(N > 1)
                *w = t1;
        }
        return *fail == 0;
    }
};

// z_t of a packed bank inverse S (LDS or global memory) for lane t < 48 (lanes
// above: a copy of lane 0's), R: the bank's values twice in a row in LDS.
// In parts of 96 bytes, so that the values fit beside the matrix blocks
// in the registers.
template <typename T>
__device__ __forceinline__ T packed_product(const T* __restrict__ S, const T* R)
{
    const int l = (int)__lane_id(), t = l < BD ? l : 0;
    T         z = S[t] * R[t];
    constexpr int N = 48 / sizeof(T);
#pragma unroll 1
    for(int h = 1; h < kDiag; h += N)
    {
        T a[N], m[N];
#pragma unroll
        for(int k = 0; k < N; k++)
        {
            const int d = h + k;
            a[k]        = S[(unsigned)(d * BD + t)];
            m[k]        = S[(unsigned)(d * BD + (t >= d ? t - d : t - d + BD))];
        }
#pragma unroll
        for(int k = 0; k < N; k++)
        {
            z += a[k] * R[t + h + k];
            if(h + k < kDiag - 1)  // D_24 holds both its halves
                z += m[k] * R[t - h - k + BD];
        }
    }
    return z;
}

// the same with S whole, in LDS: fewer LDS reads, for r is the same for all
// lanes (425 rows, an iteration: 13.8 us packed, 13.3 us whole)
template <typename T>
__device__ __forceinline__ T whole_product(const T* S, const T* R)
{
    S += __lane_id() < BD ? __lane_id() : 0;
    T z = 0;
#pragma unroll 12
    for(int u = 0; u < BD; u++)
        z += S[u * BD] * R[u];
    return z;
}

// LDS of a workgroup, in bytes, without the cached inverse rows and banks
template <typename T>
size_t persist_lds(int nloc, int nhalo, int nbank, const TailPlan& tp, int L, bool mas,
                   bool contact)
{
    size_t n = (size_t)(6 * (nloc + nhalo) + 9 * nloc) * sizeof(double);
    if(mas)
    {
        const int ntl = L - tp.lt;
        n += (size_t)(kRB * (tp.span / BANK) + std::max(3 * nloc * ntl, 2 * BD * kPW) + kR0 * nbank)
             * sizeof(T);
        n += (size_t)(nloc * ntl + (tp.span - tp.first) + nloc) * sizeof(int);
        n += (size_t)(nloc * ntl + nloc + 16 * nbank) * sizeof(short);
    }
    n += (size_t)nhalo * sizeof(int);
    if(contact)
        n += (size_t)3 * kPT * sizeof(double);
    return (n + 79) / 16 * 16;
}

// ctl[3] = 1 if a launch per operation is the faster way for the contact rows of
// some workgroup of the solve (one wave each).  A launch of its own, 5 us once
// per solve: inside k_pcg_persist it cost registers in every iteration (46,656
// rows: 0.7%).
__global__ void __launch_bounds__(64) k_contact_rows(const int* __restrict__ rstart,
                                                     const int* __restrict__ rp,
                                                     int* __restrict__ ctl)
{
    const int v0 = rstart[blockIdx.x], v1 = rstart[blockIdx.x + 1];
    int       len = 0;
    for(int v = v0 + (int)threadIdx.x; v < v1; v += 64)
        len = max(len, rp[v + 1] - rp[v]);
    for(int o = 32; o > 0; o >>= 1)
        len = max(len, __shfl_xor(len, o, 64));
    const long long more = (rp[v1] - rp[v0] + kPT - 1) / kPT - 1;
    if(threadIdx.x == 0 && more > 0
       && more * (kRoundNs + kRoundRowNs * min(len, kPT)) > kGainNs + (long long)kRowNs * len)
        ctl[3] = 1;
}

template <typename T, bool MAS, int kPasses>
__global__ void __launch_bounds__(kPT) k_pcg_persist(PersistArgs<T> A)
{
    extern __shared__ __align__(16) unsigned char plds[];
    __shared__ double bar_part[2 * kPW], bar_tot[2 * kPW];
    __shared__ int    fail[2], wcnt[kPW];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int b  = blockIdx.x;
    const int v0 = A.rstart[b], nloc = A.rstart[b + 1] - v0;
    const int h0 = A.hptr[b], nh = A.hptr[b + 1] - h0;
    const int n3 = 3 * nloc;
    Barrier   bar{A.slots, A.groups, b, 0u, bar_part, bar_tot, fail};
    if(tid == 0)
        fail[0] = 0, fail[1] = A.polls;
    if(A.rp2 && A.ctl[3])  // k_contact_rows
        return;

    // ---- LDS: [own | halo] p and x, own r, z, A p, then the MAS tail
    const int NL3 = 3 * A.nloc, NV = 3 * (A.nloc + A.nhalo);
    double*   pl  = reinterpret_cast<double*>(plds);
    double*   xl  = pl + NV;
    double*   rl  = xl + NV;
    double*   zl  = rl + NL3;
    double*   al  = zl + NL3;
    double*   ce  = al + NL3;  // products of the contact blocks, one per thread
    const TailPlan& tp  = A.tp;
    const int       L   = A.L;
    const int       ntl = MAS ? L - tp.lt : 0;
    // tail R (kRB per bank), products of the tail nodes, r by level-0 slot
    T*              Rs   = reinterpret_cast<T*>(ce + (A.rp2 ? 3 * kPT : 0));
    T*              zb   = Rs + kRB * (tp.span / BANK);
    T*              rs0  = zb + (MAS ? max(3 * A.nloc * ntl, 2 * BD * kPW) : 0);
    int*            hc   = reinterpret_cast<int*>(rs0 + (MAS ? kR0 * A.nbank : 0));
    int*            list = hc + A.nhalo;
    unsigned*       memb = reinterpret_cast<unsigned*>(list + A.nloc * ntl);
    unsigned*       own1 = memb + (tp.span - tp.first);
    unsigned short* fl   = reinterpret_cast<unsigned short*>(own1 + (MAS ? A.nloc : 0));
    unsigned short* at0  = fl + A.nloc * ntl;  // place of each own row in rs0
    unsigned short* lsl  = at0 + A.nloc;       // own row of each level-0 slot
    T* const        keep = reinterpret_cast<T*>(plds + A.keep_off);
    const int b0 = tp.base / BANK;
    int       bk0 = 0, nbk = 0, f0 = 0, n1 = 0, total = 0;

    for(int i = tid; i < 3 * (nloc + nh); i += kPT)
    {
        pl[i] = 0.0;
        xl[i] = 0.0;
    }
    for(int i = tid; i < nh; i += kPT)
        hc[i] = 3 * A.hcol[h0 + i];
    int  nkeep = 0, nbcache = 0;  // cached rows of tail products, cached level-0 banks
    bool whole  = false;          // the latter as 48 x 48 blocks
    int  nstage = 0;              // banks loaded again each iteration, into stage
    T*   stage  = nullptr;
    if constexpr(MAS)
    {
        bk0 = A.bstart[b], nbk = A.bstart[b + 1] - bk0;
        for(int i = tid; i < 16 * nbk; i += kPT)
        {
            const int v = A.vert_of_slot[16 * (size_t)bk0 + i];
            lsl[i]      = v >= 0 ? (unsigned short)(v - v0) : (unsigned short)0xffff;
            if(v >= 0)
                at0[v - v0] = (unsigned short)(kR0 * (i / BANK) + 3 * (i % BANK));
        }
        for(int i = tid; i < kR0 * A.nbank; i += kPT)
            rs0[i] = (T)0;
        // own level-1 nodes (consecutive): member slots
        if(nbk > 0)
        {
            f0 = A.bank_first[bk0];
            n1 = A.bank_first[bk0 + nbk - 1] + A.bank_ncl[bk0 + nbk - 1] - f0;
        }
        for(int i = tid; i < n1; i += kPT)
            own1[i] = ((unsigned)(A.child_bank[f0 + i] - bk0) << 16) | A.child_mask[f0 + i];
        for(int i = tp.first + tid; i < tp.span; i += kPT)
            memb[i - tp.first] =
                ((unsigned)(A.child_bank[tp.base + i] - b0) << 16) | A.child_mask[tp.base + i];
        for(int i = tid; i < kRB * (tp.span / BANK); i += kPT)
            Rs[i] = (T)0;
        // distinct tail nodes of the own vertices (k_mas_finish's list, made once)
        for(int l = tp.lt; l < L; l++)
        {
            const int  g    = tid < nloc ? A.chain[(size_t)(v0 + tid) * (L - 1) + l - 1] : -1;
            const int  up   = __shfl_up(g, 1, 64);
            const bool head = tid < nloc && (lane == 0 || up != g);
            const u64  m    = __ballot(head);
            if(lane == 0)
                wcnt[w] = __popcll(m);
            __syncthreads();
            int at = total + __popcll(m & ((2ull << lane) - 1ull)) - 1;
            for(int q = 0; q < kPW; q++)
            {
                at += q < w ? wcnt[q] : 0;
                total += wcnt[q];
            }
            if(tid < nloc)
                fl[(l - tp.lt) * A.nloc + tid] = (unsigned short)at;
            if(head)
                list[at] = g - tp.base;
            __syncthreads();
        }
        // inverse rows of the tail products, then level-0 banks, as many as fit
        nkeep = min(3 * total, A.cache / kRow);
        for(int f = tid / 16; f < nkeep; f += kPT / 16)
        {
            const int n = list[f / 3];
            const T*  P = A.dense + (size_t)(b0 - A.first_dense + n / BANK) * BD * BD
                         + (3 * (n % BANK) + f % 3) * BD;
            for(int u = tid % 16; u < BD; u += 16)
                keep[kRow * f + u] = P[u];
        }
        const int left = A.cache - kRow * nkeep;
        whole          = nbk * BD * BD <= left;
        nbcache        = whole ? nbk : min(nbk, left / kBankPack);
        for(int i = tid; i < nbcache * (whole ? BD * BD : kBankPack); i += kPT)
            keep[kRow * nkeep + i] =
                whole ? A.inv[(size_t)(bk0 + i / (BD * BD)) * kBankPack
                              + pack_at(i % (BD * BD) / BD, i % BD)]
                      : A.inv[(size_t)bk0 * kBankPack + i];
        stage  = reinterpret_cast<T*>(((size_t)Rs + 15) & ~(size_t)15);
        nstage = min(nbk - nbcache, (int)(rs0 - stage) / kBankPack);
    }
    // The inverses that found no place for the whole solve come into the
    // tail's buffers, which are free until level 0 is done, while the
    // workgroup waits at a barrier. 1 KB per wave and step; a step that would
    // end beyond the last bank starts earlier.  46,656 rows, an iteration: 24.6
    // us with these banks read where they are used, 21.4 us (with kBankRows).
    auto load_stage = [&]() {
        if constexpr(MAS)
        {
            constexpr int V = 16 / sizeof(T);  // values per lane
            const T*      p = A.inv + (size_t)(bk0 + nbcache) * kBankPack;
            const int     n = nstage * kBankPack;
            for(int i = 64 * V * w; i < n; i += 64 * V * kPW)
            {
                const int o = min(i, n - 64 * V);
                __builtin_amdgcn_global_load_lds(
                    (const __attribute__((address_space(1))) void*)(p + o + V * lane),
                    (__attribute__((address_space(3))) void*)(stage + o), 16, 0, 0);
            }
        }
    };
    __syncthreads();
    load_stage();
    auto put_r = [&](int i, double r) {
        rl[i] = r;
        if constexpr(MAS)
            rs0[at0[i / 3] + i % 3] = rs0[at0[i / 3] + i % 3 + BD] = (T)r;
    };
    for(int i = tid; i < n3; i += kPT)
        put_r(i, A.b[3 * (size_t)v0 + i]);
    // this thread's rows: the first kReg blocks of its lane stay in registers
    // (16 or 12 of a row's blocks; a tet mesh has about 15), the rest is read
    // again
    constexpr int kReg = kPasses == 1 ? 4 : 3;
    int    kn[kPasses], k1[kPasses], q0[kPasses], q1[kPasses], cr[kPasses][kReg];
    double Br[kPasses][kReg][9];
#pragma unroll
    for(int s = 0; s < kPasses; s++)
    {
        const int  row = s * kPassRows + tid / kRowL;
        const bool on  = row < nloc;
        const int  k0  = (on ? A.rowptr[v0 + row] : 0) + tid % kRowL;
        k1[s]          = on ? A.rowptr[v0 + row + 1] : 0;
        kn[s]          = k0 + kReg * kRowL;
        q0[s]          = on && A.rp2 ? A.rp2[v0 + row] + tid % kRowL : 0;
        q1[s]          = on && A.rp2 ? A.rp2[v0 + row + 1] : 0;
#pragma unroll
        for(int j = 0; j < kReg; j++)
        {
            const int  k  = k0 + j * kRowL;
            const bool in = k < k1[s];
            cr[s][j]      = in ? 3 * (int)A.lcol[k] : 0;
#pragma unroll
            for(int q = 0; q < 9; q++)
                Br[s][j][q] = in ? A.vals[9 * (size_t)k + q] : 0.0;
        }
    }
    __syncthreads();

    // Contact rows are a few long ones (a body's nodes, a fixed vertex under a
    // cloth): thread t takes the workgroup's t-th contact block, keeps its
    // column's p in registers and leaves the product in ce for the row to
    // sum in order; further blocks follow kPT at a time, their p read again.
    int    e0 = 0, ne = 0, je = -1;
    double pe[3] = {0.0, 0.0, 0.0};
    if(A.rp2)
    {
        e0 = A.rp2[v0];
        ne = A.rp2[v0 + nloc] - e0;
        if(tid < ne)
            je = A.cols2[e0 + tid];
    }
    auto contact_product = [&](int e, const double* u) {
        const double* B = A.vals2 + 9 * (size_t)e;
#pragma unroll
        for(int c = 0; c < 3; c++)
            ce[3 * tid + c] = B[3 * c] * u[0] + B[3 * c + 1] * u[1] + B[3 * c + 2] * u[2];
    };

    // al = A u for the own rows, u = [own | halo] in LDS, the first contact
    // products in ce; contact columns j beyond them through contact(j, u_j)
    // from global memory; returns this thread's u.A u
    auto spmv = [&](const double* u, auto&& contact) {
        const int g = tid % kRowL;
        double    d = 0.0, a[kPasses][3];
#pragma unroll
        for(int s = 0; s < kPasses; s++)
        {
            a[s][0] = a[s][1] = a[s][2] = 0.0;
            auto add = [&](const double* B, const double* x) {
                const double x0 = x[0], x1 = x[1], x2 = x[2];
                a[s][0] += B[0] * x0 + B[1] * x1 + B[2] * x2;
                a[s][1] += B[3] * x0 + B[4] * x1 + B[5] * x2;
                a[s][2] += B[6] * x0 + B[7] * x1 + B[8] * x2;
            };
#pragma unroll
            for(int j = 0; j < kReg; j++)
                add(Br[s][j], u + cr[s][j]);
            for(int k = kn[s]; k < k1[s]; k += kRowL)
            {
                double B[9];
#pragma unroll
                for(int q = 0; q < 9; q++)
                    B[q] = A.vals[9 * (size_t)k + q];
                add(B, u + 3 * (int)A.lcol[k]);
            }
        }
#pragma unroll 1
        for(int h = 0; h < ne; h += kPT)
        {
            if(h > 0)
            {
                __syncthreads();
                if(h + tid < ne)
                {
                    double x[3];
                    contact(A.cols2[e0 + h + tid], x);
                    contact_product(e0 + h + tid, x);
                }
                __syncthreads();
            }
#pragma unroll
            for(int s = 0; s < kPasses; s++)
                for(int k = q0[s] + (max(e0 + h - q0[s], 0) + kRowL - 1) / kRowL * kRowL;
                    k < min(q1[s], e0 + h + kPT); k += kRowL)
                {
                    const double* c = ce + 3 * (k - e0 - h);
                    a[s][0] += c[0];
                    a[s][1] += c[1];
                    a[s][2] += c[2];
                }
        }
#pragma unroll
        for(int s = 0; s < kPasses; s++)
        {
            const int row = s * kPassRows + tid / kRowL;
#pragma unroll
            for(int o = kRowL / 2; o > 0; o >>= 1)
            {
#pragma unroll
                for(int c = 0; c < 3; c++)
                    a[s][c] += __shfl_xor(a[s][c], o, kRowL);
            }
            if(row < nloc && g == 0)
            {
#pragma unroll
                for(int c = 0; c < 3; c++)
                {
                    al[3 * row + c] = a[s][c];
                    d += u[3 * row + c] * a[s][c];
                }
            }
        }
        return d;
    };

    double rz = 0.0, beta = 0.0, thr = 0.0;
    for(int k = 0; k < A.maxit; k++)
    {
        const bool check = k > 0 && k % A.every == 0;
        double     rr    = 0.0;
        if(k > 0)
        {
            // ---- p = z + beta p: own rows and halo
            double* const       pnow = (k & 1) ? A.p1 : A.p0;
            const double* const pold = (k & 1) ? A.p0 : A.p1;
            double ze[3] = {0.0, 0.0, 0.0};
            if(je >= 0)
            {
#pragma unroll
                for(int c = 0; c < 3; c++)
                    ze[c] = ld_agent(A.z + 3 * (size_t)je + c);
            }
            for(int i = tid; i < 3 * nh; i += kPT)
            {
                const double zj = ld_agent(A.z + hc[i / 3] + i % 3);
                pl[n3 + i]      = fma(beta, pl[n3 + i], zj);
            }
            for(int i = tid; i < n3; i += kPT)
            {
                const double p = fma(beta, pl[i], zl[i]);
                pl[i]          = p;
                if(A.rp2)
                    st_agent(pnow + 3 * (size_t)v0 + i, p);
            }
            if(je >= 0)
            {
#pragma unroll
                for(int c = 0; c < 3; c++)
                    pe[c] = fma(beta, pe[c], ze[c]);
                contact_product(e0 + tid, pe);
            }
            __syncthreads();
            // ---- A p and p.Ap
            double pap = spmv(pl, [&](int j, double* p) {
#pragma unroll
                for(int c = 0; c < 3; c++)
                {
                    p[c] = ld_agent(A.z + 3 * (size_t)j + c);
                    if(k > 1)
                        p[c] = fma(beta, ld_agent(pold + 3 * (size_t)j + c), p[c]);
                }
            });
            bar.arrive<1>(pap);
            load_stage();
            if(!bar.wait<1>(&pap))
                break;
            // ---- x += a p, r -= a Ap; at a check r = b - A x
            const double a = rz / pap;
            for(int i = tid; i < n3; i += kPT)
            {
                xl[i] += a * pl[i];
                if(!check)
                    put_r(i, rl[i] - a * al[i]);
                else
                    st_agent(A.x + 3 * (size_t)v0 + i, xl[i]);
            }
            if(check)
            {
                bar.arrive<0>();
                if(!bar.wait<0>())
                    break;
                for(int i = tid; i < 3 * nh; i += kPT)
                    xl[n3 + i] = ld_agent(A.x + hc[i / 3] + i % 3);
                if(je >= 0)
                {
                    double xe[3];
#pragma unroll
                    for(int c = 0; c < 3; c++)
                        xe[c] = ld_agent(A.x + 3 * (size_t)je + c);
                    contact_product(e0 + tid, xe);
                }
                __syncthreads();
                spmv(xl, [&](int j, double* x) {
#pragma unroll
                    for(int c = 0; c < 3; c++)
                        x[c] = ld_agent(A.x + 3 * (size_t)j + c);
                });
                __syncthreads();
                for(int i = tid; i < n3; i += kPT)
                    put_r(i, A.b[3 * (size_t)v0 + i] - al[i]);
            }
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the staged inverses
        __syncthreads();
        if(!A.use_rz && (check || k == 0))
            for(int i = tid; i < n3; i += kPT)
                rr += rl[i] * rl[i];
        // ---- z = M r
        double rzp = 0.0;
        if constexpr(!MAS)
        {
            if(tid < nloc)
            {
                const double* D  = A.dinv + 9 * (size_t)(v0 + tid);
                const double  r0 = rl[3 * tid], r1 = rl[3 * tid + 1], r2 = rl[3 * tid + 2];
#pragma unroll
                for(int c = 0; c < 3; c++)
                {
                    const double zc = D[3 * c] * r0 + D[3 * c + 1] * r1 + D[3 * c + 2] * r2;
                    zl[3 * tid + c] = zc;
                    st_agent(A.z + 3 * (size_t)(v0 + tid) + c, zc);
                    rzp += rl[3 * tid + c] * zc;
                }
            }
        }
        else
        {
            // R of the own level-1 nodes, members in node order
#pragma unroll 1
            for(int q = tid; q < 3 * n1; q += kPT)
            {
                const unsigned mk = own1[q / 3];
                const T        s  = member_sum(rs0 + kR0 * (mk >> 16), mk, q % 3);
                st_agent(A.R + 3 * (size_t)f0 + q, s);
            }
            bar.arrive<0>();
            // level-0 products between arriving and waiting
#pragma unroll 1
            for(int j = w; j < nbk; j += kPW)
            {
                const T* rv = rs0 + kR0 * j;
                T        z;
                if(whole)
                    z = whole_product(keep + kRow * nkeep + j * BD * BD, rv);
                else if(j < nbcache + nstage)
                    z = packed_product(j < nbcache ? keep + kRow * nkeep + j * kBankPack
                                                   : stage + (j - nbcache) * kBankPack,
                                       rv);
                else
                    z = packed_product(A.inv + (size_t)(bk0 + j) * kBankPack, rv);
                const int sl = lane < BD ? (int)lsl[16 * j + lane / 3] : 0xffff;
                if(sl != 0xffff)
                    zl[3 * sl + lane % 3] = (double)z;
            }
            if(!bar.wait<0>())
                break;
            // coarse levels below the tail: banks shared out over all waves
            bool ok = true;
            for(int l = 1; l < tp.lt && l < L; l++)
            {
                const int lb = (tp.count[l] + BANK - 1) / BANK;
#pragma unroll 1
                for(int j = b * kPW + w; j < lb; j += A.groups * kPW)
                {
                    const int  gb    = tp.off[l] / BANK + j;
                    const int  g     = gb * BANK + lane / 3;
                    const bool valid = lane < BD && g - tp.off[l] < tp.count[l];
                    T*         Rv    = zb + 2 * BD * w;  // free until the tail's products
                    wave_lds_sync();
                    if(lane < BD)
                        Rv[lane] = Rv[lane + BD] =
                            valid ? ld_agent(A.R + 3 * (size_t)g + lane % 3) : (T)0;
                    wave_lds_sync();
                    st_agent(A.Z + (size_t)gb * ZB + lane,
                             packed_product(A.inv + (size_t)gb * kBankPack, Rv));
                    if(l + 1 < L)
                    {
                        const int first = A.bank_first[gb], ncl = A.bank_ncl[gb];
                        if(lane < 3 * ncl)
                        {
                            const int n = first + lane / 3;
                            st_agent(A.R + 3 * (size_t)first + lane,
                                     member_sum(Rv, A.child_mask[n], lane % 3));
                        }
                    }
                }
                bar.arrive<0>();
                ok = bar.wait<0>();
                if(!ok)
                    break;
            }
            if(!ok)
                break;
            // the tail: R_lt whole, higher levels restricted in LDS, products of
            // the own vertices' nodes
            if(ntl > 0)
            {
                constexpr int W   = 8 / sizeof(T);  // R values per load
                const u64*    src = reinterpret_cast<const u64*>(A.R + 3 * (size_t)tp.base);
                const int     n8  = 3 * tp.first / W;
#pragma unroll 1
                for(int i = tid; i < n8; i += 4 * kPT)
                {
                    u64 q[4];
#pragma unroll
                    for(int e = 0; e < 4; e++)
                        q[e] = ld_agent(src + (i + e * kPT < n8 ? i + e * kPT : i));
#pragma unroll
                    for(int e = 0; e < 4; e++)
                    {
                        const int j = i + e * kPT;
                        if(j < n8)
                            *reinterpret_cast<u64*>(Rs + W * j + (kRB - BD) * (j / (BD / W))) =
                                q[e];
                    }
                }
                __syncthreads();
                for(int l = tp.lt; l + 1 < L; l++)
                {
                    const int o = tp.off[l + 1] - tp.base;
#pragma unroll 1
                    for(int q = tid; q < 3 * ((tp.count[l + 1] + BANK - 1) & -BANK); q += kPT)
                    {
                        // zeros behind the last node: inverses were staged here
                        const unsigned mk = memb[o - tp.first + q / 3];
                        const T        t  = q < 3 * tp.count[l + 1]
                                                ? member_sum(Rs + kRB * (mk >> 16), mk, q % 3)
                                                : (T)0;
                        Rs[kRB * ((o + q / 3) / BANK) + 3 * ((o + q / 3) % BANK) + q % 3] = t;
                    }
                    __syncthreads();
                }
                // four lanes per product
#pragma unroll 1
                for(int f = tid / 4; f < 3 * total; f += kPT / 4)
                {
                    const int n  = list[f / 3], h = (BD / 4) * (tid % 4);
                    const T*  rv = Rs + kRB * (n / BANK) + h;
                    T         S[BD / 4], z = 0;
                    if(f < nkeep)
                    {
#pragma unroll
                        for(int u = 0; u < BD / 4; u++)
                            S[u] = keep[kRow * f + h + u];
                    }
                    else
                    {
                        const T* P = A.dense + (size_t)(b0 - A.first_dense + n / BANK) * BD * BD
                                     + (3 * (n % BANK) + f % 3) * BD + h;
#pragma unroll
                        for(int u = 0; u < BD / 4; u++)
                            S[u] = P[u];
                    }
#pragma unroll
                    for(int u = 0; u < BD / 4; u++)
                        z += S[u] * rv[u];
                    z += __shfl_xor(z, 1, 4);
                    z += __shfl_xor(z, 2, 4);
                    if(tid % 4 == 0)
                        zb[f] = z;
                }
                __syncthreads();
            }
            for(int i = tid; i < n3; i += kPT)
            {
                const int v = i / 3, c = i % 3;
                T         z = (T)zl[i];
                for(int l = 1; l < L; l++)
                {
                    if(l < tp.lt)
                    {
                        const int g = A.chain[(size_t)(v0 + v) * (L - 1) + l - 1];
                        z += ld_agent(A.Z + (size_t)(g >> 4) * ZB + 3 * (g & 15) + c);
                    }
                    else
                        z += zb[3 * fl[(l - tp.lt) * A.nloc + v] + c];
                }
                zl[i] = (double)z;
                st_agent(A.z + 3 * (size_t)v0 + i, (double)z);
                rzp += rl[i] * (double)z;
            }
        }
        double rzn, q;
        bool   met;
        if(!A.use_rz && (check || k == 0))
        {
            bar.arrive<2>(rzp, rr);
            met = bar.wait<2>(&rzn, &q);
        }
        else
        {
            bar.arrive<1>(rzp);
            met = bar.wait<1>(&rzn);
            q   = rzn;
        }
        if(!met)
            break;
        if(k == 0)
        {
            const double qr = A.q_ref > 0.0 ? A.q_ref : q;
            thr             = A.rel2 * qr > A.abs2 ? A.rel2 * qr : A.abs2;
            if(b == 0 && tid == 0)
                A.out[0] = rzn;
            if(rzn == 0.0 || !(rzn == rzn))
                break;
        }
        else if(check)
        {
            const bool bad = !(rzn == rzn) || !(q == q);
            if(b == 0 && tid == 0)
                A.out[1] = rzn;
            if(q <= thr || bad)
            {
                if(b == 0 && tid == 0)
                {
                    A.ctl[0] = k;
                    A.ctl[1] = bad ? 1 : 0;
                }
                break;
            }
        }
        beta = k == 0 ? 0.0 : rzn / rz;
        rz   = rzn;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS is under way
    __syncthreads();
    if(fail[0] && tid == 0)
        A.ctl[2] = 1;  // a wait ran out
    for(int i = tid; i < n3; i += kPT)
        A.x[3 * (size_t)v0 + i] = xl[i];
}

// the rest of the arguments; false: the LDS of a compute unit does not hold it
template <typename T, bool MAS>
bool fit(const PersistPlan& P, Mas* mas, PersistArgs<T>& a)
{
    if constexpr(MAS)
    {
        const MasView<T> m = mas->view<T>();
        a.vert_of_slot = m.vert_of_slot, a.bank_first = m.bank_first, a.bank_ncl = m.bank_ncl;
        a.chain = m.chain, a.child_bank = m.child_bank, a.child_mask = m.child_mask;
        a.inv = m.inv, a.dense = m.dense, a.R = m.R, a.Z = m.Z, a.L = mas->levels(), a.nbank = P.banks;
        a.first_dense = mas->parts();
        a.tp = tail_plan(a.L, mas->level_sizes(), [&](int span, int levels) {
            TailPlan t;
            t.lt = a.L - levels, t.span = span;
            return persist_lds<T>(P.rows, P.halo, P.banks, t, a.L, true, a.rp2 != nullptr)
                   <= kPLds;
        });
    }
    const size_t fix = persist_lds<T>(P.rows, P.halo, P.banks, a.tp, a.L, MAS, a.rp2 != nullptr);
    if(fix > kPLds)
        return false;
    a.keep_off     = (int)fix;
    a.cache        = MAS ? (int)((kPLds - fix) / sizeof(T)) : 0;
    a.lds          = (unsigned)(MAS ? kPLds : fix);
    return true;
}

template <typename T, bool MAS>
void launch(const PersistPlan& P, PersistArgs<T> a, std::pair<hipEvent_t, hipEvent_t> ev,
            hipStream_t s)
{
    void*       args[] = {&a};
    const void* f      = P.rows <= kPassRows
                             ? reinterpret_cast<const void*>(&k_pcg_persist<T, MAS, 1>)
                             : reinterpret_cast<const void*>(&k_pcg_persist<T, MAS, 2>);
    SG_HIP(hipExtLaunchKernel(f, dim3(P.groups), dim3(kPT), args, a.lds, s, ev.first, ev.second,
                              0));
}

// The workgroups of a solve wait for each other, so all of them have to run at
// once.  A workgroup takes a compute unit (its LDS leaves no room for a second
// one), other kernels end and give theirs back, and the solves of this process
// share the units out here: a solve holds its units from before its launch
// until it has ended, and the next one in line waits until enough are free.
// Workgroups go to the XCDs in turn, so units are counted per XCD; within one,
// kernels of several streams were seen to fill it to the last unit (101 + 101,
// 63 + 63 + 63 + 63 and 248 + 6 workgroups on 256 units start within 10 us).  A
// cooperative launch would have the runtime run one such solve at a time.  ms
// per solve of several threads with a system each, cooperative launches / this /
// a launch per operation: 425 rows, 8 threads 0.95-1.05 / 0.37-0.40 / 0.60-0.72;
// 6,480 rows, 4 threads 1.58 / 1.18 / 1.73, 8 threads (whose streams share
// hardware queues) 1.59 / 1.2-1.5 / 1.00; 46,656 rows, 8 threads 3.1 / 3.1 / 3.6.
class Units
{
  public:
    void take(int n, int all)
    {
        std::unique_lock<std::mutex> lock(m_);
        const u64 me = last_++;
        cv_.wait(lock, [&] { return me == turn_ && used_ + n <= all; });
        used_ += n;
        turn_++;
        cv_.notify_all();
    }
    void give(int n)
    {
        std::lock_guard<std::mutex> lock(m_);
        used_ -= n;
        cv_.notify_all();
    }
    static Units& of(int dev)
    {
        static Units* const u = new Units[kMaxDevices];  // outlives threads at exit
        SG_CHECK(dev >= 0 && dev < kMaxDevices, -1, "device index out of range");
        return u[dev];
    }

  private:
    static constexpr int    kMaxDevices = 64;
    std::mutex              m_;
    std::condition_variable cv_;
    int                     used_ = 0;
    u64                     last_ = 0, turn_ = 0;  // the line's end and head
};

struct UnitsHeld
{
    Units& u;
    int    n;
    UnitsHeld(const PersistPlan& P)
        : u(Units::of(P.dev))
        , n(std::min((P.groups + kXcds - 1) / kXcds, P.units))
    {
        u.take(n, P.units);
    }
    ~UnitsHeld() { u.give(n); }
    UnitsHeld(const UnitsHeld&)            = delete;
    UnitsHeld& operator=(const UnitsHeld&) = delete;
};
}  // namespace

void PersistPlan::build(const Bsr& A, const std::vector<int>& part_first, hipStream_t s)
{
    groups       = 0;
    const int nb = A.nb;
    int       cus = 0;
    SG_HIP(hipGetDevice(&dev));
    SG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    units       = cus / kXcds;
    const int G = std::min(std::min(kMaxGroups, units * kXcds), std::max(1, nb / kGroupRows));
    if(nb > kMaxRows * G)
        return;
    // row ranges, cut at parts; a bank weighs as much as kBankRows rows
    const bool       mas = !part_first.empty();
    std::vector<int> rs(G + 1), bs(G + 1, 0);
    for(int g = 0; g <= G; g++)
    {
        rs[g] = (int)((long long)nb * g / G);
        if(mas)
        {
            const int np = (int)part_first.size() - 1;
            int       j  = g > 0 ? bs[g - 1] : 0;
            while(j < np && part_first[j] + kBankRows * j < (nb + kBankRows * np) * (double)g / G)
                j++;
            bs[g] = j;
            rs[g] = part_first[j];
        }
    }
    int nr = 0, nh = 0, nk = 0;
    for(int g = 0; g < G; g++)
    {
        nr = std::max(nr, rs[g + 1] - rs[g]);
        nk = std::max(nk, bs[g + 1] - bs[g]);
    }
    if(nr > kMaxRows)
        return;
    std::vector<int>            stamp(nb, -1), at(nb, 0), hp(G + 1, 0), hc;
    std::vector<unsigned short> lc(A.nnzb);
    for(int g = 0; g < G; g++)
    {
        const int own = rs[g + 1] - rs[g], h0 = (int)hc.size();
        for(int k = A.h_rowptr[rs[g]]; k < A.h_rowptr[rs[g + 1]]; k++)
        {
            const int j = A.h_cols[k];
            if(j >= rs[g] && j < rs[g + 1])
            {
                lc[k] = (unsigned short)(j - rs[g]);
                continue;
            }
            if(stamp[j] != g)
            {
                stamp[j] = g;
                at[j]    = (int)hc.size() - h0;
                hc.push_back(j);
            }
            if(own + at[j] > 0xffff)
                return;
            lc[k] = (unsigned short)(own + at[j]);
        }
        hp[g + 1] = (int)hc.size();
        nh        = std::max(nh, hp[g + 1] - hp[g]);
    }
    if(persist_lds<double>(nr, nh, nk, TailPlan{}, 0, false, true) > kPLds)
        return;
    rstart.upload(rs, s);
    bstart.upload(bs, s);
    hptr.upload(hp, s);
    hcol.upload(hc, s);
    lcol.upload(lc, s);
    slots.resize((size_t)2 * kMaxGroups * kSlotWords);
    ctl.resize(4);
    out.resize(2);
    SG_HIP(hipStreamSynchronize(s));
    rows = nr, halo = nh, banks = nk, groups = G;
}

bool persist_solve(PersistPlan& P, const SysView& S, Mas* mas, const double* dinv,
                   const double* b, double* x, double* z, double* p0, double* p1,
                   const PcgConfig& cfg, int maxit, int every, PersistResult* res, hipStream_t s,
                   Profiler* prof)
{
    if(!P.ready())
        return false;
    if(P.skip > 0)
    {
        P.skip--;
        return false;
    }
    const bool contact = S.coo && S.coo->cap > 0 && S.coo->live > 0;
    std::optional<UnitsHeld>          held;
    std::pair<hipEvent_t, hipEvent_t> ev{nullptr, nullptr};
    auto run = [&](auto zero, auto is_mas) {
        using T             = decltype(zero);
        constexpr bool MAS  = decltype(is_mas)::value;
        PersistArgs<T> a{};
        a.groups = P.groups, a.nloc = P.rows, a.nhalo = P.halo;
        a.rstart = P.rstart.data(), a.bstart = P.bstart.data();
        a.hptr = P.hptr.data(), a.hcol = P.hcol.data(), a.lcol = P.lcol.data();
        a.rowptr = S.A->rowptr.data(), a.vals = S.A->vals.data();
        if(contact)
        {
            SG_CHECK(S.coo->rows_valid, -5, "contact CSR is stale: build_rows() after assembly");
            a.rp2 = S.coo->rp.data(), a.cols2 = S.coo->rc.data(), a.vals2 = S.coo->rv.data();
        }
        a.b = b, a.x = x, a.z = z, a.p0 = p0, a.p1 = p1, a.dinv = dinv;
        a.rel2 = cfg.rel_tol * cfg.rel_tol, a.abs2 = cfg.abs_tol * cfg.abs_tol;
        a.q_ref = cfg.q_ref, a.use_rz = cfg.use_rz ? 1 : 0, a.maxit = maxit, a.every = every;
        a.slots = P.slots.data(), a.ctl = P.ctl.data(), a.out = P.out.data(), a.polls = P.polls;
        if(!fit<T, MAS>(P, mas, a))
            return false;
        held.emplace(P);
        SG_HIP(hipMemsetAsync(P.slots.data(), 0, P.slots.size() * sizeof(u64), s));
        SG_HIP(hipMemsetAsync(P.ctl.data(), 0, P.ctl.size() * sizeof(int), s));
        SG_HIP(hipMemsetAsync(P.out.data(), 0, P.out.size() * sizeof(double), s));
        if(contact)
        {
            hipLaunchKernelGGL(k_contact_rows, dim3(P.groups), dim3(64), 0, s, a.rstart, a.rp2,
                               a.ctl);
            SG_LAUNCH_CHECK();
        }
        if(prof)
            ev = prof->kernel_events("pcg");
        launch<T, MAS>(P, a, ev, s);
        return true;
    };
    const bool ran = !mas          ? run(0.0, std::false_type{})
                     : mas->fp32() ? run(0.0f, std::true_type{})
                                   : run(0.0, std::true_type{});
    if(!ran)
        return false;
    int    hc[4];
    double ho[2];
    SG_HIP(hipMemcpyAsync(hc, P.ctl.data(), sizeof(hc), hipMemcpyDeviceToHost, s));
    SG_HIP(hipMemcpyAsync(ho, P.out.data(), sizeof(ho), hipMemcpyDeviceToHost, s));
    SG_HIP(hipStreamSynchronize(s));
    if(hc[2] != 0)  // a wait ran out: every workgroup has left
    {
        P.pause = P.pause ? std::min(2 * P.pause, 1024) : 16;
        P.skip  = P.pause;
    }
    else
        P.pause = 0;
    // or too many contact blocks in one workgroup's rows
    if(hc[2] != 0 || hc[3] != 0)
    {
        if(prof)
            prof->discard("pcg", ev);
        return false;
    }
    res->stop_at = hc[0];
    res->bad     = hc[1];
    res->rz0     = ho[0];
    res->rz      = ho[1];
    return true;
}

}  // namespace sgipc
