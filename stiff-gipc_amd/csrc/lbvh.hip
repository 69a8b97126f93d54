// lbvh.hip -- linear BVH over collision faces / edges (lbvh_f / lbvh_e).
//
// Construction follows StiffGIPC/mlbvh.cu:2074-2157 (Karras 2012):
//   leaf AABBs (:1149-1204), scene box (calcMaxBV :1745), keys
//   morton30(centre) << 32 | index (:1208-1227), sort, leaf/internal nodes
//   (:1229-1269, determine_range :135, find_split :198), bottom-up refit (:1271).
// Built with -ffp-contract=off: keys, node arrays and boxes are bit-identical
// to the CPU restatement.
//
// The key sort is this file's own LSD radix sort on 8-bit digits (keys only:
// the primitive index is the key's low word).  Each 256-thread block ranks
// its 2048-key tile stably with wave64 multi-split: eight ballots give every
// lane the mask of same-digit peers, per-wave digit counts are combined in
// LDS.  Digits above the index width and above the 30-bit Morton code are
// skipped, so a 50k-primitive tree needs 6 passes.
#include <climits>

#include "sgipc.h"
#include "sim_kernels.h"

namespace sgipc
{

constexpr int kSortThreads = 256;
constexpr int kSortItems   = 8;
constexpr int kSortTile    = kSortThreads * kSortItems;

__global__ void k_leaf_aabb(int n, int arity, const uint32_t* __restrict__ prims,
                            const double* __restrict__ x, const double* __restrict__ dx,
                            double alpha, double* __restrict__ leaf)
{
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if(e >= n)
        return;
    double up[3] = {-1e32, -1e32, -1e32}, lo[3] = {1e32, 1e32, 1e32};
    for(int k = 0; k < arity; k++)
    {
        uint32_t v = prims[(size_t)arity * e + k];
        for(int c = 0; c < 3; c++)
        {
            double p = x[3 * (size_t)v + c];
            lo[c]    = (p < lo[c]) ? p : lo[c];
            up[c]    = (up[c] < p) ? p : up[c];
            if(dx)
            {
                double q = p - dx[3 * (size_t)v + c] * alpha;
                lo[c]    = (q < lo[c]) ? q : lo[c];
                up[c]    = (up[c] < q) ? q : up[c];
            }
        }
    }
    for(int c = 0; c < 3; c++)
    {
        leaf[6 * (size_t)e + c]     = up[c];
        leaf[6 * (size_t)e + 3 + c] = lo[c];
    }
}

// min/max reduction of the leaf boxes: per-block partials then one block
__global__ void __launch_bounds__(256) k_box_partial(int n, const double* __restrict__ leaf,
                                                     double* __restrict__ part)
{
    __shared__ double s[6][4];
    int    e = blockIdx.x * blockDim.x + threadIdx.x;
    double v[6];
    for(int c = 0; c < 3; c++)
    {
        v[c]     = (e < n) ? leaf[6 * (size_t)e + c] : -1e32;
        v[3 + c] = (e < n) ? leaf[6 * (size_t)e + 3 + c] : 1e32;
    }
    for(int c = 0; c < 3; c++)
    {
        v[c]     = wave_max(v[c]);
        v[3 + c] = wave_min(v[3 + c]);
    }
    if(__lane_id() == 0)
        for(int c = 0; c < 6; c++)
            s[c][threadIdx.x >> 6] = v[c];
    __syncthreads();
    if(threadIdx.x < 6)
    {
        int    c = threadIdx.x;
        double r = s[c][0];
        for(int w = 1; w < 4; w++)
            r = (c < 3) ? ((r < s[c][w]) ? s[c][w] : r) : ((s[c][w] < r) ? s[c][w] : r);
        part[6 * (size_t)blockIdx.x + c] = r;
    }
}

__global__ void __launch_bounds__(256) k_box_final(int nb, const double* __restrict__ part,
                                                   double* __restrict__ scene)
{
    __shared__ double s[6][4];
    double v[6] = {-1e32, -1e32, -1e32, 1e32, 1e32, 1e32};
    for(int i = threadIdx.x; i < nb; i += blockDim.x)
        for(int c = 0; c < 6; c++)
        {
            double p = part[6 * (size_t)i + c];
            v[c]     = (c < 3) ? ((v[c] < p) ? p : v[c]) : ((p < v[c]) ? p : v[c]);
        }
    for(int c = 0; c < 3; c++)
    {
        v[c]     = wave_max(v[c]);
        v[3 + c] = wave_min(v[3 + c]);
    }
    if(__lane_id() == 0)
        for(int c = 0; c < 6; c++)
            s[c][threadIdx.x >> 6] = v[c];
    __syncthreads();
    if(threadIdx.x < 6)
    {
        int    c = threadIdx.x;
        double r = s[c][0];
        for(int w = 1; w < 4; w++)
            r = (c < 3) ? ((r < s[c][w]) ? s[c][w] : r) : ((s[c][w] < r) ? s[c][w] : r);
        scene[c] = r;
    }
}

__device__ __forceinline__ uint32_t expand_bits(uint32_t v)
{
    v = (v * 0x00010001u) & 0xFF0000FFu;
    v = (v * 0x00000101u) & 0x0F00F00Fu;
    v = (v * 0x00000011u) & 0xC30C30C3u;
    v = (v * 0x00000005u) & 0x49249249u;
    return v;
}

__device__ __forceinline__ double clamp_ref(double v, double lo, double hi)
{
    double a = (v < lo) ? lo : v;  // std::max(v, lo)
    return (hi < a) ? hi : a;      // std::min(a, hi)
}

__device__ __forceinline__ uint32_t morton_code(double x, double y, double z)
{
    const double res = 1024.0;
    x                = clamp_ref(x * res, 0.0, res - 1.0);
    y                = clamp_ref(y * res, 0.0, res - 1.0);
    z                = clamp_ref(z * res, 0.0, res - 1.0);
    return (expand_bits((uint32_t)x) << 2) + (expand_bits((uint32_t)y) << 1)
           + expand_bits((uint32_t)z);
}

// Morton code of box e's centre, then e
__device__ __forceinline__ uint64_t morton_key(int e, const double* __restrict__ leaf,
                                               const double* scene)
{
    double lo[3] = {scene[3], scene[4], scene[5]};
    double sz[3] = {scene[0] - lo[0], scene[1] - lo[1], scene[2] - lo[2]};
    double c[3];
    for(int k = 0; k < 3; k++)
        c[k] = (leaf[6 * (size_t)e + k] + leaf[6 * (size_t)e + 3 + k]) * 0.5;
    uint64_t mc = morton_code((c[0] - lo[0]) / sz[0], (c[1] - lo[1]) / sz[1], (c[2] - lo[2]) / sz[2]);
    return (mc << 32) | (uint64_t)(uint32_t)e;
}

__global__ void k_morton(int n, const double* __restrict__ leaf, const double* __restrict__ scene,
                         uint64_t* __restrict__ keys)
{
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if(e < n)
        keys[e] = morton_key(e, leaf, scene);
}

// ------------------------------------------------------------ radix sort
__global__ void __launch_bounds__(kSortThreads) k_sort_hist(int n, int shift,
                                                            const uint64_t* __restrict__ keys,
                                                            unsigned* __restrict__ hist, int nblk)
{
    __shared__ unsigned h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    int base = blockIdx.x * kSortTile;
    for(int j = 0; j < kSortItems; j++)
    {
        int i = base + j * kSortThreads + threadIdx.x;
        if(i < n)
            atomicAdd(&h[(keys[i] >> shift) & 0xFF], 1u);
    }
    __syncthreads();
    hist[(size_t)threadIdx.x * nblk + blockIdx.x] = h[threadIdx.x];
}

// exclusive scan of hist (digit-major, 256 * nblk entries: a multiple of 4),
// one workgroup: tiles of 4096 entries, 4 consecutive per thread (one 16-byte
// load, coalesced across the workgroup), the next tile's load issued before
// the current tile is scanned; a running carry joins the tiles
__global__ void __launch_bounds__(1024) k_sort_scan(int total, unsigned* __restrict__ hist)
{
    __shared__ unsigned wsum[16];
    uint4*     h4    = reinterpret_cast<uint4*>(hist);
    const int  n4    = total >> 2;
    const int  t     = threadIdx.x;
    const int  w     = t >> 6;
    unsigned   carry = 0;
    uint4      cur   = t < n4 ? h4[t] : make_uint4(0u, 0u, 0u, 0u);
    for(int b4 = 0; b4 < n4; b4 += 1024)
    {
        const int i4  = b4 + t;
        uint4     nxt = (i4 + 1024 < n4) ? h4[i4 + 1024] : make_uint4(0u, 0u, 0u, 0u);
        unsigned  s0 = cur.x, s1 = s0 + cur.y, s2 = s1 + cur.z, s3 = s2 + cur.w;
        unsigned  s  = s3;  // inclusive scan of the per-thread sums
        for(int o = 1; o < 64; o <<= 1)
        {
            unsigned u = __shfl_up(s, o, 64);
            if((int)__lane_id() >= o)
                s += u;
        }
        if(__lane_id() == 63)
            wsum[w] = s;
        __syncthreads();
        if(t < 16)
        {
            unsigned ws = wsum[t];
            for(int o = 1; o < 16; o <<= 1)
            {
                unsigned u = __shfl_up(ws, o, 16);
                if(t >= o)
                    ws += u;
            }
            wsum[t] = ws;
        }
        __syncthreads();
        unsigned excl = s - s3 + (w > 0 ? wsum[w - 1] : 0u) + carry;
        if(i4 < n4)
            h4[i4] = make_uint4(excl, excl + s0, excl + s1, excl + s2);
        carry += wsum[15];
        __syncthreads();  // wsum is rewritten by the next tile
        cur = nxt;
    }
}

// stable scatter: keys are visited in tile order (round j, then thread);
// with KV each key's 32-bit value moves with it
template <bool KV>
__global__ void __launch_bounds__(kSortThreads) k_sort_scatter(int n, int shift,
                                                               const uint64_t* __restrict__ in,
                                                               uint64_t* __restrict__ out,
                                                               const unsigned* __restrict__ hist,
                                                               int nblk,
                                                               const uint32_t* __restrict__ vin,
                                                               uint32_t* __restrict__ vout)
{
    __shared__ unsigned base_d[256];
    __shared__ unsigned wcnt[4][256];
    const int lane = __lane_id();
    const int w    = threadIdx.x >> 6;
    base_d[threadIdx.x] = hist[(size_t)threadIdx.x * nblk + blockIdx.x];
    const int tile      = blockIdx.x * kSortTile;
    for(int j = 0; j < kSortItems; j++)
    {
        for(int q = 0; q < 4; q++)
            wcnt[q][threadIdx.x] = 0;
        __syncthreads();
        int      i    = tile + j * kSortThreads + threadIdx.x;
        bool     live = i < n;
        uint64_t k    = live ? in[i] : 0;
        unsigned d    = (unsigned)((k >> shift) & 0xFF);
        unsigned long long peers = __ballot(live);
#pragma unroll
        for(int b = 0; b < 8; b++)
        {
            unsigned long long m = __ballot((d >> b) & 1u);
            peers &= ((d >> b) & 1u) ? m : ~m;
        }
        unsigned long long lt   = (lane == 0) ? 0ull : (peers & ((~0ull) >> (64 - lane)));
        unsigned           rank = (unsigned)__popcll(lt);
        if(live && rank == 0)
            wcnt[w][d] = (unsigned)__popcll(peers);
        __syncthreads();
        if(live)
        {
            unsigned off = base_d[d] + rank;
            for(int q = 0; q < w; q++)
                off += wcnt[q][d];
            out[off] = k;
            if(KV)
                vout[off] = vin[i];
        }
        __syncthreads();
        base_d[threadIdx.x] += wcnt[0][threadIdx.x] + wcnt[1][threadIdx.x] + wcnt[2][threadIdx.x]
                               + wcnt[3][threadIdx.x];
        __syncthreads();
    }
}

// The whole sort in one workgroup, for up to 1024 J keys: a pass over one digit
// is a few microseconds of work here, against three launches of 2 to 6 us and
// the gaps between them.  A thread holds J keys (element 64 J w + 64 j + lane in
// the current order); ranks come from ballots and per-wave digit counters, so a
// pass is stable, and the keys move through LDS.  What: the keys, pairs, or the
// keys made here from the n leaf boxes (their common box into scene, Morton
// codes; see k_box_partial, k_morton).
enum
{
    SORT_KEYS  = 0,
    SORT_PAIRS = 1,
    SORT_BOXES = 2
};
constexpr int kSmallThreads = 1024;

template <int J, int What>
constexpr size_t kSmallLds = (size_t)kSmallThreads * J * (What == SORT_PAIRS ? 12 : 8)
                             + (kSmallThreads / 64 + 1) * 256 * sizeof(unsigned);

template <int J, int What>
__global__ void __launch_bounds__(kSmallThreads)
    k_sort_small(int n, int lo, int hi, uint64_t* __restrict__ keys, uint32_t* __restrict__ vals,
                 const double* __restrict__ leaf, double* __restrict__ scene)
{
    constexpr int NW = kSmallThreads / 64;
    extern __shared__ __align__(16) unsigned char sort_lds[];
    uint64_t* lk    = reinterpret_cast<uint64_t*>(sort_lds);
    unsigned* cnt   = reinterpret_cast<unsigned*>(lk + kSmallThreads * J);  // [wave][digit]
    unsigned* dbase = cnt + 256 * NW;
    uint32_t* lv    = dbase + 256;
    __shared__ double   box[6][NW], sc[6];
    __shared__ unsigned wsum[4];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int i0 = 64 * J * w + lane;
    uint64_t  k[J];
    uint32_t  v[J];
    if constexpr(What == SORT_BOXES)
    {
        double b[6] = {-1e32, -1e32, -1e32, 1e32, 1e32, 1e32};
#pragma unroll
        for(int j = 0; j < J; j++)
            if(i0 + 64 * j < n)
                for(int c = 0; c < 6; c++)
                {
                    const double p = leaf[6 * (size_t)(i0 + 64 * j) + c];
                    b[c] = (c < 3) ? ((b[c] < p) ? p : b[c]) : ((p < b[c]) ? p : b[c]);
                }
        for(int c = 0; c < 6; c++)
        {
            const double r = c < 3 ? wave_max(b[c]) : wave_min(b[c]);
            if(lane == 0)
                box[c][w] = r;
        }
        __syncthreads();
        if(t < 6)
        {
            double r = box[t][0];
            for(int q = 1; q < NW; q++)
                r = (t < 3) ? ((r < box[t][q]) ? box[t][q] : r)
                            : ((box[t][q] < r) ? box[t][q] : r);
            scene[t] = sc[t] = r;
        }
        __syncthreads();
#pragma unroll
        for(int j = 0; j < J; j++)
            k[j] = i0 + 64 * j < n ? morton_key(i0 + 64 * j, leaf, sc) : 0;
    }
    else
    {
#pragma unroll
        for(int j = 0; j < J; j++)
        {
            const bool live = i0 + 64 * j < n;
            k[j]            = live ? keys[i0 + 64 * j] : 0;
            if(What == SORT_PAIRS)
                v[j] = live ? vals[i0 + 64 * j] : 0;
        }
    }
#pragma unroll 1
    for(int sh = lo; sh < hi; sh += 8)
    {
        unsigned* my = cnt + 256 * w;
        unsigned  r[J];
        for(int q = 0; q < 4; q++)
            my[64 * q + lane] = 0;
        wave_lds_sync();
#pragma unroll
        for(int j = 0; j < J; j++)
        {
            const bool         live  = i0 + 64 * j < n;
            const unsigned     d     = (unsigned)(k[j] >> sh) & 0xFF;
            unsigned long long peers = __ballot(live);
#pragma unroll
            for(int b = 0; b < 8; b++)
            {
                const unsigned long long m = __ballot((d >> b) & 1u);
                peers &= ((d >> b) & 1u) ? m : ~m;
            }
            const unsigned rank = (unsigned)__popcll(peers & ((1ull << lane) - 1ull));
            const unsigned c    = my[d];
            wave_lds_sync();
            if(live && rank == 0)
                my[d] = c + (unsigned)__popcll(peers);
            wave_lds_sync();
            r[j] = c + rank;
        }
        __syncthreads();
        // digit t: its waves' counters become offsets; then the digits' offsets
        unsigned tot = 0, s = 0;
        if(t < 256)
        {
            unsigned c[NW];
#pragma unroll
            for(int q = 0; q < NW; q++)
                c[q] = cnt[256 * q + t];
#pragma unroll
            for(int q = 0; q < NW; q++)
            {
                cnt[256 * q + t] = tot;
                tot += c[q];
            }
            s = tot;
            for(int o = 1; o < 64; o <<= 1)
            {
                const unsigned u = __shfl_up(s, o, 64);
                if(lane >= o)
                    s += u;
            }
            if(lane == 63)
                wsum[w] = s;
        }
        __syncthreads();
        if(t < 256)
        {
            for(int q = 0; q < w; q++)
                s += wsum[q];
            dbase[t] = s - tot;
        }
        __syncthreads();
#pragma unroll
        for(int j = 0; j < J; j++)
            if(i0 + 64 * j < n)
            {
                const unsigned d   = (unsigned)(k[j] >> sh) & 0xFF;
                const unsigned off = dbase[d] + my[d] + r[j];
                lk[off]            = k[j];
                if(What == SORT_PAIRS)
                    lv[off] = v[j];
            }
        __syncthreads();
#pragma unroll
        for(int j = 0; j < J; j++)
            if(i0 + 64 * j < n)
            {
                k[j] = lk[i0 + 64 * j];
                if(What == SORT_PAIRS)
                    v[j] = lv[i0 + 64 * j];
            }
    }
#pragma unroll
    for(int j = 0; j < J; j++)
        if(i0 + 64 * j < n)
        {
            keys[i0 + 64 * j] = k[j];
            if(What == SORT_PAIRS)
                vals[i0 + 64 * j] = v[j];
        }
}

// --------------------------------------------------------- Karras build
__device__ __forceinline__ int cub64(uint64_t a, uint64_t b) { return __clzll(a ^ b); }

__global__ void k_leaf_nodes(int n, const uint64_t* __restrict__ keys, uint32_t* __restrict__ nodes,
                             const double* __restrict__ leaf, double* __restrict__ bvs, int arity,
                             const uint32_t* __restrict__ prims, const int* __restrict__ body,
                             int2* __restrict__ lbody)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= n)
        return;
    if(i < n - 1)
    {
        uint32_t* nd = nodes + 4 * (size_t)i;
        nd[0] = nd[1] = nd[2] = nd[3] = 0xFFFFFFFFu;
    }
    uint32_t  el = (uint32_t)(keys[i] & 0xFFFFFFFFull);
    uint32_t* nd = nodes + 4 * (size_t)(i + n - 1);
    nd[0] = nd[1] = nd[2] = 0xFFFFFFFFu;
    nd[3]                 = el;
    const int b = body[prims[(size_t)arity * el]];
    lbody[i]    = make_int2(b, b);
    for(int c = 0; c < 6; c++)
        bvs[6 * (size_t)(i + n - 1) + c] = leaf[6 * (size_t)el + c];
}

__global__ void k_internal_nodes(int n, const uint64_t* __restrict__ code, uint32_t* __restrict__ nodes,
                                 int* __restrict__ rng)
{
    int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if(idx >= n - 1)
        return;
    int first, last;
    if(idx == 0)
    {
        first = 0;
        last  = n - 1;
    }
    else
    {
        uint64_t self = code[idx];
        int      Ld   = cub64(self, code[idx - 1]);
        int      Rd   = cub64(self, code[idx + 1]);
        int      d    = (Rd > Ld) ? 1 : -1;
        int      dmin = Ld < Rd ? Ld : Rd;
        int      lmax = 2;
        int      delta = -1;
        int      it    = idx + d * lmax;
        if(0 <= it && it < n)
            delta = cub64(self, code[it]);
        while(delta > dmin)
        {
            lmax <<= 1;
            it    = idx + d * lmax;
            delta = -1;
            if(0 <= it && it < n)
                delta = cub64(self, code[it]);
        }
        int l = 0;
        for(int t = lmax >> 1; t > 0; t >>= 1)
        {
            it    = idx + (l + t) * d;
            delta = -1;
            if(0 <= it && it < n)
                delta = cub64(self, code[it]);
            if(delta > dmin)
                l += t;
        }
        int j = idx + l * d;
        first = d < 0 ? j : idx;
        last  = d < 0 ? idx : j;
    }
    int gamma;
    {
        uint64_t fc = code[first], lc = code[last];
        if(fc == lc)
            gamma = (first + last) >> 1;
        else
        {
            int dn     = cub64(fc, lc);
            int split  = first;
            int stride = last - first;
            do
            {
                stride     = (stride + 1) >> 1;
                int middle = split + stride;
                if(middle < last && cub64(fc, code[middle]) > dn)
                    split = middle;
            } while(stride > 1);
            gamma = split;
        }
    }
    rng[2 * (size_t)idx]     = first < last ? first : last;
    rng[2 * (size_t)idx + 1] = first < last ? last : first;
    uint32_t L = (uint32_t)gamma, R = (uint32_t)gamma + 1;
    if(min(first, last) == gamma)
        L += n - 1;
    if(max(first, last) == gamma + 1)
        R += n - 1;
    nodes[4 * (size_t)idx + 1] = L;
    nodes[4 * (size_t)idx + 2] = R;
    nodes[4 * (size_t)L]       = (uint32_t)idx;
    nodes[4 * (size_t)R]       = (uint32_t)idx;
}

// ------------------------------------------------------------------ refit
// Internal node i covers the sorted leaves [first_i, last_i] (Karras), so its
// box is the union of those leaf boxes.  Unions are exact (max/min), so the
// boxes are bit-identical to a bottom-up refit whatever the order.  Instead
// of walking up with atomics and device-wide fences, every node is computed
// independently from the aligned power-of-two groups of leaves (level k: one
// box per 2^k leaves): a range is at most two groups per level, so the longest
// chain is 2 log2(n) boxes.  (With two levels of 64-groups a node scanned up
// to 255 boxes one after the other: 84 us per tree of 387k edges.)  The
// groups also carry the smallest and largest body id of their primitives.

// one thread per entry of the input level (m entries); a wave makes the six
// levels above it
__global__ void __launch_bounds__(256) k_box_levels(int m, const double* __restrict__ in,
                                                    const int2* __restrict__ inb,
                                                    double* __restrict__ agg,
                                                    int2* __restrict__ aggb, BoxLevels lv, int k0)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double    v[6];
    int2      b = make_int2(INT_MAX, INT_MIN);
    if(i < m)
    {
        for(int c = 0; c < 6; c++)
            v[c] = in[6 * (size_t)i + c];
        b = inb[i];
    }
    else
        for(int c = 0; c < 3; c++)
        {
            v[c]     = -INFINITY;
            v[3 + c] = INFINITY;
        }
#pragma unroll
    for(int k = 0; k < 6; k++)
    {
        const int o = 1 << k;
#pragma unroll
        for(int c = 0; c < 3; c++)
        {
            double a = __shfl_xor(v[c], o, 64), d = __shfl_xor(v[3 + c], o, 64);
            v[c]     = (v[c] < a) ? a : v[c];
            v[3 + c] = (d < v[3 + c]) ? d : v[3 + c];
        }
        b.x = min(b.x, __shfl_xor(b.x, o, 64));
        b.y = max(b.y, __shfl_xor(b.y, o, 64));
        if(i < m && (i & (2 * o - 1)) == 0)
        {
            const size_t g = (size_t)lv.off[k0 + k + 1] + (i >> (k + 1));
#pragma unroll
            for(int c = 0; c < 6; c++)
                agg[6 * g + c] = v[c];
            aggb[g] = b;
        }
    }
}

// the next float below / above x unless x is a float
__device__ __forceinline__ float float_down(double x)
{
    float f = (float)x;
    if((double)f > x)
        f = f > 0.0f ? __uint_as_float(__float_as_uint(f) - 1u)
                     : (f < 0.0f ? __uint_as_float(__float_as_uint(f) + 1u) : -1e-45f);
    return f;
}
__device__ __forceinline__ float float_up(double x) { return -float_down(-x); }

// one thread per node: internal nodes' boxes, and every node's half of its
// parent's traversal record (box rounded outwards to FP32)
__global__ void __launch_bounds__(256) k_refit(int n, const int* __restrict__ rng,
                                               const uint32_t* __restrict__ nodes,
                                               const int2* __restrict__ lbody,
                                               const double* __restrict__ agg,
                                               const int2* __restrict__ aggb, BoxLevels lv,
                                               double* __restrict__ bvs,
                                               NodeHalf* __restrict__ rec)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= 2 * n - 1)
        return;
    const uint32_t parent = nodes[4 * (size_t)i];
    const double*  leaf   = bvs + 6 * (size_t)(n - 1);
    double         v[6];
    int2           b;
    if(i >= n - 1)
    {
        for(int c = 0; c < 6; c++)
            v[c] = bvs[6 * (size_t)i + c];
        b = lbody[i - (n - 1)];
    }
    else
    {
        for(int c = 0; c < 3; c++)
        {
            v[c]     = -INFINITY;
            v[3 + c] = INFINITY;
        }
        b        = make_int2(INT_MAX, INT_MIN);
        auto add = [&](int k, int j) {
            const double* p = k == 0 ? leaf + 6 * (size_t)j : agg + 6 * (size_t)(lv.off[k] + j);
            const int2    q = k == 0 ? lbody[j] : aggb[lv.off[k] + j];
#pragma unroll
            for(int c = 0; c < 3; c++)
            {
                v[c]     = (v[c] < p[c]) ? p[c] : v[c];
                v[3 + c] = (p[3 + c] < v[3 + c]) ? p[3 + c] : v[3 + c];
            }
            b.x = min(b.x, q.x);
            b.y = max(b.y, q.y);
        };
        int l = rng[2 * (size_t)i], r = rng[2 * (size_t)i + 1] + 1;
        for(int k = 0; l < r; k++)
        {
            if(l & 1)
                add(k, l++);
            if(r & 1)
                add(k, --r);
            l >>= 1;
            r >>= 1;
        }
        double* o = bvs + 6 * (size_t)i;
        for(int c = 0; c < 6; c++)
            o[c] = v[c];
    }
    if(parent == 0xFFFFFFFFu)
        return;
    NodeHalf h;
    for(int c = 0; c < 3; c++)
    {
        h.up[c] = float_up(v[c]);
        h.lo[c] = float_down(v[3 + c]);
    }
    h.child = i >= n - 1 ? (0x80000000u | (uint32_t)(i - (n - 1))) : (uint32_t)i;
    h.body  = b.x == b.y && b.x != -1 ? b.x : kMixedBody;
    rec[2 * (size_t)parent + (nodes[4 * (size_t)parent + 1] == (uint32_t)i ? 0 : 1)] = h;
}

void Lbvh::init(int n_, int arity_, const uint32_t* prims_, const int* body_)
{
    n     = n_;
    arity = arity_;
    prims = prims_;
    body  = body_;
    if(n <= 0)
        return;
    leaf.resize(6 * (size_t)n);
    bvs.resize(6 * (size_t)(2 * n - 1));
    nodes.resize(4 * (size_t)(2 * n - 1));
    rec.resize(2 * (size_t)(n > 1 ? n - 1 : 1));
    keys.resize(n);
    keys_alt.resize(n);
    lbody.resize(n);
    rng.resize(2 * (size_t)(n > 1 ? n - 1 : 1));
    levels    = BoxLevels{};
    int total = 0, m = n;
    // six levels per launch, past the first level of one box
    for(int k = 1; k < kBoxLevels; k++)
    {
        m             = (m + 1) / 2;
        levels.off[k] = total;
        total += m;
    }
    agg.resize(6 * (size_t)total);
    aggb.resize(total);
    hist.resize(radix_sort_hist_size(n));
    scene.resize(6);
    partial.resize(6 * (size_t)grid_for(n, 256));
}

// exclusive scan of the digit-major histogram (256 digits x nblk tiles), in
// place: one workgroup for short histograms, the three-launch tiled scan
// (tile sums, their scan, apply; its tile sums after the histogram) for long
// ones, where one workgroup's sequential rounds take longer than two launches
static void sort_scan(unsigned* hist, int nblk, hipStream_t s)
{
    const int total = 256 * nblk;
    if(nblk < 128)
        hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(1024), 0, s, total, hist);
    else
        scan_exclusive_u32(total, hist, hist, hist + total, s);
}

// the sort in one workgroup; false: too many keys for it.  Boxes, keys and four
// passes: 14.5 us up to 2,048 boxes against 15 launches of together 52 us and
// the gaps between them (a Newton iteration on a 425-vertex bar has about five
// such sorts: 2.5 -> 2.3 ms).  Sixteen keys per thread no longer fit the
// registers: 81 us for 14,000 boxes, 15 launches take 66 us and their gaps, and
// the iteration was not faster; so the line lies at eight.
template <int What>
static bool sort_small(int n, int lo, int hi, uint64_t* keys, uint32_t* vals, const double* leaf,
                       double* scene, hipStream_t s)
{
    auto go = [&](auto kern, size_t lds) {
        hipLaunchKernelGGL(kern, dim3(1), dim3(kSmallThreads), lds, s, n, lo, hi, keys, vals, leaf,
                           scene);
        SG_LAUNCH_CHECK();
        return true;
    };
    if(n <= 2 * kSmallThreads)
        return go(k_sort_small<2, What>, kSmallLds<2, What>);
    if(n <= 4 * kSmallThreads)
        return go(k_sort_small<4, What>, kSmallLds<4, What>);
    if(n <= 8 * kSmallThreads)
        return go(k_sort_small<8, What>, kSmallLds<8, What>);
    return false;
}

// stable LSD radix sort of n 64-bit keys on the 8-bit digits from bit lo to
// bit hi (exclusive); the result ends in keys (alt: scratch of n keys, hist:
// radix_sort_hist_size(n) counters)
void radix_sort_keys(uint64_t* keys, uint64_t* alt, unsigned* hist, int n, int lo, int hi,
                     hipStream_t s)
{
    if(n <= 1 || sort_small<SORT_KEYS>(n, lo, hi, keys, nullptr, nullptr, nullptr, s))
        return;
    int       nblk = (n + kSortTile - 1) / kSortTile;
    uint64_t* a    = keys;
    uint64_t* b    = alt;
    for(int sh = lo; sh < hi; sh += 8)
    {
        hipLaunchKernelGGL(k_sort_hist, dim3(nblk), dim3(kSortThreads), 0, s, n, sh, a, hist, nblk);
        sort_scan(hist, nblk, s);
        hipLaunchKernelGGL(k_sort_scatter<false>, dim3(nblk), dim3(kSortThreads), 0, s, n, sh, a, b,
                           hist, nblk, nullptr, nullptr);
        SG_LAUNCH_CHECK();
        std::swap(a, b);
    }
    if(a != keys)
        SG_HIP(hipMemcpyAsync(keys, a, n * sizeof(uint64_t), hipMemcpyDeviceToDevice, s));
}

void radix_sort_pairs(uint64_t* keys, uint64_t* kalt, uint32_t* vals, uint32_t* valt,
                      unsigned* hist, int n, int lo, int hi, hipStream_t s)
{
    if(n <= 1 || sort_small<SORT_PAIRS>(n, lo, hi, keys, vals, nullptr, nullptr, s))
        return;
    int       nblk = (n + kSortTile - 1) / kSortTile;
    uint64_t* a    = keys;
    uint64_t* b    = kalt;
    uint32_t* va   = vals;
    uint32_t* vb   = valt;
    for(int sh = lo; sh < hi; sh += 8)
    {
        hipLaunchKernelGGL(k_sort_hist, dim3(nblk), dim3(kSortThreads), 0, s, n, sh, a, hist, nblk);
        sort_scan(hist, nblk, s);
        hipLaunchKernelGGL(k_sort_scatter<true>, dim3(nblk), dim3(kSortThreads), 0, s, n, sh, a, b,
                           hist, nblk, va, vb);
        SG_LAUNCH_CHECK();
        std::swap(a, b);
        std::swap(va, vb);
    }
    if(a != keys)
    {
        SG_HIP(hipMemcpyAsync(keys, a, n * sizeof(uint64_t), hipMemcpyDeviceToDevice, s));
        SG_HIP(hipMemcpyAsync(vals, va, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
    }
}

int radix_key_bits(uint64_t max_key)
{
    int b = 0;
    while(b < 64 && (max_key >> b))
        b++;
    return (b + 7) / 8 * 8;
}

size_t radix_sort_hist_size(int n)
{
    const int total = 256 * ((n + kSortTile - 1) / kSortTile);
    return (size_t)total + scan_tmp_size(total);
}

void Lbvh::build(const double* x, const double* dx, double alpha, hipStream_t s)
{
    if(n <= 0)
        return;
    hipLaunchKernelGGL(k_leaf_aabb, dim3(grid_for(n, 256)), dim3(256), 0, s, n, arity, prims, x,
                       dx, alpha, leaf.data());
    // the keys enter in index order and every pass is stable, so sorting the
    // 30 Morton bits alone orders by (morton, index)
    if(!sort_small<SORT_BOXES>(n, 32, 62, keys.data(), nullptr, leaf.data(), scene.data(), s))
    {
        unsigned nb = grid_for(n, 256);
        hipLaunchKernelGGL(k_box_partial, dim3(nb), dim3(256), 0, s, n, leaf.data(),
                           partial.data());
        hipLaunchKernelGGL(k_box_final, dim3(1), dim3(256), 0, s, (int)nb, partial.data(),
                           scene.data());
        hipLaunchKernelGGL(k_morton, dim3(grid_for(n, 256)), dim3(256), 0, s, n, leaf.data(),
                           scene.data(), keys.data());
        SG_LAUNCH_CHECK();
        radix_sort_keys(keys.data(), keys_alt.data(), hist.data(), n, 32, 62, s);
    }
    hipLaunchKernelGGL(k_leaf_nodes, dim3(grid_for(n, 256)), dim3(256), 0, s, n, keys.data(),
                       nodes.data(), leaf.data(), bvs.data(), arity, prims, body, lbody.data());
    if(n > 1)
    {
        hipLaunchKernelGGL(k_internal_nodes, dim3(grid_for(n - 1, 256)), dim3(256), 0, s, n,
                           keys.data(), nodes.data(), rng.data());
        int m = n;
        for(int k = 0; m > 1; k += 6)
        {
            SG_CHECK(k + 6 < kBoxLevels, SGIPC_ECAPACITY, "too many primitives for the box levels");
            hipLaunchKernelGGL(k_box_levels, dim3(grid_for(m, 256)), dim3(256), 0, s, m,
                               k == 0 ? bvs.data() + 6 * (size_t)(n - 1)
                                      : agg.data() + 6 * (size_t)levels.off[k],
                               k == 0 ? lbody.data() : aggb.data() + levels.off[k], agg.data(),
                               aggb.data(), levels, k);
            m = (m + 63) / 64;
        }
        hipLaunchKernelGGL(k_refit, dim3(grid_for(2 * n - 1, 256)), dim3(256), 0, s, n, rng.data(),
                           nodes.data(), lbody.data(), agg.data(), aggb.data(), levels, bvs.data(),
                           rec.data());
    }
    SG_LAUNCH_CHECK();
}

}  // namespace sgipc
