// contact.hip -- proximity and CCD candidate queries on the LBVHs.
//
//   k_query_vf   surface vertex vs face tree  (_selfQuery_vf, mlbvh.cu:1308-1408)
//   k_query_ee   edge leaf vs edge tree       (_selfQuery_ee, mlbvh.cu:1511-1634)
//   k_ccd_vf/ee  swept candidates             (_selfQuery_*_ccd, mlbvh.cu:1410-1740)
//   k_edge_tri   segment-triangle intersection (_edgeTriIntersectionQuery,
//                GIPC.cu:8188-8302, segTriIntersect :961-1013)
// Classification and codes follow _checkPTintersection / _checkEEintersection
// (mlbvh.cu:537-1062, smooth == false).  Built with -ffp-contract=off so the
// pair multiset equals the CPU restatement's.
//
// One wave per 64 queries, one query per lane.  A traversal step loads one
// 64-byte record (both children's boxes in FP32, rounded outwards); the exact
// FP64 box test decides at the leaves, which gives the same leaves as FP64
// tests all the way down (a leaf's box is inside its ancestors').  Proximity
// and CCD queries skip subtrees whose primitives all belong to the query's
// own body: such pairs are never candidates, and in scenes of many bodies
// they are most of what a query meets.  The leaves that a wave's walks meet
// are collected and tested 64 at a time, whichever query they belong to.
// Records are claimed with one counter update per wave and event.  Bound by
// the dependent record loads of the walk.  64 cubes in contact (73,728 edges,
// 40,573 pairs), each leaf tested where it is met / collected: edge-edge
// 397 / 130 us, vertex-face 195 / 61 us, swept 331 / 77 and 152 / 52 us,
// edge-triangle 226 / 116 us.
//
// The traversal stack lives in LDS as stk[depth][lane] (bank-conflict free),
// its rarely reached upper part (a 64-bit-key Karras tree is at most 64 deep)
// in the lane's private memory.
#include "sim_kernels.h"

namespace sgipc
{

constexpr int kStackLds = 20;
constexpr int kStackMax = 64;

__device__ __forceinline__ bool overlap(const double* l, const double* r, double gap)
{
    // l, r: {upper xyz, lower xyz} (mlbvh.cu:31-40)
    for(int c = 0; c < 3; c++)
        if((r[3 + c] - l[c]) >= gap || (l[3 + c] - r[c]) >= gap)
            return false;
    return true;
}

// one counter update for the active lanes of the wave; this lane's slot
__device__ __forceinline__ unsigned claim(unsigned* counter)
{
    const unsigned long long m      = __ballot(1);
    const int                lane   = (int)__lane_id();
    const int                leader = __ffsll((long long)m) - 1;
    unsigned                 base   = 0;
    if(lane == leader)
        base = atomicAdd(counter, (unsigned)__popcll(m));
    base = __shfl(base, leader, 64);
    return base + (unsigned)__popcll(m & ((1ull << lane) - 1ull));
}

struct PairSink
{
    int4*     pairs;
    int4*     raw;
    unsigned* cnt;  // [0] total, [2] PP, [3] PE, [4] PT + EE
    int       cap;
    int*      overflow;
    unsigned  type[3] = {0, 0, 0};  // this lane's PP, PE, PT + EE records
    __device__ void emit(int4 code, int4 rawc, int slot_type)
    {
        unsigned o = claim(cnt);
        if((int)o >= cap)
        {
            atomicExch(overflow, 1);
            return;
        }
        pairs[o] = code;
        raw[o]   = rawc;
        type[0] += slot_type == 2 ? 1u : 0u;
        type[1] += slot_type == 3 ? 1u : 0u;
        type[2] += slot_type == 4 ? 1u : 0u;
    }
    // every lane of the wave, after its last record
    __device__ void flush()
    {
        for(int k = 0; k < 3; k++)
        {
            unsigned t = type[k];
            for(int o = 32; o > 0; o >>= 1)
                t += __shfl_xor(t, o, 64);
            if(__lane_id() == 0 && t)
                atomicAdd(cnt + 2 + k, t);
        }
    }
};

__device__ void check_pt(const double* x, int id0, int id1, int id2, int id3, double dHat,
                         PairSink& sk)
{
    V3   v0 = ld3(x + 3 * id0), v1 = ld3(x + 3 * id1), v2 = ld3(x + 3 * id2), v3 = ld3(x + 3 * id3);
    int  t  = dtype_pt(v0, v1, v2, v3);
    int4 raw = make_int4(-id0 - 1, id1, id2, id3);
    switch(t)
    {
        case 0:
            if(d_pp(v0, v1) < dHat)
                sk.emit(make_int4(-id0 - 1, id1, -1, -1), raw, 2);
            break;
        case 1:
            if(d_pp(v0, v2) < dHat)
                sk.emit(make_int4(-id0 - 1, id2, -1, -1), raw, 2);
            break;
        case 2:
            if(d_pp(v0, v3) < dHat)
                sk.emit(make_int4(-id0 - 1, id3, -1, -1), raw, 2);
            break;
        case 3:
            if(d_pe(v0, v1, v2) < dHat)
                sk.emit(make_int4(-id0 - 1, id1, id2, -1), raw, 3);
            break;
        case 4:
            if(d_pe(v0, v2, v3) < dHat)
                sk.emit(make_int4(-id0 - 1, id2, id3, -1), raw, 3);
            break;
        case 5:
            if(d_pe(v0, v3, v1) < dHat)
                sk.emit(make_int4(-id0 - 1, id3, id1, -1), raw, 3);
            break;
        case 6:
            if(d_pt(v0, v1, v2, v3) < dHat)
                sk.emit(make_int4(-id0 - 1, id1, id2, id3), raw, 4);
            break;
        default: break;
    }
}

__device__ __forceinline__ double epx(V3 r0, V3 r1, V3 r2, V3 r3)
{
    return 1e-3 * sqn(r0 - r1) * sqn(r2 - r3);
}

__device__ void check_ee(const double* x, const double* xr, int id0, int id1, int id2, int id3,
                         int obj, double dHat, PairSink& sk)
{
    V3   v0 = ld3(x + 3 * id0), v1 = ld3(x + 3 * id1), v2 = ld3(x + 3 * id2), v3 = ld3(x + 3 * id3);
    int  t   = dtype_ee(v0, v1, v2, v3);
    int4 raw = make_int4(id0, id1, id2, id3);
    auto flag01 = [&]() {
        double cr = sqn(cross(v0 - v1, v2 - v3));
        return (cr < epx(ld3(xr + 3 * id0), ld3(xr + 3 * id1), ld3(xr + 3 * id2),
                         ld3(xr + 3 * id3)))
                   ? -obj - 2
                   : -1;
    };
    auto flag23 = [&]() {
        double cr = sqn(cross(v2 - v3, v0 - v1));
        return (cr < epx(ld3(xr + 3 * id2), ld3(xr + 3 * id3), ld3(xr + 3 * id0),
                         ld3(xr + 3 * id1)))
                   ? -obj - 2
                   : -1;
    };
    switch(t)
    {
        case 0:
            if(d_pp(v0, v2) < dHat)
                sk.emit(make_int4(-id0 - 1, id2, -1, flag01()), raw, 2);
            break;
        case 1:
            if(d_pp(v0, v3) < dHat)
                sk.emit(make_int4(-id0 - 1, id3, -1, flag01()), raw, 2);
            break;
        case 2:
            if(d_pe(v0, v2, v3) < dHat)
                sk.emit(make_int4(-id0 - 1, id2, id3, flag01()), raw, 3);
            break;
        case 3:
            if(d_pp(v1, v2) < dHat)
                sk.emit(make_int4(-id1 - 1, id2, -1, flag01()), raw, 2);
            break;
        case 4:
            if(d_pp(v1, v3) < dHat)
                sk.emit(make_int4(-id1 - 1, id3, -1, flag01()), raw, 2);
            break;
        case 5:
            if(d_pe(v1, v2, v3) < dHat)
                sk.emit(make_int4(-id1 - 1, id2, id3, flag01()), raw, 3);
            break;
        case 6:
            if(d_pe(v2, v0, v1) < dHat)
                sk.emit(make_int4(-id2 - 1, id0, id1, flag23()), raw, 3);
            break;
        case 7:
            if(d_pe(v3, v0, v1) < dHat)
                sk.emit(make_int4(-id3 - 1, id0, id1, flag23()), raw, 3);
            break;
        case 8:
            if(d_ee(v0, v1, v2, v3) < dHat)
                sk.emit(make_int4(id0, id1, id2, id3), raw, 4);
            break;
        default: break;
    }
}

__device__ __forceinline__ bool vf_ok(const int* body, const int* bt, int v, uint3 f)
{
    if(!((body[v] != body[f.x]) || (body[v] == -1)))
        return false;
    if(v == (int)f.x || v == (int)f.y || v == (int)f.z)
        return false;
    if(bt[v] >= 2 && bt[f.x] >= 2 && bt[f.y] >= 2 && bt[f.z] >= 2)
        return false;
    return true;
}

__device__ __forceinline__ bool ee_ok(const int* body, const int* bt, uint2 a, uint2 b, int self,
                                      int obj)
{
    if(self == obj)
        return false;
    if(!((body[a.x] != body[b.x]) || (body[a.x] == -1)))
        return false;
    if(a.x == b.x || a.x == b.y || a.y == b.x || a.y == b.y || obj < self)
        return false;
    if(bt[a.x] >= 2 && bt[a.y] >= 2 && bt[b.x] >= 2 && bt[b.y] >= 2)
        return false;
    return true;
}

// what a traversal reads of a tree
struct Tree
{
    int             n;
    const NodeHalf* rec;
    const double*   leaf;  // sorted leaf boxes
    const uint64_t* keys;  // low word: element of the sorted leaf
    __device__ uint32_t element(int s) const { return (uint32_t)keys[s]; }
};

static Tree tree_of(const Lbvh& b)
{
    return Tree{b.n, b.rec.data(), b.bvs.data() + 6 * (size_t)(b.n > 0 ? b.n - 1 : 0),
                b.keys.data()};
}

// the float below / above x by at least one step
__device__ __forceinline__ float below(double x)
{
    const float f = (float)x;
    return f - fmaxf(fabsf(f) * 2.4e-7f, 1e-37f);
}

// LDS of a wave's queries
struct WaveQueries
{
    uint32_t stk[kStackLds][64];  // traversal stacks
    uint32_t own[3][64];          // what a leaf visit needs of its query
    double   q[6][64];            // query boxes
    uint32_t item[3 * 64];        // leaves to visit: sorted leaf
    uint8_t  of[3 * 64];          // and query (lane)
};

// visit(query lane, sorted leaf) for every leaf whose box overlaps the
// query's box q within gap; live: this lane has a query.  Called by all lanes
// of a wave.  The leaves that the 64 walks meet are collected and visited 64
// at a time, one per lane and of whichever query: a visit's chain of loads
// then holds up the wave once for 64 leaves, not once for each step in
// which some lane met one.  A visit that returns true ends the wave's walks.
// Leaves at sorted positions up to `after` are left out: a self query of the
// tree from its sorted leaf `after` then meets every unordered pair of leaves
// once, from the earlier one.  qbody: skip subtrees of this body (kMixedBody:
// none).
template <typename Visit>
__device__ __forceinline__ void traverse(const Tree& T, bool live, const double (&q)[6], double gap,
                                         int qbody, WaveQueries& W, Visit&& visit, int after = -1)
{
    const int lane = threadIdx.x;
#pragma unroll
    for(int c = 0; c < 6; c++)
        W.q[c][lane] = q[c];
    // the query box grown by gap and rounded outwards
    float ql[3], qu[3];
#pragma unroll
    for(int c = 0; c < 3; c++)
    {
        qu[c] = -below(-(q[c] + gap));
        ql[c] = below(q[3 + c] - gap);
    }
    auto hit = [&](const NodeHalf& h) {
        bool ok = qbody == kMixedBody || h.body != qbody;
#pragma unroll
        for(int c = 0; c < 3; c++)
            ok = ok && !(h.lo[c] > qu[c]) && !(h.up[c] < ql[c]);
        return ok;
    };
    int  n   = 0;  // collected leaves
    auto put = [&](bool on, uint32_t leaf) {
        const unsigned long long m = __ballot(on);
        const int                o = n + __popcll(m & ((1ull << lane) - 1ull));
        if(on)
        {
            W.item[o] = leaf & 0x7fffffffu;
            W.of[o]   = (uint8_t)lane;
        }
        n += __popcll(m);
    };
    // the last (up to) 64 collected leaves
    auto take = [&]() {
        wave_lds_sync();
        const int c  = n < 64 ? n : 64;
        bool      ok = false;
        if(lane < c)
        {
            const int s = (int)W.item[n - c + lane], o = W.of[n - c + lane];
            double    b[6];
#pragma unroll
            for(int k = 0; k < 6; k++)
                b[k] = W.q[k][o];
            ok = overlap(b, T.leaf + 6 * (size_t)s, gap) && visit(o, s);
        }
        n -= c;
        wave_lds_sync();
        return __any(ok) != 0;
    };
    uint32_t deep[kStackMax - kStackLds];
    int      sp   = 0;
    uint32_t node = 0;
    bool     more = live && T.n > 1 && after < T.n - 1;
    if(T.n == 1)
        put(live && after < 0, 0u);
    while(__any(more))
    {
        bool     pl = false, pr = false;
        uint32_t cl = 0, cr = 0;
        if(more)
        {
            const NodeHalf L = T.rec[2 * (size_t)node], R = T.rec[2 * (size_t)node + 1];
            const bool     hl = hit(L) && (int)(L.child & 0x7fffffffu) > after, hr = hit(R);
            cl = L.child, cr = R.child;
            pl = hl && (cl >> 31), pr = hr && (cr >> 31);
            const bool il = hl && !pl, ir = hr && !pr;
            if(il && ir)
            {
                if(sp < kStackLds)
                    W.stk[sp++][lane] = cr;
                else if(sp < kStackMax)
                    deep[sp++ - kStackLds] = cr;
            }
            if(il || ir)
                node = il ? cl : cr;
            else if(sp == 0)
                more = false;
            else
            {
                sp--;
                if(sp < kStackLds)
                    node = W.stk[sp][lane];
                else
                    node = deep[sp - kStackLds];
            }
        }
        put(pl, cl);
        put(pr, cr);
        bool stop = false;
        while(n >= 64 && !stop)
            stop = take();
        if(stop)
            return;
    }
    if(n > 0)
        take();
}

__device__ __forceinline__ int query_body(int b) { return b == -1 ? kMixedBody : b; }

__global__ void __launch_bounds__(64) k_query_vf(int ns, const uint32_t* __restrict__ surf,
                                                 const uint3* __restrict__ faces,
                                                 const int* __restrict__ body,
                                                 const int* __restrict__ bt,
                                                 const double* __restrict__ x, Tree tree,
                                                 double dHat, PairSink sk)
{
    __shared__ WaveQueries W;
    const int  i    = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < ns;
    const int  v    = (int)surf[live ? i : 0];
    const double q[6] = {x[3 * v], x[3 * v + 1], x[3 * v + 2], x[3 * v], x[3 * v + 1], x[3 * v + 2]};
    W.own[0][threadIdx.x] = (uint32_t)v;
    traverse(tree, live, q, sqrt(dHat), query_body(body[v]), W, [&](int o, int s) {
        const int v = (int)W.own[0][o];
        uint3     f = faces[tree.element(s)];
        if(vf_ok(body, bt, v, f))
            check_pt(x, v, f.x, f.y, f.z, dHat, sk);
        return false;
    });
    sk.flush();
}

// Edge-edge pairs: each edge queries the edge tree from its own sorted leaf
// for the leaves after it, and a pair is emitted with its lower edge index
// first, as the reference emits it from that edge's query (obj > self).
__global__ void __launch_bounds__(64) k_query_ee(int ne, const uint2* __restrict__ edges,
                                                 const int* __restrict__ body,
                                                 const int* __restrict__ bt,
                                                 const double* __restrict__ x,
                                                 const double* __restrict__ xr, Tree tree,
                                                 double dHat, PairSink sk)
{
    __shared__ WaveQueries W;
    const int  i    = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < ne;
    const int  il   = live ? i : 0;
    const int  self = (int)tree.element(il);
    double     q[6];
    for(int c = 0; c < 6; c++)
        q[c] = tree.leaf[6 * (size_t)il + c];
    const uint2 e = edges[self];
    W.own[0][threadIdx.x] = (uint32_t)self;
    W.own[1][threadIdx.x] = e.x;
    W.own[2][threadIdx.x] = e.y;
    traverse(
        tree, live, q, sqrt(dHat), query_body(body[e.x]), W,
        [&](int p, int s) {
            const int   self = (int)W.own[0][p];
            const uint2 e    = make_uint2(W.own[1][p], W.own[2][p]);
            const int   obj  = (int)tree.element(s);
            const int   lo   = self < obj ? self : obj;
            const int   hi   = self < obj ? obj : self;
            const uint2 o    = edges[obj];
            const uint2 a = lo == self ? e : o, b = lo == self ? o : e;
            if(ee_ok(body, bt, a, b, lo, hi))
                check_ee(x, xr, a.x, a.y, b.x, b.y, hi, dHat, sk);
            return false;
        },
        i);
    sk.flush();
}

struct CandSink
{
    int4*     out;
    unsigned* cnt;
    int       cap;
    int*      overflow;
    __device__ void emit(int4 c)
    {
        unsigned o = claim(cnt);
        if((int)o >= cap)
        {
            atomicExch(overflow, 1);
            return;
        }
        out[o] = c;
    }
};

__global__ void __launch_bounds__(64) k_ccd_vf(int ns, const uint32_t* __restrict__ surf,
                                               const uint3* __restrict__ faces,
                                               const int* __restrict__ body,
                                               const int* __restrict__ bt,
                                               const double* __restrict__ x,
                                               const double* __restrict__ dx, double alpha,
                                               Tree tree, double dHat, CandSink sk)
{
    __shared__ WaveQueries W;
    const int  i    = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < ns;
    const int  v    = (int)surf[live ? i : 0];
    double     q[6];
    for(int c = 0; c < 3; c++)
    {
        double a = x[3 * v + c], b = x[3 * v + c] - dx[3 * v + c] * alpha;
        q[c]     = (a < b) ? b : a;   // upper: combines(v - dx alpha) after (v, v)
        q[3 + c] = (b < a) ? b : a;
    }
    W.own[0][threadIdx.x] = (uint32_t)v;
    traverse(tree, live, q, sqrt(dHat), query_body(body[v]), W, [&](int o, int s) {
        const int v = (int)W.own[0][o];
        uint3     f = faces[tree.element(s)];
        if(((body[v] != body[f.x]) || (body[v] == -1))
           && !(bt[v] >= 2 && bt[f.x] >= 2 && bt[f.y] >= 2 && bt[f.z] >= 2)
           && v != (int)f.x && v != (int)f.y && v != (int)f.z)
            sk.emit(make_int4(-v - 1, f.x, f.y, f.z));
        return false;
    });
}

__global__ void __launch_bounds__(64) k_ccd_ee(int ne, const uint2* __restrict__ edges,
                                               const int* __restrict__ body,
                                               const int* __restrict__ bt, Tree tree, double dHat,
                                               CandSink sk)
{
    __shared__ WaveQueries W;
    const int  i    = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < ne;
    const int  il   = live ? i : 0;
    const int  self = (int)tree.element(il);
    double     q[6];
    for(int c = 0; c < 6; c++)
        q[c] = tree.leaf[6 * (size_t)il + c];
    const uint2 e = edges[self];
    W.own[0][threadIdx.x] = (uint32_t)self;
    W.own[1][threadIdx.x] = e.x;
    W.own[2][threadIdx.x] = e.y;
    traverse(
        tree, live, q, sqrt(dHat), query_body(body[e.x]), W,
        [&](int p, int s) {
            const int   self = (int)W.own[0][p];
            const uint2 e    = make_uint2(W.own[1][p], W.own[2][p]);
            const int   obj  = (int)tree.element(s);
            const int   lo   = self < obj ? self : obj;
            const int   hi   = self < obj ? obj : self;
            const uint2 o    = edges[obj];
            const uint2 a = lo == self ? e : o, b = lo == self ? o : e;
            if(ee_ok(body, bt, a, b, lo, hi))
                sk.emit(make_int4(a.x, a.y, b.x, b.y));
            return false;
        },
        i);
}

__device__ bool seg_tri(V3 e0, V3 e1, V3 t0, V3 t1, V3 t2)
{
    V3 c0 = t1 - t0, c1 = t2 - t0, c2 = e0 - e1;
    V3 n  = cross(c0, c1);
    if(dot(n, e0 - t0) * dot(n, e1 - t0) > 0)
        return false;
    double det = det_cols(c0, c1, c2);
    // segTriIntersect's |det| < 1e-20, plus a scale-relative test so that an
    // edge lying in the triangle's plane (coplanar surface faces) is rejected
    // whatever the mesh size; the absolute constant alone lets round-off
    // determinants through at centimetre scales
    double sc = sqrt(sqn(c0) * sqn(c1) * sqn(c2));
    if(fabs(det) < 1e-20 || fabs(det) <= 1e-12 * sc)
        return false;
    V3     b = e0 - t0;
    double u = det_cols(b, c1, c2) / det, v = det_cols(c0, b, c2) / det,
           t = det_cols(c0, c1, b) / det;
    return (u >= 0.0 && v >= 0.0 && u + v <= 1.0 && t >= 0.0 && t <= 1.0);
}

// one lane per face, in the face tree's sorted order (neighbouring lanes
// walk neighbouring parts of the edge tree)
__global__ void __launch_bounds__(64) k_edge_tri(int nf, const uint3* __restrict__ faces,
                                                 const uint2* __restrict__ edges,
                                                 const int* __restrict__ bt,
                                                 const double* __restrict__ x, Tree ftree,
                                                 Tree tree, int* hit)
{
    __shared__ WaveQueries W;
    const int  i    = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < nf;
    const int  il   = live ? i : 0;
    const uint3 f   = faces[ftree.element(il)];
    double      q[6];
    for(int c = 0; c < 6; c++)
        q[c] = ftree.leaf[6 * (size_t)il + c];
    W.own[0][threadIdx.x] = f.x;
    W.own[1][threadIdx.x] = f.y;
    W.own[2][threadIdx.x] = f.z;
    traverse(tree, live, q, 0.0, kMixedBody, W, [&](int o, int s) {
        const uint3 F = make_uint3(W.own[0][o], W.own[1][o], W.own[2][o]);
        const uint2 E = edges[tree.element(s)];
        if(F.x == E.x || F.x == E.y || F.y == E.x || F.y == E.y || F.z == E.x || F.z == E.y)
            return false;
        if(bt[F.x] >= 2 && bt[F.y] >= 2 && bt[F.z] >= 2 && bt[E.x] >= 2 && bt[E.y] >= 2)
            return false;
        const bool found = seg_tri(ld3(x + 3 * E.x), ld3(x + 3 * E.y), ld3(x + 3 * F.x),
                                   ld3(x + 3 * F.y), ld3(x + 3 * F.z));
        if(found)
            atomicExch(hit, 1);
        return found;
    });
}

__global__ void k_ground_intersect(const unsigned* __restrict__ gcount,
                                   const uint32_t* __restrict__ gp, const double* __restrict__ x,
                                   V3 n, double off, int* hit)
{
    unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if(i >= *gcount)
        return;
    double dist = dot(n, ld3(x + 3 * gp[i])) - off;
    if(dist < 0)
        atomicExch(hit, 1);
}

// ----------------------------------------------------------------- launch
void launch_query_proximity(const SimDev& d, const Lbvh& bf, const Lbvh& be, const double* xr,
                            hipStream_t s)
{
    SG_HIP(hipMemsetAsync(d.pcount, 0, 5 * sizeof(unsigned), s));
    PairSink sk{d.pairs, d.pairs_raw, d.pcount, d.pair_cap, d.overflow};
    if(d.nf > 0 && d.ns > 0)
        hipLaunchKernelGGL(k_query_vf, dim3(grid_for(d.ns, 64)), dim3(64), 0, s, d.ns, d.surf,
                           (const uint3*)d.faces, d.body, d.btype, d.x, tree_of(bf), d.dHat, sk);
    if(d.ne > 1)
        hipLaunchKernelGGL(k_query_ee, dim3(grid_for(d.ne, 64)), dim3(64), 0, s, d.ne,
                           (const uint2*)d.edges, d.body, d.btype, d.x, xr, tree_of(be), d.dHat,
                           sk);
    SG_LAUNCH_CHECK();
}

void launch_query_ccd(const SimDev& d, const Lbvh& bf, const Lbvh& be, const double* dx,
                      double alpha, int4* cand, unsigned* ccount, int cap, int* overflow,
                      hipStream_t s)
{
    SG_HIP(hipMemsetAsync(ccount, 0, sizeof(unsigned), s));
    CandSink sk{cand, ccount, cap, overflow};
    if(d.nf > 0 && d.ns > 0)
        hipLaunchKernelGGL(k_ccd_vf, dim3(grid_for(d.ns, 64)), dim3(64), 0, s, d.ns, d.surf,
                           (const uint3*)d.faces, d.body, d.btype, d.x, dx, alpha, tree_of(bf),
                           d.dHat, sk);
    if(d.ne > 1)
        hipLaunchKernelGGL(k_ccd_ee, dim3(grid_for(d.ne, 64)), dim3(64), 0, s, d.ne,
                           (const uint2*)d.edges, d.body, d.btype, tree_of(be), d.dHat, sk);
    SG_LAUNCH_CHECK();
}

void launch_edge_tri(const SimDev& d, const Lbvh& bf, const Lbvh& be, int* hit, hipStream_t s)
{
    if(d.nf == 0 || d.ne == 0)
        return;
    hipLaunchKernelGGL(k_edge_tri, dim3(grid_for(d.nf, 64)), dim3(64), 0, s, d.nf,
                       (const uint3*)d.faces, (const uint2*)d.edges, d.btype, d.x, tree_of(bf),
                       tree_of(be), hit);
    SG_LAUNCH_CHECK();
}

void launch_ground_intersect(const SimDev& d, int* hit, hipStream_t s)
{
    if(!d.use_ground || d.ns == 0)
        return;
    hipLaunchKernelGGL(k_ground_intersect, dim3(grid_for(d.ns, 256)), dim3(256), 0, s, d.gcount,
                       d.gp, d.x, d.gn, d.goff, hit);
    SG_LAUNCH_CHECK();
}

}  // namespace sgipc
