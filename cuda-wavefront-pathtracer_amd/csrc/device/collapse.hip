// device/collapse.hip - H-PLOC nodes -> compressed BVH8 on the device (see collapse.h).
#include "device/collapse.h"
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>

namespace cwp {

namespace {

constexpr int kPMax = 3;                 // primitives per wide leaf (the collapse's pMax)
constexpr float kCNode = 1.f, kCPrim = 0.3f;
constexpr unsigned char kDecLeaf = 0, kDecNode = 1, kDecPrev = 2, kDecDist = 10;
constexpr float kInf = 3e38f;
constexpr int kWaitVmcnt0 = 0x0F70;      // s_waitcnt vmcnt(0)

// The wide levels 0 .. kTopLevels - 1 (at most 8^l nodes each), and every level of a tree of at most kOneBlock primitives, run
// in one workgroup: a launch per level, three with the numbering, costs more than such a level's work. Whole collapse of n
// random boxes, ms: kTopLevels 2 / 4 / 6 at n = 12,000 0.358 / 0.395 / 0.437, 100,000 0.421 / 0.465 / 1.44, 500,000 0.571 / 0.618
// / 3.84 (level 2 has up to 64 nodes, 8 waves' work, but level 3 up to 512). One workgroup / launches: 1,000 primitives 0.220 /
// 0.281, 8,192 0.320 / 0.366, 12,000 0.369 / 0.380, 20,000 0.453 / 0.393.
constexpr int kTopLevels = 2, kOneBlock = 8192;

// scratch arrays carved out of one allocation (binary nodes: N = 2n - 1; wide nodes: at most n)
struct Scratch {
    int* parent; int* flag;                             // per binary node: parent; 256 x parent count + climb arrivals
    float* cost;                                        // per internal node, 8 floats: primitives (int bits), cost as 1..7 wide roots
    unsigned char* dec;                                 // per binary node, 8 bytes: [0] split of 8 roots, [1..7] decisions
    int* wBin; int* wSlot; int* wChild; int* wNInt; int* wLp; int* wT; int* wTP; int* wS; int* wP; int* wIdx;
    unsigned char* wLeaf;
    int* ctl;                                           // [0] error, [1] levels run by the one-workgroup launch
    int* lv; int* num;                                  // per level: first wide node, wide nodes
};

__device__ __forceinline__ Vec3 boxLo(const Vec4* hn, int h) { return xyz(hn[2 * h]); }
__device__ __forceinline__ Vec3 boxHi(const Vec4* hn, int h) { return xyz(hn[2 * h + 1]); }
__device__ __forceinline__ int leftOf(const Vec4* hn, int h) { return asInt(hn[2 * h].w); }
__device__ __forceinline__ int rightOf(const Vec4* hn, int h) { return asInt(hn[2 * h + 1].w); }
// AABB::area of the host: 0 for an empty box, else 2 (dx dy + dy dz + dz dx)
__device__ __forceinline__ float areaOf(Vec3 lo, Vec3 hi) {
    if (hi.x < lo.x) return 0.f;
    const Vec3 d = hi - lo;
    return 2.f * (d.x * d.y + d.y * d.z + d.z * d.x);
}

// --------------------------------------------------------------------------------------------------- checks
__global__ void k_cb_check(const Vec4* __restrict__ hn, int n, Scratch W) {
    const int N = 2 * n - 1;
    for (int h = blockIdx.x * blockDim.x + threadIdx.x; h < N; h += gridDim.x * blockDim.x) {
        const int l = leftOf(hn, h), r = rightOf(hn, h);
        if (h < n) {
            if (l < 0 || l >= n || r != -1) atomicOr(&W.ctl[0], 1);
        } else if (l < 0 || r < 0 || l >= h || r >= h) {
            atomicOr(&W.ctl[0], 2);
        } else {
            W.parent[l] = h; W.parent[r] = h;
            atomicAdd(&W.flag[l], 256); atomicAdd(&W.flag[r], 256);
        }
    }
}
__global__ void k_cb_check2(int n, Scratch W) {
    const int N = 2 * n - 1;
    for (int h = blockIdx.x * blockDim.x + threadIdx.x; h < N; h += gridDim.x * blockDim.x)
        if (W.flag[h] != (h == N - 1 ? 0 : 256)) atomicOr(&W.ctl[0], 4);
}

// --------------------------------------------------------------------------------------------------- cost tables
// Costs and decisions cross waves through device-coherent accesses (relaxed device-scope atomics), ordered by a
// vmcnt(0) wait before each arrival counter, as in the H-PLOC climb.
__device__ __forceinline__ void st2(float* p, float a, float b) {
    __hip_atomic_store((uint64_t*)p, (uint64_t)__float_as_uint(a) | ((uint64_t)__float_as_uint(b) << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ld2(const float* p, float& a, float& b) {
    const uint64_t v = __hip_atomic_load((const uint64_t*)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    a = __uint_as_float((uint32_t)v); b = __uint_as_float((uint32_t)(v >> 32));
}
// the table of binary node h: its primitives and its costs as 1..7 roots. A leaf's follows from its box (it costs
// A count cPrim at every width), so leaves store none.
__device__ __forceinline__ int costTable(const Vec4* hn, int n, const float* cost, int h, float c[8]) {
    if (h < n) {
        const float cl = areaOf(boxLo(hn, h), boxHi(hn, h)) * (float)1 * kCPrim;
        for (int i = 1; i < 8; i++) c[i] = cl;
        return 1;
    }
    const float* t = cost + 8 * (size_t)(h - n);
    float p;
    ld2(t, p, c[1]); ld2(t + 2, c[2], c[3]); ld2(t + 4, c[4], c[5]); ld2(t + 6, c[6], c[7]);
    return __float_as_int(p);
}
__device__ __forceinline__ void stD(unsigned char* p, const unsigned char d[8]) {
    const uint64_t v = (uint64_t)d[0] | ((uint64_t)d[1] << 8) | ((uint64_t)d[2] << 16) | ((uint64_t)d[3] << 24) |
                       ((uint64_t)d[4] << 32) | ((uint64_t)d[5] << 40) | ((uint64_t)d[6] << 48) | ((uint64_t)d[7] << 56);
    __hip_atomic_store((uint64_t*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One lane per leaf climbs to the root; the second lane to arrive at a node computes its table from both children
// (collapseCWBVH's bottom-up pass: leaves cost A count cPrim at every width; an internal node's cost as i roots is
// the best split of i roots between its children, or the cost as fewer roots; as 1 root it is the better of a leaf
// (at most pMax primitives) and an internal wide node over the best split of 8 roots). A table is one 32-byte record of
// four 64-bit coherent accesses, and leaves have none: with 4-byte accesses and leaf tables 2.02 M primitives took 721 us.
__global__ void __launch_bounds__(256) k_cb_dp(const Vec4* __restrict__ hn, int n, Scratch W) {
    const int h0 = blockIdx.x * blockDim.x + threadIdx.x;
    if (h0 >= n || W.ctl[0]) return;   // not a tree: the parents cannot be followed
    const int root = 2 * n - 2;
    int cur = h0;
    while (cur != root) {
        const int par = W.parent[cur];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);   // this lane's tables performed before the arrival
        if ((atomicAdd(&W.flag[par], 1) & 255) == 0) break;   // first to arrive: the sibling's lane computes the parent
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        float cl[8], cr[8];
        const int p = costTable(hn, n, W.cost, leftOf(hn, par), cl) + costTable(hn, n, W.cost, rightOf(hn, par), cr);
        const float A = areaOf(boxLo(hn, par), boxHi(hn, par));
        float dist[9]; int dk[9];
        for (int j = 2; j <= 8; j++) {
            dist[j] = kInf; dk[j] = 1;
            for (int k = 1; k < j; k++) { const float v = cl[k] + cr[j - k]; if (v < dist[j]) { dist[j] = v; dk[j] = k; } }
        }
        const float cLeaf = p <= kPMax ? A * (float)p * kCPrim : kInf;
        const float cInt = dist[8] + A * kCNode;
        float c[8];
        unsigned char d[8];
        if (cLeaf <= cInt) { c[1] = cLeaf; d[1] = kDecLeaf; } else { c[1] = cInt; d[1] = kDecNode; }
        d[0] = (unsigned char)dk[8];
        for (int i = 2; i < 8; i++) {
            if (dist[i] < c[i - 1]) { c[i] = dist[i]; d[i] = (unsigned char)(kDecDist + dk[i]); }
            else { c[i] = c[i - 1]; d[i] = kDecPrev; }
        }
        float* t = W.cost + 8 * (size_t)(par - n);
        st2(t, __int_as_float(p), c[1]); st2(t + 2, c[2], c[3]); st2(t + 4, c[4], c[5]); st2(t + 6, c[6], c[7]);
        stD(W.dec + 8 * (size_t)(par - n), d);
        cur = par;
    }
}

// --------------------------------------------------------------------------------------------------- wide nodes
__device__ __forceinline__ uint64_t decOf(const Scratch& W, int n, int h) { return *(const uint64_t*)(W.dec + 8 * (size_t)(h - n)); }
__device__ __forceinline__ int decAt(uint64_t d, int i) { return (int)((d >> (8 * i)) & 255u); }
// the roots node h contributes where its table is asked for i: i, or fewer where fewer cost as much; d: its decisions
__device__ __forceinline__ int rootsOf(const Scratch& W, int n, int h, int i, uint64_t& d) {
    if (h < n) return 1;
    d = decOf(W, n, h);
    while (i > 1 && decAt(d, i) == kDecPrev) i--;
    return i;
}
// the j-th binary root of the wide node over binary node b (left to right, the host's recursion order), -1: fewer roots
__device__ __forceinline__ int wideRoot(const Vec4* hn, int n, const Scratch& W, int b, int j) {
    uint64_t d = decOf(W, n, b);
    const int k8 = decAt(d, 0);
    int nd = leftOf(hn, b), i = rootsOf(W, n, nd, k8, d);
    if (j >= i) {
        j -= i;
        nd = rightOf(hn, b);
        i = rootsOf(W, n, nd, 8 - k8, d);
        if (j >= i) return -1;
    }
    while (i > 1) {   // d: the split of nd's i roots
        const int k = decAt(d, i) - kDecDist, r = rightOf(hn, nd), rest = i - k;
        nd = leftOf(hn, nd);
        i = rootsOf(W, n, nd, k, d);
        if (j >= i) { j -= i; nd = r; i = rootsOf(W, n, nd, rest, d); }
    }
    return nd;
}

// The wide nodes [start, end) of level l, eight lanes each: lane j of a node finds the node's j-th child (decision
// root) and holds its costs for the eight slots; greedy octant slot assignment (repeatedly the (child, free slot)
// pair of lowest -dot(child centre - node centre, slot direction), the lowest child and slot among equals), leaf flags,
// and the next level's records appended after this level's (one atomic per wave). The root is a single leaf when its
// table chose a leaf (at most pMax primitives) or n == 1. A lane per node held the 8 x 8 costs and the recursion in
// scratch memory: 1.2 ms for the twelve levels of 2.02 M primitives.
__device__ __forceinline__ void cbLevel(const Vec4* __restrict__ hn, int n, int l, int start, int end, int wave, int waves, int cap,
                                        const Scratch& W) {
    const int lane = (int)(threadIdx.x & 63u), j = lane & 7, g = lane >> 3;
    for (int X0 = start + wave * 8; X0 < end; X0 += waves * 8) {   // wave-uniform bound
        const int X = X0 + g;
        const bool on = X < end;
        const int b = on ? W.wBin[X] : 2 * n - 2;
        const bool asLeaf = X == 0 && (n == 1 || decAt(decOf(W, n, 2 * n - 2), 1) == kDecLeaf);
        int ch = -1;
        if (on) ch = asLeaf ? (j == 0 ? b : -1) : wideRoot(hn, n, W, b, j);
        float cost[8];
        for (int s = 0; s < 8; s++) cost[s] = kInf;
        if (ch >= 0) {
            const Vec3 pc = (boxLo(hn, b) + boxHi(hn, b)) * 0.5f;
            const Vec3 cc = (boxLo(hn, ch) + boxHi(hn, ch)) * 0.5f - pc;
            for (int s = 0; s < 8; s++)
                cost[s] = -(cc.x * (s & 1 ? -1.f : 1.f) + cc.y * (s & 2 ? -1.f : 1.f) + cc.z * (s & 4 ? -1.f : 1.f));
        }
        int slot = -1;
        unsigned taken = 0;   // per node: slots given away
        for (int it = 0; it < 8; it++) {
            float v = kInf;
            int at = -1;
            if (ch >= 0 && slot < 0)
                for (int s = 0; s < 8; s++)
                    if (!((taken >> s) & 1u) && cost[s] < v) { v = cost[s]; at = s; }
            float bv = v;   // the node's lowest cost and the first lane that holds it
            int who = at >= 0 ? j : 8;
            for (int o = 1; o < 8; o <<= 1) {
                const float ov = __shfl_xor(bv, o, 8);
                const int ow = __shfl_xor(who, o, 8);
                if (ow < 8 && (who == 8 || ov < bv || (ov == bv && ow < who))) { bv = ov; who = ow; }
            }
            const unsigned wait = (unsigned)(__ballot(ch >= 0 && slot < 0) >> (8 * g)) & 255u;
            if (who == 8) {   // costs that compare with nothing (NaN, beyond the range): the first child, the first slot
                who = wait ? __builtin_ctz(wait) : 8;
                at = __builtin_ctz(~taken);
            }
            at = __shfl(at, who & 7, 8);
            if (wait) {
                if (j == who) slot = at;
                taken |= 1u << at;
            }
        }
        const bool lf = ch >= 0 && (asLeaf || ch < n || decAt(decOf(W, n, ch), 1) == kDecLeaf);
        const bool inner = ch >= 0 && !lf;
        unsigned leaf = lf ? 1u << slot : 0u, mid = inner ? 1u << slot : 0u;
        int lp = lf ? (ch < n ? 1 : __float_as_int(W.cost[8 * (size_t)(ch - n)])) : 0;
        for (int o = 1; o < 8; o <<= 1) { leaf |= __shfl_xor(leaf, o, 8); mid |= __shfl_xor(mid, o, 8); lp += __shfl_xor(lp, o, 8); }
        const uint64_t mm = __ballot(inner);
        const int total = (int)__builtin_popcountll(mm);
        int first = 0;
        if (total) {
            if (lane == 0) first = atomicAdd(&W.num[l + 1], total);
            first = end + __builtin_amdgcn_readfirstlane(first);
            if (first + total > cap) { if (lane == 0) atomicOr(&W.ctl[0], 8); return; }
        }
        if (on) {
            if (ch >= 0) W.wSlot[8 * (size_t)X + slot] = ch;
            if (!((taken >> j) & 1u)) W.wSlot[8 * (size_t)X + j] = -1;
            if (j == 0) { W.wLeaf[X] = (unsigned char)leaf; W.wNInt[X] = (int)__builtin_popcount(mid); W.wLp[X] = lp; }
            if (inner) {
                const int ord = (int)__builtin_popcount(mid & ((1u << slot) - 1u));
                const int to = first + (int)__builtin_popcountll(mm & ((1ull << (8 * g)) - 1ull)) + ord;
                W.wBin[to] = ch;
                W.wChild[8 * (size_t)X + ord] = to;
            }
        }
    }
}

// subtree totals of internal children and leaf primitives, one level at a time from the deepest
__device__ __forceinline__ void cbTotals(int X, const Scratch& W) {
    int t = W.wNInt[X], tp = W.wLp[X];
    for (int j = 0; j < W.wNInt[X]; j++) { const int c = W.wChild[8 * (size_t)X + j]; t += W.wT[c]; tp += W.wTP[c]; }
    W.wT[X] = t; W.wTP[X] = tp;
}
// the host's numbering, one level at a time from the root: its stack pops a node, appends the node's internal
// children (child base) and leaf primitives (triangle base), pushes the internal children in slot order and so visits
// them in decreasing slot order
__device__ __forceinline__ void cbOffsets(int X, const Scratch& W) {
    const int m = W.wNInt[X];
    int s = W.wS[X] + m, p = W.wP[X] + W.wLp[X];
    for (int j = m - 1; j >= 0; j--) {   // later slots are visited first
        const int c = W.wChild[8 * (size_t)X + j];
        W.wS[c] = s; W.wP[c] = p;
        W.wIdx[c] = 1 + W.wS[X] + j;
        s += W.wT[c]; p += W.wTP[c];
    }
}
// Level l's range is on the device (the host waits for none): [lv[l], lv[l] + num[l]), where num[l] was counted by level
// l - 1. Levels the one-workgroup launch has run, and everything after an error, are skipped.
__global__ void __launch_bounds__(256) k_cb_level(const Vec4* __restrict__ hn, int n, int l, int cap, Scratch W) {
    if (W.ctl[0] || l < W.ctl[1]) return;
    const int start = W.lv[l], end = min(start + W.num[l], cap);
    if (blockIdx.x == 0 && threadIdx.x == 0) { W.lv[l + 1] = end; W.num[l + 2] = 0; }
    cbLevel(hn, n, l, start, end, (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6), (int)(gridDim.x * (blockDim.x >> 6)), cap, W);
}
// the numbering waits until every level has run: after an error, or while level `levels` (the first one not launched; 0:
// the one-workgroup launch ran them all) holds nodes, there is none
__device__ __forceinline__ bool cbUnfinished(int levels, const Scratch& W) { return W.ctl[0] || (levels > 0 && W.num[levels] != 0); }
__global__ void __launch_bounds__(256) k_cb_totals(int l, int levels, Scratch W) {
    if (cbUnfinished(levels, W) || l < W.ctl[1]) return;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < W.num[l]; k += gridDim.x * blockDim.x) cbTotals(W.lv[l] + k, W);
}
__global__ void __launch_bounds__(256) k_cb_offsets(int l, int levels, Scratch W) {
    if (cbUnfinished(levels, W) || l < W.ctl[1]) return;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < W.num[l]; k += gridDim.x * blockDim.x) cbOffsets(W.lv[l] + k, W);
}
// the first levels in one workgroup: up to `most`, or fewer when the tree ends (down: the levels; up: totals, then offsets)
constexpr int kTopBlock = 1024;
__global__ void __launch_bounds__(kTopBlock) k_cb_top_down(const Vec4* __restrict__ hn, int n, int most, int cap, Scratch W) {
    if (W.ctl[0]) return;
    int start = 0, end = 1, l = 0;
    if (threadIdx.x == 0) {
        W.wBin[0] = 2 * n - 2; W.wS[0] = 0; W.wP[0] = 0; W.wIdx[0] = 0;
        W.lv[0] = 0; W.num[0] = 1; W.num[1] = 0;
    }
    __syncthreads();
    for (; l < most && end > start; l++) {
        if (threadIdx.x == 0) { W.lv[l + 1] = end; W.num[l + 2] = 0; }
        __threadfence_block();
        __syncthreads();
        cbLevel(hn, n, l, start, end, (int)(threadIdx.x >> 6), kTopBlock / 64, cap, W);
        __threadfence_block();
        __syncthreads();
        const int next = __hip_atomic_load(&W.num[l + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        start = end; end = min(end + next, cap);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        W.ctl[1] = l;
        if (end == start)   // the tree has ended: the levels after it are empty for whoever asks
            for (int m = l + 1; m <= kTopLevels + 1; m++) { W.lv[m] = end; W.num[m] = 0; }
    }
}
__global__ void __launch_bounds__(kTopBlock) k_cb_top_up(int levels0, Scratch W) {
    if (cbUnfinished(levels0, W)) return;
    const int levels = W.ctl[1];
    for (int l = levels - 1; l >= 0; l--) {
        for (int k = threadIdx.x; k < W.num[l]; k += kTopBlock) cbTotals(W.lv[l] + k, W);
        __threadfence_block();
        __syncthreads();
    }
    for (int l = 0; l < levels; l++) {
        for (int k = threadIdx.x; k < W.num[l]; k += kTopBlock) cbOffsets(W.lv[l] + k, W);
        __threadfence_block();
        __syncthreads();
    }
}

__device__ int quantExpD(float ext, float lo, float hi) {
    if (!(ext > 0.f)) return -100;
    int e = (int)ceilf((float)log2((double)(ext / 255.f)));   // the correctly rounded single-precision log2
    if (e < -100) e = -100;
    while (lo + 255.f * ldexpf(1.f, e) < hi) e++;
    return e;
}
__device__ int quantD(float v, float o, float sc, bool up) {
    const float f = (v - o) / sc;
    const int i = up ? (int)ceilf(f) : (int)floorf(f);
    return i < 0 ? 0 : (i > 255 ? 255 : i);
}
__device__ uint32_t pack4D(const int* q, int b) {
    return (uint32_t)q[b] | ((uint32_t)q[b + 1] << 8) | ((uint32_t)q[b + 2] << 16) | ((uint32_t)q[b + 3] << 24);
}

// the 80-byte node of wide node X and its leaves' primitives; levels: the levels launched
__global__ void __launch_bounds__(256) k_cb_emit(const Vec4* __restrict__ hn, int n, int levels, Scratch W, Vec4* out, int* prim) {
    const int X = blockIdx.x * blockDim.x + threadIdx.x;
    if (cbUnfinished(levels, W)) return;
    const int last = max(levels, W.ctl[1]), total = W.lv[last];   // every wide node precedes the first empty level
    if (X >= total) return;
    const int b = W.wBin[X];
    const Vec3 lo = boxLo(hn, b), hi = boxHi(hn, b);
    const Vec3 ext = hi - lo;
    const int ex = quantExpD(ext.x, lo.x, hi.x), ey = quantExpD(ext.y, lo.y, hi.y), ez = quantExpD(ext.z, lo.z, hi.z);
    const float sx = ldexpf(1.f, ex), sy = ldexpf(1.f, ey), sz = ldexpf(1.f, ez);
    int qlox[8], qloy[8], qloz[8], qhix[8], qhiy[8], qhiz[8], meta[8];
    const int triBase = W.wP[X], childBase = 1 + W.wS[X];
    const unsigned leaf = W.wLeaf[X];
    unsigned imask = 0;
    int off = 0;
    for (int s = 0; s < 8; s++) {
        qlox[s] = qloy[s] = qloz[s] = qhix[s] = qhiy[s] = qhiz[s] = 0; meta[s] = 0;
        const int cn = W.wSlot[8 * (size_t)X + s];
        if (cn < 0) continue;
        const Vec3 cl = boxLo(hn, cn), chh = boxHi(hn, cn);
        qlox[s] = quantD(cl.x, lo.x, sx, false); qhix[s] = quantD(chh.x, lo.x, sx, true);
        qloy[s] = quantD(cl.y, lo.y, sy, false); qhiy[s] = quantD(chh.y, lo.y, sy, true);
        qloz[s] = quantD(cl.z, lo.z, sz, false); qhiz[s] = quantD(chh.z, lo.z, sz, true);
        if ((leaf >> s) & 1u) {   // the binary subtree's primitives, left to right
            int st[8], sp = 0, cnt = 0;
            st[sp++] = cn;
            while (sp > 0) {   // at most pMax leaves: the stack never holds more than pMax + 1 entries
                const int h = st[--sp];
                if (h < n) { if (triBase + off + cnt < n) prim[triBase + off + cnt] = leftOf(hn, h); cnt++; }
                else if (sp < 7) { st[sp++] = rightOf(hn, h); st[sp++] = leftOf(hn, h); }
            }
            meta[s] = 0x80 | ((cnt - 1) << 5) | off;
            off += cnt;
        } else { meta[s] = 0x40; imask |= 1u << s; }
    }
    const uint32_t ew = (uint32_t)(ex + 127) | ((uint32_t)(ey + 127) << 8) | ((uint32_t)(ez + 127) << 16) | (imask << 24);
    if (W.wIdx[X] >= total) return;   // the numbering covers [0, total) exactly
    Vec4* o = out + 5 * (size_t)W.wIdx[X];
    o[0] = v4(lo.x, lo.y, lo.z, asFloatU(ew));
    o[1] = v4(asFloat(childBase), asFloat(triBase), asFloatU(pack4D(meta, 0)), asFloatU(pack4D(meta, 4)));
    const uint32_t u[12] = { pack4D(qlox, 0), pack4D(qlox, 4), pack4D(qloy, 0), pack4D(qloy, 4), pack4D(qloz, 0), pack4D(qloz, 4),
                             pack4D(qhix, 0), pack4D(qhix, 4), pack4D(qhiy, 0), pack4D(qhiy, 4), pack4D(qhiz, 0), pack4D(qhiz, 4) };
    for (int j = 0; j < 3; j++) o[2 + j] = v4(asFloatU(u[4 * j]), asFloatU(u[4 * j + 1]), asFloatU(u[4 * j + 2]), asFloatU(u[4 * j + 3]));
}

#define CCHK(x)                                                                                                        \
    do {                                                                                                               \
        hipError_t e_ = (x);                                                                                           \
        if (e_ != hipSuccess) { err = std::string(#x) + ": " + hipGetErrorString(e_); return false; }                  \
    } while (0)

float hostArea(Vec3 lo, Vec3 hi) {
    if (hi.x < lo.x) return 0.f;
    const Vec3 d = hi - lo;
    return 2.f * (d.x * d.y + d.y * d.z + d.z * d.x);
}

constexpr int kFirstLevels = 16;   // levels queued before the host looks at the counts
constexpr size_t kLevelPad = 64;   // level records past the deepest possible level: the first levels of a small tree
Scratch carve(void* mem, int n) {
    const size_t N = 2 * (size_t)n - 1, M = (size_t)n;
    char* p = (char*)mem;
    auto take = [&](size_t bytes) { char* q = p; p += (bytes + 255) & ~(size_t)255; return (void*)q; };
    Scratch W;
    W.ctl = (int*)take(64);
    W.parent = (int*)take(N * 4); W.flag = (int*)take(N * 4);
    W.cost = (float*)take(M * 32); W.dec = (unsigned char*)take(M * 8);
    W.wBin = (int*)take(M * 4); W.wSlot = (int*)take(M * 32); W.wChild = (int*)take(M * 32); W.wNInt = (int*)take(M * 4);
    W.wLp = (int*)take(M * 4); W.wT = (int*)take(M * 4); W.wTP = (int*)take(M * 4); W.wS = (int*)take(M * 4);
    W.wP = (int*)take(M * 4); W.wIdx = (int*)take(M * 4); W.wLeaf = (unsigned char*)take(M);
    W.lv = (int*)take((M + kLevelPad) * 4); W.num = (int*)take((M + kLevelPad) * 4);
    return W;
}
size_t scratchBytes(int n) {
    const size_t N = 2 * (size_t)n - 1, M = (size_t)n;
    auto r = [](size_t b) { return (b + 255) & ~(size_t)255; };
    return r(64) + 2 * r(N * 4) + r(M * 32) + r(M * 8) + 2 * r(M * 32) + 8 * r(M * 4) + r(M) + 2 * r((M + kLevelPad) * 4) + 256;
}

}  // namespace

CwbvhCollapser::~CwbvhCollapser() { release(); }

void CwbvhCollapser::release() {
    if (mem_) hipFree(mem_);
    mem_ = nullptr; cap_ = 0; bytes_ = 0;
}

bool CwbvhCollapser::reserve(int n, std::string& err) {
    if (n <= cap_) return true;
    release();
    bytes_ = scratchBytes(n);
    CCHK(hipMalloc(&mem_, bytes_));
    cap_ = n;
    return true;
}

bool CwbvhCollapser::run(const Vec4* hn, int n, Vec4* nodesOut, int* primOut, void* stream, int& numNodes, int& depth,
                         std::string& err) {
    if (n < 1 || !hn || !nodesOut || !primOut) { err = "CWBVH collapse: bad arguments"; return false; }
    if (n > (1 << 28)) { err = "CWBVH collapse: too many primitives"; return false; }
    if (!reserve(n, err)) return false;
    hipStream_t st = (hipStream_t)stream;
    const Scratch W = carve(mem_, n);
    const int N = 2 * n - 1;
    CCHK(hipMemsetAsync(W.ctl, 0, 64, st));
    CCHK(hipMemsetAsync(W.flag, 0, (size_t)N * 4, st));
    const int gN = std::min((N + 255) / 256, 4096);
    k_cb_check<<<gN, 256, 0, st>>>(hn, n, W);
    k_cb_check2<<<gN, 256, 0, st>>>(n, W);
    if (n > 1) k_cb_dp<<<(n + 255) / 256, 256, 0, st>>>(hn, n, W);
    // As many levels as an ordinary tree has (2.02 M primitives: 12; an empty level costs 3 us) are queued with the
    // numbering behind them, so the host waits once before it knows the tree's end. A deeper tree's numbering kernels do
    // nothing then: batches of level launches follow, each as long as all before it (at most 1,024), with a look at the counts
    // after each, and the numbering is queued once more when the last level is known. So a tree of L levels takes 3 L
    // launches (with the numbering behind every 16 levels they were L^2 / 16): chains of 9,000 / 20,000 primitives (1,286 /
    // 2,857 levels) 407 / 1,918 -> 46 / 86 ms, of 400,000 1.6 s.
    const bool one = n <= kOneBlock;
    const int top = one ? kOneBlock : kTopLevels;
    auto grid = [&](int l, int perNode) {   // level l holds at most 8^l nodes
        const long long nodes = l < 8 ? std::min<long long>(1ll << (3 * l), n) : n;
        return (int)std::max<long long>(1, std::min<long long>((nodes * perNode + 255) / 256, 2048));
    };
    int levels = one ? 0 : kFirstLevels;   // levels launched
    struct { int ctl[2]; } head = {};
    int lastNum = 0;
    auto number = [&]() {
        for (int l = levels - 1; l >= kTopLevels; l--) k_cb_totals<<<grid(l, 1), 256, 0, st>>>(l, levels, W);
        k_cb_top_up<<<1, kTopBlock, 0, st>>>(levels, W);
        for (int l = kTopLevels; l < levels; l++) k_cb_offsets<<<grid(l, 1), 256, 0, st>>>(l, levels, W);
        k_cb_emit<<<(n + 255) / 256, 256, 0, st>>>(hn, n, levels, W, nodesOut, primOut);
    };
    k_cb_top_down<<<1, kTopBlock, 0, st>>>(hn, n, top, n, W);
    for (int l = kTopLevels; l < levels; l++) k_cb_level<<<grid(l, 8), 256, 0, st>>>(hn, n, l, n, W);
    number();
    for (bool again = false;; again = true) {
        CCHK(hipMemcpyAsync(&head, W.ctl, sizeof head, hipMemcpyDeviceToHost, st));
        if (!one) CCHK(hipMemcpyAsync(&lastNum, W.num + levels, 4, hipMemcpyDeviceToHost, st));
        CCHK(hipStreamSynchronize(st));
        if (head.ctl[0] & 7) { err = "CWBVH collapse: the H-PLOC nodes are not a tree over [0, n) (code " + std::to_string(head.ctl[0]) + ")"; return false; }
        if (head.ctl[0]) { err = "CWBVH collapse: more wide nodes than primitives (code " + std::to_string(head.ctl[0]) + ")"; return false; }
        if (one || lastNum == 0) { if (again) number(); break; }
        if (levels >= n) { err = "CWBVH collapse: wide tree deeper than its primitive count"; return false; }
        // up to the last level such a tree can have, n - 1 (the level records reach kLevelPad beyond it)
        for (int k = std::min(std::min(levels, 1024), n - levels); k > 0; k--, levels++)
            k_cb_level<<<grid(levels, 8), 256, 0, st>>>(hn, n, levels, n, W);
    }
    // the non-empty levels (a prefix), their end
    const int run = std::max(levels, head.ctl[1]);
    std::vector<int> num(run + 1), lv(run + 1);
    CCHK(hipMemcpyAsync(num.data(), W.num, num.size() * 4, hipMemcpyDeviceToHost, st));
    CCHK(hipMemcpyAsync(lv.data(), W.lv, lv.size() * 4, hipMemcpyDeviceToHost, st));
    unsigned char rootDec[2] = { 0, 0 };
    if (n > 1) {
        CCHK(hipMemcpyAsync(rootDec, W.dec + 8 * (size_t)(n - 2), 2, hipMemcpyDeviceToHost, st));
        CCHK(hipMemcpyAsync(&rootCost_, W.cost + 8 * (size_t)(n - 2) + 1, 4, hipMemcpyDeviceToHost, st));
    }
    CCHK(hipStreamSynchronize(st));
    CCHK(hipGetLastError());
    rootLeaf_ = n == 1 || rootDec[1] == kDecLeaf;
    depth = 0;
    while (depth < run && num[depth] > 0) depth++;
    numNodes = lv[run];
    return true;
}

bool cwbvhFromHplocHost(const Vec4* hnodes, int n, std::vector<Vec4>& nodes, std::vector<int>& prim, int& depth,
                        double& gpuMs, float& sah, std::string& err) {
    if (n < 1) { err = "CWBVH collapse: no primitives"; return false; }
    const size_t N = 2 * (size_t)n - 1;
    Vec4 *dH = nullptr, *dN = nullptr;
    int* dP = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    CwbvhCollapser C;
    bool ok = false;
    do {
        if (hipMalloc(&dH, N * 2 * sizeof(Vec4)) != hipSuccess || hipMalloc(&dN, (size_t)n * 5 * sizeof(Vec4)) != hipSuccess ||
            hipMalloc(&dP, (size_t)n * 4) != hipSuccess) { err = "CWBVH collapse: out of device memory"; break; }
        if (hipMemcpy(dH, hnodes, N * 2 * sizeof(Vec4), hipMemcpyHostToDevice) != hipSuccess) { err = "CWBVH collapse: upload failed"; break; }
        if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) { err = "CWBVH collapse: events"; break; }
        int nn = 0;
        if (!C.run(dH, n, dN, dP, nullptr, nn, depth, err)) break;   // first run: loads the kernels (not timed)
        hipEventRecord(e0, nullptr);
        if (!C.run(dH, n, dN, dP, nullptr, nn, depth, err)) break;
        hipEventRecord(e1, nullptr);
        if (hipEventSynchronize(e1) != hipSuccess) { err = "CWBVH collapse failed"; break; }
        float ms = 0;
        hipEventElapsedTime(&ms, e0, e1);
        gpuMs = ms;
        {   // the host collapse's SAH: the root's cost (an internal wide root; or a leaf root plus one node) over its area
            const Vec4 rl = hnodes[2 * (2 * (size_t)n - 2)], rh = hnodes[2 * (2 * (size_t)n - 2) + 1];
            const float Ar = hostArea(xyz(rl), xyz(rh));
            const bool leafRoot = n == 1 || C.rootIsLeaf();
            sah = Ar > 0 ? (leafRoot ? (Ar * (float)n * kCPrim + Ar * kCNode) / Ar : C.rootCost() / Ar) : 0.f;
        }
        nodes.resize((size_t)nn * 5); prim.resize((size_t)n);
        if (hipMemcpy(nodes.data(), dN, nodes.size() * sizeof(Vec4), hipMemcpyDeviceToHost) != hipSuccess ||
            hipMemcpy(prim.data(), dP, prim.size() * 4, hipMemcpyDeviceToHost) != hipSuccess) { err = "CWBVH collapse: download failed"; break; }
        ok = true;
    } while (false);
    if (e0) hipEventDestroy(e0);
    if (e1) hipEventDestroy(e1);
    if (dH) hipFree(dH);
    if (dN) hipFree(dN);
    if (dP) hipFree(dP);
    return ok;
}

}  // namespace cwp
