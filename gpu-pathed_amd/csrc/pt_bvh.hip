// pt_bvh.hip -- GPU BVH builder for gfx950.
//
// 1. 63-bit Morton codes of primitive centroids (21 bits per axis) + primitive AABBs
// 2. stable LSD radix sort of (code, index), 8 passes of 8 bits; ranking inside a tile with
//    wave64 ballots (one 64-bit mask per key bit)
// 3. a binary tree over the sorted primitives, one of
//    - LBVH: Karras 2012 binary radix tree (one thread per internal node; equal codes ordered
//      by index), then a bottom-up AABB refit (atomic arrival counter per node; the second
//      child to arrive merges);
//    - PLOC (Meister & Bittner 2018, parallel locally-ordered clustering): every cluster of the
//      Morton-ordered list finds the neighbour within PLOC_RADIUS positions whose merged box
//      has the least surface area; mutual nearest neighbours merge; the list is compacted with
//      a prefix sum; repeat until one cluster is left.  The primitives are then put in the
//      tree's depth-first leaf order so every subtree covers a contiguous range.
// 4. collapse into a 4-wide BVH of 128-byte nodes, on the GPU: subtrees of <= PT_LEAF_MAX
//    primitives become leaf ranges of the primitive array, and which internal nodes become
//    4-wide nodes is chosen to minimise a surface-area cost (bottom-up dynamic programme over
//    the binary tree with arrival counters; then the nodes are written level by level from
//    the root, the live children of a node at consecutive indices).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "pt_gpu.h"

namespace pt {

namespace {

constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortThreads * kSortItems;

__device__ __forceinline__ uint64_t spread21(uint32_t v) {
    uint64_t x = v & 0x1fffffULL;
    x = (x | x << 32) & 0x1f00000000ffffULL;
    x = (x | x << 16) & 0x1f0000ff0000ffULL;
    x = (x | x << 8) & 0x100f00f00f00f00fULL;
    x = (x | x << 4) & 0x10c30c30c30c30c3ULL;
    x = (x | x << 2) & 0x1249249249249249ULL;
    return x;
}

struct Box {
    float lo[3], hi[3];
};

__device__ __forceinline__ Box primBox(const float4 *prims, int i) {
    const float4 a = prims[3 * i], b = prims[3 * i + 1], c = prims[3 * i + 2];
    Box bx;
    if (asInt(b.w) == PT_TAG_SPHERE) {
        const float r = b.x;
        bx.lo[0] = a.x - r; bx.lo[1] = a.y - r; bx.lo[2] = a.z - r;
        bx.hi[0] = a.x + r; bx.hi[1] = a.y + r; bx.hi[2] = a.z + r;
    } else {
        bx.lo[0] = fminf(a.x, fminf(b.x, c.x)); bx.hi[0] = fmaxf(a.x, fmaxf(b.x, c.x));
        bx.lo[1] = fminf(a.y, fminf(b.y, c.y)); bx.hi[1] = fmaxf(a.y, fmaxf(b.y, c.y));
        bx.lo[2] = fminf(a.z, fminf(b.z, c.z)); bx.hi[2] = fmaxf(a.z, fmaxf(b.z, c.z));
    }
    // widen by a few ulps so rounding in the slab test cannot cull a watertight hit
    for (int k = 0; k < 3; k++) {
        const float e = fmaxf(fabsf(bx.lo[k]), fabsf(bx.hi[k])) * 2.0e-6f + 1.0e-30f;
        bx.lo[k] -= e;
        bx.hi[k] += e;
    }
    return bx;
}

__global__ void k_morton(const float4 *prims, int n, float3 lo, float3 ext, uint64_t *keys, uint32_t *vals, float *boxes) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const Box b = primBox(prims, i);
    float c[3];
    const float e[3] = {ext.x, ext.y, ext.z}, l[3] = {lo.x, lo.y, lo.z};
    uint64_t key = 0;
    for (int k = 0; k < 3; k++) {
        c[k] = 0.5f * (b.lo[k] + b.hi[k]);
        float u = e[k] > 0.f ? (c[k] - l[k]) / e[k] : 0.5f;
        u = fminf(fmaxf(u, 0.f), 1.f);
        const uint32_t q = min((uint32_t)(u * 2097152.0f), 2097151u);
        key |= spread21(q) << (2 - k);
    }
    keys[i] = key;
    vals[i] = (uint32_t)i;
    for (int k = 0; k < 3; k++) {
        boxes[6 * i + k] = b.lo[k];
        boxes[6 * i + 3 + k] = b.hi[k];
    }
}

// --- radix sort -----------------------------------------------------------------------
__global__ __launch_bounds__(kSortThreads) void k_sort_hist(const uint64_t *keys, int n, int shift, int numTiles, uint32_t *hist) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int base = blockIdx.x * kSortTile;
    for (int it = 0; it < kSortItems; it++) {
        const int idx = base + it * kSortThreads + threadIdx.x;
        if (idx < n) atomicAdd(&h[(keys[idx] >> shift) & 255], 1u);
    }
    __syncthreads();
    hist[threadIdx.x * numTiles + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(kSortThreads) void k_sort_scatter(const uint64_t *keysIn, const uint32_t *valsIn, uint64_t *keysOut, uint32_t *valsOut,
                                                               const uint32_t *offsets, int n, int shift, int numTiles) {
    __shared__ uint32_t running[256];
    __shared__ uint32_t base[256];
    __shared__ uint32_t waveCnt[4][256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    base[tid] = offsets[tid * numTiles + blockIdx.x];
    running[tid] = 0;
    const uint64_t ltMask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int it = 0; it < kSortItems; it++) {
        for (int w = 0; w < 4; w++) waveCnt[w][tid] = 0;
        __syncthreads();
        const int idx = blockIdx.x * kSortTile + it * kSortThreads + tid;
        const bool valid = idx < n;
        const uint64_t key = valid ? keysIn[idx] : 0ull;
        const uint32_t val = valid ? valsIn[idx] : 0u;
        const uint32_t digit = (uint32_t)(key >> shift) & 255u;
        uint64_t m = __ballot(valid);
        for (int b = 0; b < 8; b++) {
            const bool bit = (digit >> b) & 1u;
            const uint64_t bb = __ballot(bit);
            m &= bit ? bb : ~bb;
        }
        const uint32_t rank = (uint32_t)__popcll(m & ltMask);
        if (valid && rank == 0) waveCnt[wave][digit] = (uint32_t)__popcll(m);
        __syncthreads();
        if (valid) {
            uint32_t pre = running[digit];
            for (int w = 0; w < wave; w++) pre += waveCnt[w][digit];
            const uint32_t pos = base[digit] + pre + rank;
            keysOut[pos] = key;
            valsOut[pos] = val;
        }
        __syncthreads();
        running[tid] += waveCnt[0][tid] + waveCnt[1][tid] + waveCnt[2][tid] + waveCnt[3][tid];
        __syncthreads();
    }
}

// The whole sort by one block for up to kSortTile keys: a key's place is the number of keys that
// come before it, counted over the keys in LDS (2048 keys: 4M comparisons, about as long as two
// of the 24 launches of the radix passes).
constexpr int kSortSmallThreads = 1024;
__global__ __launch_bounds__(kSortSmallThreads) void k_sort_small(const uint64_t *keysIn, const uint32_t *valsIn, uint64_t *keysOut, uint32_t *valsOut,
                                                                  int n) {
    __shared__ uint64_t k[kSortTile];
    for (int i = threadIdx.x; i < n; i += kSortSmallThreads) k[i] = keysIn[i];
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kSortSmallThreads) {
        const uint64_t key = k[i];
        int pos = 0;
        for (int j = 0; j < n; j++) pos += k[j] < key || (k[j] == key && j < i) ? 1 : 0;
        keysOut[pos] = key;
        valsOut[pos] = valsIn[i];
    }
}

__global__ void k_gather(const float4 *prims, const float *boxes, const uint32_t *order, int n, float4 *primsOut, float *boxesOut) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t s = order[i];
    primsOut[3 * i] = prims[3 * s];
    primsOut[3 * i + 1] = prims[3 * s + 1];
    primsOut[3 * i + 2] = prims[3 * s + 2];
    for (int k = 0; k < 6; k++) boxesOut[6 * i + k] = boxes[6 * s + k];
}

// --- Karras 2012 hierarchy --------------------------------------------------------------
__device__ __forceinline__ int delta(const uint64_t *keys, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    const uint64_t a = keys[i], b = keys[j];
    if (a == b) return 64 + __clz((uint32_t)(i ^ j));
    return __clzll(a ^ b);
}

// child encoding during the build: >= 0 internal node, < 0 leaf ~primitive
__global__ void k_karras(const uint64_t *keys, int n, int2 *children, int *cnt, int *firstLeaf, int *parentNode, int *parentLeaf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(keys, n, i, i - d);
    int lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = delta(keys, n, i, j);
    int s = 0;
    int t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int gamma = i + s * d + min(d, 0);
    const int first = min(i, j), last = max(i, j);
    int left, right;
    if (first == gamma) {
        left = ~gamma;
        parentLeaf[gamma] = i;
    } else {
        left = gamma;
        parentNode[gamma] = i;
    }
    if (last == gamma + 1) {
        right = ~(gamma + 1);
        parentLeaf[gamma + 1] = i;
    } else {
        right = gamma + 1;
        parentNode[gamma + 1] = i;
    }
    children[i] = make_int2(left, right);
    cnt[i] = last - first + 1;
    firstLeaf[i] = first;
    if (i == 0) parentNode[0] = -1;
}

// All primitives in one leaf below a single 4-wide root (n <= PT_LEAF_MAX).
__global__ void k_write_single(const float *leafBoxes, int n, float4 *nodes) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    float lo[3] = {1e30f, 1e30f, 1e30f}, hi[3] = {-1e30f, -1e30f, -1e30f};
    for (int i = 0; i < n; i++)
        for (int k = 0; k < 3; k++) {
            lo[k] = fminf(lo[k], leafBoxes[6 * i + k]);
            hi[k] = fmaxf(hi[k], leafBoxes[6 * i + 3 + k]);
        }
    for (int k = 0; k < 3; k++) {
        nodes[2 * k] = make_float4(lo[k], 1e30f, 1e30f, 1e30f);
        nodes[2 * k + 1] = make_float4(hi[k], -1e30f, -1e30f, -1e30f);
    }
    nodes[6] = make_float4(asFloat(~(((n - 1) << PT_LEAF_COUNT_SHIFT) | 0)), asFloat(PT_EMPTY_CHILD), asFloat(PT_EMPTY_CHILD),
                           asFloat(PT_EMPTY_CHILD));
    nodes[7] = make_float4(0.f, 0.f, 0.f, 0.f);
}

__global__ void k_fill_int(int *p, int n, int v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

inline int blocks(int64_t n, int t) { return (int)((n + t - 1) / t); }

// --- prefix sums ------------------------------------------------------------------------
// Exclusive scan of m values in place, the total written to data[m]: tiles of kScanTile values
// scanned in LDS (one per block), the tile totals scanned by one block, then added back.
constexpr int kScanThreads = 256;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;

template <class T> __device__ T blockExclusiveScan(T v, T *sh, T *total) {
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int off = 1; off < kScanThreads; off <<= 1) {
        const T x = t >= off ? sh[t - off] : (T)0;
        __syncthreads();
        sh[t] += x;
        __syncthreads();
    }
    const T incl = sh[t];
    *total = sh[kScanThreads - 1];
    __syncthreads();
    return incl - v;
}

template <class T> __global__ __launch_bounds__(kScanThreads) void k_scan_tiles(T *data, int m, T *tileSums, const int *mDev) {
    __shared__ T sh[kScanThreads];
    if (mDev) m = *mDev;
    const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    T v[kScanItems];
    T sum = 0;
    for (int k = 0; k < kScanItems; k++) {
        v[k] = base + k < m ? data[base + k] : (T)0;
        sum += v[k];
    }
    T total;
    T run = blockExclusiveScan<T>(sum, sh, &total);
    for (int k = 0; k < kScanItems; k++) {
        if (base + k < m) data[base + k] = run;
        run += v[k];
    }
    if (threadIdx.x == 0) tileSums[blockIdx.x] = total;
}

// one block: exclusive scan of the tile totals (any count), total to tileSums[tiles]
template <class T> __global__ __launch_bounds__(kScanThreads) void k_scan_totals(T *tileSums, int tiles) {
    __shared__ T sh[kScanThreads];
    T carry = 0;
    for (int b0 = 0; b0 < tiles; b0 += kScanThreads) {
        const int i = b0 + threadIdx.x;
        const T v = i < tiles ? tileSums[i] : (T)0;
        T total;
        const T ex = blockExclusiveScan<T>(v, sh, &total);
        if (i < tiles) tileSums[i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) tileSums[tiles] = carry;
}

template <class T> __global__ void k_scan_add(T *data, int m, const T *tileSums, int tiles, const int *mDev) {
    if (mDev) m = *mDev;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) data[i] += tileSums[i / kScanTile];
    if (i == 0) data[m] = tileSums[tiles];
}

// The same by one block, for counts that a block's few passes cover sooner than three launches.
constexpr int kScanSmall = 8 * kScanTile;
template <class T> __global__ __launch_bounds__(kScanThreads) void k_scan_small(T *data, int m, const int *mDev) {
    __shared__ T sh[kScanThreads];
    if (mDev) m = *mDev;
    T carry = 0;
    for (int b0 = 0; b0 < m; b0 += kScanTile) {
        const int base = b0 + threadIdx.x * kScanItems;
        T v[kScanItems], sum = 0, total;
        for (int k = 0; k < kScanItems; k++) {
            v[k] = base + k < m ? data[base + k] : (T)0;
            sum += v[k];
        }
        T run = carry + blockExclusiveScan<T>(sum, sh, &total);
        for (int k = 0; k < kScanItems; k++) {
            if (base + k < m) data[base + k] = run;
            run += v[k];
        }
        carry += total;
    }
    if (threadIdx.x == 0) data[m] = carry;
}

// data holds m + 1 entries; tmp at least tiles(m) + 1.  mDev: the count is on the device, at
// most m.
template <class T> void exclusiveScan(T *data, int m, T *tmp, hipStream_t stream, const int *mDev = nullptr) {
    if (m <= kScanSmall) {
        k_scan_small<T><<<1, kScanThreads, 0, stream>>>(data, m, mDev);
    } else {
        const int tiles = std::max(1, (m + kScanTile - 1) / kScanTile);
        k_scan_tiles<T><<<tiles, kScanThreads, 0, stream>>>(data, m, tmp, mDev);
        k_scan_totals<T><<<1, kScanThreads, 0, stream>>>(tmp, tiles);
        k_scan_add<T><<<std::max(1, (m + 255) / 256), 256, 0, stream>>>(data, m, tmp, tiles, mDev);
    }
    PT_HIP_TRY(hipGetLastError());
}
inline int scanTmpEntries(int m) { return (m + kScanTile - 1) / kScanTile + 2; }

// --- binary tree shared by both builders --------------------------------------------------
// children: >= 0 internal node, < 0 ~leaf (leaf = position in the Morton order); cnt and
// first: primitives below an internal node and the position of the first in the final
// primitive order; leafPos: final position of a leaf and posLeaf its inverse (nullptr: the
// Morton position).
struct BinTree {
    int n = 0, root = 0;
    const int2 *children = nullptr;
    const float *nodeBoxes = nullptr, *leafBoxes = nullptr;
    const int *cnt = nullptr, *first = nullptr, *leafPos = nullptr, *posLeaf = nullptr;
    const int *parentNode = nullptr, *parentLeaf = nullptr;
};

__device__ __forceinline__ int childCount(const BinTree &t, int c) { return c < 0 ? 1 : t.cnt[c]; }

__device__ __forceinline__ float boxArea6(const float *b) {
    const float dx = b[3] - b[0], dy = b[4] - b[1], dz = b[5] - b[2];
    return dx * dy + dy * dz + dz * dx;
}

// --- PLOC --------------------------------------------------------------------------------
constexpr int PLOC_RADIUS = 16;
constexpr int kPlocThreads = 256;

__global__ void k_ploc_init(int n, const float *leafBoxes, int *clusters, float *cbox) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    clusters[i] = ~i;
    for (int k = 0; k < 6; k++) cbox[6 * i + k] = leafBoxes[6 * i + k];
}

// Nearest neighbour of every cluster among the PLOC_RADIUS positions on either side: least
// surface area of the merged box, ties to the lower position.
__global__ __launch_bounds__(kPlocThreads) void k_ploc_nn(const float *cbox, int m, int *nn) {
    __shared__ float sb[(kPlocThreads + 2 * PLOC_RADIUS) * 6];
    const int start = blockIdx.x * kPlocThreads;
    for (int k = threadIdx.x; k < (kPlocThreads + 2 * PLOC_RADIUS) * 6; k += kPlocThreads) {
        const int pos = start - PLOC_RADIUS + k / 6;
        sb[k] = pos >= 0 && pos < m ? cbox[(int64_t)pos * 6 + k % 6] : 0.f;
    }
    __syncthreads();
    const int i = start + threadIdx.x;
    if (i >= m) return;
    const float *bi = &sb[(threadIdx.x + PLOC_RADIUS) * 6];
    float best = INFINITY;
    int bj = i;
    const int j0 = max(0, i - PLOC_RADIUS), j1 = min(m - 1, i + PLOC_RADIUS);
    for (int j = j0; j <= j1; j++) {
        if (j == i) continue;
        const float *bj6 = &sb[(j - start + PLOC_RADIUS) * 6];
        float u[6];
        for (int k = 0; k < 3; k++) {
            u[k] = fminf(bi[k], bj6[k]);
            u[3 + k] = fmaxf(bi[3 + k], bj6[3 + k]);
        }
        const float d = boxArea6(u);
        if (d < best) {
            best = d;
            bj = j;
        }
    }
    nn[i] = bj;
}

// Merge pairs (2k, 2k + 1): the fallback for an iteration in which no two clusters chose each
// other (never observed; it keeps the loop finite).
__global__ void k_ploc_pairs(int m, int *nn) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int j = i ^ 1;
    nn[i] = j < m ? j : i;
}

// keep flag (low 32 bits) and new-node flag (high 32 bits) per cluster position
__global__ void k_ploc_flags(const int *nn, int m, unsigned long long *flags) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int j = nn[i];
    const bool mutual = j != i && nn[j] == i;
    const unsigned long long keep = mutual && i > j ? 0ull : 1ull;
    const unsigned long long leader = mutual && i < j ? 1ull : 0ull;
    flags[i] = keep | leader << 32;
}

__global__ void k_ploc_merge(const int *clusters, const float *cbox, const int *nn, int m, const unsigned long long *pre, int nodeBase,
                             int *clustersOut, float *cboxOut, int2 *children, float *nodeBoxes, int *cnt, int *parentNode, int *parentLeaf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int j = nn[i];
    const bool mutual = j != i && nn[j] == i;
    if (mutual && i > j) return;
    const int pos = (int)(pre[i] & 0xffffffffull);
    const float *a = &cbox[6 * (size_t)i];
    if (!mutual) {
        clustersOut[pos] = clusters[i];
        for (int k = 0; k < 6; k++) cboxOut[6 * (size_t)pos + k] = a[k];
        return;
    }
    const int id = nodeBase + (int)(pre[i] >> 32);
    const int l = clusters[i], r = clusters[j];
    const float *b = &cbox[6 * (size_t)j];
    float u[6];
    for (int k = 0; k < 3; k++) {
        u[k] = fminf(a[k], b[k]);
        u[3 + k] = fmaxf(a[3 + k], b[3 + k]);
    }
    children[id] = make_int2(l, r);
    for (int k = 0; k < 6; k++) {
        nodeBoxes[6 * (size_t)id + k] = u[k];
        cboxOut[6 * (size_t)pos + k] = u[k];
    }
    cnt[id] = (l < 0 ? 1 : cnt[l]) + (r < 0 ? 1 : cnt[r]);
    if (l < 0) parentLeaf[~l] = id; else parentNode[l] = id;
    if (r < 0) parentLeaf[~r] = id; else parentNode[r] = id;
    clustersOut[pos] = id;
}

// depth-first leaf order: a leaf's position is the number of leaves in the left subtrees its
// root path passes
__global__ void k_leaf_positions(BinTree t, int *leafPos) {
    const int leaf = blockIdx.x * blockDim.x + threadIdx.x;
    if (leaf >= t.n) return;
    int off = 0, cur = ~leaf, p = t.parentLeaf[leaf];
    // a root path has fewer than n nodes; the step bound only guards against a malformed tree
    for (int steps = 0; p >= 0 && steps < t.n; steps++) {
        const int2 c = t.children[p];
        if (c.y == cur) off += childCount(t, c.x);
        cur = p;
        p = t.parentNode[p];
    }
    leafPos[leaf] = off;
}

// first position of every internal node: written by its leftmost leaf
__global__ void k_node_first(BinTree t, int *first) {
    const int leaf = blockIdx.x * blockDim.x + threadIdx.x;
    if (leaf >= t.n) return;
    const int o = t.leafPos[leaf];
    int cur = ~leaf, p = t.parentLeaf[leaf];
    for (int steps = 0; p >= 0 && t.children[p].x == cur && steps < t.n; steps++) {
        first[p] = o;
        cur = p;
        p = t.parentNode[p];
    }
}

__global__ void k_scatter_prims(const float4 *in, const int *leafPos, int n, float4 *out, int *posLeaf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int o = leafPos[i];
    posLeaf[o] = i;
    out[3 * (size_t)o] = in[3 * (size_t)i];
    out[3 * (size_t)o + 1] = in[3 * (size_t)i + 1];
    out[3 * (size_t)o + 2] = in[3 * (size_t)i + 2];
}

// --- 4-wide collapse -----------------------------------------------------------------------
// A 4-wide node costs kNodeCost x its area, a leaf kPrimCost x its area x its primitives.
// Bottom up, every live internal node (more than PT_LEAF_MAX primitives) gets the cheapest way
// to spend 1..3 child slots of its parent on its subtree: one slot is the node itself as a
// 4-wide node (W), two or three spread its subtree over its children (S2, S3), opening it.
constexpr float kNodeCost = 1.0f;
constexpr float kPrimCost = 0.6f;

struct CollapseTables {
    float *W, *S2, *S3;
    unsigned char *split;   // 3 per node: slots of the left child when the children share 2..4
    unsigned char *opened;  // bit k: spreading over k + 2 slots opens the node
};

__device__ __forceinline__ bool liveChild(const BinTree &t, int c) { return c >= 0 && t.cnt[c] > PT_LEAF_MAX; }
__device__ __forceinline__ const float *boxOf(const BinTree &t, int c) {
    return c >= 0 ? &t.nodeBoxes[6 * (size_t)c] : &t.leafBoxes[6 * (size_t)(~c)];
}

// --- bottom-up pass over the binary tree -----------------------------------------------------
// Every internal node once both its children are done: its box (LBVH; PLOC has them already),
// its collapse costs and its height.  One thread per leaf climbs towards the root; the second
// arrival at a node computes it.
//
// What a step costs is making a child's results visible to whichever thread comes second: between
// workgroups that takes agent-scope fences (each XCD has its own L2), which at two per leaf and
// node was all of the pass's time (1.31M leaves: 7.4 ms for the boxes and 7.9 ms more for the
// costs; 2.5 ms with only the subtrees that span 1024-leaf tiles done that way).  So no node is
// shared between workgroups: a workgroup does the subtrees that lie wholly inside its kClimbTile
// consecutive leaf positions and notes the nodes it leaves its tile at, the next launch's
// workgroups carry on from those in tiles kClimbFan times as long, until one tile holds the
// tree (1.31M leaves: three launches).
//
// Then it is the chain of dependent loads per level that counts.  In global memory it was parent,
// its range, arrival, children, their results, 3 us a level (295 + 157 + 162 us); a node's place is
// now loaded while its child is computed, the first launch's results, nine in ten, meet in LDS, and
// a climb keeps the child that it comes from (81 + 111 us).
constexpr int kClimbTile = 1024;
constexpr int kClimbFan = 64;

struct ClimbArgs {
    BinTree t;
    CollapseTables tb;
    float *nodeBoxes;   // BOXES: written here (t.nodeBoxes)
    int *height;        // internal nodes on the longest path from the node down, itself included
    int *arrivals;      // per internal node, 0 on entry
    // nodes outside their tile that a tile's subtrees have arrived at: from the tile's first
    // position on, their number per tile; of this launch and of the one before
    int *left[2], *leftCount[2];
};

// What a parent needs of a child: a leaf, or an internal node that has been computed.
struct Subtree {
    float box[6];
    float W, S2, S3;
    int cnt, height;   // leaves, and internal nodes on the longest path down
    __device__ __forceinline__ float cost(int slots, float leafCost) const {
        return cnt <= PT_LEAF_MAX ? leafCost : slots == 1 ? W : slots == 2 ? S2 : S3;
    }
};

// Internal node p from its children x and y; its results go to the global tables, and back.
template <bool BOXES> __device__ __forceinline__ Subtree climbNode(const ClimbArgs &a, int p, int cnt, const Subtree &x, const Subtree &y) {
    Subtree r;
    for (int k = 0; k < 3; k++) {
        r.box[k] = fminf(x.box[k], y.box[k]);
        r.box[3 + k] = fmaxf(x.box[3 + k], y.box[3 + k]);
    }
    if constexpr (BOXES)
        for (int k = 0; k < 6; k++) a.nodeBoxes[6 * (size_t)p + k] = r.box[k];
    r.cnt = cnt;
    r.height = 1 + max(x.height, y.height);
    a.height[p] = r.height;
    r.W = r.S2 = r.S3 = 0.f;
    if (cnt <= PT_LEAF_MAX) return r;
    const float lx = kPrimCost * boxArea6(x.box) * (float)x.cnt, ly = kPrimCost * boxArea6(y.box) * (float)y.cnt;
    float share[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j = 2; j <= 4; j++) {
        float best = INFINITY;
        int bi = 1;
        for (int i = 1; i < j; i++) {
            const float v = x.cost(min(i, 3), lx) + y.cost(min(j - i, 3), ly);
            if (v < best) {
                best = v;
                bi = i;
            }
        }
        share[j] = best;
        a.tb.split[3 * (size_t)p + (j - 2)] = (unsigned char)bi;
    }
    r.W = kNodeCost * boxArea6(r.box) + share[4];
    r.S2 = fminf(r.W, share[2]);
    r.S3 = fminf(r.W, share[3]);
    a.tb.W[p] = r.W;
    a.tb.S2[p] = r.S2;
    a.tb.S3[p] = r.S3;
    a.tb.opened[p] = (unsigned char)((share[2] < r.W ? 1 : 0) | (share[3] < r.W ? 2 : 0));
    return r;
}

// A node's place in the tree.  A climb loads its next node's while it waits for the present one.
struct Place {
    int first, cnt, parent;
    int2 children;
};
__device__ __forceinline__ Place placeOf(const BinTree &t, int p) {
    if (p < 0) return Place{0, 0, -1, make_int2(0, 0)};
    return Place{t.first[p], t.cnt[p], t.parentNode[p], t.children[p]};
}

__device__ __forceinline__ Subtree leafSubtree(const ClimbArgs &a, int leaf) {
    Subtree s;
    for (int k = 0; k < 6; k++) s.box[k] = a.t.leafBoxes[6 * (size_t)leaf + k];
    s.W = s.S2 = s.S3 = 0.f;
    s.cnt = 1;
    s.height = 0;
    return s;
}
__device__ __forceinline__ Subtree globalSubtree(const ClimbArgs &a, int c) {
    if (c < 0) return leafSubtree(a, ~c);
    Subtree s;
    for (int k = 0; k < 6; k++) s.box[k] = a.nodeBoxes[6 * (size_t)c + k];
    s.W = a.tb.W[c];
    s.S2 = a.tb.S2[c];
    s.S3 = a.tb.S3[c];
    s.cnt = a.t.cnt[c];
    s.height = a.height[c];
    return s;
}

// The first launch over an LBVH, whose node numbers are positions of their subtrees' ends: a tile's
// nodes meet in LDS, and the global tables are only written, without a wait.
__global__ __launch_bounds__(kClimbTile) void k_climb_tiles(ClimbArgs a) {
    __shared__ float box[6][kClimbTile], cost[3][kClimbTile];
    __shared__ int cnt[kClimbTile], height[kClimbTile], arrivals[kClimbTile];
    __shared__ int out;
    if (threadIdx.x == 0) out = 0;
    arrivals[threadIdx.x] = 0;
    __syncthreads();
    const int begin = (int)(blockIdx.x * kClimbTile), end = min(begin + kClimbTile, a.t.n);
    const int pos = begin + (int)threadIdx.x;
    if (pos < end) {
        int p = a.t.parentLeaf[pos], from = ~pos;
        Subtree s = leafSubtree(a, pos);
        Place at = placeOf(a.t, p);
        // a node inside the tile has all its leaves there, so its two arrivals are of this workgroup
        while (p >= 0 && at.first >= begin && at.first + at.cnt <= end) {
            if (from >= 0) {
                const int k = from - begin;
                for (int j = 0; j < 6; j++) box[j][k] = s.box[j];
                cost[0][k] = s.W;
                cost[1][k] = s.S2;
                cost[2][k] = s.S3;
                cnt[k] = s.cnt;
                height[k] = s.height;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
            if (__hip_atomic_fetch_add(&arrivals[p - begin], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0) {
                p = -1;
                break;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            const Place next = placeOf(a.t, at.parent);
            const bool left = at.children.x == from;
            const int c = left ? at.children.y : at.children.x;
            Subtree o;
            if (c < 0) {
                o = leafSubtree(a, ~c);
            } else {
                const int k = c - begin;
                for (int j = 0; j < 6; j++) o.box[j] = box[j][k];
                o.W = cost[0][k];
                o.S2 = cost[1][k];
                o.S3 = cost[2][k];
                o.cnt = cnt[k];
                o.height = height[k];
            }
            s = left ? climbNode<true>(a, p, at.cnt, s, o) : climbNode<true>(a, p, at.cnt, o, s);
            from = p;
            p = at.parent;
            at = next;
        }
        if (p >= 0) a.left[1][begin + atomicAdd(&out, 1)] = p;
    }
    __syncthreads();
    if (threadIdx.x == 0) a.leftCount[1][blockIdx.x] = out;
}

// One launch of the pass over tiles of `tile` leaf positions; in: the parity of the launch before,
// whose tiles were `sub` long (0: the first launch, from the leaves).
template <bool BOXES> __global__ __launch_bounds__(kClimbTile) void k_climb(ClimbArgs a, int tile, int sub, int in) {
    __shared__ int out;
    if (threadIdx.x == 0) out = 0;
    __syncthreads();
    const int64_t begin64 = (int64_t)blockIdx.x * tile;
    const int begin = (int)begin64, end = (int)min(begin64 + tile, (int64_t)a.t.n);
    auto climb = [&](int p) {
        Place at = placeOf(a.t, p);
        while (p >= 0 && at.first >= begin && at.first + at.cnt <= end) {
            __threadfence_block();
            if (__hip_atomic_fetch_add(&a.arrivals[p], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0) return;
            __threadfence_block();
            const Place next = placeOf(a.t, at.parent);
            climbNode<BOXES>(a, p, at.cnt, globalSubtree(a, at.children.x), globalSubtree(a, at.children.y));
            p = at.parent;
            at = next;
        }
        // a tile of n positions is left at most n times: every time for another subtree
        if (p >= 0) a.left[1 - in][begin + atomicAdd(&out, 1)] = p;
    };
    if (sub == 0) {
        const int pos = begin + (int)threadIdx.x;
        if (pos < end) climb(a.t.parentLeaf[a.t.posLeaf ? a.t.posLeaf[pos] : pos]);
    } else {
        constexpr int kPer = kClimbTile / kClimbFan;
        const int s = (int)threadIdx.x / kPer;
        const int64_t from = begin64 + (int64_t)s * sub;
        if (from < end) {
            const int n = a.leftCount[in][blockIdx.x * kClimbFan + s];
            for (int k = (int)threadIdx.x % kPer; k < n; k += kPer) climb(a.left[in][from + k]);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) a.leftCount[1 - in][blockIdx.x] = out;
}

template <bool BOXES> void climbTree(const ClimbArgs &a, hipStream_t stream) {
    int in = 0;
    int64_t sub = 0;
    for (int64_t tile = kClimbTile;; tile *= kClimbFan) {
        const int len = (int)std::min<int64_t>(tile, INT32_MAX);
        if (BOXES && sub == 0) k_climb_tiles<<<blocks(a.t.n, len), kClimbTile, 0, stream>>>(a);
        else k_climb<BOXES><<<blocks(a.t.n, len), kClimbTile, 0, stream>>>(a, len, (int)sub, in);
        PT_HIP_TRY(hipGetLastError());
        if (tile >= a.t.n) return;
        sub = tile;
        in = 1 - in;
    }
}

// The children of the 4-wide node made from binary node x: its two children sharing four
// slots, opened where the cost tables say so, in left-to-right order.
__device__ int wideChildren(const BinTree &t, const CollapseTables &tb, int x, int *kids) {
    int stackNode[4], stackSlots[4], sp = 0, nk = 0;
    const int2 c = t.children[x];
    const int i4 = tb.split[3 * (size_t)x + 2];
    stackNode[sp] = c.y;
    stackSlots[sp++] = 4 - i4;
    stackNode[sp] = c.x;
    stackSlots[sp++] = i4;
    while (sp > 0) {
        sp--;
        const int y = stackNode[sp], s = stackSlots[sp];
        if (!liveChild(t, y) || s == 1 || !(tb.opened[y] & (1 << (s - 2)))) {
            kids[nk++] = y;
            continue;
        }
        const int i = tb.split[3 * (size_t)y + (s - 2)];
        const int2 cy = t.children[y];
        stackNode[sp] = cy.y;
        stackSlots[sp++] = s - i;
        stackNode[sp] = cy.x;
        stackSlots[sp++] = i;
    }
    return nk;
}

// A level of 4-wide nodes: how many, and the index of the first.
struct WideLevel {
    int m, base;
};

constexpr int kNoKid = INT32_MAX;

// The 4-wide node made from binary node x: its children and how many of them are live.
__device__ int4 wideNode(const BinTree &t, const CollapseTables &tb, int x, unsigned *live) {
    int kids[4];
    const int nk = wideChildren(t, tb, x, kids);
    unsigned c = 0;
    for (int k = 0; k < nk; k++) c += liveChild(t, kids[k]) ? 1u : 0u;
    *live = c;
    return make_int4(kids[0], kids[1], nk > 2 ? kids[2] : kNoKid, nk > 3 ? kids[3] : kNoKid);
}

__global__ void k_level_root(BinTree t, CollapseTables tb, int4 *frontier, unsigned *live, WideLevel *levels) {
    frontier[0] = wideNode(t, tb, t.root, &live[0]);
    levels[0] = WideLevel{1, 0};
}

// Writes a level's nodes, four lanes a node, one per child; rank: the exclusive sums of the
// nodes' live children.  A live child goes to the next level at its base + its rank; its lane
// works out its children (opening a child is a chain of dependent loads: a thread per node did
// up to four in a row).
__global__ __launch_bounds__(256) void k_level_write(BinTree t, CollapseTables tb, const int4 *frontier, WideLevel *levels, const unsigned *rank,
                                                     int4 *next, unsigned *nextLive, float4 *nodes) {
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) >> 2, k = threadIdx.x & 3;
    const WideLevel lv = levels[0];
    if (i == 0 && k == 0) levels[1] = WideLevel{lv.m > 0 ? (int)rank[lv.m] : 0, lv.base + lv.m};
    if (i >= lv.m) return;
    const int y = ((const int *)frontier)[4 * (size_t)i + k];
    const bool live = y != kNoKid && liveChild(t, y);
    const unsigned group = (unsigned)(__ballot(live) >> (threadIdx.x & 60)) & 15u;
    const int r = (int)rank[i] + __popc(group & ((1u << k) - 1u));
    float *o = (float *)&nodes[(size_t)PT_NODE_F4 * (lv.base + i)] + k;
    int ref = PT_EMPTY_CHILD;
    if (y == kNoKid) {
        // an inverted box: every slab test misses it
        for (int a = 0; a < 3; a++) {
            o[8 * a] = 1e30f;
            o[8 * a + 4] = -1e30f;
        }
    } else {
        const float *b = boxOf(t, y);
        for (int a = 0; a < 3; a++) {
            o[8 * a] = b[a];
            o[8 * a + 4] = b[3 + a];
        }
        if (live) {
            ref = lv.base + lv.m + r;
            next[r] = wideNode(t, tb, y, &nextLive[r]);
        } else {
            const int cnt = childCount(t, y);
            const int first = y < 0 ? (t.leafPos ? t.leafPos[~y] : ~y) : t.first[y];
            ref = ~(((cnt - 1) << PT_LEAF_COUNT_SHIFT) | first);
        }
    }
    o[24] = asFloat(ref);
    o[28] = 0.f;
}

constexpr int kLevelGroup = 32;   // levels queued without a look at the last one's size, at most
// Working arrays of the collapse of a tree of ni internal nodes.
struct CollapseWork {
    unsigned *live[2], *scanTmp;
    int4 *front[2];
    WideLevel *levels;
    float4 *nodes;   // every 4-wide node stands for a distinct live internal node: at most ni of them
    void want(WorkArrays &w, int ni) {
        w.want(scanTmp, (size_t)scanTmpEntries(ni + 1));
        for (int k = 0; k < 2; k++) {
            w.want(live[k], (size_t)ni + 1);
            w.want(front[k], (size_t)ni);
        }
        w.want(levels, (size_t)ni + kLevelGroup + 1);   // a level has a node at least
        w.want(nodes, (size_t)PT_NODE_F4 * ni);
    }
};

// Collapses the binary tree into 4-wide nodes (root = node 0); returns the node count and the
// number of levels.  The levels' sizes stay on the device: a group of levels is queued with
// grids for the most nodes they can have, then the host looks whether the tree has ended (a
// wait per level took half of the collapse).
int collapseWide(const BinTree &t, const CollapseTables &tb, const CollapseWork &cw, DevBuf &nodes, hipStream_t stream, int *levels) {
    const int ni = t.n - 1;
    k_level_root<<<1, 1, 0, stream>>>(t, tb, cw.front[0], cw.live[0], cw.levels);
    // a full tree of n / 2 two-primitive leaves has this many levels; a group more where it is deeper
    int group = 1;
    for (int64_t w = 4; w * 2 < t.n; w *= 4) group++;
    group = std::min(group, kLevelGroup);
    int level = 0, cur = 0;
    int64_t most = 1;
    WideLevel lv{1, 0};
    while (lv.m > 0) {
        if (level > ni) throw HipFailure("BVH collapse: more levels than internal nodes");
        for (int k = 0; k < group; k++, level++) {
            exclusiveScan<unsigned>(cw.live[cur], (int)most, cw.scanTmp, stream, &cw.levels[level].m);
            k_level_write<<<blocks(4 * most, 256), 256, 0, stream>>>(t, tb, cw.front[cur], cw.levels + level, cw.live[cur], cw.front[1 - cur],
                                                                 cw.live[1 - cur], cw.nodes);
            PT_HIP_TRY(hipGetLastError());
            most = std::min<int64_t>(4 * most, ni);
            cur = 1 - cur;
        }
        PT_HIP_TRY(hipMemcpyAsync(&lv, cw.levels + level, sizeof lv, hipMemcpyDeviceToHost, stream));
        PT_HIP_TRY(hipStreamSynchronize(stream));
        most = lv.m;
        group = 4;
    }
    std::vector<WideLevel> all(level + 1);
    PT_HIP_TRY(hipMemcpyAsync(all.data(), cw.levels, sizeof(WideLevel) * all.size(), hipMemcpyDeviceToHost, stream));
    nodes.alloc(sizeof(float4) * PT_NODE_F4 * (size_t)lv.base);
    PT_HIP_TRY(hipMemcpyAsync(nodes.p, cw.nodes, sizeof(float4) * PT_NODE_F4 * (size_t)lv.base, hipMemcpyDeviceToDevice, stream));
    PT_HIP_TRY(hipStreamSynchronize(stream));
    *levels = 0;
    while (*levels < level && all[*levels].m > 0) ++*levels;
    return lv.base;
}

}  // namespace

size_t scanEntries(int m) { return (size_t)scanTmpEntries(m); }
void scanCounts(uint32_t *data, int m, uint32_t *tmp, hipStream_t stream) { exclusiveScan<uint32_t>(data, m, tmp, stream); }

int deviceCUs() {
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return 256;
    return prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
}

void buildBvh(const float4 *primsIn, int n, const float lo[3], const float hi[3], DevBuf &nodes, float4 *primsSorted, hipStream_t stream,
              BvhInfo *info, int builder) {
    info->numNodes = 0;
    info->depth = 0;
    info->binaryDepth = 0;
    if (n <= 0) return;
    const int numTiles = blocks(n, kSortTile), counters = 256 * numTiles;
    const int ni = std::max(1, n - 1);
    WorkArrays work;
    uint64_t *keys[2];
    uint32_t *vals[2], *hist, *histTmp;
    float *boxes, *boxes2, *nodeBoxes;
    int2 *children;
    int *cnt, *first, *parentNode, *parentLeaf, *leafPos = nullptr, *posLeaf = nullptr;
    ClimbArgs climb;
    CollapseWork cw;
    for (int k = 0; k < 2; k++) {
        work.want(keys[k], n);
        work.want(vals[k], n);
    }
    work.want(hist, (size_t)counters + 1);
    work.want(histTmp, (size_t)scanTmpEntries(counters));
    work.want(boxes, (size_t)6 * n);
    work.want(boxes2, (size_t)6 * n);
    work.want(nodeBoxes, (size_t)6 * ni);
    work.want(children, ni);
    work.want(cnt, ni);
    work.want(first, ni);
    work.want(parentNode, ni);
    work.want(parentLeaf, n);
    work.want(climb.tb.W, ni);
    work.want(climb.tb.S2, ni);
    work.want(climb.tb.S3, ni);
    work.want(climb.tb.split, (size_t)3 * ni);
    work.want(climb.tb.opened, ni);
    work.want(climb.height, ni);
    work.want(climb.arrivals, ni);
    for (int k = 0; k < 2; k++) {
        work.want(climb.left[k], n);
        work.want(climb.leftCount[k], (size_t)blocks(n, kClimbTile) + kClimbFan);
    }
    if (builder == PT_BVH_PLOC) {
        work.want(leafPos, n);
        work.want(posLeaf, n);
    }
    cw.want(work, ni);
    work.alloc();
    const float3 flo = make_float3(lo[0], lo[1], lo[2]);
    const float3 ext = make_float3(hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]);
    const bool small = n <= kSortTile;
    k_morton<<<blocks(n, 256), 256, 0, stream>>>(primsIn, n, flo, ext, keys[small], vals[small], boxes);
    PT_HIP_TRY(hipGetLastError());
    if (small) k_sort_small<<<1, kSortSmallThreads, 0, stream>>>(keys[1], vals[1], keys[0], vals[0], n);
    for (int pass = 0; pass < (small ? 0 : 8); pass++) {
        const int shift = pass * 8, in = pass & 1;
        k_sort_hist<<<numTiles, kSortThreads, 0, stream>>>(keys[in], n, shift, numTiles, hist);
        // one block scanned the 256 x tiles counters before: 290 us a pass at 1.31M primitives
        // against 11 us for the tiled scan
        exclusiveScan<uint32_t>(hist, counters, histTmp, stream);
        k_sort_scatter<<<numTiles, kSortThreads, 0, stream>>>(keys[in], vals[in], keys[1 - in], vals[1 - in], hist, n, shift, numTiles);
    }
    // the sorted data is in the first pair
    k_gather<<<blocks(n, 256), 256, 0, stream>>>(primsIn, boxes, vals[0], n, primsSorted, boxes2);
    PT_HIP_TRY(hipGetLastError());
    if (n <= PT_LEAF_MAX) {
        nodes.alloc(sizeof(float4) * PT_NODE_F4);
        k_write_single<<<1, 64, 0, stream>>>(boxes2, n, nodes.as<float4>());
        PT_HIP_TRY(hipGetLastError());
        PT_HIP_TRY(hipStreamSynchronize(stream));
        info->numNodes = 1;
        info->depth = 1;
        info->binaryDepth = n > 1 ? 1 : 0;
        return;
    }
    BinTree t;
    t.n = n;
    t.children = children;
    t.nodeBoxes = nodeBoxes;
    t.leafBoxes = boxes2;
    t.cnt = cnt;
    t.first = first;
    t.parentNode = parentNode;
    t.parentLeaf = parentLeaf;
    if (builder == PT_BVH_PLOC) {
        k_fill_int<<<blocks(ni, 256), 256, 0, stream>>>(parentNode, ni, -1);
        // clusters start as the Morton-ordered leaves; each iteration merges mutual nearest
        // neighbours, whose new nodes take the next indices in position order
        DevBuf clus[2], cbox[2], nn, flags, scanTmp, primsTmp;
        for (int k = 0; k < 2; k++) {
            clus[k].alloc(sizeof(int) * n);
            cbox[k].alloc(sizeof(float) * 6 * n);
        }
        nn.alloc(sizeof(int) * n);
        flags.alloc(sizeof(unsigned long long) * ((size_t)n + 1));
        scanTmp.alloc(sizeof(unsigned long long) * (size_t)scanTmpEntries(n + 1));
        k_ploc_init<<<blocks(n, 256), 256, 0, stream>>>(n, boxes2, clus[0].as<int>(), cbox[0].as<float>());
        int m = n, nodeBase = 0, cur = 0;
        while (m > 1) {
            k_ploc_nn<<<blocks(m, kPlocThreads), kPlocThreads, 0, stream>>>(cbox[cur].as<float>(), m, nn.as<int>());
            for (int attempt = 0; attempt < 2; attempt++) {
                if (attempt == 1) k_ploc_pairs<<<blocks(m, 256), 256, 0, stream>>>(m, nn.as<int>());
                k_ploc_flags<<<blocks(m, 256), 256, 0, stream>>>(nn.as<int>(), m, flags.as<unsigned long long>());
                exclusiveScan<unsigned long long>(flags.as<unsigned long long>(), m, scanTmp.as<unsigned long long>(), stream);
                unsigned long long tot = 0;
                PT_HIP_TRY(hipMemcpyAsync(&tot, flags.as<unsigned long long>() + m, sizeof tot, hipMemcpyDeviceToHost, stream));
                PT_HIP_TRY(hipStreamSynchronize(stream));
                const int merged = (int)(tot >> 32);
                if (merged == 0 && attempt == 0) continue;  // no mutual pair: merge neighbours pairwise
                if (merged == 0 || nodeBase + merged > ni) throw HipFailure("PLOC: clustering made no progress");
                k_ploc_merge<<<blocks(m, 256), 256, 0, stream>>>(clus[cur].as<int>(), cbox[cur].as<float>(), nn.as<int>(), m,
                                                                 flags.as<unsigned long long>(), nodeBase, clus[1 - cur].as<int>(),
                                                                 cbox[1 - cur].as<float>(), children, nodeBoxes,
                                                                 cnt, parentNode, parentLeaf);
                PT_HIP_TRY(hipGetLastError());
                nodeBase += merged;
                m = (int)(tot & 0xffffffffull);
                cur = 1 - cur;
                break;
            }
        }
        if (nodeBase != ni) throw HipFailure("PLOC: the tree does not have n - 1 internal nodes");
        t.root = ni - 1;  // the last merge
        // depth-first leaf order, then every internal node's first position
        k_leaf_positions<<<blocks(n, 256), 256, 0, stream>>>(t, leafPos);
        t.leafPos = leafPos;
        k_node_first<<<blocks(n, 256), 256, 0, stream>>>(t, first);
        primsTmp.alloc(sizeof(float4) * 3 * (size_t)n);
        PT_HIP_TRY(hipMemcpyAsync(primsTmp.p, primsSorted, sizeof(float4) * 3 * (size_t)n, hipMemcpyDeviceToDevice, stream));
        k_scatter_prims<<<blocks(n, 256), 256, 0, stream>>>(primsTmp.as<float4>(), leafPos, n, primsSorted, posLeaf);
        t.posLeaf = posLeaf;
        PT_HIP_TRY(hipGetLastError());
        PT_HIP_TRY(hipStreamSynchronize(stream));  // primsTmp is freed on leaving this block
    } else {
        k_karras<<<blocks(ni, 256), 256, 0, stream>>>(keys[0], n, children, cnt, first, parentNode, parentLeaf);
        PT_HIP_TRY(hipGetLastError());
        t.root = 0;
    }
    climb.t = t;
    climb.nodeBoxes = nodeBoxes;
    k_fill_int<<<blocks(ni, 256), 256, 0, stream>>>(climb.arrivals, ni, 0);
    if (builder == PT_BVH_PLOC) climbTree<false>(climb, stream);
    else climbTree<true>(climb, stream);
    int levels = 1, height = 0;
    PT_HIP_TRY(hipMemcpyAsync(&height, climb.height + t.root, sizeof height, hipMemcpyDeviceToHost, stream));
    const int count = collapseWide(t, climb.tb, cw, nodes, stream, &levels);
    // the working arrays are freed on return
    PT_HIP_TRY(hipStreamSynchronize(stream));
    info->numNodes = count;
    info->depth = levels;
    info->binaryDepth = height;
}

}  // namespace pt
