// GPU BVH construction, refit and linear blend skinning for gfx950.
//
// Replaces OptiX's acceleration-structure build and update
// (src/optix/optix_ray_tracer.cu:213-359 build, :443-463 update) and the
// skinning lambda of Scene::update_gscene (src/scene/scene.cu:336-395).
//
// Build (deterministic: every decision uses integers, an exact total-order
// min/max on floats, or float formulas evaluated in a fixed order, so the
// bytes are reproducible by a host execution of the same steps):
//   1. triangle boxes, box centroids, centroid bounds (two-level reduction)
//   2. 63-bit Morton codes of centroids, stable radix sort of (code, id)
//   3. Karras (HPG 2012) binary radix tree, index tie-break for equal codes
//   4. bottom-up pass by radix-tree depth (deepest first, nodes ordered by
//      depth, runs of small levels in one launch): boxes, primitive counts, SAH costs, collapse-to-leaf
//      decisions (leaves of <= max_leaf triangles)
//   5. frontier of the highest subtrees with <= T primitives ("clusters")
//   6. top of the tree rebuilt with a 16-bin SAH sweep over the clusters, by
//      levels, breadth-first node numbering at the end
//   7. emit 64-byte nodes (two child boxes per node) and the triangles in
//      Morton order (48 bytes each, primitive and mesh id in the w lanes)
// Refit keeps the topology and recomputes child boxes bottom-up by levels.
// Kernel boundaries (barriers in a run of small levels) order them: per-node device-scope fences
// (an L2 write-back and invalidate each on gfx950) made the arrival-counter
// form of these passes several times slower.
#include "srt_internal.h"
#include <hipcub/hipcub.hpp>
#include <cstdio>
#include <algorithm>

namespace srt {

// total order on floats (-0 < +0): key, inverse, min/max
SRT_D uint32_t fkey(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
SRT_D float fromkey(uint32_t k) { return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k); }
SRT_D float kmin(float a, float b) { return (fkey(b) < fkey(a)) ? b : a; }
SRT_D float kmax(float a, float b) { return (fkey(b) > fkey(a)) ? b : a; }

struct DBox { float lo[3], hi[3]; };
SRT_D DBox empty_box() {
    DBox b;
    for (int i = 0; i < 3; i++) { b.lo[i] = __builtin_huge_valf(); b.hi[i] = -__builtin_huge_valf(); }
    return b;
}
SRT_D void grow(DBox& b, const DBox& o) {
    for (int i = 0; i < 3; i++) { b.lo[i] = kmin(b.lo[i], o.lo[i]); b.hi[i] = kmax(b.hi[i], o.hi[i]); }
}
SRT_D float box_area(const DBox& b) {
    float dx = b.hi[0] - b.lo[0], dy = b.hi[1] - b.lo[1], dz = b.hi[2] - b.lo[2];
    if (!(dx >= 0.0f)) return 0.0f;
    return 2.0f * ((dx * dy + dy * dz) + dz * dx);
}

// SoA box storage
struct BoxArr { float *lox, *loy, *loz, *hix, *hiy, *hiz; };
SRT_D DBox ldbox(const BoxArr& a, size_t i) {
    DBox b;
    b.lo[0] = a.lox[i]; b.lo[1] = a.loy[i]; b.lo[2] = a.loz[i];
    b.hi[0] = a.hix[i]; b.hi[1] = a.hiy[i]; b.hi[2] = a.hiz[i];
    return b;
}
SRT_D void stbox(const BoxArr& a, size_t i, const DBox& b) {
    a.lox[i] = b.lo[0]; a.loy[i] = b.lo[1]; a.loz[i] = b.lo[2];
    a.hix[i] = b.hi[0]; a.hiy[i] = b.hi[1]; a.hiz[i] = b.hi[2];
}

// ---------------------------------------------------------------------------
// 1. triangle boxes + centroid bounds
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_tri_boxes(const float* pos, const uint32_t* idx, int n, BoxArr tb, float* cen,
                                                   uint32_t* partial) {
    __shared__ uint32_t red[6][256];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    DBox cb = empty_box();
    if (i < n) {
        DBox b = empty_box();
        for (int v = 0; v < 3; v++) {
            const float* p = pos + 3 * (size_t)idx[3 * (size_t)i + v];
            for (int a = 0; a < 3; a++) { b.lo[a] = kmin(b.lo[a], p[a]); b.hi[a] = kmax(b.hi[a], p[a]); }
        }
        stbox(tb, i, b);
        for (int a = 0; a < 3; a++) {
            float c = (b.lo[a] + b.hi[a]) * 0.5f;
            cen[3 * (size_t)i + a] = c;
            cb.lo[a] = c; cb.hi[a] = c;
        }
    }
    for (int a = 0; a < 3; a++) { red[a][threadIdx.x] = fkey(cb.lo[a]); red[3 + a][threadIdx.x] = fkey(cb.hi[a]); }
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            for (int a = 0; a < 3; a++) {
                red[a][threadIdx.x] = min(red[a][threadIdx.x], red[a][threadIdx.x + s]);
                red[3 + a][threadIdx.x] = max(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + s]);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < 6) partial[6 * (size_t)blockIdx.x + threadIdx.x] = red[threadIdx.x][0];
}

__global__ void __launch_bounds__(256) k_reduce_bounds(const uint32_t* partial, int nblocks, uint32_t* out6) {
    __shared__ uint32_t red[6][256];
    uint32_t lo[3] = {0xffffffffu, 0xffffffffu, 0xffffffffu}, hi[3] = {0u, 0u, 0u};
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x)
        for (int a = 0; a < 3; a++) { lo[a] = min(lo[a], partial[6 * (size_t)b + a]); hi[a] = max(hi[a], partial[6 * (size_t)b + 3 + a]); }
    for (int a = 0; a < 3; a++) { red[a][threadIdx.x] = lo[a]; red[3 + a][threadIdx.x] = hi[a]; }
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int a = 0; a < 3; a++) {
                red[a][threadIdx.x] = min(red[a][threadIdx.x], red[a][threadIdx.x + s]);
                red[3 + a][threadIdx.x] = max(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) out6[threadIdx.x] = red[threadIdx.x][0];
}

// ---------------------------------------------------------------------------
// 2. Morton codes (21 bits per axis, x in the highest bit of each triple)
// ---------------------------------------------------------------------------
SRT_D uint64_t expand_bits21(uint32_t v) {
    uint64_t x = v & 0x1fffffu;
    x = (x | (x << 32)) & 0x1f00000000ffffULL;
    x = (x | (x << 16)) & 0x1f0000ff0000ffULL;
    x = (x | (x << 8)) & 0x100f00f00f00f00fULL;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ULL;
    x = (x | (x << 2)) & 0x1249249249249249ULL;
    return x;
}
SRT_D uint32_t morton_axis(float c, float lo, float ext) {
    float t = (ext > 0.0f) ? (c - lo) / ext : 0.0f;
    float q = t * 2097152.0f;
    return (q >= 2097151.0f) ? 2097151u : (q > 0.0f ? (uint32_t)q : 0u);
}
__global__ void __launch_bounds__(256) k_morton(const float* cen, const uint32_t* cb6, int n, uint64_t* keys, uint32_t* vals) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t q[3];
    for (int a = 0; a < 3; a++) {
        float lo = fromkey(cb6[a]), hi = fromkey(cb6[3 + a]);
        q[a] = morton_axis(cen[3 * (size_t)i + a], lo, hi - lo);
    }
    keys[i] = (expand_bits21(q[0]) << 2) | (expand_bits21(q[1]) << 1) | expand_bits21(q[2]);
    vals[i] = (uint32_t)i;
}

// ---------------------------------------------------------------------------
// 3. Karras radix tree
// ---------------------------------------------------------------------------
SRT_D int kdelta(const uint64_t* c, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    uint64_t a = c[i], b = c[j];
    if (a != b) return __clzll((long long)(a ^ b));
    return 64 + __clz((int)((uint32_t)i ^ (uint32_t)j));
}
// child refs: >= 0 internal node, < 0 leaf (-k-1)
__global__ void __launch_bounds__(256) k_karras(const uint64_t* sc, int n, int32_t* kl, int32_t* kr, int32_t* kfirst,
                                                int32_t* par_int, int32_t* par_leaf) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    int d = (kdelta(sc, n, i, i + 1) - kdelta(sc, n, i, i - 1)) >= 0 ? 1 : -1;
    int dmin = kdelta(sc, n, i, i - d);
    int lmax = 2;
    while (kdelta(sc, n, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (kdelta(sc, n, i, i + (l + t) * d) > dmin) l += t;
    int j = i + l * d;
    int dnode = kdelta(sc, n, i, j);
    int sp = 0, t = l;
    do {
        t = (t + 1) / 2;
        if (kdelta(sc, n, i, i + (sp + t) * d) > dnode) sp += t;
    } while (t > 1);
    int gamma = i + sp * d + min(d, 0);
    int lo = min(i, j), hi = max(i, j);
    int32_t left = (lo == gamma) ? -(gamma + 1) : gamma;
    int32_t right = (hi == gamma + 1) ? -(gamma + 2) : gamma + 1;
    kl[i] = left;
    kr[i] = right;
    kfirst[i] = lo;
    if (left < 0) par_leaf[-left - 1] = i; else par_int[left] = i;
    if (right < 0) par_leaf[-right - 1] = i; else par_int[right] = i;
}

// ---------------------------------------------------------------------------
// 4. bottom-up boxes / counts / SAH costs / collapse
// ---------------------------------------------------------------------------
struct KArr {
    BoxArr box;
    int32_t* count;
    float* cost;
    int32_t* collapse;
};
// Nodes ordered by level: a stable counting sort with one 8-bit key per node.
// The trees' levels fit 8 bits (a radix tree's common prefixes grow with every
// level, so it has at most 63 + 32 of them; a binary tree deeper than kMaxDepth
// is refused), so one pass orders the nodes: histograms of pieces of
// kLevelPiece nodes, one scan per level over the pieces, and the ranks within
// each piece, 64 nodes at a time by matching keys across the wave.  Bound by
// the two reads of the keys and one write of the ids; it took the place of a
// library radix sort and of a search for the levels' first nodes: for the
// radix tree of 1M triangles (16-bit keys, two passes of 18 launches) about
// 170 us, now 36 us.
constexpr int kLevels = 256;
constexpr int kLevelNone = 255;         // unused node slots: after every level
constexpr int kLevelPiece = 4096;
SRT_D uint8_t level_key(int level) { return (uint8_t)min(level, kLevelNone - 1); }
__global__ void __launch_bounds__(256) k_level_hist(int n, const uint8_t* key, int pieces, int32_t* hist) {
    __shared__ int32_t s_h[kLevels];
    const int tid = threadIdx.x;
    s_h[tid] = 0;
    __syncthreads();
    const int b = blockIdx.x * kLevelPiece, e = min(b + kLevelPiece, n);
    for (int i = b + tid; i < e; i += 256) atomicAdd(&s_h[key[i]], 1);
    __syncthreads();
    hist[(size_t)tid * pieces + blockIdx.x] = s_h[tid];
}
// inclusive scan over a workgroup of 256 threads; `s_w` holds its waves' sums
SRT_D int32_t block_scan256(int32_t v, int32_t* s_w) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int d = 1; d < 64; d <<= 1) {
        const int32_t u = __shfl_up(v, d);
        if (lane >= d) v += u;
    }
    __syncthreads();
    if (lane == 63) s_w[wv] = v;
    __syncthreads();
    for (int w = 0; w < wv; w++) v += s_w[w];
    return v;
}
// workgroup L: the pieces' counts of level L become their first ranks within
// the level, the sum its size
__global__ void __launch_bounds__(256) k_level_scan(int pieces, int32_t* hist, int32_t* size) {
    __shared__ int32_t s_w[4];
    __shared__ int32_t s_run;
    const int tid = threadIdx.x;
    int32_t* row = hist + (size_t)blockIdx.x * pieces;
    int32_t run = 0;
    for (int start = 0; start < pieces; start += 256) {
        const int i = start + tid;
        const int32_t v = i < pieces ? row[i] : 0;
        const int32_t incl = block_scan256(v, s_w);
        if (i < pieces) row[i] = run + incl - v;
        if (tid == 255) s_run = incl;
        __syncthreads();
        run += s_run;
    }
    if (tid == 0) size[blockIdx.x] = run;
}
// `ids`: node at each position; `number`: position of each node (or null);
// `first`: first position of every level, kLevels + 1 entries
__global__ void __launch_bounds__(256) k_level_rank(int n, const uint8_t* key, int pieces, const int32_t* hist,
                                                    const int32_t* size, uint32_t* ids, int32_t* number, int32_t* first) {
    __shared__ int32_t s_w[4];
    __shared__ int32_t s_next[4][kLevels];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int32_t mine = size[tid];
    const int32_t incl = block_scan256(mine, s_w);
    if (blockIdx.x == 0) {
        first[tid] = incl - mine;
        if (tid == kLevels - 1) first[kLevels] = incl;
    }
    for (int w = 0; w < 4; w++) s_next[w][tid] = 0;
    __syncthreads();
    constexpr int kRun = kLevelPiece / 4;         // consecutive nodes of one wave
    const int b = blockIdx.x * kLevelPiece + wv * kRun, e = min(b + kRun, n);
    for (int i = b + lane; i < e; i += 64) atomicAdd(&s_next[wv][key[i]], 1);
    __syncthreads();
    {
        int32_t at = incl - mine + hist[(size_t)tid * pieces + blockIdx.x];
        for (int w = 0; w < 4; w++) {
            const int32_t k = s_next[w][tid];
            s_next[w][tid] = at;
            at += k;
        }
    }
    __syncthreads();
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int start = b; start < e; start += 64) {
        const int i = start + lane;
        const int k = i < e ? (int)key[i] : -1;
        unsigned long long todo = __ballot(k >= 0);
        int32_t at = 0;
        while (todo) {
            const int d = __builtin_amdgcn_readlane(k, __ffsll(todo) - 1);
            const unsigned long long same = __ballot(k == d);
            const int32_t base = s_next[wv][d];
            if (k == d) at = base + __popcll(same & below);
            if (lane == 0) s_next[wv][d] = base + __popcll(same);
            __builtin_amdgcn_wave_barrier();      // the next match may be of the same level
            todo &= ~same;
        }
        if (k >= 0) {
            ids[at] = (uint32_t)i;
            if (number) number[i] = at;
        }
    }
}
// Depth of radix-tree node i below the root (node 0)
__global__ void __launch_bounds__(256) k_radix_depth(int m, const int32_t* par_int, uint8_t* key) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    int depth = 0;
    for (int p = par_int[i]; p >= 0; p = par_int[p]) depth++;
    key[i] = level_key(depth);
}
// One depth of the bottom-up pass (deepest first): box, triangle count, SAH
// cost and collapse decision of each node from its two children, which the
// previous launch (or the triangle boxes) provides.
SRT_D void bottom_up_node(int p, const uint32_t* order, const BoxArr& tb, const int32_t* kl, const int32_t* kr, const KArr& K,
                          int max_leaf, float c_trav, float c_isect) {
    DBox bl, br;
    int cl, cr;
    float costl, costr;
    int32_t L = kl[p], R = kr[p];
    if (L < 0) { int q = -L - 1; bl = ldbox(tb, order[q]); cl = 1; costl = c_isect * 1.0f * box_area(bl); }
    else { bl = ldbox(K.box, L); cl = K.count[L]; costl = K.cost[L]; }
    if (R < 0) { int q = -R - 1; br = ldbox(tb, order[q]); cr = 1; costr = c_isect * 1.0f * box_area(br); }
    else { br = ldbox(K.box, R); cr = K.count[R]; costr = K.cost[R]; }
    DBox b = bl;
    grow(b, br);
    int cnt = cl + cr;
    float sa = box_area(b);
    float ci = c_trav * sa + costl + costr;
    float cf = c_isect * (float)cnt * sa;
    int col = (cnt <= max_leaf) && (cf <= ci);
    stbox(K.box, p, b);
    K.count[p] = cnt;
    K.cost[p] = col ? cf : ci;
    K.collapse[p] = col;
}
__global__ void __launch_bounds__(256) k_bottom_up_level(const uint32_t* ids, int count, const uint32_t* order, BoxArr tb,
                                                         const int32_t* kl, const int32_t* kr, KArr K, int max_leaf,
                                                         float c_trav, float c_isect) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < count) bottom_up_node((int)ids[k], order, tb, kl, kr, K, max_leaf, c_trav, c_isect);
}
// Passes over the levels of a tree, deepest first, have many levels of few
// nodes (the deepest ones, and those near the root), and a launch for each costs
// more than its nodes.  One workgroup takes a run of consecutive levels of at
// most kRunNodes nodes, with a barrier between two levels: the writes of a
// level are seen by the next one through the CU's own cache.  Of the 34 levels
// of the 1M-triangle field's radix tree 15 are in two such runs; a frame of the
// skinned tube (skin, refit, render) takes 2.82 ms instead of 2.88, a rebuild
// of the field, bound elsewhere, the same within its noise.
constexpr int kRunNodes = 1024;
constexpr int kRunLevels = 64;
struct LevelRun {
    int32_t levels;
    int32_t first[kRunLevels], end[kRunLevels];      // deepest first
};
template <class Node> SRT_D void run_levels(const LevelRun& run, const uint32_t* ids, Node&& node) {
    for (int r = 0; r < run.levels; r++) {
        const int k = run.first[r] + (int)threadIdx.x;
        if (k < run.end[r]) node((int)ids[k]);
        __syncthreads();
    }
}
__global__ void __launch_bounds__(kRunNodes) k_bottom_up_run(LevelRun run, const uint32_t* ids, const uint32_t* order, BoxArr tb,
                                                             const int32_t* kl, const int32_t* kr, KArr K, int max_leaf,
                                                             float c_trav, float c_isect) {
    run_levels(run, ids, [&](int p) { bottom_up_node(p, order, tb, kl, kr, K, max_leaf, c_trav, c_isect); });
}

// ---------------------------------------------------------------------------
// 5. cluster frontier (marks the first sorted position of each cluster)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_frontier(int n, int T, const int32_t* kfirst, const int32_t* kcount, const int32_t* par_int,
                                                  const int32_t* par_leaf, int32_t* mark) {
    int x = blockIdx.x * blockDim.x + threadIdx.x;
    // x < n-1: internal node x; n-1 <= x < 2n-1: leaf x-(n-1)
    if (x >= 2 * n - 1) return;
    int32_t ref, first, cnt, parent;
    if (x < n - 1) { ref = x; first = kfirst[x]; cnt = kcount[x]; parent = par_int[x]; }
    else { int k = x - (n - 1); ref = -(k + 1); first = k; cnt = 1; parent = par_leaf[k]; }
    if (cnt > T) return;
    if (parent >= 0 && kcount[parent] <= T) return;
    mark[first] = ref;
}

// cluster items for the top-level SAH
struct Items {
    BoxArr box;
    float *cx, *cy, *cz;
    int32_t* count;
    int32_t* ref;
};
__global__ void __launch_bounds__(256) k_items(int m, const int32_t* cl, const uint32_t* order, BoxArr tb, KArr K,
                                               const int32_t* kfirst, int top, Items it) {
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= m) return;
    int32_t c = cl[q];
    DBox b;
    int cnt;
    int32_t ref;
    if (c < 0) {
        int k = -c - 1;
        b = ldbox(tb, order[k]); cnt = 1; ref = leaf_ref((uint32_t)k, 1u);
    } else {
        b = ldbox(K.box, c); cnt = K.count[c];
        ref = K.collapse[c] ? leaf_ref((uint32_t)kfirst[c], (uint32_t)cnt) : top + c;
    }
    stbox(it.box, q, b);
    it.cx[q] = (b.lo[0] + b.hi[0]) * 0.5f;
    it.cy[q] = (b.lo[1] + b.hi[1]) * 0.5f;
    it.cz[q] = (b.lo[2] + b.hi[2]) * 0.5f;
    it.count[q] = cnt;
    it.ref[q] = ref;
}

SRT_D void set_child(BvhNode* nd, int side, const DBox& b, int32_t ref) {
    if (side == 0) {
        nd->a.x = b.lo[0]; nd->a.y = b.hi[0]; nd->a.z = b.lo[1]; nd->a.w = b.hi[1];
        nd->c.x = b.lo[2]; nd->c.y = b.hi[2];
        nd->d.x = ref;
    } else {
        nd->b.x = b.lo[0]; nd->b.y = b.hi[0]; nd->b.z = b.lo[1]; nd->b.w = b.hi[1];
        nd->c.z = b.lo[2]; nd->c.w = b.hi[2];
        nd->d.y = ref;
    }
}

// ---------------------------------------------------------------------------
// 6. top-level binned SAH over the clusters, breadth-first
// ---------------------------------------------------------------------------
// A split of a node's item range [b, e) at `mid` is the only one with this
// boundary in the whole tree, so the node's record is kept under its boundary
// and needs no number until the end: nodes are numbered breadth-first, left
// before right, which is the order of (level, boundary), one counting sort.
// No level therefore waits for the number of nodes of the one before it, and
// the host reads nothing until all are split.  A node's split depends only on
// its own items, so the tree is the one a sequential build produces.
//   wide levels  (the first ones, where every node has thousands of items):
//                chunks of kWideChunk items bin into their node's accumulators,
//                one wave per node chooses the split, the chunks partition
//   middle levels: one launch per level; a node of more than kBlockItems items
//                is split by a workgroup, one of more than kSmallItems by a wave
//   small nodes  (two to kSmallItems items): one wave builds the whole subtree
//                in LDS
// Items are read from it[level & 1] and written, partitioned, to the other.
// Lane 16 a + k of a wave holds bin k of axis a when a split is chosen; the
// boxes and centroid bounds of a node's children are unions of bins, so a level
// reads its items once to bin and once to partition them.
// Before, per level: bounds, bins by LDS atomics, partition, child boxes, a
// scan that numbered the children and a wait for their count, with one wave
// per node down to two items: 3.0 ms of the 4.7 ms of a rebuild of the
// 1M-triangle field (347 thousand clusters, 26 levels); now 1.1 ms.
constexpr int kBins = 16;
constexpr int kTopWaves = 4;           // waves of a workgroup
// 3 axes x 21 items are one wave's split candidates
constexpr int kSmallItems = 21;
// four waves share a node that one would work on for more than four rounds of 64
// items: a rebuild of the 1M-triangle field takes 3.00 ms, 3.04 ms with a line at 128 or at 512
constexpr int kBlockItems = 256;
// A wide level of the 1M-triangle field takes 35 us whatever its nodes' sizes, a
// level of middle nodes as long as its largest node: with seven wide levels
// instead of nine (1300 items per node on average) the rebuild takes 3.09 ms.
constexpr int kWideLevels = 9;
constexpr int kWideMin = 1024;         // items per node on average down to which levels are wide
constexpr int kWideChunk = 512;        // two rounds of a wave's 64 items
constexpr int kWideCopies = 8;         // accumulators of a node: chunks of a node share an address eight times less
constexpr int kRegions = 64;           // small nodes are listed by region of the items, each with its own counter
constexpr int kRegionBlocks = 32;       // two workgroups a SIMD
constexpr int kAccWords = 14;          // box lo xyz, hi xyz, centroid lo xyz, hi xyz (keys), triangles, items

SRT_D int bin_of(float c, float lo, float scale) {
    int bi = (int)((c - lo) * scale);
    if (bi > kBins - 1) bi = kBins - 1;
    if (bi < 0) bi = 0;
    return bi;
}
SRT_D float item_c(const Items& it, int a, int i) { return a == 0 ? it.cx[i] : (a == 1 ? it.cy[i] : it.cz[i]); }
SRT_D void copy_item(const Items& s, int i, const Items& d, int j) {
    d.box.lox[j] = s.box.lox[i]; d.box.loy[j] = s.box.loy[i]; d.box.loz[j] = s.box.loz[i];
    d.box.hix[j] = s.box.hix[i]; d.box.hiy[j] = s.box.hiy[i]; d.box.hiz[j] = s.box.hiz[i];
    d.cx[j] = s.cx[i]; d.cy[j] = s.cy[i]; d.cz[j] = s.cz[i];
    d.count[j] = s.count[i]; d.ref[j] = s.ref[i];
}
SRT_D void wave_sync() {      // LDS of one wave: its accesses stay in order, the compiler must keep them so
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// word q of an accumulator: identity, union
SRT_D uint32_t acc_empty(int q) {
    return q >= 12 ? 0u : (q % 6 < 3 ? fkey(__builtin_huge_valf()) : fkey(-__builtin_huge_valf()));
}
SRT_D uint32_t acc_union(int q, uint32_t x, uint32_t y) { return q >= 12 ? x + y : (q % 6 < 3 ? min(x, y) : max(x, y)); }
// the value of the lane CTRL names within a row of 16 lanes, `old` where there is none
template <int CTRL> SRT_D uint32_t row_get(uint32_t old, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, 0xf, 0xf, false);
}
constexpr int kRowShl = 0x100, kRowShr = 0x110;       // + lanes
// a value that is the same in all lanes, held in a scalar register: loops over it need no per-lane exit
SRT_D int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
SRT_D uint32_t read_lane(uint32_t v, int lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, lane); }
// minimum over the wave, in every lane
SRT_D uint32_t wave_min_u32(uint32_t v) {
    v = min(v, row_get<kRowShr + 1>(~0u, v));
    v = min(v, row_get<kRowShr + 2>(~0u, v));
    v = min(v, row_get<kRowShr + 4>(~0u, v));
    v = min(v, row_get<kRowShr + 8>(~0u, v));
    return min(min(read_lane(v, 15), read_lane(v, 31)), min(read_lane(v, 47), read_lane(v, 63)));
}

struct alignas(16) TopTask {
    int32_t b, e;           // items; e == b: none
    int32_t up;             // 2 * parent's boundary + side, 0 for the root
    uint32_t cb[6];         // centroid bounds (keys): lo xyz, hi xyz
};
struct SmallTask {
    int32_t b, e, up, level;
};
// A child is another node (its boundary, written when that node is split), a
// given ref, or the item at a position of it[0] or it[1].
constexpr int kChildNode = 0, kChildRef = 1, kChildItem = 2;
struct alignas(64) TopRec {
    float box[2][6];        // child boxes: lo xyz, hi xyz
    int32_t child[2];
    int32_t kind[2];
};
struct WideSplit {
    int32_t axis, split, mid;
    float lo, scale;
};
struct TopBuild {
    int m;                  // items
    int wide_levels;
    Items it[2];
    TopRec* rec;            // by boundary, 1 .. m - 1
    uint8_t* level;         // of boundary p at p - 1
    TopTask* wide[2];       // 2^L slots: the children of slot t are 2 t and 2 t + 1
    TopTask* mid[2];        // slot of a node: the multiple of kSmallItems + 1 in its range, see mid_slot
    SmallTask* small;       // by regions
    int32_t* nsmall;        // per region, 256 bytes apart
    int32_t* any;           // [L]: level L has middle nodes
    uint32_t* cb;           // centroid bounds of all items (keys)
    uint32_t* acc;          // wide nodes' accumulators [slot][copy][word][lane 0 .. 47]
    int32_t* chunk_items;   // items per chunk and lane (bin) of a wide level
    WideSplit* wsplit;
};
// Nodes of a level are disjoint ranges of more than kSmallItems items, so each
// holds a multiple of kSmallItems + 1 that no other one holds: a slot without a
// counter.
__host__ __device__ inline int mid_slot(int b) { return (b + kSmallItems) / (kSmallItems + 1); }
__host__ __device__ inline int mid_slots(int m) { return m / (kSmallItems + 1) + 1; }
// first item and first list entry of a region: nodes start at least two items apart
__host__ __device__ inline int region_first(int m, int r) { return (int)(((int64_t)r * m + kRegions - 1) / kRegions); }
__host__ __device__ inline int region_base(int m, int r) { return region_first(m, r) / 2 + r; }
SRT_D int region_of(int m, int b) { return (int)((int64_t)b * kRegions / m); }

// one child of the node split at `mid` on level L (one lane)
SRT_D void top_child(const TopBuild& B, int L, int mid, int side, int b, int e, const uint32_t* cb, int wide_slot) {
    TopRec* r = B.rec + mid;
    if (e - b == 1) {
        r->child[side] = b;
        r->kind[side] = kChildItem + ((L + 1) & 1);
        return;
    }
    r->kind[side] = kChildNode;
    const int32_t up = 2 * mid + side;
    if (e - b <= kSmallItems) {
        const int reg = region_of(B.m, b);
        const int q = atomicAdd(B.nsmall + reg * 64, 1);
        B.small[region_base(B.m, reg) + q] = {b, e, up, L + 1};
        return;
    }
    TopTask t;
    t.b = b; t.e = e; t.up = up;
    for (int q = 0; q < 6; q++) t.cb[q] = cb[q];
    if (wide_slot >= 0) {
        B.wide[(L + 1) & 1][wide_slot] = t;
    } else {
        B.mid[(L + 1) & 1][mid_slot(b)] = t;
        B.any[L + 1] = 1;
    }
}
// the node of task t split at `mid`: `side` holds the children's boxes and
// centroid bounds (one lane)
SRT_D void top_node(const TopBuild& B, int L, const TopTask& t, int mid, const uint32_t side[2][12], int wide_slot) {
    TopRec* r = B.rec + mid;
    for (int s = 0; s < 2; s++)
        for (int q = 0; q < 6; q++) r->box[s][q] = fromkey(side[s][q]);
    B.level[mid - 1] = level_key(L);
    if (t.up) B.rec[t.up >> 1].child[t.up & 1] = mid;
    top_child(B, L, mid, 0, t.b, mid, side[0] + 6, wide_slot);
    top_child(B, L, mid, 1, mid, t.e, side[1] + 6, wide_slot < 0 ? -1 : wide_slot + 1);
}

// Bins in LDS, R copies of each word next to each other: neighbouring items
// mostly share a bin, and the lanes of a wave that do add to R different banks
// (one copy per wave, as before, took a wide level of the 1M-triangle field
// 35 us, lanes that own a bin and look at every item 24 to 43 us, 16 copies
// 13 us).  A workgroup shares 16 copies, a wave on its own has 4 of the same
// memory.
constexpr int kAccTotal = kAccWords * 48;
constexpr int kBlockCopies = 16, kWaveCopies = kBlockCopies / kTopWaves;
template <int R> SRT_D void bins_clear(uint32_t* s, int tid, int threads) {
    for (int i = 4 * tid; i < kAccTotal * R; i += 4 * threads) {
        const uint32_t v = acc_empty(i / (48 * R));
        *(uint4*)(s + i) = make_uint4(v, v, v, v);
    }
}
// the wave's items [b, e)
template <int R> SRT_D void bins_add(const Items& it, int b, int e, const uint32_t* cb, uint32_t* s) {
    const int lane = __lane_id();
    float lo[3], ext[3], scale[3];
    for (int a = 0; a < 3; a++) {
        lo[a] = fromkey(cb[a]);
        ext[a] = fromkey(cb[3 + a]) - lo[a];
        scale[a] = ext[a] > 0.0f ? (float)kBins / ext[a] : 0.0f;
    }
    for (int i = b + lane; i < e; i += 64) {
        const DBox ib = ldbox(it.box, i);
        const float c[3] = {it.cx[i], it.cy[i], it.cz[i]};
        const uint32_t tris = (uint32_t)it.count[i];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            if (!(ext[a] > 0.0f)) continue;
            uint32_t* p = s + (16 * a + bin_of(c[a], lo[a], scale[a])) * R + lane % R;
            for (int q = 0; q < 3; q++) {
                atomicMin(p + q * (48 * R), fkey(ib.lo[q]));
                atomicMax(p + (3 + q) * (48 * R), fkey(ib.hi[q]));
                atomicMin(p + (6 + q) * (48 * R), fkey(c[q]));
                atomicMax(p + (9 + q) * (48 * R), fkey(c[q]));
            }
            atomicAdd(p + 12 * (48 * R), tris);
            atomicAdd(p + 13 * (48 * R), 1u);
        }
    }
}
// word q of bin l (0 .. 47); the copies in an order that spreads the lanes over the banks
template <int R> SRT_D uint32_t bins_word(const uint32_t* s, int q, int l) {
    uint32_t v = acc_empty(q);
    for (int c = 0; c < R; c++) v = acc_union(q, v, s[(q * 48 + l) * R + (c + l) % R]);
    return v;
}
// SAH over the 15 bin boundaries of each axis (cost = area x triangles per side
// of the boundary) from the lanes' bins: the first minimum in (axis, boundary)
// order.  Returns its lane, -1 when no boundary separates items (every extent
// zero or every item in one bin); `side` gets the children's words.
SRT_D int sah_choose_wave(const uint32_t* acc, const uint32_t* cb, uint32_t side[2][kAccWords]) {
    static_assert(kBins == 16, "a row of 16 lanes per axis");
    const int lane = __lane_id();
    const int a = lane >> 4, k = lane & 15;
    uint32_t pre[kAccWords], suf[kAccWords];
    for (int q = 0; q < kAccWords; q++) {
        const uint32_t none = acc_empty(q);
        uint32_t p = acc[q], s = acc[q];
        p = acc_union(q, p, row_get<kRowShr + 1>(none, p));
        s = acc_union(q, s, row_get<kRowShl + 1>(none, s));
        p = acc_union(q, p, row_get<kRowShr + 2>(none, p));
        s = acc_union(q, s, row_get<kRowShl + 2>(none, s));
        p = acc_union(q, p, row_get<kRowShr + 4>(none, p));
        s = acc_union(q, s, row_get<kRowShl + 4>(none, s));
        p = acc_union(q, p, row_get<kRowShr + 8>(none, p));
        s = acc_union(q, s, row_get<kRowShl + 8>(none, s));
        pre[q] = p;
        suf[q] = row_get<kRowShl + 1>(none, s);         // the right side of boundary k starts at bin k + 1
    }
    DBox lb, rb;
    for (int q = 0; q < 3; q++) {
        lb.lo[q] = fromkey(pre[q]); lb.hi[q] = fromkey(pre[3 + q]);
        rb.lo[q] = fromkey(suf[q]); rb.hi[q] = fromkey(suf[3 + q]);
    }
    const int axis = min(a, 2);
    const uint32_t klo = axis == 0 ? cb[0] : (axis == 1 ? cb[1] : cb[2]);
    const uint32_t khi = axis == 0 ? cb[3] : (axis == 1 ? cb[4] : cb[5]);
    uint32_t key = ~0u;
    if (a < 3 && k < kBins - 1 && fromkey(khi) - fromkey(klo) > 0.0f && pre[12] != 0 && suf[12] != 0) {
        const float cost = box_area(lb) * (float)(int32_t)pre[12] + box_area(rb) * (float)(int32_t)suf[12];
        if (cost < __builtin_huge_valf()) key = __float_as_uint(cost);
    }
    const uint32_t best = wave_min_u32(key);
    if (best == ~0u) return -1;
    const int w = uniform(__ffsll(__ballot(key == best)) - 1);
    for (int q = 0; q < kAccWords; q++) {
        side[0][q] = read_lane(pre[q], w);
        side[1][q] = read_lane(suf[q], w);
    }
    return w;
}
// the words of the items [b, e) by one wave, for a node without a boundary
SRT_D void union_items(const Items& it, int b, int e, uint32_t* out) {
    uint32_t v[12];
    for (int q = 0; q < 12; q++) v[q] = acc_empty(q);
    for (int i = b + __lane_id(); i < e; i += 64) {
        const DBox ib = ldbox(it.box, i);
        for (int a = 0; a < 3; a++) {
            const uint32_t c = fkey(item_c(it, a, i));
            v[a] = min(v[a], fkey(ib.lo[a]));
            v[3 + a] = max(v[3 + a], fkey(ib.hi[a]));
            v[6 + a] = min(v[6 + a], c);
            v[9 + a] = max(v[9 + a], c);
        }
    }
    for (int q = 0; q < 12; q++) {
        for (int d = 32; d > 0; d >>= 1) v[q] = acc_union(q, v[q], (uint32_t)__shfl_xor((int)v[q], d));
        out[q] = read_lane(v[q], 0);
    }
}
// the wave's items [b, e), stable: left ones from `l`, right ones from `r`
SRT_D void partition_items(const Items& src, const Items& dst, int b, int e, int axis, float lo, float scale, int split,
                           int l, int r) {
    const int lane = __lane_id();
    b = uniform(b);
    e = uniform(e);
    const unsigned long long below = (1ull << lane) - 1ull;
    for (int start = b; start < e; start += 64) {
        const int i = start + lane;
        const bool has = i < e;
        const bool left = has && bin_of(item_c(src, axis, i), lo, scale) <= split;
        const unsigned long long ml = __ballot(left), mr = __ballot(has && !left);
        if (has) copy_item(src, i, dst, left ? l + __popcll(ml & below) : r + __popcll(mr & below));
        l += __popcll(ml);
        r += __popcll(mr);
    }
}
// One node of a middle level by W waves (each takes a consecutive part of the
// items); with W > 1 every wave of the workgroup calls it with the same task.
template <int W>
SRT_D void split_task(const TopBuild& B, int L, const TopTask& t, int wv, uint32_t* s_bins, int32_t* s_left) {
    constexpr int R = W == 1 ? kWaveCopies : kBlockCopies;
    const int lane = __lane_id();
    const Items &src = B.it[L & 1], &dst = B.it[(L + 1) & 1];
    const int per = (t.e - t.b + W * 64 - 1) / (W * 64) * 64;
    const int b = uniform(W == 1 ? t.b : min(t.b + wv * per, t.e)), e = uniform(W == 1 ? t.e : min(b + per, t.e));
    uint32_t* bins = W == 1 ? s_bins + wv * (kAccTotal * kWaveCopies) : s_bins;
    bins_clear<R>(bins, W == 1 ? lane : (int)threadIdx.x, 64 * W);
    if (W > 1) __syncthreads();
    else wave_sync();
    bins_add<R>(src, b, e, t.cb, bins);
    if (W > 1) __syncthreads();
    else wave_sync();
    uint32_t acc[kAccWords];
    for (int q = 0; q < kAccWords; q++) acc[q] = lane < 48 ? bins_word<R>(bins, q, lane) : acc_empty(q);
    uint32_t side[2][kAccWords];
    const int w = uniform(sah_choose_wave(acc, t.cb, side));
    int mid = (t.b + t.e) / 2;
    if (w >= 0) {
        mid = t.b + (int)side[0][13];
        const int axis = w >> 4;
        const float lo = fromkey(axis == 0 ? t.cb[0] : (axis == 1 ? t.cb[1] : t.cb[2]));
        const float ext = fromkey(axis == 0 ? t.cb[3] : (axis == 1 ? t.cb[4] : t.cb[5])) - lo;
        int before = 0;
        if (W > 1) {
            int32_t left = 0;
            for (int i = b + lane; i < e; i += 64)
                left += bin_of(item_c(src, axis, i), lo, (float)kBins / ext) <= (w & 15) ? 1 : 0;
            for (int d = 32; d > 0; d >>= 1) left += __shfl_xor(left, d);
            if (lane == 0) s_left[wv] = left;
            __syncthreads();
            for (int v = 0; v < wv; v++) before += s_left[v];
        }
        partition_items(src, dst, b, e, axis, lo, (float)kBins / ext, w & 15, t.b + before, mid + (b - t.b) - before);
    } else {
        for (int i = b + lane; i < e; i += 64) copy_item(src, i, dst, i);
        union_items(src, t.b, mid, side[0]);
        union_items(src, mid, t.e, side[1]);
    }
    if (wv == 0 || W == 1) {
        if (lane == 0) {
            const uint32_t* s0 = side[0];
            const uint32_t* s1 = side[1];
            uint32_t sd[2][12];
            for (int q = 0; q < 12; q++) {
                sd[0][q] = s0[q];
                sd[1][q] = s1[q];
            }
            top_node(B, L, t, mid, sd, -1);
        }
    }
}
// workgroup g: kMidSlots slots of the level, nodes of more than kBlockItems
// items by all waves, then the others by one wave each.  Bound by the latency
// of a node's chain (load, bin, scan, choose, partition); with one slot a wave
// most workgroups of a level were empty and a level took at least 48 us.
constexpr int kMidSlots = 16;
__global__ void __launch_bounds__(64 * kTopWaves) k_top_mid(TopBuild B, int L, int slots) {
    __shared__ alignas(16) uint32_t s_bins[kAccTotal * kBlockCopies];
    __shared__ TopTask s_task[kMidSlots];
    __shared__ int32_t s_left[kTopWaves];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    // every wave knows the slots in use; wave 0 takes the tasks out of them
    const int slot = blockIdx.x * kMidSlots + lane;
    TopTask* p = B.mid[L & 1] + slot;
    TopTask mine;
    mine.b = mine.e = 0;
    if (wv == 0 && lane < kMidSlots) {
        if (slot < slots) {
            mine = *p;
            if (mine.e > mine.b) p->b = p->e = 0;    // the list of level L + 2
        }
        s_task[lane] = mine;
    }
    __syncthreads();
    int n = 0;
    if (lane < kMidSlots) n = s_task[lane].e - s_task[lane].b;
    for (unsigned long long big = __ballot(n > kBlockItems); big; big &= big - 1) {
        split_task<kTopWaves>(B, L, s_task[__ffsll(big) - 1], wv, s_bins, s_left);
        __syncthreads();
    }
    int k = 0;
    for (unsigned long long some = __ballot(n > 0 && n <= kBlockItems); some; some &= some - 1)
        if (k++ % kTopWaves == wv) split_task<1>(B, L, s_task[__ffsll(some) - 1], wv, s_bins, s_left);
}
// Subtrees of two to kSmallItems items, one wave each.  With so few items the
// candidates are the items themselves: lane 21 a + i is the boundary after item
// i's bin of axis a (an empty bin's boundary costs the same as the one before
// it), it looks at every item once and has both sides' boxes and counts, with
// no bins and no scan.  Nodes of two items, a third of all, are left to the
// end and split by a lane each.  Bound by instructions, about 300 for a node.
__global__ void __launch_bounds__(64 * kTopWaves) k_top_small(TopBuild B) {
    static_assert(3 * kSmallItems <= 64, "one lane per axis and item");
    struct alignas(16) Item {
        uint32_t w[12];     // box and centroid keys, triangles, ref
    };
    __shared__ Item s_item[kTopWaves][kSmallItems];
    __shared__ int32_t s_bin[kTopWaves][64];
    __shared__ int4 s_stack[kTopWaves][kSmallItems];
    __shared__ int4 s_pair[kTopWaves][kSmallItems / 2];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int axis = lane / kSmallItems, li = lane % kSmallItems, ax = min(axis, 2);
    const int reg = blockIdx.x / kRegionBlocks, first = blockIdx.x % kRegionBlocks * kTopWaves + wv;
    const unsigned long long below = (1ull << lane) - 1ull;
    Item* item = s_item[wv];
    const int count = B.nsmall[reg * 64], base = region_base(B.m, reg);
    for (int k = first; k < count; k += kRegionBlocks * kTopWaves) {
        const SmallTask t = B.small[base + k];
        const Items& it = B.it[t.level & 1];
        const int total = t.e - t.b;
        wave_sync();
        if (lane < total) {
            const int i = t.b + lane;
            Item v;
            const DBox ib = ldbox(it.box, i);
            for (int a = 0; a < 3; a++) {
                v.w[a] = fkey(ib.lo[a]);
                v.w[3 + a] = fkey(ib.hi[a]);
                v.w[6 + a] = fkey(item_c(it, a, i));
            }
            v.w[9] = (uint32_t)it.count[i];
            v.w[10] = (uint32_t)it.ref[i];
            v.w[11] = 0;
            item[lane] = v;
        }
        if (lane == 0) {
            s_stack[wv][0] = make_int4(0, total, t.up, t.level);
            s_pair[wv][0] = make_int4(0, total, t.up, t.level);
        }
        wave_sync();
        int sp = total > 2 ? 1 : 0, pairs = total > 2 ? 0 : 1;
        while (sp > 0) {
            sp--;
            const int4 f = s_stack[wv][sp];
            const int b = uniform(f.x), e = uniform(f.y);
            const int n = e - b;
            uint32_t mn = ~0u, mx = 0u;
            for (int j = b; j < e; j++) {
                const uint32_t c = item[j].w[6 + ax];
                mn = min(mn, c);
                mx = max(mx, c);
            }
            const float lo = fromkey(mn), ext = fromkey(mx) - lo;
            const bool on = axis < 3 && li < n && ext > 0.0f;
            int bin = kBins;
            if (on) bin = bin_of(fromkey(item[b + li].w[6 + ax]), lo, (float)kBins / ext);
            s_bin[wv][lane] = bin;
            wave_sync();
            // lane j < n: item j and its bins of the three axes
            const Item v = item[min(b + lane, kSmallItems - 1)];
            const int own = min(lane, kSmallItems - 1);
            const uint32_t bins = (uint32_t)s_bin[wv][own] | (uint32_t)s_bin[wv][kSmallItems + own] << 8 |
                                  (uint32_t)s_bin[wv][2 * kSmallItems + own] << 16;
            uint32_t l[6], r[6];
            int32_t lc = 0, rc = 0;
            for (int q = 0; q < 6; q++) l[q] = r[q] = acc_empty(q);
            for (int j = 0; j < n; j++) {
                uint32_t x[6];
                for (int q = 0; q < 6; q++) x[q] = read_lane(v.w[q], j);
                const int32_t tris = (int32_t)read_lane(v.w[9], j);
                if ((int)((read_lane(bins, j) >> (8 * ax)) & 0xffu) <= bin) {
                    for (int q = 0; q < 6; q++) l[q] = acc_union(q, l[q], x[q]);
                    lc += tris;
                } else {
                    for (int q = 0; q < 6; q++) r[q] = acc_union(q, r[q], x[q]);
                    rc += tris;
                }
            }
            uint32_t key = ~0u;
            if (on && bin < kBins - 1 && lc != 0 && rc != 0) {
                DBox lb, rb;
                for (int q = 0; q < 3; q++) {
                    lb.lo[q] = fromkey(l[q]); lb.hi[q] = fromkey(l[3 + q]);
                    rb.lo[q] = fromkey(r[q]); rb.hi[q] = fromkey(r[3 + q]);
                }
                const float cost = box_area(lb) * (float)lc + box_area(rb) * (float)rc;
                if (cost < __builtin_huge_valf()) key = __float_as_uint(cost);
            }
            const uint32_t best = wave_min_u32(key);
            int w = 0, nl = (t.b + b + t.b + e) / 2 - (t.b + b);
            bool left = lane < nl;
            if (best != ~0u) {
                // the first minimum in (axis, boundary) order
                const uint32_t code = key == best ? (uint32_t)(16 * axis + bin) : ~0u;
                const uint32_t pick = wave_min_u32(code);
                w = __ffsll(__ballot(code == pick)) - 1;
                left = lane < n && s_bin[wv][(int)(pick >> 4) * kSmallItems + min(lane, kSmallItems - 1)] <= (int)(pick & 15u);
                nl = __popcll(__ballot(left));
            } else {
                for (int q = 0; q < 6; q++) l[q] = r[q] = acc_empty(q);
                for (int j = 0; j < n; j++)
                    for (int q = 0; q < 6; q++) {
                        const uint32_t x = read_lane(v.w[q], j);
                        if (j < nl) l[q] = acc_union(q, l[q], x);
                        else r[q] = acc_union(q, r[q], x);
                    }
            }
            const unsigned long long ml = __ballot(left), mr = __ballot(lane < n && !left);
            wave_sync();
            if (lane < n) item[b + (left ? __popcll(ml & below) : nl + __popcll(mr & below))] = v;
            wave_sync();
            const int mid = t.b + b + nl;
            TopRec* rec = B.rec + mid;
            if (lane == w)
                for (int q = 0; q < 6; q++) {
                    rec->box[0][q] = fromkey(l[q]);
                    rec->box[1][q] = fromkey(r[q]);
                }
            const bool li1 = nl == 1, ri1 = n - nl == 1;
            if (lane == 0) {
                B.level[mid - 1] = level_key(f.w);
                if (f.z) B.rec[f.z >> 1].child[f.z & 1] = mid;
                rec->kind[0] = li1 ? kChildRef : kChildNode;
                rec->kind[1] = ri1 ? kChildRef : kChildNode;
                if (li1) rec->child[0] = (int32_t)item[b].w[10];
                if (ri1) rec->child[1] = (int32_t)item[e - 1].w[10];
                const int4 lt = make_int4(b, b + nl, 2 * mid, f.w + 1), rt = make_int4(b + nl, e, 2 * mid + 1, f.w + 1);
                int at = sp, pat = pairs;
                if (n - nl == 2) s_pair[wv][pat++] = rt;
                else if (!ri1) s_stack[wv][at++] = rt;
                if (nl == 2) s_pair[wv][pat++] = lt;
                else if (!li1) s_stack[wv][at++] = lt;
            }
            sp += (nl > 2 ? 1 : 0) + (n - nl > 2 ? 1 : 0);
            pairs += (nl == 2 ? 1 : 0) + (n - nl == 2 ? 1 : 0);
            wave_sync();
        }
        // The nodes of two items, one lane each: every boundary costs the same,
        // so the first axis whose bins differ splits them, in bin order.
        if (lane < pairs) {
            const int4 f = s_pair[wv][lane];
            const Item v0 = item[f.x], v1 = item[f.x + 1];
            bool split = false, swap = false;
            for (int a = 0; a < 3; a++) {
                const float c0 = fromkey(v0.w[6 + a]), c1 = fromkey(v1.w[6 + a]);
                const float lo = fromkey(min(v0.w[6 + a], v1.w[6 + a]));
                const float ext = fromkey(max(v0.w[6 + a], v1.w[6 + a])) - lo;
                if (split || !(ext > 0.0f)) continue;
                const float scale = (float)kBins / ext;
                const int b0 = bin_of(c0, lo, scale), b1 = bin_of(c1, lo, scale);
                split = b0 != b1;
                swap = b1 < b0;
            }
            DBox x0, x1;
            for (int q = 0; q < 3; q++) {
                x0.lo[q] = fromkey(v0.w[q]); x0.hi[q] = fromkey(v0.w[3 + q]);
                x1.lo[q] = fromkey(v1.w[q]); x1.hi[q] = fromkey(v1.w[3 + q]);
            }
            const float cost = box_area(x0) * (float)(int32_t)v0.w[9] + box_area(x1) * (float)(int32_t)v1.w[9];
            swap = swap && cost < __builtin_huge_valf();       // else the items keep their order
            const int mid = t.b + f.x + 1;
            TopRec rec;
            for (int q = 0; q < 3; q++) {
                rec.box[0][q] = swap ? x1.lo[q] : x0.lo[q];
                rec.box[0][3 + q] = swap ? x1.hi[q] : x0.hi[q];
                rec.box[1][q] = swap ? x0.lo[q] : x1.lo[q];
                rec.box[1][3 + q] = swap ? x0.hi[q] : x1.hi[q];
            }
            rec.child[0] = (int32_t)(swap ? v1.w[10] : v0.w[10]);
            rec.child[1] = (int32_t)(swap ? v0.w[10] : v1.w[10]);
            rec.kind[0] = rec.kind[1] = kChildRef;
            B.rec[mid] = rec;
            B.level[mid - 1] = level_key(f.w);
            if (f.z) B.rec[f.z >> 1].child[f.z & 1] = mid;
        }
    }
}

// Chunks of a wide level: s_first[t] .. s_first[t + 1] are slot t's (at most 256 slots).  Returns their number.
SRT_D int wide_chunks(int ntask, const TopTask* task, int32_t* s_first) {
    __shared__ int32_t s_w[4];
    const int t = threadIdx.x;
    const int v = t < ntask ? (task[t].e - task[t].b + kWideChunk - 1) / kWideChunk : 0;
    s_first[t + 1] = block_scan256(v, s_w);
    if (t == 0) s_first[0] = 0;
    __syncthreads();
    return s_first[ntask];
}
SRT_D int wide_slot_of(const int32_t* s_first, int g) {
    int lo = 0, hi = 255;                 // the slot with s_first[slot] <= g < s_first[slot + 1]
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (g < s_first[mid + 1]) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}
static_assert((1 << (kWideLevels - 1)) <= 256 && kTopWaves == 4, "a wide level's slots are scanned by one workgroup");
__global__ void __launch_bounds__(64 * kTopWaves) k_top_wide_bins(TopBuild B, int L) {
    __shared__ int32_t s_first[257];
    __shared__ alignas(16) uint32_t s_bins[kAccTotal * kBlockCopies];
    const int tid = threadIdx.x, wv = tid >> 6, g = blockIdx.x;
    const TopTask* task = B.wide[L & 1];
    if (g >= wide_chunks(1 << L, task, s_first)) return;
    const int t = wide_slot_of(s_first, g);
    const TopTask tk = task[t];
    const int b = tk.b + (g - s_first[t]) * kWideChunk, e = min(b + kWideChunk, tk.e);
    constexpr int kPart = kWideChunk / kTopWaves;
    bins_clear<kBlockCopies>(s_bins, tid, 64 * kTopWaves);
    __syncthreads();
    const int wb = min(b + wv * kPart, e);
    bins_add<kBlockCopies>(B.it[L & 1], wb, min(wb + kPart, e), tk.cb, s_bins);
    __syncthreads();
    uint32_t* out = B.acc + ((size_t)t * kWideCopies + g % kWideCopies) * kAccTotal;
    for (int j = tid; j < kAccTotal; j += 64 * kTopWaves) {
        const int q = j / 48, l = j % 48;
        const uint32_t v = bins_word<kBlockCopies>(s_bins, q, l);
        if (q == 13) B.chunk_items[(size_t)g * 48 + l] = (int32_t)v;
        if (v == acc_empty(q)) continue;
        if (q >= 12) atomicAdd(out + j, v);
        else if (q % 6 < 3) atomicMin(out + j, v);
        else atomicMax(out + j, v);
    }
}
// workgroup (one wave) t: the split of slot t, its children, and its accumulators empty again
__global__ void __launch_bounds__(64) k_top_wide_sah(TopBuild B, int L) {
    const int t = blockIdx.x, lane = threadIdx.x;
    const TopTask tk = B.wide[L & 1][t];
    const bool more = L + 1 < B.wide_levels;
    if (more && lane < 2) {
        TopTask* c = B.wide[(L + 1) & 1] + 2 * t + lane;
        c->b = c->e = 0;
    }
    if (tk.e <= tk.b) return;
    __syncthreads();                      // the children below replace the empty slots
    uint32_t acc[kAccWords];
    for (int q = 0; q < kAccWords; q++) acc[q] = acc_empty(q);
    if (lane < 48)
        for (int c = 0; c < kWideCopies; c++) {
            uint32_t* p = B.acc + ((size_t)t * kWideCopies + c) * kAccTotal + lane;
            for (int q = 0; q < kAccWords; q++) {
                acc[q] = acc_union(q, acc[q], p[q * 48]);
                p[q * 48] = acc_empty(q);
            }
        }
    uint32_t side[2][kAccWords];
    const int w = sah_choose_wave(acc, tk.cb, side);
    const Items& src = B.it[L & 1];
    int mid = (tk.b + tk.e) / 2;
    WideSplit s = {-1, 0, mid, 0.0f, 0.0f};
    if (w >= 0) {
        mid = tk.b + (int)side[0][13];
        const int axis = w >> 4;
        const float lo = fromkey(axis == 0 ? tk.cb[0] : (axis == 1 ? tk.cb[1] : tk.cb[2]));
        const float ext = fromkey(axis == 0 ? tk.cb[3] : (axis == 1 ? tk.cb[4] : tk.cb[5])) - lo;
        s = {axis, w & 15, mid, lo, (float)kBins / ext};
    } else {
        union_items(src, tk.b, mid, side[0]);
        union_items(src, mid, tk.e, side[1]);
    }
    if (lane == 0) {
        uint32_t sd[2][12];
        for (int q = 0; q < 12; q++) {
            sd[0][q] = side[0][q];
            sd[1][q] = side[1][q];
        }
        B.wsplit[t] = s;
        top_node(B, L, tk, mid, sd, more ? 2 * t : -1);
    }
}
__global__ void __launch_bounds__(64 * kTopWaves) k_top_wide_scatter(TopBuild B, int L) {
    __shared__ int32_t s_first[257];
    __shared__ int32_t s_left[kTopWaves], s_before[kTopWaves];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = blockIdx.x;
    const TopTask* task = B.wide[L & 1];
    if (g >= wide_chunks(1 << L, task, s_first)) return;
    const int t = wide_slot_of(s_first, g), f = s_first[t];
    const int tb = task[t].b, b = tb + (g - f) * kWideChunk, e = min(b + kWideChunk, task[t].e);
    const WideSplit s = B.wsplit[t];
    const Items &src = B.it[L & 1], &dst = B.it[(L + 1) & 1];
    if (s.axis < 0) {
        for (int i = b + tid; i < e; i += 64 * kTopWaves) copy_item(src, i, dst, i);
        return;
    }
    // left items of the node's chunks before this one, and of the waves' parts of it
    int32_t before = 0;
    for (int j = tid; j < (g - f) * 16; j += 64 * kTopWaves)
        if ((j & 15) <= s.split) before += B.chunk_items[(size_t)(f + (j >> 4)) * 48 + 16 * s.axis + (j & 15)];
    for (int d = 32; d > 0; d >>= 1) before += __shfl_xor(before, d);
    constexpr int kPart = kWideChunk / kTopWaves;
    const int wb = min(b + wv * kPart, e), we = min(wb + kPart, e);
    int32_t left = 0;
    for (int i = wb + lane; i < we; i += 64) left += bin_of(item_c(src, s.axis, i), s.lo, s.scale) <= s.split ? 1 : 0;
    for (int d = 32; d > 0; d >>= 1) left += __shfl_xor(left, d);
    if (lane == 0) {
        s_left[wv] = left;
        s_before[wv] = before;
    }
    __syncthreads();
    int l = 0;
    for (int w = 0; w < kTopWaves; w++) l += s_before[w] + (w < wv ? s_left[w] : 0);
    partition_items(src, dst, wb, we, s.axis, s.lo, s.scale, s.split, tb + l, s.mid + (wb - tb) - l);
}

// empty lists, counters and accumulators (slots: middle slots; words: of the wide accumulators)
__global__ void __launch_bounds__(256) k_top_clear(TopBuild B, int slots, int words) {
    const int i0 = blockIdx.x * 256 + threadIdx.x, stride = gridDim.x * 256;
    for (int i = i0; i < 2 * slots; i += stride) {
        TopTask* t = B.mid[i >= slots ? 1 : 0] + (i >= slots ? i - slots : i);
        t->b = t->e = 0;
    }
    for (int i = i0; i < kRegions * 64; i += stride) B.nsmall[i] = 0;
    for (int i = i0; i < kLevels; i += stride) B.any[i] = 0;
    for (int i = i0; i < 6; i += stride) B.cb[i] = acc_empty(i);
    for (int i = i0; i < words; i += stride) B.acc[i] = acc_empty(i / 48 % kAccWords);
}
// centroid bounds of all items
__global__ void __launch_bounds__(256) k_top_bounds(TopBuild B) {
    __shared__ uint32_t s_cb[4][6];
    uint32_t v[6];
    for (int q = 0; q < 6; q++) v[q] = acc_empty(q);
    for (int i = blockIdx.x * 256 + threadIdx.x; i < B.m; i += gridDim.x * 256)
        for (int a = 0; a < 3; a++) {
            const uint32_t c = fkey(item_c(B.it[0], a, i));
            v[a] = min(v[a], c);
            v[3 + a] = max(v[3 + a], c);
        }
    for (int q = 0; q < 6; q++) {
        for (int d = 32; d > 0; d >>= 1) v[q] = acc_union(q, v[q], (uint32_t)__shfl_xor((int)v[q], d));
        if ((threadIdx.x & 63) == 0) s_cb[threadIdx.x >> 6][q] = v[q];
    }
    __syncthreads();
    const int q = threadIdx.x;
    if (q < 6) {
        uint32_t x = s_cb[0][q];
        for (int w = 1; w < 4; w++) x = acc_union(q, x, s_cb[w][q]);
        if (q < 3) atomicMin(B.cb + q, x);
        else atomicMax(B.cb + q, x);
    }
}
__global__ void k_top_root(TopBuild B) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    TopTask t;
    t.b = 0; t.e = B.m; t.up = 0;
    for (int q = 0; q < 6; q++) t.cb[q] = B.cb[q];
    if (B.wide_levels > 0) {
        B.wide[0][0] = t;
    } else if (B.m > kSmallItems) {
        B.mid[0][mid_slot(0)] = t;
    } else {
        B.small[0] = {0, B.m, 0, 0};
        B.nsmall[0] = 1;
    }
}
// node r: the r-th boundary in (level, boundary) order
__global__ void __launch_bounds__(256) k_top_write(TopBuild B, const uint32_t* ids, const int32_t* number, BvhNode* nodes) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= B.m - 1) return;
    const TopRec rec = B.rec[ids[r] + 1];
    for (int side = 0; side < 2; side++) {
        DBox bx;
        for (int k = 0; k < 3; k++) { bx.lo[k] = rec.box[side][k]; bx.hi[k] = rec.box[side][3 + k]; }
        const int32_t c = rec.child[side], kind = rec.kind[side];
        int32_t ref = c;
        if (kind == kChildNode) ref = number[c - 1];
        else if (kind >= kChildItem) ref = kind == kChildItem ? B.it[0].ref[c] : B.it[1].ref[c];
        set_child(nodes + r, side, bx, ref);
    }
}

// ---------------------------------------------------------------------------
// 7. emit the Karras nodes that remain, triangles, parents, depth
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_emit(int n, int T, int top, int max_leaf, const int32_t* kl, const int32_t* kr,
                                              const int32_t* kfirst, const int32_t* par_int, const uint32_t* order, BoxArr tb,
                                              KArr K, BvhNode* nodes, int32_t* valid) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    if (K.count[i] > T || K.collapse[i]) return;
    for (int p = par_int[i]; p >= 0 && K.count[p] <= max_leaf; p = par_int[p])
        if (K.collapse[p]) return;
    BvhNode* nd = nodes + top + i;
    int32_t ch[2] = {kl[i], kr[i]};
    for (int side = 0; side < 2; side++) {
        int32_t c = ch[side];
        DBox b;
        int32_t ref;
        if (c < 0) { int k = -c - 1; b = ldbox(tb, order[k]); ref = leaf_ref((uint32_t)k, 1u); }
        else {
            b = ldbox(K.box, c);
            ref = K.collapse[c] ? leaf_ref((uint32_t)kfirst[c], (uint32_t)K.count[c]) : top + c;
        }
        set_child(nd, side, b, ref);
    }
    valid[top + i] = 1;
}

// Sorted triangle records for the traversal and the 128-byte shading records
// of the same triangles (positions, material, vertex normals and tangents),
// rewritten after every skinning step.
struct TriSrc {
    const float *pos, *nrm, *tan;
    const uint32_t* idx;
    const int32_t *tri_mesh, *mesh_mat;
};
__global__ void __launch_bounds__(256) k_tris(int n, const uint32_t* order, TriSrc src, float4* tris, float4* rec) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    uint32_t p = order[k];
    const uint32_t* ix = src.idx + 3 * (size_t)p;
    const float* a = src.pos + 3 * (size_t)ix[0];
    const float* b = src.pos + 3 * (size_t)ix[1];
    const float* c = src.pos + 3 * (size_t)ix[2];
    const int32_t mesh = src.tri_mesh[p];
    const int32_t mat = src.mesh_mat[mesh];
    tris[3 * (size_t)k + 0] = make_float4(a[0], a[1], a[2], __uint_as_float(p));
    tris[3 * (size_t)k + 1] = make_float4(b[0], b[1], b[2], __int_as_float(mesh));
    tris[3 * (size_t)k + 2] = make_float4(c[0], c[1], c[2], __int_as_float(mat));
    // shading record (layout at DevScene::tri_rec)
    float nv[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, t[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int v = 0; v < 3; v++) {
        for (int j = 0; j < 3; j++) {
            if (src.nrm) nv[3 * v + j] = src.nrm[3 * (size_t)ix[v] + j];
            if (src.tan) t[3 * v + j] = src.tan[3 * (size_t)ix[v] + j];
        }
    }
    float4* r = rec + 8 * (size_t)k;
    r[0] = make_float4(a[0], a[1], a[2], __int_as_float(mat));
    r[1] = make_float4(b[0], b[1], b[2], nv[0]);
    r[2] = make_float4(c[0], c[1], c[2], nv[1]);
    r[3] = make_float4(nv[2], nv[3], nv[4], nv[5]);
    r[4] = make_float4(nv[6], nv[7], nv[8], t[0]);
    r[5] = make_float4(t[1], t[2], t[3], t[4]);
    r[6] = make_float4(t[5], t[6], t[7], t[8]);
    r[7] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}
static void launch_tris(SceneRec* s, hipStream_t st) {
    TriSrc src;
    src.pos = (const float*)s->pos.p;
    src.nrm = s->has_nrm ? (const float*)s->nrm.p : nullptr;
    src.tan = s->has_tan ? (const float*)s->tan.p : nullptr;
    src.idx = (const uint32_t*)s->idx.p;
    src.tri_mesh = (const int32_t*)s->tri_mesh.p;
    src.mesh_mat = (const int32_t*)s->mesh_mat.p;
    const int n = s->nf;
    k_tris<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(n, (const uint32_t*)s->order.p, src, (float4*)s->tris.p,
                                                        (float4*)s->tri_rec.p);
}

// parents in the final tree: parent index * 2 + side, -1 for the root
__global__ void __launch_bounds__(256) k_final_parents(int num_nodes, const BvhNode* nodes, const int32_t* valid, int32_t* parent) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_nodes || !valid[i]) return;
    int4 d = nodes[i].d;
    if (d.x >= 0) parent[d.x] = 2 * i;
    if (d.y >= 0) parent[d.y] = 2 * i + 1;
}

// ---------------------------------------------------------------------------
// refit: leaf boxes from the current triangles, then boxes bottom-up
// ---------------------------------------------------------------------------
SRT_D DBox leaf_box(const float4* tris, int32_t ref) {
    DBox b = empty_box();
    uint32_t f = leaf_first(ref), c = leaf_count(ref);
    for (uint32_t k = f; k < f + c; k++)
        for (int v = 0; v < 3; v++) {
            float4 p = tris[3 * (size_t)k + v];
            b.lo[0] = kmin(b.lo[0], p.x); b.hi[0] = kmax(b.hi[0], p.x);
            b.lo[1] = kmin(b.lo[1], p.y); b.hi[1] = kmax(b.hi[1], p.y);
            b.lo[2] = kmin(b.lo[2], p.z); b.hi[2] = kmax(b.hi[2], p.z);
        }
    return b;
}
SRT_D DBox node_union(const BvhNode* nd) {
    DBox l, r;
    float4 a = nd->a, b = nd->b, c = nd->c;
    l.lo[0] = a.x; l.hi[0] = a.y; l.lo[1] = a.z; l.hi[1] = a.w; l.lo[2] = c.x; l.hi[2] = c.y;
    r.lo[0] = b.x; r.hi[0] = b.y; r.lo[1] = b.z; r.hi[1] = b.w; r.lo[2] = c.z; r.hi[2] = c.w;
    grow(l, r);
    return l;
}
// Level of every binary-tree node (root = 0; kLevelNone for unused slots)
__global__ void __launch_bounds__(256) k_node_level(int num_nodes, const int32_t* valid, const int32_t* parent,
                                                    uint8_t* key) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= num_nodes) return;
    if (!valid[i]) {
        key[i] = (uint8_t)kLevelNone;
        return;
    }
    int level = 0;
    for (int p = parent[i]; p >= 0; p = parent[p >> 1]) level++;
    key[i] = level_key(level);
}
// One level of the bottom-up refit (deepest level first): each node takes its
// leaf children's boxes from the current triangles and its inner children's
// boxes as the union of their two child boxes, written by the previous launch.
// Kernel boundaries order the levels, so no device-wide fences are needed.
SRT_D void refit_node(int p, BvhNode* nodes, const float4* tris) {
    BvhNode* nd = nodes + p;
    const int4 d = nd->d;
    const DBox l = d.x < 0 ? leaf_box(tris, d.x) : node_union(nodes + d.x);
    const DBox r = d.y < 0 ? leaf_box(tris, d.y) : node_union(nodes + d.y);
    set_child(nd, 0, l, d.x);
    set_child(nd, 1, r, d.y);
}
__global__ void __launch_bounds__(256) k_refit_level(const uint32_t* ids, int count, BvhNode* nodes,
                                                     const float4* tris) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < count) refit_node((int)ids[k], nodes, tris);
}
__global__ void __launch_bounds__(kRunNodes) k_refit_run(LevelRun run, const uint32_t* ids, BvhNode* nodes,
                                                         const float4* tris) {
    run_levels(run, ids, [&](int p) { refit_node(p, nodes, tris); });
}

// ---------------------------------------------------------------------------
// 4-wide tree collapsed from the binary tree.  The binary leaves stay leaves;
// which binary inner nodes become 4-wide nodes is chosen by a bottom-up
// dynamic program that minimises the summed surface area of the 4-wide nodes
// (the surface-area estimate of the node steps of a traversal; the leaves'
// triangle tests do not depend on the choice).  Per binary inner node x:
//   W(x)    = area(x) + G(x, 4)    x as a 4-wide node
//   G(x, k) = min over j in 1..k-1 of H(l, j) + H(r, k - j)
//   H(c, j) = 0 for a leaf, W(c) for j = 1, min(W(c), G(c, j)) for j > 1
// (H(c, j): subtree c in at most j child slots, c kept as one slot or opened).
// The 4-wide nodes are then emitted top-down by levels following the stored
// choices (ties keep a child whole, and give the left child the fewest
// slots).  Nodes are numbered level by level in order (deterministic); boxes
// are copies of binary-tree boxes, so both trees give every ray the same box
// tests.
// ---------------------------------------------------------------------------
SRT_D DBox child_box(const BvhNode& nd, int side) {
    DBox b;
    if (side == 0) {
        b.lo[0] = nd.a.x; b.hi[0] = nd.a.y; b.lo[1] = nd.a.z; b.hi[1] = nd.a.w; b.lo[2] = nd.c.x; b.hi[2] = nd.c.y;
    } else {
        b.lo[0] = nd.b.x; b.hi[0] = nd.b.y; b.lo[1] = nd.b.z; b.hi[1] = nd.b.w; b.lo[2] = nd.c.z; b.hi[2] = nd.c.w;
    }
    return b;
}
struct Kids4 {
    int32_t ref[4], src[4];
    int n;
};
// dynamic-program tables per binary inner node: W, G(k) for k = 2, 3, 4, and
// the slots given to the left child for each k (2 bits each)
struct C4Dp {
    float* W;
    float* G;            // 3 per node
    uint32_t* J;         // bits 2(k-2) .. 2(k-2)+1: left slots for k
};
SRT_D float c4_H(const C4Dp& dp, int32_t c, int j) {
    if (c < 0) return 0.0f;
    const float w = dp.W[c];
    if (j == 1) return w;
    const float g = dp.G[3 * (size_t)c + (j - 2)];
    return g < w ? g : w;
}
SRT_D void c4_dp_node(int x, const BvhNode* nodes, const C4Dp& dp) {
    const BvhNode nd = nodes[x];
    DBox b = child_box(nd, 0);
    grow(b, child_box(nd, 1));
    const int32_t l = nd.d.x, r = nd.d.y;
    uint32_t jbits = 0;
    float g4 = 0.0f;
    for (int k = 2; k <= 4; k++) {
        float best = __builtin_huge_valf();
        int bj = 1;
        for (int j = 1; j < k; j++) {
            const float v = c4_H(dp, l, j) + c4_H(dp, r, k - j);
            if (v < best) { best = v; bj = j; }
        }
        dp.G[3 * (size_t)x + (k - 2)] = best;
        jbits |= (uint32_t)bj << (2 * (k - 2));
        if (k == 4) g4 = best;
    }
    dp.J[x] = jbits;
    dp.W[x] = box_area(b) + g4;
}
__global__ void __launch_bounds__(256) k_c4_dp(const uint32_t* ids, int count, const BvhNode* nodes, C4Dp dp) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) c4_dp_node((int)ids[i], nodes, dp);
}
__global__ void __launch_bounds__(kRunNodes) k_c4_dp_run(LevelRun run, const uint32_t* ids, const BvhNode* nodes, C4Dp dp) {
    run_levels(run, ids, [&](int x) { c4_dp_node(x, nodes, dp); });
}
// children of the 4-wide node made from binary node x: subtree (c, j) is kept
// as one slot when c is a leaf, j == 1 or opening it is not cheaper, else
// opened into its children with the stored split of j slots
SRT_D Kids4 collapse_children(const BvhNode* nodes, int32_t x, const C4Dp& dp) {
    Kids4 k;
    k.n = 0;
    for (int j = 0; j < 4; j++) { k.ref[j] = 0; k.src[j] = -1; }
    int32_t st_ref[4], st_src[4], st_j[4];
    int sp = 0;
    const BvhNode nd = nodes[x];
    const int jl = min(max((int)(dp.J[x] >> 4) & 3, 1), 3);      // k = 4; every split gives each side a slot
    st_ref[sp] = nd.d.y; st_src[sp] = (x << 1) | 1; st_j[sp] = 4 - jl; sp++;
    st_ref[sp] = nd.d.x; st_src[sp] = x << 1; st_j[sp] = jl; sp++;
    while (sp > 0) {
        sp--;
        const int32_t c = st_ref[sp], src = st_src[sp];
        const int j = st_j[sp];
        const bool open = c >= 0 && j > 1 && dp.G[3 * (size_t)c + (j - 2)] < dp.W[c];
        if (!open) {
            k.ref[k.n] = c;
            k.src[k.n] = src;
            k.n++;
            continue;
        }
        const BvhNode nc = nodes[c];
        const int cl = min(max((int)(dp.J[c] >> (2 * (j - 2))) & 3, 1), j - 1);
        st_ref[sp] = nc.d.y; st_src[sp] = (c << 1) | 1; st_j[sp] = j - cl; sp++;
        st_ref[sp] = nc.d.x; st_src[sp] = c << 1; st_j[sp] = cl; sp++;
    }
    // slots by decreasing box area (stable): any-hit traversals visit the hit
    // children in slot order, the likeliest to hold an occluder first
    float area[4];
    for (int j = 0; j < k.n; j++) area[j] = box_area(child_box(nodes[k.src[j] >> 1], k.src[j] & 1));
    for (int a = 1; a < k.n; a++)
        for (int b = a; b > 0 && area[b] > area[b - 1]; b--) {
            const float ta = area[b]; area[b] = area[b - 1]; area[b - 1] = ta;
            const int32_t tr = k.ref[b]; k.ref[b] = k.ref[b - 1]; k.ref[b - 1] = tr;
            const int32_t ts = k.src[b]; k.src[b] = k.src[b - 1]; k.src[b - 1] = ts;
        }
    return k;
}
// One level of the collapse is two launches that take its size from the device,
// so the levels follow each other without the host: k_c4_count gives workgroup
// g the g-th piece of the level and counts the inner children of its nodes
// (exclusive within the piece, and the piece's sum), k_c4_emit adds the sums of
// the pieces before its own, so the next level is numbered in order.
// sizes[L]: nodes of level L; bases[L]: their first number.  16 levels of the
// 1M-triangle field took 1.3 ms with a library scan, two copies and a wait for
// each, now 0.5 ms; bound by the chains of reads through the binary nodes.
constexpr int kC4Grid = 256;            // pieces of a level: a workgroup per CU, one read of the sums per thread
SRT_D int c4_piece(int nf) { return (nf + (int)gridDim.x * 256 - 1) / ((int)gridDim.x * 256) * 256; }
__global__ void __launch_bounds__(256) k_c4_count(int L, const int32_t* sizes, const int32_t* level, const BvhNode* nodes,
                                                  C4Dp dp, int32_t* off, int32_t* sums) {
    __shared__ int32_t s_w[4];
    __shared__ int32_t s_last;
    const int tid = threadIdx.x, nf = sizes[L], piece = c4_piece(nf);
    const int b = blockIdx.x * piece, e = min(b + piece, nf);
    int32_t run = 0;
    for (int start = b; start < e; start += 256) {
        const int i = start + tid;
        int32_t m = 0;
        if (i < e) {
            const Kids4 k = collapse_children(nodes, level[i], dp);
            for (int j = 0; j < k.n; j++) m += (k.ref[j] >= 0) ? 1 : 0;
        }
        const int32_t incl = block_scan256(m, s_w);
        if (i < e) off[i] = run + incl - m;
        if (tid == 255) s_last = incl;
        __syncthreads();
        run += s_last;
    }
    if (tid == 0) sums[blockIdx.x] = run;
}
SRT_D void set4(Bvh4Node& o, int j, const DBox& b) {
    float* lx = &o.lox.x; float* hx = &o.hix.x; float* ly = &o.loy.x; float* hy = &o.hiy.x;
    float* lz = &o.loz.x; float* hz = &o.hiz.x;
    lx[j] = b.lo[0]; hx[j] = b.hi[0]; ly[j] = b.lo[1]; hy[j] = b.hi[1]; lz[j] = b.lo[2]; hz[j] = b.hi[2];
}
SRT_D void c4_node(const BvhNode* nodes, const Kids4& k, int32_t q, int32_t base_next, Bvh4Node* out,
                   int32_t* next_level) {
    Bvh4Node o;
    int32_t* ref = &o.ref.x;
    int32_t* src = &o.src.x;
    DBox empty;
    empty.lo[0] = empty.lo[1] = empty.lo[2] = __builtin_huge_valf();
    empty.hi[0] = empty.hi[1] = empty.hi[2] = -__builtin_huge_valf();
    for (int j = 0; j < 4; j++) {
        if (j < k.n) {
            const int32_t sx = k.src[j];
            set4(o, j, child_box(nodes[sx >> 1], sx & 1));
            src[j] = sx;
            if (k.ref[j] >= 0) {
                next_level[q] = k.ref[j];
                ref[j] = base_next + q;
                q++;
            } else {
                ref[j] = k.ref[j];
            }
        } else {
            set4(o, j, empty);
            src[j] = -1;
            ref[j] = 0;
        }
    }
    *out = o;
}
__global__ void __launch_bounds__(256) k_c4_emit(int L, int32_t* sizes, int32_t* bases, const int32_t* level,
                                                 const BvhNode* nodes, C4Dp dp, const int32_t* off, const int32_t* sums,
                                                 Bvh4Node* out, int32_t* next_level) {
    __shared__ int32_t s_before[4], s_all[4];
    const int tid = threadIdx.x, nf = sizes[L], base = bases[L], piece = c4_piece(nf);
    int32_t before = 0, all = 0;
    for (int g = tid; g < (int)gridDim.x; g += 256) {
        const int32_t v = sums[g];
        all += v;
        before += g < (int)blockIdx.x ? v : 0;
    }
    for (int d = 32; d > 0; d >>= 1) {
        all += __shfl_xor(all, d);
        before += __shfl_xor(before, d);
    }
    if ((tid & 63) == 0) {
        s_all[tid >> 6] = all;
        s_before[tid >> 6] = before;
    }
    __syncthreads();
    if (blockIdx.x == 0 && tid == 0) {
        sizes[L + 1] = s_all[0] + s_all[1] + s_all[2] + s_all[3];
        bases[L + 1] = base + nf;
    }
    before = s_before[0] + s_before[1] + s_before[2] + s_before[3];
    const int b = blockIdx.x * piece, e = min(b + piece, nf);
    for (int i = b + tid; i < e; i += 256)
        c4_node(nodes, collapse_children(nodes, level[i], dp), before + off[i], base + nf, out + base + i, next_level);
}
// after a binary-tree refit: each wide child box is copied from its binary slot again
__global__ void __launch_bounds__(256) k_refit4(int n4, const BvhNode* nodes, Bvh4Node* nodes4) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n4) return;
    Bvh4Node o = nodes4[i];
    const int32_t* src = &o.src.x;
    for (int j = 0; j < 4; j++)
        if (src[j] >= 0) set4(o, j, child_box(nodes[src[j] >> 1], src[j] & 1));
    nodes4[i] = o;
}

// the radix root's triangle count, collapse decision and first triangle, and the number of clusters, for one copy
// (four copies and two waits took 0.1 ms of a 1M-triangle rebuild's 3.0)
__global__ void k_build_facts(KArr K, const int32_t* kfirst, const int32_t* nsel, int32_t* out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    out[0] = K.count[0];
    out[1] = K.collapse[0];
    out[2] = kfirst[0];
    out[3] = nsel ? *nsel : 1;
}

__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// scene.cu:362-392: skinned position / normal / tangent from up to 4 bones
__global__ void __launch_bounds__(256) k_skin(int nv, const float* op, const float* on, const float* ot, const int32_t* bid,
                                              const float* bw, int nb, const float* bones, float* pos, float* nrm, float* tan) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nv) return;
    f3 v = mk(0.0f), nn = mk(0.0f), tt = mk(0.0f);
    f3 ov = ld3(op + 3 * (size_t)i);
    f3 onn = on ? ld3(on + 3 * (size_t)i) : mk(0.0f);
    f3 ott = ot ? ld3(ot + 3 * (size_t)i) : mk(0.0f);
    for (int j = 0; j < 4; j++) {
        int id = bid[4 * (size_t)i + j];
        float w = bw[4 * (size_t)i + j];
        if (id == -1) {
            if (j == 0) { v = ov; nn = onn; tt = ott; }
            break;
        }
        if (id >= nb) continue;
        const float* m = bones + 12 * (size_t)id;
        f3 pp = mk(m[0] * ov.x + m[1] * ov.y + m[2] * ov.z + m[3], m[4] * ov.x + m[5] * ov.y + m[6] * ov.z + m[7],
                   m[8] * ov.x + m[9] * ov.y + m[10] * ov.z + m[11]);
        v = v + pp * w;
        f3 pn = mk(m[0] * onn.x + m[1] * onn.y + m[2] * onn.z, m[4] * onn.x + m[5] * onn.y + m[6] * onn.z,
                   m[8] * onn.x + m[9] * onn.y + m[10] * onn.z);
        nn = nn + pn * w;
        f3 pt = mk(m[0] * ott.x + m[1] * ott.y + m[2] * ott.z, m[4] * ott.x + m[5] * ott.y + m[6] * ott.z,
                   m[8] * ott.x + m[9] * ott.y + m[10] * ott.z);
        tt = tt + pt * w;
    }
    pos[3 * (size_t)i] = v.x; pos[3 * (size_t)i + 1] = v.y; pos[3 * (size_t)i + 2] = v.z;
    if (nrm) { nrm[3 * (size_t)i] = nn.x; nrm[3 * (size_t)i + 1] = nn.y; nrm[3 * (size_t)i + 2] = nn.z; }
    if (tan) { tan[3 * (size_t)i] = tt.x; tan[3 * (size_t)i + 1] = tt.y; tan[3 * (size_t)i + 2] = tt.z; }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {
// Build scratch: 256-byte aligned slices bumped out of 16 MiB (or larger)
// device chunks.  The chunks go back to the context when the build ends and
// the next build takes them again (the smallest kept chunk that fits), so a
// rebuild of the same scene calls neither hipMalloc nor hipFree: each hipFree
// of a chunk cost about 0.25 ms of host time, 18 chunks for a 1M-triangle
// rebuild.  Kernels of a build still queued when its chunks go back are
// ordered before the next build's by the context's stream.
struct Tmp {
    static constexpr size_t kChunk = (size_t)16 << 20;
    srt_ctx* c;
    std::vector<DevBuf> chunks;
    size_t used = 0, cap = 0;      // of the last chunk
    bool failed = false;           // some get() returned nullptr
    explicit Tmp(srt_ctx* cc) : c(cc) {}
    ~Tmp() {
        if (!c->keep_build_scratch) {
            for (auto& b : chunks) dev_free(c, b);
            return;
        }
        std::lock_guard<std::mutex> g(c->scratch_mu);
        for (auto& b : chunks) c->build_scratch.push_back(b);
    }
    bool take_kept(size_t size, DevBuf& out) {
        std::lock_guard<std::mutex> g(c->scratch_mu);
        auto& kept = c->build_scratch;
        int best = -1;
        for (int i = 0; i < (int)kept.size(); i++)
            if (kept[i].bytes >= size && (best < 0 || kept[i].bytes < kept[best].bytes)) best = i;
        if (best < 0) return false;
        out = kept[best];
        kept.erase(kept.begin() + best);
        return true;
    }
    template <class T> T* get(size_t count) {
        const size_t bytes = (std::max<size_t>(count, 1) * sizeof(T) + 255) & ~(size_t)255;
        if (chunks.empty() || used + bytes > cap) {
            DevBuf b;
            const size_t size = std::max(bytes, kChunk);
            if (!take_kept(size, b) && dev_alloc(c, b, size)) {
                failed = true;
                return nullptr;
            }
            chunks.push_back(b);
            used = 0;
            cap = b.bytes;
        }
        T* p = (T*)((char*)chunks.back().p + used);
        used += bytes;
        return p;
    }
};
inline unsigned nblk(int64_t n, int b = 256) { return (unsigned)std::max<int64_t>(1, (n + b - 1) / b); }
// The levels 0 .. levels - 1 that start at `first`, deepest first: `level(L)` for one of many nodes, `run(r)` for
// consecutive ones of few.
template <class Level, class Run> void by_levels(const int32_t* first, int levels, Level&& level, Run&& run) {
    LevelRun r;
    r.levels = 0;
    for (int L = levels - 1; L >= 0; L--) {
        const bool few = first[L + 1] - first[L] <= kRunNodes;
        if (few) {
            r.first[r.levels] = first[L];
            r.end[r.levels] = first[L + 1];
            r.levels++;
        }
        if (r.levels > 0 && (!few || L == 0 || r.levels == kRunLevels)) {
            run(r);
            r.levels = 0;
        }
        if (!few) level(L);
    }
}
// node ids of `n` keyed nodes in level order; `number` (or null) the nodes' positions, `first` (or null) the levels'
// first positions on the host (kLevels + 1), for which it waits
int order_levels(srt_ctx* c, Tmp& tmp, int n, const uint8_t* key, uint32_t* ids, int32_t* number,
                 std::vector<int32_t>* first) {
    const int pieces = (int)nblk(n, kLevelPiece);
    int32_t* hist = tmp.get<int32_t>((size_t)kLevels * pieces);
    int32_t* size = tmp.get<int32_t>(kLevels);
    int32_t* dfirst = tmp.get<int32_t>(kLevels + 1);
    if (tmp.failed) return set_err(c, SRT_E_OOM, "level scratch");
    hipStream_t st = c->stream;
    k_level_hist<<<pieces, 256, 0, st>>>(n, key, pieces, hist);
    k_level_scan<<<kLevels, 256, 0, st>>>(pieces, hist, size);
    k_level_rank<<<pieces, 256, 0, st>>>(n, key, pieces, hist, size, ids, number, dfirst);
    if (!first) return SRT_OK;
    first->resize(kLevels + 1);
    if (int r = hip_check(c, hipMemcpyAsync(first->data(), dfirst, 4 * first->size(), hipMemcpyDeviceToHost, st), "copy"))
        return r;
    return hip_check(c, hipStreamSynchronize(st), "level order");
}
}  // namespace

int bvh_build(srt_ctx* c, SceneRec* s, int max_leaf, int cluster_size) {
    if (max_leaf < 1 || max_leaf > kMaxLeaf) return set_err(c, SRT_E_LIMIT, "max_leaf must be in [1, %d]", kMaxLeaf);
    const int n = s->nf;
    if (n < 1) return set_err(c, SRT_E_INVALID, "scene has no triangles");
    if ((int64_t)n > kMaxTriangles) return set_err(c, SRT_E_LIMIT, "too many triangles for the leaf encoding");
    hipStream_t st = c->stream;
    // default: clusters of at most 4 triangles under the binned-SAH top (at
    // most 2^18 clusters): 3.5 % faster traversal than 64 on the 1M-triangle
    // field, for a build of about 3 ns per triangle
    // a cluster holds at least a leaf's triangles: a collapsed (leaf) subtree
    // never spans the cluster frontier
    const int T = std::max(max_leaf, cluster_size > 0 ? cluster_size : std::max(kAutoClusterMin, n / kAutoClusterDiv));
    const float c_trav = 1.0f, c_isect = 1.0f;
    Tmp tmp(c);
    // boxes & centroids
    BoxArr tb;
    tb.lox = tmp.get<float>(n); tb.loy = tmp.get<float>(n); tb.loz = tmp.get<float>(n);
    tb.hix = tmp.get<float>(n); tb.hiy = tmp.get<float>(n); tb.hiz = tmp.get<float>(n);
    float* cen = tmp.get<float>(3 * (size_t)n);
    unsigned nb = nblk(n);
    uint32_t* partial = tmp.get<uint32_t>(6 * (size_t)nb);
    uint32_t* cb6 = tmp.get<uint32_t>(6);
    uint64_t* keys = tmp.get<uint64_t>(n);
    uint64_t* keys2 = tmp.get<uint64_t>(n);
    uint32_t* vals = tmp.get<uint32_t>(n);
    int32_t* kl = tmp.get<int32_t>(n);
    int32_t* kr = tmp.get<int32_t>(n);
    int32_t* kfirst = tmp.get<int32_t>(n);
    int32_t* par_int = tmp.get<int32_t>(n);
    int32_t* par_leaf = tmp.get<int32_t>(n);
    KArr K;
    K.box.lox = tmp.get<float>(n); K.box.loy = tmp.get<float>(n); K.box.loz = tmp.get<float>(n);
    K.box.hix = tmp.get<float>(n); K.box.hiy = tmp.get<float>(n); K.box.hiz = tmp.get<float>(n);
    K.count = tmp.get<int32_t>(n); K.cost = tmp.get<float>(n); K.collapse = tmp.get<int32_t>(n);
    int32_t* tri_mesh = (int32_t*)s->tri_mesh.p;
    if (tmp.failed || !cen || !K.collapse) return set_err(c, SRT_E_OOM, "BVH build scratch exceeds the HBM budget");

    // final outputs: the scene is without a tree until all of them are written
    s->has_bvh = false;
    if (dev_realloc(c, s->order, (size_t)n * 4) || dev_realloc(c, s->tris, (size_t)n * 48)) return SRT_E_OOM;
    uint32_t* order = (uint32_t*)s->order.p;

    k_tri_boxes<<<nb, 256, 0, st>>>((const float*)s->pos.p, (const uint32_t*)s->idx.p, n, tb, cen, partial);
    k_reduce_bounds<<<1, 256, 0, st>>>(partial, (int)nb, cb6);
    k_morton<<<nb, 256, 0, st>>>(cen, cb6, n, keys, vals);
    {
        size_t tbytes = 0;
        (void)hipcub::DeviceRadixSort::SortPairs(nullptr, tbytes, keys, keys2, vals, order, n, 0, 63, st);
        void* tstore = tmp.get<char>(tbytes);
        if (tmp.failed || !tstore) return set_err(c, SRT_E_OOM, "sort scratch");
        if (int r = hip_check(c, hipcub::DeviceRadixSort::SortPairs(tstore, tbytes, keys, keys2, vals, order, n, 0, 63, st), "radix sort"))
            return r;
    }
    k_fill_i32<<<nblk(n), 256, 0, st>>>(par_int, n, -1);
    if (n > 1) {
        k_karras<<<nblk(n - 1), 256, 0, st>>>(keys2, n, kl, kr, kfirst, par_int, par_leaf);
        // bottom-up by depth: the n - 1 radix-tree nodes ordered by depth
        const int m = n - 1;
        uint8_t* dkey = tmp.get<uint8_t>(m);
        uint32_t* dids = tmp.get<uint32_t>(m);
        if (tmp.failed) return set_err(c, SRT_E_OOM, "depth scratch");
        k_radix_depth<<<nblk(m), 256, 0, st>>>(m, par_int, dkey);
        std::vector<int32_t> df;
        if (int r = order_levels(c, tmp, m, dkey, dids, nullptr, &df)) return r;
        int dmax = 0;
        while (dmax + 1 < kLevels && df[dmax + 1] < m) dmax++;
        if (dmax >= kLevelNone - 1) return set_err(c, SRT_E_LIMIT, "radix tree depth %d exceeds %d", dmax, kLevelNone - 2);
        for (int D = 0; D <= dmax; D++)
            if (df[D + 1] == df[D]) return set_err(c, SRT_E_STATE, "radix tree depth %d is empty", D);
        by_levels(df.data(), dmax + 1,
                  [&](int D) {
                      const int count = df[D + 1] - df[D];
                      k_bottom_up_level<<<nblk(count), 256, 0, st>>>(dids + df[D], count, order, tb, kl, kr, K, max_leaf,
                                                                     c_trav, c_isect);
                  },
                  [&](const LevelRun& run) {
                      k_bottom_up_run<<<1, kRunNodes, 0, st>>>(run, dids, order, tb, kl, kr, K, max_leaf, c_trav, c_isect);
                  });
    }
    // clusters
    int m = 1;
    int32_t* clusters = nullptr;
    int32_t* nsel = tmp.get<int32_t>(1);
    int32_t* facts = tmp.get<int32_t>(4);
    if (tmp.failed) return set_err(c, SRT_E_OOM, "cluster scratch");
    if (n > 1 && n > T) {
        int32_t* mark = tmp.get<int32_t>(n);
        clusters = tmp.get<int32_t>(n);
        if (tmp.failed || !nsel) return set_err(c, SRT_E_OOM, "cluster scratch");
        k_fill_i32<<<nblk(n), 256, 0, st>>>(mark, n, 0x7fffffff);
        k_frontier<<<nblk(2 * (int64_t)n - 1), 256, 0, st>>>(n, T, kfirst, K.count, par_int, par_leaf, mark);
        struct NotSentinel {
            __host__ __device__ bool operator()(const int32_t& x) const { return x != 0x7fffffff; }
        };
        size_t tbytes = 0;
        (void)hipcub::DeviceSelect::If(nullptr, tbytes, mark, clusters, nsel, n, NotSentinel(), st);
        void* tstore = tmp.get<char>(tbytes);
        if (tmp.failed || !tstore) return set_err(c, SRT_E_OOM, "select scratch");
        if (int r = hip_check(c, hipcub::DeviceSelect::If(tstore, tbytes, mark, clusters, nsel, n, NotSentinel(), st), "select"))
            return r;
    }
    // what the host needs of it: the root's triangles, whether it is a leaf, and the number of clusters
    int32_t root_count = 1, root_collapse = 0, root_first = 0;
    if (n > 1) {
        k_build_facts<<<1, 64, 0, st>>>(K, kfirst, clusters ? nsel : nullptr, facts);
        int32_t h[4];
        if (int r = hip_check(c, hipMemcpyAsync(h, facts, sizeof h, hipMemcpyDeviceToHost, st), "copy")) return r;
        if (int r = hip_check(c, hipStreamSynchronize(st), "bvh build (sort/tree/clusters)")) return r;
        root_count = h[0];
        root_collapse = h[1];
        root_first = h[2];
        m = h[3];
    }
    const int top = m - 1;
    const int num_nodes = std::max(top + std::max(n - 1, 0), 1);
    if (dev_realloc(c, s->nodes, (size_t)num_nodes * sizeof(BvhNode)) ||
        dev_realloc(c, s->node_parent, (size_t)num_nodes * 4) || dev_realloc(c, s->level_nodes, (size_t)num_nodes * 4) ||
        dev_realloc(c, s->node_valid, (size_t)num_nodes * 4))
        return SRT_E_OOM;
    BvhNode* nodes = (BvhNode*)s->nodes.p;
    int32_t* valid = (int32_t*)s->node_valid.p;
    k_fill_i32<<<nblk((int64_t)num_nodes * 16), 256, 0, st>>>((int32_t*)nodes, (int64_t)num_nodes * 16, 0);
    k_fill_i32<<<nblk(num_nodes), 256, 0, st>>>(valid, num_nodes, 0);

    int32_t root;
    if (m > 1) {
        TopBuild B;
        B.m = m;
        B.wide_levels = 0;
        while (B.wide_levels < kWideLevels && (m >> B.wide_levels) > kWideMin) B.wide_levels++;
        for (Items& x : B.it) {
            x.box.lox = tmp.get<float>(m); x.box.loy = tmp.get<float>(m); x.box.loz = tmp.get<float>(m);
            x.box.hix = tmp.get<float>(m); x.box.hiy = tmp.get<float>(m); x.box.hiz = tmp.get<float>(m);
            x.cx = tmp.get<float>(m); x.cy = tmp.get<float>(m); x.cz = tmp.get<float>(m);
            x.count = tmp.get<int32_t>(m); x.ref = tmp.get<int32_t>(m);
        }
        const int slots = mid_slots(m), wide_slots = 1 << std::max(B.wide_levels - 1, 0);
        const int acc_words = B.wide_levels > 0 ? wide_slots * kWideCopies * kAccTotal : 0;
        B.rec = tmp.get<TopRec>(m);
        B.level = tmp.get<uint8_t>(m);
        for (int k = 0; k < 2; k++) {
            B.wide[k] = tmp.get<TopTask>(wide_slots);
            B.mid[k] = tmp.get<TopTask>(slots);
        }
        B.small = tmp.get<SmallTask>((size_t)region_base(m, kRegions));
        B.nsmall = tmp.get<int32_t>(kRegions * 64);
        B.any = tmp.get<int32_t>(kLevels);
        B.cb = tmp.get<uint32_t>(6);
        B.acc = tmp.get<uint32_t>(acc_words);
        B.chunk_items = tmp.get<int32_t>(((size_t)m / kWideChunk + wide_slots) * 48);
        B.wsplit = tmp.get<WideSplit>(wide_slots);
        uint32_t* ids = tmp.get<uint32_t>(m);
        int32_t* number = tmp.get<int32_t>(m);
        if (tmp.failed) return set_err(c, SRT_E_OOM, "top-level scratch");
        k_items<<<nblk(m), 256, 0, st>>>(m, clusters, order, tb, K, kfirst, top, B.it[0]);
        k_top_clear<<<std::min(nblk(std::max(2 * slots, acc_words)), 1024u), 256, 0, st>>>(B, slots, acc_words);
        k_top_bounds<<<std::min(nblk(m), 128u), 256, 0, st>>>(B);
        k_top_root<<<1, 64, 0, st>>>(B);
        int L = 0;
        for (; L < B.wide_levels; L++) {
            // every chunk but a node's last one is full
            const int chunks = m / kWideChunk + (1 << L);
            k_top_wide_bins<<<chunks, 64 * kTopWaves, 0, st>>>(B, L);
            k_top_wide_sah<<<1 << L, 64, 0, st>>>(B, L);
            k_top_wide_scatter<<<chunks, 64 * kTopWaves, 0, st>>>(B, L);
        }
        // The middle levels of a tree half as deep again as a balanced one are
        // queued at once, then four at a time until a level has no middle node:
        // an empty one costs up to 13 us, a wait 45 us (the 1M-triangle field has
        // 23 levels above its small nodes, a balanced tree would have 14).
        int balanced = 0;
        while ((m >> balanced) > kSmallItems) balanced++;
        for (int to = 3 * balanced / 2 + 2; balanced > 0; to += 4) {
            if (to >= kLevelNone) return set_err(c, SRT_E_LIMIT, "BVH depth exceeds the traversal limit %d", kMaxDepth);
            for (; L < to; L++)
                k_top_mid<<<nblk(slots, kMidSlots), 64 * kTopWaves, 0, st>>>(B, L, slots);
            int32_t more = 0;
            if (int r = hip_check(c, hipMemcpyAsync(&more, B.any + L, 4, hipMemcpyDeviceToHost, st), "top level")) return r;
            if (int r = hip_check(c, hipStreamSynchronize(st), "top level")) return r;
            if (!more) break;
        }
        k_top_small<<<kRegions * kRegionBlocks, 64 * kTopWaves, 0, st>>>(B);
        if (int r = order_levels(c, tmp, top, B.level, ids, number, nullptr)) return r;
        k_top_write<<<nblk(top), 256, 0, st>>>(B, ids, number, nodes);
        k_fill_i32<<<nblk(top), 256, 0, st>>>(valid, top, 1);
        root = 0;
    } else if (n == 1) {
        root = leaf_ref(0u, 1u);
    } else {
        root = root_collapse ? leaf_ref((uint32_t)root_first, (uint32_t)root_count) : top + 0;
    }
    if (n > 1)
        k_emit<<<nblk(n - 1), 256, 0, st>>>(n, T, top, max_leaf, kl, kr, kfirst, par_int, order, tb, K, nodes, valid);
    if (dev_realloc(c, s->tri_rec, (size_t)n * 8 * sizeof(float4))) return SRT_E_OOM;
    launch_tris(s, st);
    int32_t* parent = (int32_t*)s->node_parent.p;
    k_fill_i32<<<nblk(num_nodes), 256, 0, st>>>(parent, num_nodes, -1);
    k_final_parents<<<nblk(num_nodes), 256, 0, st>>>(num_nodes, nodes, valid, parent);
    if (int r = hip_check(c, hipGetLastError(), "bvh launch")) return r;
    // nodes by level for the refit and the collapse; levels 0 .. depth-1 hold the inner nodes, unused slots come last
    int32_t depth = 0;
    s->level_first.assign(1, 0);
    if (root >= 0) {
        uint8_t* lkey = tmp.get<uint8_t>(num_nodes);
        if (tmp.failed) return set_err(c, SRT_E_OOM, "level scratch");
        k_node_level<<<nblk(num_nodes), 256, 0, st>>>(num_nodes, valid, parent, lkey);
        std::vector<int32_t> hf;
        if (int r = order_levels(c, tmp, num_nodes, lkey, (uint32_t*)s->level_nodes.p, nullptr, &hf)) return r;
        while (depth < kLevelNone && hf[depth] < hf[kLevelNone]) depth++;
        if (depth > kMaxDepth)
            return set_err(c, SRT_E_LIMIT, "BVH depth %d exceeds the traversal limit %d", depth, kMaxDepth);
        for (int L = 0; L < depth; L++)
            if (hf[L + 1] == hf[L]) return set_err(c, SRT_E_STATE, "BVH level %d is empty", L);
        s->level_first.assign(hf.begin(), hf.begin() + depth + 1);
    } else {
        if (int r = hip_check(c, hipStreamSynchronize(st), "bvh build")) return r;
    }
    s->root = root;
    s->num_nodes = num_nodes;
    s->max_depth = depth;
    s->num_clusters = m;
    s->num_top = top;
    s->cluster_size = T;
    s->max_leaf = max_leaf;
    if (int r = bvh4_build(c, s)) return r;
    s->has_bvh = true;
    return SRT_OK;
}

int bvh4_build(srt_ctx* c, SceneRec* s) {
    s->num_nodes4 = 0;
    s->depth4 = 0;
    if (s->root < 0) {            // a single leaf
        dev_free(c, s->nodes4);
        s->root4 = s->root;
        return SRT_OK;
    }
    hipStream_t st = c->stream;
    const int n2 = s->num_nodes;
    if (dev_realloc(c, s->nodes4, (size_t)n2 * sizeof(Bvh4Node))) return SRT_E_OOM;
    Tmp tmp(c);
    const int nlev = (int)s->level_first.size() - 1;
    if (nlev < 1) return set_err(c, SRT_E_STATE, "4-wide collapse without the binary tree's levels");
    int32_t* lev[2] = {tmp.get<int32_t>(n2), tmp.get<int32_t>(n2)};
    int32_t* off = tmp.get<int32_t>(n2);
    int32_t* sums = tmp.get<int32_t>(kC4Grid);
    // at most as many 4-wide levels as binary ones
    int32_t* sizes = tmp.get<int32_t>(2 * (size_t)(nlev + 2));
    int32_t* bases = sizes + nlev + 2;
    C4Dp dp;
    dp.W = tmp.get<float>(n2);
    dp.G = tmp.get<float>(3 * (size_t)n2);
    dp.J = tmp.get<uint32_t>(n2);
    if (tmp.failed) return SRT_E_OOM;
    // the dynamic program, deepest level first (levels 0 .. depth-1 hold the inner nodes)
    const uint32_t* level_nodes = (const uint32_t*)s->level_nodes.p;
    by_levels(s->level_first.data(), nlev,
              [&](int L) {
                  const int first = s->level_first[L], count = s->level_first[L + 1] - first;
                  k_c4_dp<<<nblk(count), 256, 0, st>>>(level_nodes + first, count, (const BvhNode*)s->nodes.p, dp);
              },
              [&](const LevelRun& run) {
                  k_c4_dp_run<<<1, kRunNodes, 0, st>>>(run, level_nodes, (const BvhNode*)s->nodes.p, dp);
              });
    k_fill_i32<<<1, 64, 0, st>>>(lev[0], 1, s->root);
    k_fill_i32<<<1, 64, 0, st>>>(sizes, 1, 1);
    k_fill_i32<<<1, 64, 0, st>>>(bases, 1, 0);
    // A 4-wide node spans one to three binary levels on its deepest path: a
    // little over half of the binary levels are queued at once (the 1M-triangle
    // field: 27 binary, 16 4-wide levels), then four at a time until a level is
    // empty.  An empty level costs about 10 us, a wait for the count 45 us.
    Bvh4Node* out = (Bvh4Node*)s->nodes4.p;
    std::vector<int32_t> h(2 * (size_t)(nlev + 2));
    int levels = 0, queued = 0;
    for (int more = 3 * nlev / 5 + 1; ; more = 4) {
        for (const int to = std::min(queued + more, nlev); queued < to; queued++) {
            // level L has at most 4^L nodes
            const int64_t most = queued < 10 ? (int64_t)1 << (2 * queued) : n2;
            const int grid = (int)std::min<int64_t>(kC4Grid, nblk(std::min<int64_t>(most, n2)));
            const int32_t* from = lev[queued & 1];
            k_c4_count<<<grid, 256, 0, st>>>(queued, sizes, from, (const BvhNode*)s->nodes.p, dp, off, sums);
            k_c4_emit<<<grid, 256, 0, st>>>(queued, sizes, bases, from, (const BvhNode*)s->nodes.p, dp, off, sums, out,
                                            lev[(queued & 1) ^ 1]);
        }
        if (int r = hip_check(c, hipMemcpyAsync(h.data(), sizes, 4 * h.size(), hipMemcpyDeviceToHost, st), "count")) return r;
        if (int r = hip_check(c, hipStreamSynchronize(st), "collapse")) return r;
        while (levels < queued && h[levels] > 0) levels++;
        if (levels < queued || h[queued] == 0) break;
        if (queued >= nlev) return set_err(c, SRT_E_STATE, "4-wide collapse deeper than the binary tree");
    }
    const int base = h[(size_t)nlev + 2 + levels - 1] + h[levels - 1];
    if (!nodes4_fit((int64_t)base, c->max_wide_nodes)) {
        // beyond 32-bit buffer offsets: keep the binary tree only
        dev_free(c, s->nodes4);
        s->root4 = s->root;
        return SRT_OK;
    }
    s->root4 = 0;
    s->num_nodes4 = base;
    s->depth4 = levels;
    return hip_check(c, hipGetLastError(), "collapse launch");
}

int bvh_refit(srt_ctx* c, SceneRec* s) {
    if (!s->has_bvh) return set_err(c, SRT_E_STATE, "refit before build");
    hipStream_t st = c->stream;
    const int n = s->nf;
    launch_tris(s, st);
    if (s->root >= 0) {
        const int levels = (int)s->level_first.size() - 1;
        const uint32_t* level_nodes = (const uint32_t*)s->level_nodes.p;
        by_levels(s->level_first.data(), levels,
                  [&](int L) {
                      const int first = s->level_first[L], count = s->level_first[L + 1] - first;
                      k_refit_level<<<nblk(count), 256, 0, st>>>(level_nodes + first, count, (BvhNode*)s->nodes.p,
                                                                 (const float4*)s->tris.p);
                  },
                  [&](const LevelRun& run) {
                      k_refit_run<<<1, kRunNodes, 0, st>>>(run, level_nodes, (BvhNode*)s->nodes.p, (const float4*)s->tris.p);
                  });
        if (s->num_nodes4 > 0)
            k_refit4<<<nblk(s->num_nodes4), 256, 0, st>>>(s->num_nodes4, (const BvhNode*)s->nodes.p,
                                                          (Bvh4Node*)s->nodes4.p);
    }
    if (int r = hip_check(c, hipGetLastError(), "refit launch")) return r;
    return hip_check(c, hipStreamSynchronize(st), "refit");
}

int skin_vertices(srt_ctx* c, SceneRec* s, const float* bones_3x4, int nb) {
    if (!s->bone_ids.p) return set_err(c, SRT_E_STATE, "no skin weights set on this scene");
    if (nb < 0 || nb > 4096) return set_err(c, SRT_E_LIMIT, "bone count %d outside [0, 4096]", nb);
    hipStream_t st = c->stream;
    if (s->nbones < nb || !s->bones.p) {
        dev_free(c, s->bones);
        if (dev_alloc(c, s->bones, (size_t)std::max(nb, 1) * 48)) return SRT_E_OOM;
        s->nbones = nb;
    }
    if (nb > 0)
        if (int r = hip_check(c, hipMemcpyAsync(s->bones.p, bones_3x4, (size_t)nb * 48, hipMemcpyHostToDevice, st), "bones upload"))
            return r;
    hipEvent_t ev;
    prof_begin(c, "skin", &ev);
    k_skin<<<nblk(s->nv), 256, 0, st>>>(s->nv, (const float*)s->orig_pos.p, (const float*)s->orig_nrm.p,
                                        (const float*)s->orig_tan.p, (const int32_t*)s->bone_ids.p, (const float*)s->bone_w.p,
                                        nb, (const float*)s->bones.p, (float*)s->pos.p, (float*)s->nrm.p, (float*)s->tan.p);
    prof_end(c, "skin", ev, s->nv);
    return hip_check(c, hipGetLastError(), "skin launch");
}

}  // namespace srt
