/*
 * build.hip - octree construction on the GPU (qbt_build_octree).
 *
 * Produces, node for node, the array that inserting points 0..n-1 in index
 * order with octree_insert_point (src/qubatron/octree.c:95-147) produces, and
 * its compact layout (layout.hip's format):
 *
 *  - every point's octet path is computed with the reference's fp32 formula
 *    ((int)(p/size)%2 with size halved per level, octree.c:102-109) and
 *    packed into a key, 3 bits per level, first level highest (32-bit keys
 *    up to 10 levels, else 64-bit);
 *  - a stable radix sort groups equal prefixes while keeping index order. A
 *    sorted position starts a new node at every depth from the first octet
 *    that differs from the key before it, so its nodes are ranks: position i
 *    heads group #{j < i that start one at depth <= d} of depth d. One pass
 *    counts the starts per wave and depth, a scan turns the counts into
 *    ranks, a second pass writes every node's record, depth after depth,
 *    each depth in key order, which is the breadth-first hierarchical order
 *    of the compact layout: the children of a node are the consecutive nodes
 *    [first child, first child of the next node);
 *  - the node of a depth-d prefix is created by the smallest point index in
 *    its group (the first inserter, slot 8): the minimum over its children,
 *    from the leaves up (a leaf group's smallest index is its first, the sort
 *    being stable). A node whose first inserter is not its parent's is the
 *    first that this point creates, and the point creates one node more at
 *    every depth below it;
 *  - so the node index of a point's first node is 1 + the nodes of all
 *    earlier points (an exclusive scan of the per-point counts in index
 *    order), and a node with its parent's first inserter has its parent's
 *    index + 1: from the root down, every node hands its children their
 *    indices and writes its child block.
 *
 * HBM is the bound, half of it the scattered writes of child blocks and
 * reference map (node order is point order, record order is key order).
 * Whole calls, depth 12: 10M points (29M nodes) 3.3 ms with kept scratch and
 * 3.8 without, against 6.1 and 13.4 with a reduction by key, a scan and four
 * scatter passes per depth; 2M points (8M nodes) 0.89 against 2.0; 90M
 * points (158M nodes) 22.7 against 51. Scratch is 24 bytes a point (20 up to
 * 10 levels).
 */
#include <hip/hip_runtime.h>

#include <cstring>

#include <rocprim/rocprim.hpp>

#include "qbt.h"
#include "qbt_internal.hpp"

#pragma clang fp contract(off)

/* Scratch blocks of the builder: allocating and freeing scratch each time
 * costs a large part of a build (the reference rebuilds its dynamic tree
 * every frame). Each build carves its buffers from the blocks in order,
 * adding a block where none fits. A dynamic-tree build keeps its blocks, up to kKeepBytes, for the next
 * per-frame rebuild; a static build releases them when it ends. Kept blocks
 * are idle between builds, and qbt_ctx::dev_alloc releases them (trim)
 * before it would report QBT_ENOMEM. */
struct BuildState {
    std::vector<DevBuf> blocks;
    bool                active = false; /* a build is carving from the blocks */
};

void qbt_ctx::builder_free()
{
    if (build)
        for (auto& b : build->blocks) dev_free(b);
    delete build;
    build = nullptr;
}

bool qbt_ctx::builder_trim()
{
    if (!build || build->active || build->blocks.empty()) return false;
    (void) hipStreamSynchronize(stream);
    for (auto& b : build->blocks) dev_free(b);
    build->blocks.clear();
    return true;
}

namespace {

constexpr int kMaxBuildLevels = 21; /* 3 bits per level in a 64-bit key */

/* the octet path of a point. The reference divides by the cell size of each
 * level, which halves exactly: the quotients are the first one doubled level
 * by level, bit for bit (a quotient too small for a normal number truncates
 * to 0 at every level either way), so there is one division per axis; the
 * last, largest quotient decides whether all of them fit an int. */
template <class K>
__global__ void k_paths(const float* __restrict__ xyz, size_t n, float edge, int L, K* __restrict__ keys,
                        uint32_t* __restrict__ vals, unsigned int* __restrict__ bad)
{
    size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float half = edge / 2.0f;
    float       qx = xyz[3 * i] / half, qy = xyz[3 * i + 1] / half, qz = xyz[3 * i + 2] / half;
    const float up = ldexpf(1.0f, L > 0 ? L - 1 : 0);
    /* outside the int range (or NaN) the reference's conversion is undefined */
    bool ok = L == 0 || (fabsf(qx * up) < 2147483520.0f && fabsf(qy * up) < 2147483520.0f && fabsf(qz * up) < 2147483520.0f);
    K    key = 0;
    for (int l = 0; l < L; l++) {
        int o  = ok ? (int) qx % 2 : 0;
        int yi = ok ? (int) qy % 2 : 1;
        int zi = ok ? (int) qz % 2 : 1;
        if (yi == 0) o += 2;
        if (zi == 0) o += 4;
        if (o < 0) ok = false;
        key = (key << 3) | (K) (o & 7);
        qx *= 2.0f, qy *= 2.0f, qz *= 2.0f;
    }
    if (!ok) atomicAdd(bad, 1u);
    keys[i] = key;
    vals[i] = (uint32_t) i;
}

constexpr int kWaveKeys = 1024; /* sorted positions per wave of the counting and emitting passes */

/* the depth from which sorted position i starts new nodes: L + 1 for a key
 * equal to the one before it (and past the end) */
template <class K>
__device__ __forceinline__ int start_depth(const K* __restrict__ keys, size_t i, size_t n, int L, K& key)
{
    if (i >= n) return L + 1;
    key = keys[i];
    if (i == 0) return 1;
    const uint64_t x = (uint64_t) (key ^ keys[i - 1]);
    return x == 0ull ? L + 1 : L - (63 - __clzll((long long) x)) / 3;
}

/* cnt[(d - 1) * nw + w] = nodes that wave w's positions start at depth d */
template <class K>
__global__ void __launch_bounds__(256) k_count_starts(const K* __restrict__ keys, size_t n, int L,
                                                      uint32_t* __restrict__ cnt, uint32_t nw)
{
    const uint32_t w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (w >= nw) return;
    uint32_t c[kMaxBuildLevels] = {};
    for (int k = 0; k < kWaveKeys / 64; k++) {
        K         key = 0;
        const int d0  = start_depth<K>(keys, (size_t) w * kWaveKeys + (size_t) k * 64 + lane, n, L, key);
#pragma unroll
        for (int d = 1; d <= kMaxBuildLevels; d++)
            if (d <= L) c[d - 1] += (uint32_t) __popcll(__ballot(d0 <= d));
    }
#pragma unroll
    for (int d = 1; d <= kMaxBuildLevels; d++)
        if (d <= L && lane == (uint32_t) d) cnt[(size_t) (d - 1) * nw + w] = c[d - 1];
}

/* in place: exclusive scan of the nw counts of row blockIdx.x, its total to total[row] */
__global__ void __launch_bounds__(1024) k_scan_rows(uint32_t* __restrict__ cnt, uint32_t nw, uint32_t* __restrict__ total)
{
    __shared__ uint32_t ws[16];
    uint32_t*           b    = cnt + (size_t) blockIdx.x * nw;
    const int           lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t            carry = 0;
    for (uint32_t base = 0; base < nw; base += 4096) {
        const uint32_t i = base + 4 * threadIdx.x;
        uint32_t       v[4], s = 0;
        for (int k = 0; k < 4; k++) {
            v[k] = s;
            s += i + k < nw ? b[i + k] : 0u;
        }
        uint32_t x = s; /* inclusive scan within the wave */
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) ws[w] = x;
        __syncthreads();
        uint32_t before = carry, all = 0;
        for (int k = 0; k < 16; k++) {
            if (k < w) before += ws[k];
            all += ws[k];
        }
        __syncthreads();
        for (int k = 0; k < 4; k++)
            if (i + k < nw) b[i + k] = before + x - s + v[k];
        carry += all;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

/* off[d] = the first record of depth d (off[0] = 0, off[1] = 1), off[L + 1] the record count */
struct Depths {
    uint32_t off[kMaxBuildLevels + 3];
};

/* Every node's record {first child, its octet}; the smallest point index of
 * a leaf's group to model. Leaves' records hold no first child. */
template <class K>
__global__ void __launch_bounds__(256) k_emit_records(const K* __restrict__ keys, const uint32_t* __restrict__ vals,
                                                      size_t n, int L, Depths D, const uint32_t* __restrict__ rank,
                                                      uint32_t nw, uint2* __restrict__ rec, int* __restrict__ model)
{
    const uint32_t w = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (w >= nw) return;
    uint32_t at[kMaxBuildLevels] = {}; /* the next record of each depth */
#pragma unroll
    for (int d = 1; d <= kMaxBuildLevels; d++)
        if (d <= L) at[d - 1] = __builtin_amdgcn_readfirstlane(D.off[d] + rank[(size_t) (d - 1) * nw + w]);
    for (int k = 0; k < kWaveKeys / 64; k++) {
        const size_t i   = (size_t) w * kWaveKeys + (size_t) k * 64 + lane;
        K            key = 0;
        const int    d0  = start_depth<K>(keys, i, n, L, key);
        uint32_t     below = 0; /* this position's record one depth deeper */
#pragma unroll
        for (int d = kMaxBuildLevels; d >= 1; d--) {
            if (d > L) continue;
            const uint64_t m = __ballot(d0 <= d);
            if (d0 <= d) {
                const uint32_t c = at[d - 1] + __builtin_amdgcn_mbcnt_hi((uint32_t) (m >> 32),
                                                                         __builtin_amdgcn_mbcnt_lo((uint32_t) m, 0u));
                rec[c]           = make_uint2(below, (uint32_t) (key >> (3 * (L - d))) & 7u);
                if (d == L) model[c] = (int) vals[i];
                below = c;
            }
            at[d - 1] += (uint32_t) __popcll(m);
        }
    }
}

/* From the leaves up, one node of depth d (0 the root): its first inserter,
 * the smallest of its children's, to model; the number of nodes that the
 * first inserter of every other child creates (that child's and one at each
 * depth below it) to count. */
__device__ __forceinline__ void up_node(const Depths& D, int L, int d, uint32_t c, const uint2* __restrict__ rec,
                                        int* __restrict__ model, uint32_t* __restrict__ count)
{
    const uint32_t lo = d == 0 ? 1u : rec[c].x, hi = c + 1 < D.off[d + 1] ? rec[c + 1].x : D.off[d + 2];
    int            f  = -1;
    if (d > 0) {
        f = model[lo];
        for (uint32_t k = lo + 1; k < hi; k++) f = min(f, model[k]);
        model[c] = f;
    }
    for (uint32_t k = lo; k < hi; k++) {
        const int g = model[k];
        if (g != f) count[g] = (uint32_t) (L - d);
    }
}

/* From the root down, one node of depth d: indices to its children (ref,
 * r2c), its child block, its record in its final form; the leaves' records
 * are cleared by their parents. (One thread per point's chain of nodes,
 * whose indices are consecutive, writes fewer lines but reads the records
 * out of order: 10M points 2.50 ms against 1.98 for these launches and
 * k_own_nodes.) */
__device__ __forceinline__ void down_node(const Depths& D, int L, int d, uint32_t c, uint2* __restrict__ rec,
                                          const int* __restrict__ model, const uint32_t* __restrict__ base,
                                          int* __restrict__ ref, int* __restrict__ r2c, int4* __restrict__ child)
{
    const uint32_t lo = d == 0 ? 1u : rec[c].x, hi = c + 1 < D.off[d + 1] ? rec[c + 1].x : D.off[d + 2];
    const int      f = d == 0 ? -1 : model[c], idx = d == 0 ? 0 : ref[c];
    int            s0 = 0, s1 = 0, s2 = 0, s3 = 0, s4 = 0, s5 = 0, s6 = 0, s7 = 0; /* slots by value: no scratch array */
    uint32_t       mask = 0;
    for (uint32_t k = lo; k < hi; k++) {
        const int g  = model[k];
        const int ki = g == f ? idx + 1 : (int) (1u + base[g]);
        const int o  = (int) rec[k].y;
        ref[k]       = ki;
        if (r2c) r2c[ki] = (int) k;
        s0 = o == 0 ? ki : s0, s1 = o == 1 ? ki : s1, s2 = o == 2 ? ki : s2, s3 = o == 3 ? ki : s3;
        s4 = o == 4 ? ki : s4, s5 = o == 5 ? ki : s5, s6 = o == 6 ? ki : s6, s7 = o == 7 ? ki : s7;
        mask |= 1u << o;
        if (d == L - 1) rec[k] = make_uint2(0u, 0u);
    }
    rec[c]                      = make_uint2(lo, mask | mask << 8); /* live = alloc */
    child[2 * (size_t) idx]     = make_int4(s0, s1, s2, s3);
    child[2 * (size_t) idx + 1] = make_int4(s4, s5, s6, s7);
}

__global__ void k_up(Depths D, int L, int d, const uint2* __restrict__ rec, int* __restrict__ model,
                     uint32_t* __restrict__ count)
{
    const uint32_t c = D.off[d] + blockIdx.x * blockDim.x + threadIdx.x;
    if (c < D.off[d + 1]) up_node(D, L, d, c, rec, model, count);
}

__global__ void k_down(Depths D, int L, int d, uint2* __restrict__ rec, const int* __restrict__ model,
                       const uint32_t* __restrict__ base, int* __restrict__ ref, int* __restrict__ r2c,
                       int4* __restrict__ child)
{
    const uint32_t c = D.off[d] + blockIdx.x * blockDim.x + threadIdx.x;
    if (c < D.off[d + 1]) down_node(D, L, d, c, rec, model, base, ref, r2c, child);
}

/* the top of the tree, depths top .. 0, in one block (a launch per depth
 * costs more than these few nodes) */
__global__ void __launch_bounds__(1024) k_up_top(Depths D, int L, int top, const uint2* __restrict__ rec,
                                                 int* __restrict__ model, uint32_t* __restrict__ count)
{
    for (int d = top; d >= 0; d--) {
        for (uint32_t c = D.off[d] + threadIdx.x; c < D.off[d + 1]; c += blockDim.x) up_node(D, L, d, c, rec, model, count);
        __syncthreads();
    }
    if (threadIdx.x == 0) model[0] = 0;
}

__global__ void __launch_bounds__(1024) k_down_top(Depths D, int L, int top, uint2* __restrict__ rec,
                                                   const int* __restrict__ model, const uint32_t* __restrict__ base,
                                                   int* __restrict__ ref, int* __restrict__ r2c, int4* __restrict__ child)
{
    if (threadIdx.x == 0) {
        ref[0] = 0;
        if (r2c) r2c[0] = 0;
    }
    for (int d = 0; d <= top; d++) {
        for (uint32_t c = D.off[d] + threadIdx.x; c < D.off[d + 1]; c += blockDim.x)
            down_node(D, L, d, c, rec, model, base, ref, r2c, child);
        __syncthreads();
    }
}

/* Slot 8 of every node (its point, in index order) and an empty child block
 * for it, which the nodes with children overwrite (k_down). A block's points
 * own one run of nodes; its threads write it in node order, the run's owners
 * laid out in LDS, so whole lines are written: 10M points 204 us, against
 * 352 when only the leaves' blocks are written. */
constexpr int kOwnRun = 2048; /* nodes of a run laid out at once */
__global__ void __launch_bounds__(256) k_own_nodes(const uint32_t* __restrict__ count,
                                                   const uint32_t* __restrict__ base, size_t n,
                                                   int4* __restrict__ child, int* __restrict__ model)
{
    __shared__ int      own[kOwnRun];
    __shared__ uint32_t ends[2];
    const size_t        i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t      c = i < n ? count[i] : 0u, b = i < n ? 1u + base[i] : 0u;
    if (i == 0) model[0] = 0;
    if (threadIdx.x == 0) ends[0] = b;
    if (i + 1 == n || (i < n && threadIdx.x == 255)) ends[1] = b + c;
    __syncthreads();
    const uint32_t lo = ends[0], hi = ends[1];
    for (uint32_t at = lo; at < hi; at += kOwnRun) {
        for (uint32_t k = 0; k < c; k++)
            if (b + k - at < (uint32_t) kOwnRun) own[b + k - at] = (int) i;
        __syncthreads();
        const uint32_t m = min((uint32_t) kOwnRun, hi - at);
        for (uint32_t j = threadIdx.x; j < m; j += blockDim.x) model[at + j] = own[j];
        for (uint32_t j = threadIdx.x; j < 2 * m; j += blockDim.x) child[2 * (size_t) at + j] = make_int4(0, 0, 0, 0);
        __syncthreads();
    }
}

/* a tree of the root alone */
__global__ void k_root_only(int4* __restrict__ child, int* __restrict__ model, uint2* __restrict__ rec,
                            int* __restrict__ model_c, int* __restrict__ ref, int* __restrict__ r2c)
{
    child[0] = child[1] = make_int4(0, 0, 0, 0);
    model[0]            = 0;
    rec[0]              = make_uint2(0u, 0u);
    model_c[0]          = 0;
    ref[0]              = 0;
    r2c[0]              = 0;
}

__global__ void k_zero_words(uint32_t* p, size_t n)
{
    size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

inline unsigned nblk(size_t n) { return (unsigned) ((n + 255) / 256); }

} // namespace

#define HIPCHK(x) QBT_HIPCHK(x)

/* one build's scratch, carved from the context's builder blocks */
constexpr size_t kBlockBytes = (size_t) 64 << 20;
constexpr size_t kKeepBytes  = (size_t) 2 << 30;
struct Scratch {
    qbt_ctx*    c;
    BuildState* bs;
    size_t      bi = 0, off = 0;
    bool        keep; /* keep the blocks for the next build (dynamic tree) */
    Scratch(qbt_ctx* cc, bool keep_blocks) : c(cc), bs(cc->build), keep(keep_blocks) { bs->active = true; }
    ~Scratch()
    {
        /* the caller has synchronised the stream (or no kernel uses a block
         * yet); a dynamic build keeps the first blocks up to kKeepBytes */
        size_t kept = 0, i = 0;
        if (keep)
            for (; i < bs->blocks.size() && kept + bs->blocks[i].cap <= kKeepBytes; i++) kept += bs->blocks[i].cap;
        for (size_t j = i; j < bs->blocks.size(); j++) c->dev_free(bs->blocks[j]);
        bs->blocks.resize(i);
        bs->active = false;
    }
    void* get(size_t bytes, int* rc)
    {
        bytes = ((bytes ? bytes : 16) + 255) & ~(size_t) 255;
        for (; bi < bs->blocks.size(); bi++, off = 0) {
            if (off + bytes <= bs->blocks[bi].cap) {
                void* p = (char*) bs->blocks[bi].p + off;
                off += bytes;
                *rc = QBT_OK;
                return p;
            }
        }
        DevBuf b;
        *rc = c->dev_alloc(b, bytes > kBlockBytes ? bytes : kBlockBytes);
        if (*rc) return nullptr;
        bs->blocks.push_back(b);
        bi  = bs->blocks.size() - 1;
        off = bytes;
        return b.p;
    }
};

template <class K>
static int build_t(qbt_ctx* c, int t, float edge, int levels, size_t n, size_t* nodes_out)
{
    hipStream_t s  = c->stream;
    const int   L  = levels;
    int         rc = QBT_OK;
    TreeBuf&     tr = c->tree[t];
    CompactTree& cm = tr.cmp;
    if (!c->build) c->build = new BuildState();
    Scratch    sc(c, t == 1);
    Depths     D{};
    size_t     total = 1;
    D.off[1]         = 1;
    const bool       any = n > 0 && L > 0;
    K *              k0 = nullptr, *k1 = nullptr;
    uint32_t *       v0 = nullptr, *v1 = nullptr, *cnt = nullptr, *tot = nullptr;
    void*            tmp = nullptr;
    size_t           tb  = 0;
    const uint32_t   nw  = (uint32_t) ((n + kWaveKeys - 1) / kWaveKeys);
    /* 1. paths, the stable sort, and the node count of every depth; one
     * readback for the build (with the number of points outside the int
     * range: the sort of their keys is harmless) */
    if (n > 0) {
        size_t t2 = 0;
        if (any) {
            HIPCHK(rocprim::radix_sort_pairs(nullptr, tb, k0, k1, v0, v1, n, 0, 3 * L, s));
            HIPCHK(rocprim::exclusive_scan(nullptr, t2, v0, v1, 0u, n, rocprim::plus<uint32_t>(), s));
        }
        tb = t2 > tb ? t2 : tb;
        /* one allocation: the two key arrays (the first one later holds the
         * per-point counts and their scan, 8 bytes a point), the two value
         * arrays, the counts per wave and depth, totals, library scratch */
        auto         al = [](size_t bytes) { return (bytes + 255) & ~(size_t) 255; };
        const size_t o_k1 = al(n * 8), o_v0 = o_k1 + al(n * sizeof(K)), o_v1 = o_v0 + al(n * 4), o_cnt = o_v1 + al(n * 4);
        const size_t o_tot = o_cnt + al((size_t) nw * 4 * (L ? L : 1)), o_tmp = o_tot + 256;
        char*        sp    = (char*) sc.get(o_tmp + al(tb), &rc);
        if (rc) return rc;
        k0 = (K*) sp, k1 = (K*) (sp + o_k1), v0 = (uint32_t*) (sp + o_v0), v1 = (uint32_t*) (sp + o_v1);
        cnt = (uint32_t*) (sp + o_cnt), tot = (uint32_t*) (sp + o_tot), tmp = sp + o_tmp;
        uint32_t* bad = tot + 32;
        k_zero_words<<<1, 64, 0, s>>>(tot, 64);
        k_paths<K><<<nblk(n), 256, 0, s>>>((const float*) c->pts[t].xyz.p, n, edge, L, k0, v0, bad);
        HIPCHK(hipGetLastError());
        if (any) {
            size_t b = tb;
            HIPCHK(rocprim::radix_sort_pairs(tmp, b, k0, k1, v0, v1, n, 0, 3 * L, s));
            k_count_starts<K><<<(nw + 3) / 4, 256, 0, s>>>(k1, n, L, cnt, nw);
            k_scan_rows<<<L, 1024, 0, s>>>(cnt, nw, tot);
            HIPCHK(hipGetLastError());
        }
        uint32_t h[64];
        HIPCHK(hipMemcpyAsync(h, tot, sizeof(h), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        if (h[32]) return QBT_ERANGE;
        for (int d = 1; any && d <= L; d++) total += h[d - 1];
        if (total >= (size_t) INT32_MAX) return QBT_ENOTSUP;
        for (int d = 1; any && d <= L; d++) D.off[d + 1] = D.off[d] + h[d - 1];
    }
    /* 2. the arrays: the node array and, unless its 30-bit first-child
     * indices overflow, the compact layout (its arrays hold the records
     * while the tree is built; scratch does otherwise). The arrays are
     * replaced or overwritten from here on, and nothing clears them first: a
     * build that fails below leaves no tree, and what a later upload does not
     * write is checked and laid out as new */
    const bool cmp = total < (1u << 30);
    if ((rc = c->flush_pending(t, true))) return rc; /* held uploads go with the old array */
    tr.n           = 0;
    tr.validated   = false;
    tr.full_check  = true;
    tr.cmp_stale   = true;
    tr.patch.clear();
    cm.ok = false, cm.n = 0, cm.ref_n = 0;
    if (total > tr.cap_nodes) {
        const size_t cap = total + total / 4 + 1024;
        c->dev_free(tr.child);
        c->dev_free(tr.model);
        tr.cap_nodes = 0;
        if ((rc = c->dev_alloc(tr.child, cap * 32)) || (rc = c->dev_alloc(tr.model, cap * 4))) return rc;
        tr.cap_nodes = cap;
    }
    uint2* rec;
    int *  model_c, *ref, *r2c;
    if (cmp) {
        if ((rc = c->compact_reserve(t, total, total))) return rc;
        rec = (uint2*) cm.rec.p, model_c = (int*) cm.model.p, ref = (int*) cm.ref.p, r2c = (int*) cm.r2c.p;
    } else {
        rec     = (uint2*) sc.get(total * 8, &rc);
        model_c = rc ? nullptr : (int*) sc.get(total * 4, &rc);
        ref     = rc ? nullptr : (int*) sc.get(total * 4, &rc);
        r2c     = nullptr;
        if (rc) return rc;
    }
    int4* child = (int4*) tr.child.p;
    int*  model = (int*) tr.model.p;
    if (!any) {
        k_root_only<<<1, 1, 0, s>>>(child, model, rec, model_c, ref, r2c);
    } else {
        /* 3. records, first inserters and their node counts, node indices;
         * the sort's first key array is free: per-point counts and their scan */
        uint32_t *count = (uint32_t*) k0, *base = count + n;
        int       top   = 0; /* the deepest depth with few nodes: done by one block */
        while (top + 1 < L && D.off[top + 2] - D.off[top + 1] <= 1024) top++;
        k_zero_words<<<nblk(n), 256, 0, s>>>(count, n);
        k_emit_records<K><<<(nw + 3) / 4, 256, 0, s>>>(k1, v1, n, L, D, cnt, nw, rec, model_c);
        for (int d = L - 1; d > top; d--)
            k_up<<<nblk(D.off[d + 1] - D.off[d]), 256, 0, s>>>(D, L, d, rec, model_c, count);
        k_up_top<<<1, 1024, 0, s>>>(D, L, top, rec, model_c, count);
        HIPCHK(hipGetLastError());
        size_t b = tb;
        HIPCHK(rocprim::exclusive_scan(tmp, b, count, base, 0u, n, rocprim::plus<uint32_t>(), s));
        k_own_nodes<<<nblk(n), 256, 0, s>>>(count, base, n, child, model);
        k_down_top<<<1, 1024, 0, s>>>(D, L, top, rec, model_c, base, ref, r2c, child);
        for (int d = top + 1; d < L; d++)
            k_down<<<nblk(D.off[d + 1] - D.off[d]), 256, 0, s>>>(D, L, d, rec, model_c, base, ref, r2c, child);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s));
    /* every child index above is a node index below total: nothing to check */
    tr.n          = total;
    tr.validated  = true;
    tr.full_check = false;
    tr.dirty_lo = tr.dirty_hi = 0;
    tr.vdirty.clear();
    tr.vdirty_over = false;
    tr.cmp_stale = !cmp;
    if (cmp) cm.ok = true, cm.n = total, cm.ref_n = total;
    if (nodes_out) *nodes_out = total;
    return QBT_OK;
}

extern "C" int qbt_build_octree(qbt_ctx* c, int tree, const float basecube[4], int levels, size_t npoints,
                                size_t* nodes_out)
{
    if (!c || !basecube) return QBT_EINVAL;
    if (tree != QBT_BUFFER_STATIC_OCTREE && tree != QBT_BUFFER_DYNAMIC_OCTREE) return QBT_EINVAL;
    if (levels < 0 || levels > kMaxBuildLevels) return QBT_ENOTSUP;
    const int t = tree == QBT_BUFFER_STATIC_OCTREE ? 0 : 1;
    if (npoints > c->pts[t].n || npoints >= (size_t) UINT32_MAX) return QBT_EINVAL;
    HIPCHK(hipSetDevice(c->device));
    return 3 * levels <= 32 ? build_t<uint32_t>(c, t, basecube[3], levels, npoints, nodes_out)
                            : build_t<uint64_t>(c, t, basecube[3], levels, npoints, nodes_out);
}
