/*
 * layout.hip - compact, breadth-first device layout of an uploaded octree.
 *
 * The reference numbers nodes in creation order (octree.c:121-124), which
 * for scanned or generated scenes scatters the children of a node over the
 * whole array: every 32-byte child block the traversal reads sits in its own
 * cache line. The relayout renumbers nodes level by level, children of a
 * node contiguous and in octet order, and stores per node only
 *
 *     rec  = { index of the first child, live | alloc << 8 }  (8 bytes)
 *     model = slot 8 of the reference node                     (4 bytes)
 *     ref  = the reference node index                          (4 bytes)
 *
 * where alloc marks the slots of the node's child block and live the
 * children that exist (equal after a relayout; an in-place range update can
 * clear a live bit), so child o of node j is
 * rec.x + popcount(alloc & ((1 << o) - 1)). Every level
 * comes out in hierarchical octet order, so nodes that are close in space are
 * close in memory and rays of neighbouring pixels share cache lines.
 * Traversal results are unchanged (the same children exist, the same leaves
 * carry the same slot 8); reported leaf indices are mapped back through ref.
 *
 * Only a proper tree can be renumbered this way: if a node is reachable
 * twice (shared child, cycle) the relayout reports failure and the direct
 * layout is used.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "qbt.h"
#include "qbt_internal.hpp"

#define HIPCHK(x) QBT_HIPCHK(x)

namespace {

/* ---------------- relayout ------------------------------------------------
 *
 * Level by level: the nodes of level d are records [lev[d], lev[d + 1]), in
 * hierarchical octet order, and their children, in the same order, are level
 * d + 1: per level, the children of every 256 nodes counted, the counts
 * scanned, the records written and the children linked. The bounds stay on
 * the device, so a run of levels is enqueued without a readback (the grid
 * covers what a level can hold); the first levels, 4096 nodes at most, are
 * one launch of one block. */
enum { LY_BAD = 0, LY_LEV = 2, LY_WORDS = 80 }; /* state words: failures, then lev[0 ..] */
constexpr int kTopLevels = 5;  /* levels of the one-block launch: 1 + 8 + .. + 4096 nodes */
constexpr int kMaxLevels = 64; /* deeper than any octree: a cycle */

__global__ void k_lay_init(int* __restrict__ r2c, size_t n, uint32_t* __restrict__ oon, unsigned* __restrict__ st)
{
    const size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) r2c[i] = i == 0 ? 0 : -1; /* -1: not in the tree */
    if (i < LY_WORDS) st[i] = i == LY_LEV + 1 ? 1u : 0u; /* level 0: record 0, the root */
    if (i == 0) oon[0] = 0u;
}

__device__ __forceinline__ uint32_t row_mask(int4 a, int4 b)
{
    return (a.x > 0 ? 1u : 0u) | (a.y > 0 ? 2u : 0u) | (a.z > 0 ? 4u : 0u) | (a.w > 0 ? 8u : 0u) |
           (b.x > 0 ? 16u : 0u) | (b.y > 0 ? 32u : 0u) | (b.z > 0 ? 64u : 0u) | (b.w > 0 ? 128u : 0u);
}

struct LayArgs {
    const int4* child;
    const int*  model;
    uint32_t    n; /* nodes of the array, and room in the arrays below */
    uint32_t*   oon; /* record -> reference node */
    uint2*      rec;
    int *       model_c, *ref, *r2c;
    unsigned*   st;
};

/* record j of reference node o, whose children become the records from
 * `first` on: each is claimed in r2c (a node reached twice: not a tree) */
__device__ __forceinline__ void lay_record(const LayArgs& A, uint32_t j, uint32_t o, int4 a, int4 b, uint32_t m,
                                           uint32_t first)
{
    A.rec[j]     = make_uint2(m ? first : 0u, m | m << 8); /* live = alloc */
    A.model_c[j] = A.model[o];
    A.ref[j]     = (int) o;
    const int c[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t  nj   = first;
    bool      bad  = false;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        if (!((m >> q) & 1u)) continue;
        if (nj < A.n) {
            bad |= atomicExch(&A.r2c[c[q]], (int) nj) != -1;
            A.oon[nj] = (uint32_t) c[q];
        }
        nj++;
    }
    if (bad) atomicOr(&A.st[LY_BAD], 1u);
}

/* exclusive scan of v over the block's threads; *all the total. ws: one word per wave */
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* ws, uint32_t* all)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint32_t  x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    __syncthreads(); /* ws is free again */
    if (lane == 63) ws[w] = x;
    __syncthreads();
    uint32_t before = 0, sum = 0;
    for (int k = 0; k < nw; k++) {
        if (k < w) before += ws[k];
        sum += ws[k];
    }
    *all = sum;
    return before + x - v;
}

/* the end of level d + 1: more records than nodes means shared children */
__device__ __forceinline__ void close_level(const LayArgs& A, int d, uint32_t hi, uint32_t total)
{
    const bool over = total > A.n - hi;
    if (over) atomicOr(&A.st[LY_BAD], 1u);
    A.st[LY_LEV + d + 2] = over ? hi : hi + total;
}

__global__ void __launch_bounds__(1024) k_lay_top(LayArgs A)
{
    __shared__ uint32_t ws[16];
    uint32_t            lo = 0, hi = 1;
    for (int d = 0; d < kTopLevels && hi > lo; d++) {
        uint32_t total = 0;
        for (uint32_t base = lo; base < hi; base += blockDim.x) {
            const uint32_t j = base + threadIdx.x;
            uint32_t       o = 0, m = 0;
            int4           a = make_int4(0, 0, 0, 0), b = a;
            if (j < hi) {
                o = A.oon[j];
                a = A.child[2 * (size_t) o], b = A.child[2 * (size_t) o + 1];
                m = row_mask(a, b);
            }
            uint32_t       all;
            const uint32_t off = block_scan((uint32_t) __popc(m), ws, &all);
            if (j < hi) lay_record(A, j, o, a, b, m, hi + total + off);
            total += all;
        }
        if (threadIdx.x == 0) close_level(A, d, hi, total);
        __syncthreads();
        lo = hi;
        if (total <= A.n - hi) hi += total; /* else not a tree: no more levels */
        if (threadIdx.x == 0 && hi == lo) /* the tree ends here: the levels below are empty */
            for (int k = d + 2; k <= kTopLevels + 1; k++) A.st[LY_LEV + k] = hi;
    }
}

__global__ void __launch_bounds__(256) k_lay_count(LayArgs A, int d, uint32_t* __restrict__ bsum)
{
    __shared__ uint32_t ws[4];
    const uint32_t lo = A.st[LY_LEV + d], hi = A.st[LY_LEV + d + 1];
    const uint64_t j  = (uint64_t) lo + (uint64_t) blockIdx.x * 256 + threadIdx.x;
    if ((uint64_t) lo + (uint64_t) blockIdx.x * 256 >= hi) return; /* uniform */
    uint32_t c = 0;
    if (j < hi) {
        const uint32_t o = A.oon[j];
        c = (uint32_t) __popc(row_mask(A.child[2 * (size_t) o], A.child[2 * (size_t) o + 1]));
    }
    uint32_t all;
    (void) block_scan(c, ws, &all);
    if (threadIdx.x == 0) bsum[blockIdx.x] = all;
}

/* in place: exclusive scan of the level's block counts; closes the next level */
__global__ void __launch_bounds__(1024) k_lay_scan(LayArgs A, int d, uint32_t* __restrict__ bsum)
{
    __shared__ uint32_t ws[16];
    const uint32_t      lo = A.st[LY_LEV + d], hi = A.st[LY_LEV + d + 1], nb = (hi - lo + 255u) / 256u;
    uint64_t            carry = 0; /* more than 32 bits only in an array of shared children */
    for (uint32_t base = 0; base < nb; base += 4096) {
        const uint32_t i = base + 4 * threadIdx.x;
        uint32_t       v[4], s = 0, all;
        for (int k = 0; k < 4; k++) {
            v[k] = s;
            s += i + k < nb ? bsum[i + k] : 0u;
        }
        const uint32_t off = block_scan(s, ws, &all);
        for (int k = 0; k < 4; k++)
            if (i + k < nb) bsum[i + k] = (uint32_t) carry + off + v[k];
        carry += all;
    }
    if (threadIdx.x == 0) close_level(A, d, hi, carry > 0xFFFFFFFFull ? 0xFFFFFFFFu : (uint32_t) carry);
}

__global__ void __launch_bounds__(256) k_lay_emit(LayArgs A, int d, const uint32_t* __restrict__ bsum)
{
    __shared__ uint32_t ws[4];
    const uint32_t lo = A.st[LY_LEV + d], hi = A.st[LY_LEV + d + 1];
    const uint64_t j  = (uint64_t) lo + (uint64_t) blockIdx.x * 256 + threadIdx.x;
    if ((uint64_t) lo + (uint64_t) blockIdx.x * 256 >= hi) return; /* uniform */
    uint32_t o = 0, m = 0;
    int4     a = make_int4(0, 0, 0, 0), b = a;
    if (j < hi) {
        o = A.oon[j];
        a = A.child[2 * (size_t) o], b = A.child[2 * (size_t) o + 1];
        m = row_mask(a, b);
    }
    uint32_t       all;
    const uint32_t off = block_scan((uint32_t) __popc(m), ws, &all);
    if (j < hi) lay_record(A, (uint32_t) j, o, a, b, m, hi + bsum[blockIdx.x] + off);
}

__global__ void k_fill32(uint32_t* p, size_t n, uint32_t v)
{
    size_t i = (size_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

/* ---------------- in-place patch of range uploads ------------------------ */

/* r2c entries of nodes linked by this patch carry kNew until their own
 * children are laid out */
constexpr int kNew = 1 << 30;

/* patch state words: failure, records in use, grow-list and new-list lengths */
enum { PS_FAIL = 0, PS_LEN = 1, PS_GROW = 2, PS_NEW = 3, PS_WORDS = 64 };

/* link reference node v at record p: claim r2c[v] (v must not be in the
 * tree), fill the record's ref and slot 8, and queue v for k_patch_new */
__device__ __forceinline__ void link_new(int v, uint32_t p, size_t n, const int* __restrict__ model,
                                         int* __restrict__ model_c, int* __restrict__ ref, uint2* __restrict__ rec,
                                         int* __restrict__ r2c, uint2* __restrict__ newl, uint32_t newcap,
                                         unsigned* __restrict__ ps)
{
    if (v <= 0 || (size_t) v >= n || atomicCAS(&r2c[v], -1, (int) p | kNew) != -1) { /* shared or cyclic */
        atomicOr(&ps[PS_FAIL], 1u);
        return;
    }
    ref[p]     = v;
    model_c[p] = model[v];
    rec[p]     = make_uint2(0u, 0u);
    const unsigned k = atomicAdd(&ps[PS_NEW], 1u);
    if (k < newcap) newl[k] = make_uint2((uint32_t) v, p);
    else atomicOr(&ps[PS_FAIL], 1u);
}

/* Phase 1, one node of the uploaded ranges that the layout holds (below
 * ref_n, with a record): its slot 8, and its slots against its record. A
 * zeroed slot clears the live bit (the block keeps the slot, so the ranks of
 * the others stay); a slot holding its old child again sets it. A slot that
 * now holds another node, or a slot the block lacks, needs a new block: the
 * node goes to the grow list with a snapshot of its record, and its record
 * is left to phase 2. */
__global__ void k_patch_live(const uint2* __restrict__ ranges, const uint32_t* __restrict__ roff, int nr,
                             uint32_t total, size_t ref_n, const int4* __restrict__ child,
                             const int* __restrict__ model, uint2* __restrict__ rec, int* __restrict__ model_c,
                             const int* __restrict__ ref, const int* __restrict__ r2c, uint4* __restrict__ grow,
                             unsigned* __restrict__ ps)
{
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= total) return;
    const size_t i = range_item(ranges, roff, nr, g);
    if (i >= ref_n) return; /* appended nodes are laid out below their parents */
    const int ci = r2c[i];
    if (ci < 0) return; /* not in the tree */
    model_c[ci]          = model[i];
    const uint2    r     = rec[ci];
    const uint32_t alloc = (r.y >> 8) & 0xFFu;
    const int*     c     = reinterpret_cast<const int*>(child) + 8 * i;
    uint32_t       live  = 0;
    bool           relink = false;
    for (int o = 0; o < 8; o++) {
        const uint32_t bit = 1u << o;
        const int      v   = c[o];
        if (v == 0) continue;
        if (!(alloc & bit) || ref[r.x + (uint32_t) __popc(alloc & (bit - 1u))] != v) relink = true;
        else live |= bit;
    }
    if (!relink) {
        rec[ci].y = live | alloc << 8;
        return;
    }
    const unsigned k = atomicAdd(&ps[PS_GROW], 1u);
    grow[k]          = make_uint4((uint32_t) i, (uint32_t) ci, r.x, r.y); /* at most one per item: fits */
}

/* Phase 2a, one grow-list node: a new child block at the end of the records
 * with a slot for every nonzero slot and every slot the old block had (a
 * zeroed one stays, not live); the old children's records are copied there
 * (the old block stays unused), the others linked. The node's new record is
 * left in grow[k].zw for phase 2b, since its own record may be moving in
 * this phase (its parent may be on the list). */
__global__ void k_patch_grow(uint4* __restrict__ grow, size_t n, const int4* __restrict__ child,
                             const int* __restrict__ model, uint2* __restrict__ rec, int* __restrict__ model_c,
                             int* __restrict__ ref, int* __restrict__ r2c, uint32_t cap, uint2* __restrict__ newl,
                             uint32_t newcap, unsigned* __restrict__ ps)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ps[PS_GROW]) return;
    const uint4    e     = grow[k];
    const uint32_t alloc = (e.w >> 8) & 0xFFu;
    const int*     c     = reinterpret_cast<const int*>(child) + 8 * (size_t) e.x;
    uint32_t       na    = alloc;
    for (int o = 0; o < 8; o++)
        if (c[o] > 0) na |= 1u << o;
    const uint32_t base = atomicAdd(&ps[PS_LEN], (unsigned) __popc(na));
    if ((size_t) base + (size_t) __popc(na) > cap) {
        atomicOr(&ps[PS_FAIL], 1u);
        return;
    }
    uint32_t live = 0;
    for (int o = 0; o < 8; o++) {
        const uint32_t bit = 1u << o;
        if (!(na & bit)) continue;
        const uint32_t np = base + (uint32_t) __popc(na & (bit - 1u));
        const int      v  = c[o];
        int            cur = -1;
        if (alloc & bit) { /* carry the old child's record over */
            const uint32_t op = e.z + (uint32_t) __popc(alloc & (bit - 1u));
            cur               = ref[op];
            rec[np]           = rec[op];
            model_c[np]       = model_c[op];
            ref[np]           = cur;
            if (cur > 0 && r2c[cur] == (int) op) r2c[cur] = (int) np;
        }
        if (v == 0) continue; /* zeroed: not live */
        live |= bit;
        if (v == cur) continue;
        if (cur > 0 && r2c[cur] == (int) np) r2c[cur] = -1; /* replaced: the old child leaves the tree */
        link_new(v, np, n, model, model_c, ref, rec, r2c, newl, newcap, ps);
    }
    grow[k].z = base;
    grow[k].w = live | na << 8;
}

/* Phase 2b: the grow-list nodes' records, where they are now (a node its
 * parent replaced in phase 2a has left the tree: nothing to write) */
__global__ void k_patch_commit(const uint4* __restrict__ grow, uint2* __restrict__ rec, const int* __restrict__ r2c,
                               const unsigned* __restrict__ ps)
{
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= ps[PS_GROW]) return;
    const uint4 e = grow[k];
    const int   p = r2c[e.x];
    if (p >= 0) rec[p & ~kNew] = make_uint2(e.z, e.w);
}

/* Phase 3: the subtrees below the nodes linked in phase 2, depth first, one
 * list entry per thread: each node's children get a block of records at the
 * end (live = alloc = its nonzero slots) and are claimed in r2c. */
__global__ void k_patch_new(const uint2* __restrict__ newl, uint32_t newcap, size_t n, const int4* __restrict__ child,
                            const int* __restrict__ model, uint2* __restrict__ rec, int* __restrict__ model_c,
                            int* __restrict__ ref, int* __restrict__ r2c, uint32_t cap, unsigned* __restrict__ ps)
{
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ps[PS_NEW] || e >= newcap) return;
    constexpr int kStack = 192; /* pending nodes; deeper or wider subtrees relayout instead */
    uint2         stk[kStack];
    int           sp = 0;
    stk[sp++]        = newl[e];
    while (sp > 0) {
        const uint2 u = stk[--sp];
        const int*  c = reinterpret_cast<const int*>(child) + 8 * (size_t) u.x;
        uint32_t    m = 0;
        for (int o = 0; o < 8; o++)
            if (c[o] > 0) m |= 1u << o;
        uint32_t base = 0;
        if (m) {
            base = atomicAdd(&ps[PS_LEN], (unsigned) __popc(m));
            if ((size_t) base + (size_t) __popc(m) > cap) {
                atomicOr(&ps[PS_FAIL], 1u);
                return;
            }
        }
        rec[u.y]   = make_uint2(base, m | m << 8);
        r2c[u.x]   = (int) u.y; /* laid out */
        uint32_t k = 0;
        for (int o = 0; o < 8; o++) {
            if (!((m >> o) & 1u)) continue;
            const int      v = c[o];
            const uint32_t p = base + k++;
            if ((size_t) v >= n || atomicCAS(&r2c[v], -1, (int) p | kNew) != -1 || sp >= kStack) {
                atomicOr(&ps[PS_FAIL], 1u);
                return;
            }
            ref[p]     = v;
            model_c[p] = model[v];
            stk[sp++]  = make_uint2((uint32_t) v, p);
        }
    }
}

inline unsigned nblk(size_t n) { return (unsigned) ((n + 255) / 256); }

} // namespace

int qbt_ctx::compact_reserve(int t, size_t nrec, size_t nref)
{
    CompactTree& cm = tree[t].cmp;
    int          rc;
    if (nrec > cm.cap) { /* room for the records in-place patches append */
        const size_t cap = nrec + nrec / 8 + 65536;
        cm.cap           = 0; /* a failed allocation may leave one of the three without memory */
        if ((rc = dev_alloc(cm.rec, cap * 8)) || (rc = dev_alloc(cm.model, cap * 4)) || (rc = dev_alloc(cm.ref, cap * 4)))
            return rc;
        cm.cap = cap;
    }
    if (nref > cm.r2c_cap) {
        const size_t cap = nref > tree[t].cap_nodes ? nref : tree[t].cap_nodes;
        cm.r2c_cap       = 0;
        if ((rc = dev_alloc(cm.r2c, cap * 4))) return rc;
        cm.r2c_cap = cap;
    }
    return QBT_OK;
}

/* (Re)build the compact layout of tree t. Returns QBT_OK with cmp.ok set to
 * whether the array is a proper tree; errors only on allocation/HIP
 * failures. The levels are enqueued in runs, one small synchronisation per
 * run (the first covers trees of up to 12 levels below the root); the work
 * buffers are kept for the next relayout. The render call after a whole upload
 * of a 440k-node tree, 12 levels (validation and relayout): 235 us, against
 * 790 with a library scan and two readbacks per level. */
int qbt_ctx::relayout(int t)
{
    TreeBuf&     tb = tree[t];
    CompactTree& cm = tb.cmp;
    cm.ok           = false;
    cm.n            = 0;
    cm.ref_n        = 0;
    tb.patch.clear();
    tb.relayouts++;
    const size_t n  = tb.n;
    if (n == 0 || n > (size_t) INT32_MAX) return QBT_OK;
    hipStream_t s = stream;
    int         rc;
    if ((rc = compact_reserve(t, n, n))) return rc;
    /* work buffers, carved from one kept allocation */
    auto   al    = [](size_t b) { return (b + 255) & ~(size_t) 255; };
    size_t o_oon = 0, o_sum = o_oon + al(n * 4), o_st = o_sum + al((n / 256 + 1) * 4);
    if ((rc = dev_alloc(cm.scratch, o_st + al(LY_WORDS * 4)))) return rc;
    char*     sb   = (char*) cm.scratch.p;
    uint32_t* bsum = (uint32_t*) (sb + o_sum);
    LayArgs   A{(const int4*) tb.child.p, (const int*) tb.model.p, (uint32_t) n, (uint32_t*) (sb + o_oon),
              (uint2*) cm.rec.p, (int*) cm.model.p, (int*) cm.ref.p, (int*) cm.r2c.p, (unsigned*) (sb + o_st)};
    k_lay_init<<<nblk(n > LY_WORDS ? n : LY_WORDS), 256, 0, s>>>(A.r2c, n, A.oon, A.st);
    k_lay_top<<<1, 1024, 0, s>>>(A);
    HIPCHK(hipGetLastError());
    unsigned st[LY_WORDS];
    bool     ok = false;
    int      d  = kTopLevels;
    for (int run = 13; d < kMaxLevels; run = d + 8) {
        for (; d < run && d < kMaxLevels; d++) {
            const size_t most = d < 10 ? std::min(n, (size_t) 1 << (3 * d)) : n; /* nodes a level can hold */
            k_lay_count<<<nblk(most), 256, 0, s>>>(A, d, bsum);
            k_lay_scan<<<1, 1024, 0, s>>>(A, d, bsum);
            k_lay_emit<<<nblk(most), 256, 0, s>>>(A, d, bsum);
        }
        HIPCHK(hipGetLastError());
        HIPCHK(hipMemcpyAsync(st, A.st, sizeof(st), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        if (st[LY_BAD]) break;
        if (st[LY_LEV + d] == st[LY_LEV + d + 1]) { /* level d is empty: done */
            ok = true;
            break;
        }
    }
    const uint32_t total = st[LY_LEV + d];
    /* the single-tree traversal keeps first-child indices in 30 bits */
    cm.ok    = ok && total < (1u << 30);
    cm.n     = cm.ok ? total : 0;
    cm.ref_n = cm.ok ? n : 0;
    return QBT_OK;
}

/* The range uploads since the last layout, in place: k_patch_live,
 * k_patch_grow, k_patch_commit, k_patch_new. Records are appended up to the
 * capacity; *done = false when the uploads link a node that is already in
 * the tree (shared child, cycle), need more records than the capacity holds,
 * or the layout is not current. One synchronisation reads the outcome. */
int qbt_ctx::patch_layout(int t, bool* done)
{
    TreeBuf&     tb = tree[t];
    CompactTree& cm = tb.cmp;
    *done           = false;
    if (!cm.ok || cm.ref_n == 0 || tb.n < cm.ref_n || tb.n > (size_t) INT32_MAX) return QBT_OK;
    hipStream_t  s = stream;
    int          rc;
    const size_t n = tb.n;
    /* the layout's arrays must already hold every record and reference node
     * (growing them would drop their contents; the array only outgrows them
     * by a regrowth, which relays out) */
    if (cm.n > cm.cap || n > cm.r2c_cap) return QBT_OK;
    if (cm.cap >= (1u << 30)) return QBT_OK; /* first-child indices are 30-bit */
    /* the ranges (merged on upload) below ref_n and their prefix offsets */
    std::vector<uint2>    rg;
    std::vector<uint32_t> roff;
    uint64_t              total = 0;
    std::sort(tb.patch.begin(), tb.patch.end()); /* disjoint ranges: every node once */
    std::vector<std::pair<size_t, size_t>> merged;
    for (auto& r : tb.patch) {
        if (!merged.empty() && r.first <= merged.back().second)
            merged.back().second = r.second > merged.back().second ? r.second : merged.back().second;
        else merged.push_back(r);
    }
    for (auto& r : merged) {
        const size_t lo = r.first, hi = r.second < cm.ref_n ? r.second : cm.ref_n;
        if (hi <= lo) continue;
        rg.push_back(make_uint2((uint32_t) lo, (uint32_t) hi));
        roff.push_back((uint32_t) total);
        total += hi - lo;
    }
    if (total > (1u << 28)) return QBT_OK; /* as much work as a relayout */
    /* a grow entry per dirty node, up to 8 new children each */
    const uint64_t newcap64 = total * 8 < (1u << 26) ? total * 8 + 8 : (1u << 26);
    const uint32_t newcap   = (uint32_t) newcap64;
    auto           al       = [](size_t b) { return (b + 255) & ~(size_t) 255; };
    const size_t   o_ps = 0, o_rg = o_ps + al(PS_WORDS * 4), o_ro = o_rg + al(rg.size() * 8 + 8);
    const size_t   o_gr = o_ro + al(roff.size() * 4 + 4), o_nl = o_gr + al(total * 16 + 16);
    if ((rc = dev_alloc(cm.scratch, o_nl + (size_t) newcap * 8))) return rc;
    char*     sb   = (char*) cm.scratch.p;
    unsigned* ps   = (unsigned*) (sb + o_ps);
    uint2*    drg  = (uint2*) (sb + o_rg);
    uint32_t* dro  = (uint32_t*) (sb + o_ro);
    uint4*    grow = (uint4*) (sb + o_gr);
    uint2*    newl = (uint2*) (sb + o_nl);
    unsigned  hps[PS_WORDS] = {0};
    hps[PS_LEN]             = (unsigned) cm.n;
    HIPCHK(hipMemcpyAsync(ps, hps, sizeof(hps), hipMemcpyHostToDevice, s));
    if (!rg.empty()) {
        HIPCHK(hipMemcpyAsync(drg, rg.data(), rg.size() * 8, hipMemcpyHostToDevice, s));
        HIPCHK(hipMemcpyAsync(dro, roff.data(), roff.size() * 4, hipMemcpyHostToDevice, s));
    }
    if (n > cm.ref_n) /* nodes appended since the layout: not in the tree yet */
        k_fill32<<<nblk(n - cm.ref_n), 256, 0, s>>>((uint32_t*) cm.r2c.p + cm.ref_n, n - cm.ref_n, ~0u);
    const int4* ch = (const int4*) tb.child.p;
    const int*  md = (const int*) tb.model.p;
    uint2*      rc_ = (uint2*) cm.rec.p;
    int*        mc = (int*) cm.model.p;
    int*        rf = (int*) cm.ref.p;
    int*        r2 = (int*) cm.r2c.p;
    if (total) {
        const unsigned nb = nblk(total);
        k_patch_live<<<nb, 256, 0, s>>>(drg, dro, (int) rg.size(), (uint32_t) total, cm.ref_n, ch, md, rc_, mc, rf, r2,
                                        grow, ps);
        k_patch_grow<<<nb, 256, 0, s>>>(grow, n, ch, md, rc_, mc, rf, r2, (uint32_t) cm.cap, newl, newcap, ps);
        k_patch_commit<<<nb, 256, 0, s>>>(grow, rc_, r2, ps);
        k_patch_new<<<nblk(newcap), 256, 0, s>>>(newl, newcap, n, ch, md, rc_, mc, rf, r2, (uint32_t) cm.cap, ps);
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(hps, ps, 4 * 4, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    tb.patch.clear();
    if (hps[PS_FAIL]) return QBT_OK;
    cm.n     = hps[PS_LEN];
    cm.ref_n = n;
    tb.patches++;
    *done = true;
    return QBT_OK;
}
