/*
 * trace.hpp - per-ray sparse-octree traversal for gfx950.
 *
 * Semantics (template parameter SEM): cube_trace_line of
 * src/qubatron/shaders/octree_fsh.c:138-379 (static + dynamic tree in
 * lockstep), octree_trace_line of src/qubatron/octree.c:341-537, or the
 * particle shader's copy (src/qubatron/shaders/particle_vsh.c:121-343: one
 * tree, (0, 0, 0, 0) plane-test defaults, its slot address). Results (leaf node, entry point bits,
 * miss/discard) are identical to the reference algorithm; only the storage
 * differs:
 *
 *  - The reference keeps per level the cube, four pending entry points
 *    (4 x float4) and octets, the `ispsi` word and two node indices
 *    (~108 B/level, octree_fsh.c:50-58). Here a level holds one 32-bit
 *    pending word + the node index (8 B/level, 12 with the dynamic tree) in
 *    LDS: the cube is a function of the integer cell coordinates (ix, iy, iz)
 *    of the current node, and every pending point is re-derived from the
 *    plane that produced it (same inputs, same fp32 operations, so the same
 *    bits): a mid-plane hit of that level's node, or the node's entry point,
 *    which is the point that was popped one level up (followed upwards to
 *    the root entry).
 *  - The node array is split into a 32-byte child block per node (two int4,
 *    one aligned 32 B gather per expansion) and an int32 model index array.
 *
 * Pending word: bits 0-2 count n, bits 3-5 next index k, entry j at bit
 * 8+5j: octet (3 bits) | source << 3 (0 = node entry point, 1 = z, 2 = x,
 * 3 = y mid-plane).
 *
 * Compile with -ffp-contract=off; fp32 division and sqrt correctly rounded.
 */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#pragma clang fp contract(off)

namespace qbt {

constexpr int kMaxLevel = 24;
constexpr float kFltMax = 3.402823466e+38f;

/* traversal semantics */
enum : int {
    kSemShader   = 0, /* octree_fsh.c */
    kSemCpu      = 1, /* octree.c octree_trace_line */
    kSemParticle = 2  /* particle_vsh.c */
};

/* An empty volatile asm on a value: the compiler must keep what depends on
 * it inside its branch (a rarely taken slow path would otherwise be
 * if-converted and computed on every lane). The host test build of this
 * header defines it as nothing. */
#ifndef QBT_OPAQUE
#define QBT_OPAQUE(x) asm volatile("" : "+v"(x))
#endif

enum TraceStatus : int { ST_MISS = 0, ST_HIT = 1, ST_DISCARD = -1, ST_ABORT = -2 };

struct TreeDev {
    const int4* __restrict__ child; /* direct layout: 2 per node */
    const int* __restrict__ model;  /* slot 8, 1 per node (of the layout traversed) */
    int n;                          /* node count of the layout traversed */
    const uint2* __restrict__ rec;  /* compact layout: {first child, live | alloc << 8} */
    const int* __restrict__ ref;    /* compact layout: reference node index */
};

struct AttrDev {
    const float4* __restrict__ ca; /* [2m] = colour (r,g,b,1), [2m+1] = normal (x,y,z,1) */
    int n;
};

struct SceneDev {
    TreeDev stat, dyn;
    AttrDev astat, adyn;
    float bx, by, bz, bw; /* basecube */
    int maxlevel;
    int iter_cap;
    int dyn_wide; /* both trees on compact layouts, the dynamic one of kDualRecords records or more (trace_step_c2) */
};

struct Ray {
    float px, py, pz, dx, dy, dz;
    float ix, iy, iz; /* RN(1/d) per axis (set by trace_begin), NaN where not usable */
};

/* RN(1 / d) when |d| is in [2^-20, 2^100] (the reciprocal is then a
 * normal number of magnitude at most 2^20), else NaN so that plane_k takes
 * the division */
__device__ __forceinline__ float recip_or_nan(float d)
{
    const float a = fabsf(d);
    return (a >= 0x1p-20f && a <= 0x1p+100f) ? 1.0f / d : __builtin_nanf("");
}

/* Plane test on axis k (0 x, 1 y, 2 z) at coordinate c: is_cube_xplane,
 * is_cube_yplane and is_cube_zplane (octree_fsh.c:62-99 / octree.c:302-339)
 * in one form. t = (c - p_k) / d_k; the other two coordinates are
 * p_j + d_j t, coordinate k is c; d_k == 0 gives the octree.c twin's
 * defaults (0, 0, 0, t = FLT_MAX), the particle shader's (0, 0, 0, 0)
 * (particle_vsh.c:64-65), and NaN in shader semantics (see below).
 *
 * The quotient is the correctly rounded one, as the reference's division,
 * from y = RN(1 / d_k): q = RN(a y), e = RN(a - d_k q) (one FMA),
 * t = RN(q + e y) (one FMA), a Markstein-style correction. It is taken
 * where |d_k| is in [2^-20, 2^100] (y not NaN) and |q| is in [2^-80, 2^120].
 * There |y| <= 2^20, so |a| >= |q| / (|y| (1 + 2^-24)) > 2^-101: y, q and t
 * are normal numbers and e is exact (a - d_k q is a multiple of
 * 2^(e_a - 47) >= 2^-148), so each step scales with the exponents of a and
 * d_k, and t is correct for all such operands exactly when it is for every
 * pair of significands in [1, 2). All 2^46
 * pairs are checked on the device (tests/test_gpu_quotient.py) and a sample
 * on the host (tests/test_quotient.py). Elsewhere, and where y is NaN, the
 * quotient is the division itself, on a branch that rays rarely take.
 * Everything else is selects, so that lanes of a wave do not split on the
 * axis or on d_k == 0. */
/* component k by value (a conditional over the Ray's members would select an
 * address and keep the Ray in scratch memory) */
__device__ __forceinline__ float axis3(int k, float x, float y, float z)
{
    return k == 0 ? x : (k == 1 ? y : z);
}

template <int SEM>
__device__ __forceinline__ float4 plane_k(int k, float c, const Ray& r)
{
    const float p  = axis3(k, r.px, r.py, r.pz);
    const float d  = axis3(k, r.dx, r.dy, r.dz);
    const float y  = axis3(k, r.ix, r.iy, r.iz);
    const float a  = c - p;
    const float q  = a * y;
    const float e  = __builtin_fmaf(-q, d, a);
    float       t  = __builtin_fmaf(e, y, q);
    const float aq = fabsf(q);
    const bool  ok = d != 0.0f;
    if (!(aq >= 0x1p-80f && aq <= 0x1p+120f) && ok) {
        float aa = a, dd = d;
        QBT_OPAQUE(aa);
        QBT_OPAQUE(dd);
        t = aa / dd;
    }
    const float X = r.px + r.dx * t, Y = r.py + r.dy * t, Z = r.pz + r.dz * t;
    float4      o;
    o.x = k == 0 ? c : X;
    o.y = k == 1 ? c : Y;
    o.z = k == 2 ? c : Z;
    o.w = t;
    if (SEM != kSemShader) { /* these defaults can pass the containment tests */
        o.x = ok ? o.x : 0.0f;
        o.y = ok ? o.y : 0.0f;
        o.z = ok ? o.z : 0.0f;
        o.w = ok ? o.w : (SEM == kSemCpu ? kFltMax : 0.0f);
    }
    /* Shader semantics: where d_k == 0, y is NaN and so are t and the other
     * two coordinates; every caller tests t > 0 and the containment of the
     * point before using it, and those comparisons are false for NaN just
     * as they are for the shader's FLT_MAX defaults (octree_fsh.c:64).
     * No select is spent on the defaults. */
    return o;
}

template <int SEM>
__device__ __forceinline__ float4 plane_x(float c, const Ray& r) { return plane_k<SEM>(0, c, r); }
template <int SEM>
__device__ __forceinline__ float4 plane_y(float c, const Ray& r) { return plane_k<SEM>(1, c, r); }
template <int SEM>
__device__ __forceinline__ float4 plane_z(float c, const Ray& r) { return plane_k<SEM>(2, c, r); }

struct Hit {
    float4 isp;
    int ns, nd;     /* leaf node indices (static, dynamic) as the shader holds them */
    int ix, iy, iz; /* leaf cell coordinates */
    unsigned exps;  /* node expansions */
};

/* Node cube (tlf x, y, z) at `level` with cell coordinates (ix, iy, iz).
 * GRID: every coordinate of the subdivision is an exact fp32 multiple of the
 * leaf edge (checked on the host), so x = bx + ix*w is the value the
 * reference's running sum reaches. Otherwise the running sum of the
 * reference (tlf.x += xsft*halfs, octree_fsh.c:342-347) is replayed from the
 * root along the path bits. */
template <bool GRID>
__device__ __forceinline__ void cube_at(const SceneDev& s, int level, int ix, int iy, int iz, float& x, float& y,
                                        float& z, float& w)
{
    w = ldexpf(s.bw, -level);
    if (GRID) { /* i * w is exact, so the FMA rounds as the separate add */
        x = __builtin_fmaf((float) ix, w, s.bx);
        y = __builtin_fmaf(-(float) iy, w, s.by);
        z = __builtin_fmaf(-(float) iz, w, s.bz);
    } else {
        x = s.bx, y = s.by, z = s.bz;
        for (int l = 0; l < level; l++) {
            float h  = ldexpf(s.bw, -(l + 1));
            int   sh = level - 1 - l;
            x        = x + (float) ((ix >> sh) & 1) * h;
            y        = y - (float) ((iy >> sh) & 1) * h;
            z        = z - (float) ((iz >> sh) & 1) * h;
        }
    }
}

/* Far corner (bxx, byy, bzz) and mid-planes (hx, hy, hz) of the node cube
 * (x, y, z, w), as the shader computes them (octree_fsh.c:255-256:
 * h = b + (t - b) * 0.5). On an exact grid every one of these values is a
 * multiple of the leaf edge that fp32 holds exactly, so h = t +- w / 2 is
 * the same number in one FMA. */
template <bool GRID>
__device__ __forceinline__ void cube_mid(float x, float y, float z, float w, float& bxx, float& byy, float& bzz,
                                         float& hx, float& hy, float& hz)
{
    bxx = x + w, byy = y - w, bzz = z - w;
    if (GRID) {
        hx = __builtin_fmaf(0.5f, w, x);
        hy = __builtin_fmaf(-0.5f, w, y);
        hz = __builtin_fmaf(-0.5f, w, z);
    } else {
        hx = bxx + (x - bxx) * 0.5f;
        hy = byy + (y - byy) * 0.5f;
        hz = bzz + (z - bzz) * 0.5f;
    }
}

/* Mid-plane hit `src` (1 z, 2 x, 3 y) of the node cube (x, y, z, w). */
template <int SEM, bool GRID>
__device__ __forceinline__ float4 midplane(int src, const Ray& r, float x, float y, float z, float w)
{
    float bxx, byy, bzz, hx, hy, hz;
    cube_mid<GRID>(x, y, z, w, bxx, byy, bzz, hx, hy, hz);
    const int   k = src == 1 ? 2 : src - 2; /* src 1 z, 2 x, 3 y */
    const float c = src == 1 ? hz : (src == 2 ? hx : hy);
    return plane_k<SEM>(k, c, r);
}

/* midplane() of the cube at `level` whose cell coordinates are (ix, iy,
 * iz) >> sh. On the closed-form grid only the plane's own coordinate of the
 * cube is formed, by the two FMAs that cube_at and cube_mid apply to it (the
 * sign folded into the exact product), so the bits are the same. */
template <int SEM, bool GRID>
__device__ __forceinline__ float4 midplane_cell(const SceneDev& s, const Ray& r, int src, int level, int ix, int iy,
                                                int iz, int sh)
{
    if constexpr (GRID) {
        const int   k  = src == 1 ? 2 : src - 2; /* src 1 z, 2 x, 3 y */
        const int   ci = (k == 0 ? ix : (k == 1 ? iy : iz)) >> sh;
        const float w  = ldexpf(s.bw, -level);
        const float sg = k == 0 ? 1.0f : -1.0f; /* x grows along +x, y and z along -y, -z */
        const float c0 = __builtin_fmaf(sg * (float) ci, w, axis3(k, s.bx, s.by, s.bz));
        return plane_k<SEM>(k, __builtin_fmaf(sg * 0.5f, w, c0), r);
    } else {
        float x, y, z, ww;
        cube_at<GRID>(s, level, ix >> sh, iy >> sh, iz >> sh, x, y, z, ww);
        return midplane<SEM, GRID>(src, r, x, y, z, ww);
    }
}

/* component selects by value (a conditional over lvalues selects an address
 * and forces the operands into scratch memory) */
__device__ __forceinline__ int sel(bool c, int a, int b) { return c ? a : b; }
__device__ __forceinline__ int pick4(int x, int y, int z, int w, int k)
{
    return sel(k == 0, x, sel(k == 1, y, sel(k == 2, z, w)));
}
__device__ __forceinline__ int pick8(int4 lo, int4 hi, int o)
{
    const bool h = (o & 4) != 0;
    return pick4(sel(h, hi.x, lo.x), sel(h, hi.y, lo.y), sel(h, hi.z, lo.z), sel(h, hi.w, lo.w), o & 3);
}
__device__ __forceinline__ unsigned exist_mask(int4 lo, int4 hi)
{
    return (lo.x > 0 ? 1u : 0u) | (lo.y > 0 ? 2u : 0u) | (lo.z > 0 ? 4u : 0u) | (lo.w > 0 ? 8u : 0u) |
           (hi.x > 0 ? 16u : 0u) | (hi.y > 0 ? 32u : 0u) | (hi.z > 0 ? 64u : 0u) | (hi.w > 0 ? 128u : 0u);
}

/* The child block of one node in the direct layout: 8 child indices. */
struct Block {
    int4 lo, hi;
    __device__ __forceinline__ void clear() { lo = hi = make_int4(0, 0, 0, 0); }
    __device__ __forceinline__ void load(const TreeDev& t, int i)
    {
        const int4* p = t.child + 2 * (size_t) i;
        lo            = p[0];
        hi            = p[1];
    }
    __device__ __forceinline__ unsigned mask() const { return exist_mask(lo, hi); }
    __device__ __forceinline__ int      child(int o) const { return pick8(lo, hi, o); }
};

/* Compact record: x = index of the first child; y bits 0-7 = the children
 * that exist (live), bits 8-15 = the slots of the child block (alloc): child
 * o is record x + (the number of alloc bits below o). Live is a subset of
 * alloc; they differ only where an in-place range update zeroed a slot and
 * left its record in the block. */

/* The particle shader addresses slot k of node i as texel
 * (3 i mod 8192 + k / 4, 3 i / 8192) (particle_vsh.c:110-119): the texel
 * column does not carry into the next row, so for a node whose three texels
 * straddle a row end the column passes 8191. Such a fetch is outside the
 * texture, for which GLSL ES leaves the result undefined; here it reads 0,
 * the value of a robust-access fetch. Slots 0-7 are affected only where
 * 3 i mod 8192 == 8191 (slots 4-7), the model index (slot 8) also where
 * 3 i mod 8192 == 8190. */
__device__ __forceinline__ bool particle_hi_lost(int i) { return ((uint32_t) i * 3u) % 8192u == 8191u; }
__device__ __forceinline__ bool particle_model_lost(int i) { return ((uint32_t) i * 3u) % 8192u >= 8190u; }

/* the child block of node i as the semantics SEM reads it */
template <int SEM>
__device__ __forceinline__ void load_block(Block& b, const TreeDev& t, int i)
{
    b.load(t, i);
    if (SEM == kSemParticle && particle_hi_lost(i)) b.hi = make_int4(0, 0, 0, 0);
}

/* slot k (< 8) of node i at `level` (oct_from_octets_for_index,
 * octree_fsh.c:127-136): 0 for index 0 below the root. */
template <int SEM>
__device__ __forceinline__ int child_slot(const TreeDev& t, int i, int k, int level)
{
    if (i == 0 && level > 0) return 0;
    Block b;
    load_block<SEM>(b, t, i);
    return b.child(k);
}

/* The calling lane's stack: the entry word, the node word and the dynamic
 * node word of level l are pw[l * stride], ns[l * stride], nd[l * stride]. */
struct Stack {
    uint32_t* pw;
    int* ns;
    int* nd;
    int stride;
    /* l * stride: both are far below 2^24, so a full-rate 24-bit product (a
     * 32-bit one takes four times as long) */
    __device__ __forceinline__ int at(int l) const
    {
#ifdef __HIP__
        return (int) __umul24((unsigned) l, (unsigned) stride);
#else
        return l * stride;
#endif
    }
};

/* Root entry point of a ray, recomputed from the face that trace_begin found
 * (the same operations, so the same bits): its plane, 1 x, 2 y, 3 z, 0 the ray
 * starts in the cube, and 4 for the far one. A face is three bits where the
 * point is four registers. */
template <int SEM>
__device__ __forceinline__ float4 root_entry(const SceneDev& s, const Ray& r, int face)
{
    if (face == 0) return make_float4(r.px, r.py, r.pz, 0.0f);
    const int   k = (face & 3) - 1;
    const float b = axis3(k, s.bx, s.by, s.bz), f = k == 0 ? b + s.bw : b - s.bw;
    return plane_k<SEM>(k, (face & 4) ? f : b, r);
}

/* Entry point of the node at `level` on the current path (level >= 1 uses
 * the entry popped one level up). */
template <int SEM, bool GRID>
__device__ __forceinline__ float4 entry_of(const SceneDev& s, const Ray& r, const Stack& st, int level, int ix, int iy,
                                        int iz, int face)
{
    for (int m = level; m > 0; m--) {
        uint32_t w   = st.pw[(m - 1) * st.stride];
        int      k   = (int) ((w >> 3) & 7u) - 1;
        int      src = (int) ((w >> (8 + 5 * k + 3)) & 3u);
        if (src != 0) return midplane_cell<SEM, GRID>(s, r, src, m - 1, ix, iy, iz, level - (m - 1));
    }
    return root_entry<SEM>(s, r, face);
}

/* Resumable traversal state of one ray (registers; the per-level pending
 * words and node indices live in the LDS Stack). */
struct TraceState {
    float4   entry; /* entry point of the current node */
    int      level, ix, iy, iz;
    int      ns, nd; /* current static / dynamic node */
    int      it;
    unsigned exps;
    uint32_t pend; /* bit l set while level l has pending entries; kSlowRay; bits 28-30 the root face (root_entry) */
};

enum : int { ST_CONT = 2 };

/* from this many records of the dynamic compact layout on, a stack word does
 * not hold a first child beside the block's slots (trace_step_c2) */
constexpr uint32_t kDualRecords = 1u << 24;

constexpr uint32_t kSlowRay   = 0x80000000u; /* in pend: the ray's quotients need plane_k's check */
constexpr int      kFaceShift = 28;
constexpr uint32_t kRayBits   = 0xF0000000u; /* what pend holds of the ray, not of the path */
__device__ __forceinline__ int root_face(const TraceState& t) { return (int) ((t.pend >> kFaceShift) & 7u); }

/* Whether the quotients (c - p_k) / d_k of all mid-planes of an exact grid
 * are in the domain in which plane_k needs no division (or the axis has
 * d_k == 0, in shader semantics). c is a multiple of the leaf edge u, and so
 * of 2^-43 when u >= 2^-20, and p_k is one when it is 0 or |p_k| >= 2^-20:
 * a = c - p_k is then 0 or at least 2^-43, and at most 2^62 with |p_k| and the
 * cube below 2^61. With |d_k| in [2^-20, 2^30] the quotient is 0 or in
 * [2^-74, 2^83], inside the domain; for a = 0 (+0 as every difference of equal
 * numbers) the products give 0 with the sign of d_k, as the division does. */
template <int SEM>
__device__ __forceinline__ bool quot_safe(const SceneDev& s, const Ray& r)
{
    auto axis = [](float p, float d) {
        const float a = fabsf(d), b = fabsf(p);
        return ((a >= 0x1p-20f && a <= 0x1p+30f) || (SEM == kSemShader && a == 0.0f)) &&
               ((b >= 0x1p-20f && b <= 0x1p+61f) || b == 0.0f);
    };
    const bool cube = ldexpf(s.bw, -s.maxlevel) >= 0x1p-20f && s.bw <= 0x1p+60f && fabsf(s.bx) <= 0x1p+60f &&
                      fabsf(s.by) <= 0x1p+60f && fabsf(s.bz) <= 0x1p+60f;
    return cube && axis(r.px, r.dx) && axis(r.py, r.dy) && axis(r.pz, r.dz);
}

/* plane_k's quotient without its check (quot_safe) */
__device__ __forceinline__ float quot(float c, float p, float d, float y)
{
    const float a = c - p, q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-q, d, a), y, q);
}

/* Root entry (octree_fsh.c:157-211). Returns ST_CONT, ST_HIT (maxlevel 0)
 * or ST_DISCARD. */
template <int SEM>
__device__ __forceinline__ int trace_begin(const SceneDev& s, Ray& r, TraceState& t)
{
    r.ix = recip_or_nan(r.dx);
    r.iy = recip_or_nan(r.dy);
    r.iz = recip_or_nan(r.dz);
    float4 h0 = make_float4(0.f, 0.f, 0.f, 0.f), h1 = h0;
    int    hitc = 0, f0 = 0, f1 = 0;
    {
        const float tx = s.bx, ty = s.by, tz = s.bz, tw = s.bw;
        const float rx = tx + tw, ry = ty - tw, rz = tz - tw;
        float4      a;
#define QBT_CONSIDER(face, cond)                 \
    if ((SEM != kSemCpu || a.w < kFltMax) && (cond)) { \
        if (hitc == 0) h0 = a, f0 = face;        \
        else if (hitc == 1) h1 = a, f1 = face;   \
        hitc++;                                  \
    }
        a = plane_z<SEM>(tz, r);
        QBT_CONSIDER(3, tx < a.x && a.x <= rx && ty > a.y && a.y >= ry)
        a = plane_z<SEM>(rz, r);
        QBT_CONSIDER(7, tx < a.x && a.x <= rx && ty > a.y && a.y >= ry)
        a = plane_x<SEM>(tx, r);
        QBT_CONSIDER(1, ty > a.y && a.y >= ry && tz > a.z && a.z >= rz)
        a = plane_x<SEM>(rx, r);
        QBT_CONSIDER(5, ty > a.y && a.y >= ry && tz > a.z && a.z >= rz)
        a = plane_y<SEM>(ty, r);
        QBT_CONSIDER(2, tx < a.x && a.x <= rx && tz > a.z && a.z >= rz)
        a = plane_y<SEM>(ry, r);
        QBT_CONSIDER(6, tx < a.x && a.x <= rx && tz > a.z && a.z >= rz)
#undef QBT_CONSIDER
    }
    t.exps = 0;
    if (hitc < 2) return ST_DISCARD;
    if (h0.w < 0.0f && h1.w < 0.0f) return ST_DISCARD;
    if (h1.w < h0.w) h0 = h1, f0 = f1;
    if (h0.w < 0.0f) h0 = make_float4(r.px, r.py, r.pz, 0.0f), f0 = 0;
    t.entry = h0;
    t.level = t.ix = t.iy = t.iz = 0;
    t.ns = t.nd = 0;
    t.it   = 0;
    t.pend = (quot_safe<SEM>(s, r) ? 0u : kSlowRay) | (uint32_t) f0 << kFaceShift;
    return s.maxlevel == 0 ? ST_HIT : ST_CONT;
}

/*
 * Single-tree steps on the compact layout (the hot configuration) keep a
 * different per-level encoding, so that backtracking never re-reads a node:
 *   ns word  first child index of the level's node (bits 0-29) | entries
 *            still pending (bits 30-31, 0..3)
 *   pw word  the entry being visited (bits 0-5), then up to three pending
 *            entries (bits 6-11, 12-17, 18-23); an entry is octet (3 bits) |
 *            plane << 3 (3 bits: 0 the node's entry point, 1 x, 2 y, 4 z
 *            mid-plane, the octet bit that the plane separates); bits 24-31
 *            hold the slots of the node's child block (alloc), so the child of
 *            octet o is first + (the number of those bits below o), counted
 *            when the entry is taken.
 * A per-lane bit mask marks the levels that still hold pending entries, so a
 * backtrack finds its level with one count-leading-zeros instead of a loop
 * over the stack.
 */
/* candidate src (0 entry, 1 z, 2 x, 3 y) by value: a conditional over the
 * lvalues would select an address and keep the candidates in scratch memory */
__device__ __forceinline__ float4 pick_entry(int src, float4 e, float4 z, float4 x, float4 y)
{
    float4 r = e;
    if (src == 1) r = z;
    if (src == 2) r = x;
    if (src == 3) r = y;
    return r;
}

/* the highest set bit of m, which is not 0 */
__device__ __forceinline__ int top_bit(uint32_t m) { return 31 - __builtin_clz(m); }

/* bit o of m (one bit-field extract) */
__device__ __forceinline__ bool bit_of(uint32_t m, int o) { return __builtin_amdgcn_ubfe(m, (uint32_t) o, 1u) != 0u; }

__device__ __forceinline__ void kswap(float& wa, int& ka, float& wb, int& kb)
{
    const bool sw = wb < wa; /* strict: ties keep order (octree_fsh.c:283); NaN never moves */
    const float tw = sw ? wb : wa;
    const int   tk = sw ? kb : ka;
    wb             = sw ? wa : wb;
    kb             = sw ? ka : kb;
    wa             = tw;
    ka             = tk;
}

/* The octet of a candidate point and its tie-flipped octet
 * (octree_fsh.c:292-311): the flip toggles the bit of the first axis, in
 * x, y, z order, on which the point lies on the mid-plane (the lowest set
 * bit of the on-plane mask). Key = octet | src << 3 | flipped << 5. */
__device__ __forceinline__ int octet_key(float x, float y, float z, float hx, float hy, float hz, int src)
{
    const int o  = (x > hx ? 1 : 0) | (y < hy ? 2 : 0) | (z < hz ? 4 : 0);
    const int on = (x == hx ? 1 : 0) | (y == hy ? 2 : 0) | (z == hz ? 4 : 0);
    return o | (src << 3) | ((o ^ (on & -on)) << 5);
}

/* The same keys for the three mid-plane candidates, whose coordinate on
 * their own plane is the mid-plane value itself (plane_k sets it) wherever
 * the candidate is valid, so that one comparison of each is known: z == hz
 * for the z-plane hit, x == hx for the x-plane hit, y == hy for the y-plane
 * hit. (Keys of invalid candidates are never read.) */
__device__ __forceinline__ int zplane_key(float x, float y, float hx, float hy)
{
    const int o  = (x > hx ? 1 : 0) | (y < hy ? 2 : 0);
    const int fl = x == hx ? 1 : (y == hy ? 2 : 4);
    return o | (1 << 3) | ((o ^ fl) << 5);
}
__device__ __forceinline__ int xplane_key(float y, float z, float hy, float hz)
{
    const int o = (y < hy ? 2 : 0) | (z < hz ? 4 : 0);
    return o | (2 << 3) | ((o ^ 1) << 5);
}
__device__ __forceinline__ int yplane_key(float x, float z, float hx, float hz)
{
    const int o = (x > hx ? 1 : 0) | (z < hz ? 4 : 0);
    return o | (3 << 3) | ((o ^ (x == hx ? 1 : 2)) << 5);
}

/* The kept candidates of a node, in visiting order, as 6-bit entries (first
 * one lowest), and their number: the general form, for every quotient, order
 * and tie (octree_fsh.c:251-330). mask: the live children. */
template <int SEM, bool GRID>
__device__ __forceinline__ uint32_t expand_any(const SceneDev& s, const Ray& r, const TraceState& t, uint32_t mask, int& n)
{
    float tx, ty, tz, tw, bxx, byy, bzz, hx, hy, hz;
    cube_at<GRID>(s, t.level, t.ix, t.iy, t.iz, tx, ty, tz, tw);
    cube_mid<GRID>(tx, ty, tz, tw, bxx, byy, bzz, hx, hy, hz);
    const float  qnan = __builtin_nanf("");
    const float4 az = plane_z<SEM>(hz, r);
    const float4 ax = plane_x<SEM>(hx, r);
    const float4 ay = plane_y<SEM>(hy, r);
    float        w0 = t.entry.w;
    float        w1 = (az.w > 0.0f && tx < az.x && az.x <= bxx && ty > az.y && az.y >= byy) ? az.w : qnan;
    float        w2 = (ax.w > 0.0f && ty > ax.y && ax.y >= byy && tz > ax.z && ax.z >= bzz) ? ax.w : qnan;
    float        w3 = (ay.w > 0.0f && tx < ay.x && ay.x <= bxx && tz > ay.z && ay.z >= bzz) ? ay.w : qnan;
    /* the octree.c twin's defaults for d == 0 (0, 0, 0) can pass the
     * containment tests, so it keeps the general form */
    int k0 = octet_key(t.entry.x, t.entry.y, t.entry.z, hx, hy, hz, 0);
    int k1 = SEM != kSemShader ? octet_key(az.x, az.y, az.z, hx, hy, hz, 1) : zplane_key(az.x, az.y, hx, hy);
    int k2 = SEM != kSemShader ? octet_key(ax.x, ax.y, ax.z, hx, hy, hz, 2) : xplane_key(ax.y, ax.z, hy, hz);
    int k3 = SEM != kSemShader ? octet_key(ay.x, ay.y, ay.z, hx, hy, hz, 3) : yplane_key(ay.x, ay.z, hx, hz);
    /* sort network (octree_fsh.c:283, strict: ties keep their order); NaN
     * never moves, so slot 0 stays valid */
    kswap(w0, k0, w1, k1);
    kswap(w0, k0, w2, k2);
    kswap(w0, k0, w3, k3);
    kswap(w1, k1, w2, k2);
    kswap(w1, k1, w3, k3);
    kswap(w2, k2, w3, k3);
    /* walk the sorted candidates: an octet equal to the previous valid one
     * is replaced by its flipped octet; those whose child exists are kept */
    const bool v1 = w1 == w1, v2 = w2 == w2, v3 = w3 == w3;
    const int  o0 = k0 & 7;
    const int  o1 = (k1 & 7) == o0 ? ((k1 >> 5) & 7) : (k1 & 7);
    const int  p1 = v1 ? o1 : o0;
    const int  o2 = (k2 & 7) == p1 ? ((k2 >> 5) & 7) : (k2 & 7);
    const int  p2 = v2 ? o2 : p1;
    const int  o3 = (k3 & 7) == p2 ? ((k3 >> 5) & 7) : (k3 & 7);
    auto entry = [](int o, int k) -> uint32_t { /* source 1 z, 2 x, 3 y -> plane 4, 1, 2 */
        return (uint32_t) o | ((0x2140u >> (((uint32_t) k & 0x18u) >> 1)) & 7u) << 3;
    };
    const bool t0 = bit_of(mask, o0);
    const bool t1 = v1 && bit_of(mask, o1);
    const bool t2 = v2 && bit_of(mask, o2);
    const bool t3 = v3 && bit_of(mask, o3);
    uint32_t   word = t3 ? entry(o3, k3) : 0u;
    word            = t2 ? (word << 6) | entry(o2, k2) : word;
    word            = t1 ? (word << 6) | entry(o1, k1) : word;
    word            = t0 ? (word << 6) | entry(o0, k0) : word;
    n               = (t0 ? 1 : 0) + (t1 ? 1 : 0) + (t2 ? 1 : 0) + (t3 ? 1 : 0);
    return word;
}

/* The same on an exact grid for the ray and the node in general position,
 * which is nearly always: quotients in the safe domain, no candidate before
 * the entry point, none on a second mid-plane, and the octet bits of the
 * three mid-plane hits agreeing with their order along the ray. Then each
 * crossing flips the bit of its own plane and nothing else (the reference's
 * octet by coordinates, and its tie-flipped octet where that equals the one
 * before, come to the same), and the sort needs the keys alone. false where
 * any of this does not hold: the caller takes expand_any. The traversal of
 * large frames is bound by the issue of vector instructions (195 to 225 node
 * expansions per ns), so the step is written for their number: 118 to here
 * against 173 of expand_any and the checks of its quotients, one rare branch
 * instead of four. k_primary + k_shadow of a 2160p frame of 30M points took
 * 15.38 ms with expand_any alone, 15.07 with a first form of this (the keys
 * from the hits' coordinates, 135 instructions; 62 in plane_entry), 12.83 with
 * 118 and 44, 11.88 with 35 in plane_entry (the root's entry and ancestors'
 * planes off its common path); 200k free rays 238, 209, 190 and 183 us. */
__device__ __forceinline__ bool expand_general_position(const SceneDev& s, const Ray& r, const TraceState& t,
                                                        uint32_t mask, uint32_t& word, int& n)
{
    const float w  = ldexpf(s.bw, -t.level);
    const float tx = __builtin_fmaf((float) t.ix, w, s.bx), ty = __builtin_fmaf(-(float) t.iy, w, s.by),
                tz = __builtin_fmaf(-(float) t.iz, w, s.bz);
    float bxx, byy, bzz, hx, hy, hz;
    cube_mid<true>(tx, ty, tz, w, bxx, byy, bzz, hx, hy, hz);
    const float qz = quot(hz, r.pz, r.dz, r.iz), qx = quot(hx, r.px, r.dx, r.ix), qy = quot(hy, r.py, r.dy, r.iy);
    const float zx = r.px + r.dx * qz, zy = r.py + r.dy * qz; /* the z-plane hit */
    const float xy = r.py + r.dy * qx, xz = r.pz + r.dz * qx; /* the x-plane hit */
    const float yx = r.px + r.dx * qy, yz = r.pz + r.dz * qy; /* the y-plane hit */
    const bool  vz = (qz > 0.0f) & (tx < zx) & (zx <= bxx) & (ty > zy) & (zy >= byy);
    const bool  vx = (qx > 0.0f) & (ty > xy) & (xy >= byy) & (tz > xz) & (xz >= bzz);
    const bool  vy = (qy > 0.0f) & (tx < yx) & (yx <= bxx) & (tz > yz) & (yz >= bzz);
    const float inf = __builtin_inff();
    const float wz = vz ? qz : inf, wx = vx ? qx : inf, wy = vy ? qy : inf;
    const bool  ex = t.entry.x > hx, ey = t.entry.y < hy, ez = t.entry.z < hz;
    const bool  gzx = zx > hx, gzy = zy < hy, gxy = xy < hy, gxz = xz < hz, gyx = yx > hx, gyz = yz < hz;
    /* the order of the hits; ties as the network leaves them: z, x, y, but
     * for z and x level behind y */
    const bool xbz = wx < wz, ybz = wy < wz, ybx = wy < wx;
    /* (logical operators: as numbers the conditions would go through vector
     * registers) */
    const bool slow = (t.pend & kSlowRay) != 0u, early = fminf(fminf(wz, wx), wy) < t.entry.w;
    const bool tie = (zx == hx) || (zy == hy) || (yx == hx), level = (wx == wz) && vz && ybx;
    const bool mz = vz && ((gzx != (ex != xbz)) || (gzy != (ey != ybz)));
    const bool mx = vx && ((gxz != (ez != !xbz)) || (gxy != (ey != ybx)));
    const bool my = vy && ((gyz != (ez != !ybz)) || (gyx != (ex != !ybx)));
    const bool bad = slow || early || tie || level || mz || mx || my;
    /* the crossings in order, c = plane << 3 | plane, or 24 for none (it sorts
     * last): each flips its bit of the octet before and gives its entry;
     * behind the last one an octet that the mask does not have */
    const uint32_t o0 = (ex ? 1u : 0u) | (ey ? 2u : 0u) | (ez ? 4u : 0u);
    const uint32_t cz = vz ? 36u : 24u, cx = vx ? 9u : 24u, cy = vy ? 18u : 24u;
    const uint32_t c1 = xbz ? (ybx ? cy : cx) : (ybz ? cy : cz);
    const uint32_t c3 = xbz ? (ybz ? cz : cy) : (ybx ? cx : cy);
    const uint32_t c2 = cz ^ cx ^ cy ^ c1 ^ c3;
    const uint32_t k1 = o0 ^ c1, k2 = (k1 & 7u) ^ c2, k3 = (k2 & 7u) ^ c3;
    /* the live mask once per plane: an entry's low five bits (octet and x, y
     * plane bits) are its bit, 24..31 (no candidate) are zero */
    const uint32_t m3 = mask | mask << 8 | mask << 16;
    const bool     t0 = bit_of(mask, (int) o0), t1 = bit_of(m3, (int) k1), t2 = bit_of(m3, (int) k2), t3 = bit_of(m3, (int) k3);
    uint32_t       e  = t3 ? k3 : 0u;
    e                 = t2 ? (e << 6) | k2 : e;
    e                 = t1 ? (e << 6) | k1 : e;
    word              = t0 ? (e << 6) | o0 : e;
    n                 = (t0 ? 1 : 0) + (t1 ? 1 : 0) + (t2 ? 1 : 0) + (t3 ? 1 : 0);
    return !bad;
}

/* Entry point of an entry whose plane is `plane` (1 x, 2 y, 3 or 4 z) of the
 * node at level lv of the path, with cell coordinates (sx, sy, sz):
 * midplane_cell's, the quotient unchecked where the ray allows. On an exact
 * grid the mid-plane's coordinate is one FMA: base +- (2 i + 1) w / 2 is a
 * number that fp32 holds. Plane 0, the node's own entry point (a backtracking
 * lane needs it in rare orders of a node's candidates only): the mid-plane hit
 * of the nearest node on the path entered through one (plane_of reads that of
 * a level), else the root entry. */
template <int SEM, bool GRID, class PlaneOf>
__device__ __forceinline__ float4 plane_entry(const SceneDev& s, const Ray& r, const TraceState& t, int plane, int lv,
                                              int sx, int sy, int sz, PlaneOf&& plane_of)
{
    if (!GRID || plane == 0 || (t.pend & kSlowRay) != 0u) {
        int j = lv;
        while (plane == 0 && j > 0) {
            j--;
            plane = plane_of(j);
        }
        return plane == 0 ? root_entry<SEM>(s, r, root_face(t))
                          : midplane_cell<SEM, GRID>(s, r, plane == 1 ? 2 : (plane == 2 ? 3 : 1), j, sx, sy, sz, lv - j);
    }
    const bool  px = plane == 1, py = plane == 2;
    const int   m  = 2 * sel(px, sx, sel(py, sy, sz)) + 1;
    const float h = ldexpf(s.bw, -1 - lv);
    const float bx = s.bx, by = s.by, bz = s.bz;
    const float c = __builtin_fmaf((float) m, px ? h : -h, px ? bx : (py ? by : bz));
    /* values, not the ray's members: a select between members is a load from
     * a selected address, and the ray then lives in memory */
    const float ox = r.px, oy = r.py, oz = r.pz, dx = r.dx, dy = r.dy, dz = r.dz, jx = r.ix, jy = r.iy, jz = r.iz;
    const float q = quot(c, px ? ox : (py ? oy : oz), px ? dx : (py ? dy : dz), px ? jx : (py ? jy : jz));
    const float X = r.px + r.dx * q, Y = r.py + r.dy * q, Z = r.pz + r.dz * q;
    float4      o;
    o.x = px ? c : X;
    o.y = py ? c : Y;
    o.z = (px || py) ? Z : c;
    o.w = q;
    return o;
}

/* The step does not count itself in t.it: its callers do, by the burst (the
 * compact layout is a proper tree, so a ray ends by itself; the cap is
 * reached by very deep trees only). */
template <int SEM, bool GRID>
__device__ __forceinline__ int trace_step_c1(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t)
{
    const int   level = t.level;
    const uint2 rec   = s.stat.rec[(uint32_t) t.ns]; /* node indices are non-negative: no sign extension */
    t.exps++;
    const uint32_t mask = rec.y & 0xFFu; /* live children; 0 for the root of an empty tree: no candidate taken */
    uint32_t       word = 0;
    int            n    = 0;
    if (!GRID || !expand_general_position(s, r, t, mask, word, n)) word = expand_any<SEM, GRID>(s, r, t, mask, n);
    word |= (rec.y >> 8) << 24; /* the block's slots, for the rank of an entry's child */

    /* The entry to descend into: the first kept candidate, or, backtracking
     * (octree_fsh.c:368-375), the next pending entry of the nearest ancestor
     * that has one. Descending and backtracking lanes share one path (most
     * wave-steps hold both kinds): the level they work on is lv, whose two
     * stack words every lane reads and rewrites, and the new words, the
     * pending mask and the child block are selects. */
    const bool     desc  = n > 0;
    const uint32_t below = t.pend & ~kRayBits; /* levels at and below this one have none */
    if (!desc && below == 0u) return ST_MISS;
    /* the deepest level with a pending entry, from the per-lane mask (levels
     * between it and this one have none: no loop over them) */
    const int      lv  = desc ? level : top_bit(below);
    const int      at  = st.at(lv);
    const uint32_t an  = (uint32_t) st.ns[at];
    const uint32_t pwv = st.pw[at];
    /* backtracking: the next entry of level lv becomes the current one */
    const uint32_t w   = desc ? word : ((pwv & 0xFFFFFFu) >> 6) | (pwv & 0xFF000000u);
    const uint32_t nw = desc ? rec.x | (uint32_t) (n - 1) << 30 : an - (1u << 30);
    st.pw[at] = w;
    st.ns[at] = (int) nw;
    /* bit lv: whether the level still has a pending entry */
    t.pend = (t.pend & ~(1u << lv)) | (nw >= 1u << 30 ? 1u << lv : 0u);
    const uint32_t a = nw & 0x3FFFFFFFu;
    /* Its entry point: a descending lane with plane 0 keeps its own; else that
     * of the plane, recomputed (same operations as the candidate, so the same
     * bits). */
    const int plane = (int) ((w >> 3) & 7u), sh = level - lv, o = (int) (w & 7u);
    const int sx = t.ix >> sh, sy = t.iy >> sh, sz = t.iz >> sh;
    if (!desc || plane != 0)
        t.entry = plane_entry<SEM, GRID>(s, r, t, plane, lv, sx, sy, sz,
                                         [&](int l) { return (int) ((st.pw[st.at(l)] >> 3) & 7u); });
    t.ns    = (int) (a + (uint32_t) __popc(__builtin_amdgcn_ubfe(w, 24u, (uint32_t) o))); /* first + rank */
    t.ix    = (sx << 1) | (o & 1);
    t.iy    = (sy << 1) | ((o >> 1) & 1);
    t.iz    = (sz << 1) | (o >> 2);
    t.level = lv + 1;
    return t.level == s.maxlevel ? ST_HIT : ST_CONT;
}

/* The backtrack half of trace_step_c1 on its own: leave the current node and
 * enter the next pending entry of the deepest level below t.level that has
 * one (t.pend must name one). Used where a ray's pending entries are handed
 * to another lane (split.hpp). */
template <int SEM, bool GRID>
__device__ __forceinline__ int trace_pop_c1(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t)
{
    const int      level = t.level;
    const uint32_t below = t.pend & ((1u << level) - 1u);
    const int      lv    = 31 - __clz((int) below), at = st.at(lv);
    const uint32_t an    = (uint32_t) st.ns[at];
    const uint32_t pwv   = st.pw[at];
    const uint32_t w     = ((pwv & 0xFFFFFFu) >> 6) | (pwv & 0xFF000000u);
    st.pw[at] = w;
    st.ns[at] = (int) (an - (1u << 30));
    t.pend ^= an - (1u << 30) >= 1u << 30 ? 0u : 1u << lv;
    const int sh = level - lv, o = (int) (w & 7u), sx = t.ix >> sh, sy = t.iy >> sh, sz = t.iz >> sh;
    t.entry = plane_entry<SEM, GRID>(s, r, t, (int) ((w >> 3) & 7u), lv, sx, sy, sz,
                                     [&](int l) { return (int) ((st.pw[st.at(l)] >> 3) & 7u); });
    t.ns    = (int) ((an & 0x3FFFFFFFu) + (uint32_t) __popc(__builtin_amdgcn_ubfe(w, 24u, (uint32_t) o)));
    t.ix    = (sx << 1) | (o & 1);
    t.iy    = (sy << 1) | ((o >> 1) & 1);
    t.iz    = (sz << 1) | (o >> 2);
    t.level = lv + 1;
    return t.level == s.maxlevel ? ST_HIT : ST_CONT;
}

/*
 * Both trees on their compact layouts, in the manner of trace_step_c1: one
 * path for descending and backtracking lanes, and backtracking never re-reads
 * a node. The words of a level:
 *   pw word  up to three pending entries, 8 bits each, the next one lowest
 *            (0: none): octet | plane << 3 as above | the child exists in the
 *            static tree << 6, in the dynamic one << 7; bits 24-31 the static
 *            node's slots
 *   ns word  the static node's first child (30 bits) | the plane of the entry
 *            being visited << 30 (1 x, 2 y, 3 z, 0 the node's entry point)
 *   nd word  the dynamic node's first child (24 bits) | its slots << 24; with
 *            kDualRecords records or more (SceneDev::dyn_wide) the node's
 *            index, and its record is read again on a backtrack
 * A node index is 0 where the path has left its tree. Against the direct layout's step on compact records (separate
 * descend and backtrack paths, records read again on a backtrack), 720p over
 * 5M static and 150k dynamic points: k_primary 633 -> 548 us, 719 -> 603 and
 * 202 -> 200 (three poses), k_shadow 292 -> 247, 403 -> 342, 96 -> 88. Frames
 * of 5M static points and 28.9M dynamic records (the wide words): 0.64, 0.79
 * and 1.18 ms, against 0.89, 1.09 and 1.80 with both trees on the direct
 * layout; the test of dyn_wide costs narrow frames nothing (within 0.3%).
 */
/* the plane of an entry's bits 3-5 (one-hot) as a number: 1 x, 2 y, 3 z */
__device__ __forceinline__ uint32_t plane_code(uint32_t e)
{
    const uint32_t p = (e >> 3) & 7u;
    return p - (p >> 2);
}

/* the second half of a step: entry e (8 bits) of level lv becomes the current
 * one; an, pw and ad are that level's new words (an without the plane; ad of
 * a descending lane, keep, as the narrow form has it), rd the dynamic node's
 * record where the lane descends */
template <int SEM, bool GRID>
__device__ __forceinline__ int enter_c2(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t, bool keep,
                                        int lv, uint32_t e, uint32_t pw, uint32_t an, uint32_t ad, uint2 rd)
{
    const int at = st.at(lv), level = t.level;
    const int plane = (int) plane_code(e), sh = level - lv, o = (int) (e & 7u);
    const int sx = t.ix >> sh, sy = t.iy >> sh, sz = t.iz >> sh;
    st.pw[at] = pw;
    st.ns[at] = (int) (an | (uint32_t) plane << 30);
    if (!keep || plane != 0)
        t.entry = plane_entry<SEM, GRID>(s, r, t, plane, lv, sx, sy, sz,
                                         [&](int l) { return (int) ((uint32_t) st.ns[st.at(l)] >> 30); });
    const uint32_t cs = an + (uint32_t) __popc(__builtin_amdgcn_ubfe(pw, 24u, (uint32_t) o));
    uint32_t       cd = (ad & 0xFFFFFFu) + (uint32_t) __popc(__builtin_amdgcn_ubfe(ad, 24u, (uint32_t) o));
    if (s.dyn_wide) { /* uniform */
        if (keep) ad = (uint32_t) t.nd;
        else rd = s.dyn.rec[ad];
        cd = rd.x + (uint32_t) __popc(__builtin_amdgcn_ubfe(rd.y, 8u, (uint32_t) o));
    }
    st.nd[at] = (int) ad;
    t.ns    = (e & 64u) ? (int) cs : 0;
    t.nd    = (e & 128u) ? (int) cd : 0;
    t.ix    = (sx << 1) | (o & 1);
    t.iy    = (sy << 1) | ((o >> 1) & 1);
    t.iz    = (sz << 1) | (o >> 2);
    t.level = lv + 1;
    return t.level == s.maxlevel ? ST_HIT : ST_CONT;
}

template <int SEM, bool GRID>
__device__ __forceinline__ int trace_step_c2(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t)
{
    const int      level = t.level;
    const uint2    rs = s.stat.rec[(uint32_t) t.ns], rd = s.dyn.rec[(uint32_t) t.nd]; /* the root where there is none */
    const bool     hs = t.ns != 0 || level == 0, hd = t.nd != 0 || level == 0;
    const uint32_t ms = hs ? rs.y & 0xFFu : 0u, md = hd ? rd.y & 0xFFu : 0u;
    t.exps += (hs ? 1u : 0u) + (hd ? 1u : 0u);
    uint32_t word = 0;
    int      n    = 0;
    if (!GRID || !expand_general_position(s, r, t, ms | md, word, n)) word = expand_any<SEM, GRID>(s, r, t, ms | md, n);

    const bool     desc  = n > 0;
    const uint32_t below = t.pend & ~kRayBits; /* levels at and below this one have none */
    if (!desc && below == 0u) return ST_MISS;
    const int      lv  = desc ? level : top_bit(below);
    const int      at  = st.at(lv);
    const uint32_t pwv = st.pw[at], an = (uint32_t) st.ns[at], ad = (uint32_t) st.nd[at];
    /* the entries with their trees; entries past the n-th are dropped */
    const uint32_t mm = ms << 6 | md << 15; /* bit 6 + o, 15 + o */
    auto tree_bits = [&](uint32_t e) -> uint32_t {
        const uint32_t b = mm >> (e & 7u);
        return (b & 64u) | ((b >> 8) & 128u);
    };
    const uint32_t e0 = word & 63u, e1 = (word >> 6) & 63u, e2 = (word >> 12) & 63u, e3 = (word >> 18) & 63u;
    const uint32_t p  = (e1 | tree_bits(e1)) | (e2 | tree_bits(e2)) << 8 | (e3 | tree_bits(e3)) << 16;
    const uint32_t pn = p & ((1u << ((uint32_t) (8 * n - 8) & 31u)) - 1u);
    const uint32_t e  = desc ? e0 | tree_bits(e0) : pwv & 0xFFu;
    const uint32_t w  = desc ? pn | (rs.y >> 8) << 24 : ((pwv & 0xFFFFFFu) >> 8) | (pwv & 0xFF000000u);
    /* bit lv: whether the level still has a pending entry */
    t.pend = (t.pend & ~(1u << lv)) | ((w & 0xFFFFFFu) != 0u ? 1u << lv : 0u);
    return enter_c2<SEM, GRID>(s, r, st, t, desc, lv, e, w, desc ? rs.x : an & 0x3FFFFFFFu,
                               desc ? (rd.x & 0xFFFFFFu) | (rd.y >> 8) << 24 : ad, rd);
}

/* the backtrack half of trace_step_c2 (as trace_pop_c1) */
template <int SEM, bool GRID>
__device__ __forceinline__ int trace_pop_c2(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t)
{
    const uint32_t below = t.pend & ((1u << t.level) - 1u);
    const int      lv = top_bit(below), at = st.at(lv);
    const uint32_t pwv = st.pw[at], an = (uint32_t) st.ns[at], ad = (uint32_t) st.nd[at];
    const uint32_t w   = ((pwv & 0xFFFFFFu) >> 8) | (pwv & 0xFF000000u);
    t.pend ^= ((w & 0xFFFFFFu) != 0u ? 0u : 1u) << lv;
    return enter_c2<SEM, GRID>(s, r, st, t, false, lv, pwv & 0xFFu, w, an & 0x3FFFFFFFu, ad, make_uint2(0u, 0u));
}

/* backtrack (octree_fsh.c:368-375) and pop the next pending entry of the
 * deepest level below t.level that has one; ST_MISS where none has */
template <bool DUAL, int SEM, bool GRID>
__device__ __forceinline__ int trace_pop_direct(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t)
{
    /* the deepest level with a pending entry, from the per-lane mask (bit l
     * set while level l has one; the levels between have none) */
    const int      level = t.level;
    const uint32_t below = t.pend & ((1u << level) - 1u);
    if (below == 0u) return ST_MISS;
    const int lv = 31 - __clz((int) below), sh = level - lv;
    const int ix = t.ix >> sh, iy = t.iy >> sh, iz = t.iz >> sh;
    uint32_t  w = st.pw[lv * st.stride];
    int       k = (int) ((w >> 3) & 7u), cnt = (int) (w & 7u);
    int       e = (int) ((w >> (8 + 5 * k)) & 31u);
    int       o = e & 7, src = e >> 3;
    st.pw[lv * st.stride] = (w & ~(7u << 3)) | ((uint32_t) (k + 1) << 3);
    t.pend &= k + 1 == cnt ? ~(1u << lv) : ~0u;
    float4 isp;
    if (src == 0) {
        isp = entry_of<SEM, GRID>(s, r, st, lv, ix, iy, iz, root_face(t));
    } else {
        isp = midplane_cell<SEM, GRID>(s, r, src, lv, ix, iy, iz, 0);
    }
    t.ns    = child_slot<SEM>(s.stat, st.ns[lv * st.stride], o, lv);
    t.nd    = DUAL ? child_slot<kSemShader>(s.dyn, st.nd[lv * st.stride], o, lv) : 0;
    t.ix    = (ix << 1) | (o & 1);
    t.iy    = (iy << 1) | ((o >> 1) & 1);
    t.iz    = (iz << 1) | (o >> 2);
    t.entry = isp;
    t.level = lv + 1;
    return t.level == s.maxlevel ? ST_HIT : ST_CONT;
}

/* The step on the direct layout, one tree or both; counts itself in t.it. */
template <bool DUAL, int SEM, bool GRID>
__device__ __forceinline__ int trace_step_direct(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t)
{
    if (++t.it > s.iter_cap) return ST_ABORT;
    const int level = t.level;

    /* ---- expansion of the node just entered (octree_fsh.c:251-330) ---- */
    Block sb, db;
    sb.clear();
    db.clear();
    if (t.ns != 0 || level == 0) {
        load_block<SEM>(sb, s.stat, t.ns);
        t.exps++;
    }
    if (DUAL && (t.nd != 0 || level == 0)) {
        db.load(s.dyn, t.nd);
        t.exps++;
    }
    unsigned mask = sb.mask();
    if (DUAL) mask |= db.mask();

    if (mask) {
        float tx, ty, tz, tw, bxx, byy, bzz, hx, hy, hz;
        cube_at<GRID>(s, level, t.ix, t.iy, t.iz, tx, ty, tz, tw);
        cube_mid<GRID>(tx, ty, tz, tw, bxx, byy, bzz, hx, hy, hz);

        /* candidates as (t, key) pairs, as in expand_any */
        const float  qnan = __builtin_nanf("");
        const float4 az   = plane_z<SEM>(hz, r);
        const float4 ax   = plane_x<SEM>(hx, r);
        const float4 ay   = plane_y<SEM>(hy, r);
        float        w0   = t.entry.w;
        float        w1 = (az.w > 0.0f && tx < az.x && az.x <= bxx && ty > az.y && az.y >= byy) ? az.w : qnan;
        float        w2 = (ax.w > 0.0f && ty > ax.y && ax.y >= byy && tz > ax.z && ax.z >= bzz) ? ax.w : qnan;
        float        w3 = (ay.w > 0.0f && tx < ay.x && ay.x <= bxx && tz > ay.z && ay.z >= bzz) ? ay.w : qnan;
        const int    oe = (t.entry.x > hx ? 1 : 0) | (t.entry.y < hy ? 2 : 0) | (t.entry.z < hz ? 4 : 0);
        int          k0 = oe | (oe << 5);
        int k1 = SEM != kSemShader ? octet_key(az.x, az.y, az.z, hx, hy, hz, 1) : zplane_key(az.x, az.y, hx, hy);
        int k2 = SEM != kSemShader ? octet_key(ax.x, ax.y, ax.z, hx, hy, hz, 2) : xplane_key(ax.y, ax.z, hy, hz);
        int k3 = SEM != kSemShader ? octet_key(ay.x, ay.y, ay.z, hx, hy, hz, 3) : yplane_key(ay.x, ay.z, hx, hz);
        if (w1 < w0 || w2 < w0 || w3 < w0) { /* selection-swap sort (octree_fsh.c:283); NaN never moves */
            k0 = octet_key(t.entry.x, t.entry.y, t.entry.z, hx, hy, hz, 0);
            kswap(w0, k0, w1, k1);
            kswap(w0, k0, w2, k2);
            kswap(w0, k0, w3, k3);
        }
        kswap(w1, k1, w2, k2);
        kswap(w1, k1, w3, k3);
        kswap(w2, k2, w3, k3);

        /* flip an octet equal to the previous valid one; keep those whose
         * child exists in either tree, in order, as 5-bit entries */
        const bool v1 = w1 == w1, v2 = w2 == w2, v3 = w3 == w3;
        const int  o0 = k0 & 7;
        const int  o1 = (k1 & 7) == o0 ? ((k1 >> 5) & 7) : (k1 & 7);
        const int  p1 = v1 ? o1 : o0;
        const int  o2 = (k2 & 7) == p1 ? ((k2 >> 5) & 7) : (k2 & 7);
        const int  p2 = v2 ? o2 : p1;
        const int  o3 = (k3 & 7) == p2 ? ((k3 >> 5) & 7) : (k3 & 7);
        const bool t0 = bit_of(mask, o0);
        const bool t1 = v1 && bit_of(mask, o1);
        const bool t2 = v2 && bit_of(mask, o2);
        const bool t3 = v3 && bit_of(mask, o3);
        auto ent = [](int o, int k) -> uint32_t { return (uint32_t) o | ((uint32_t) k & 0x18u); };
        uint32_t entries = t3 ? ent(o3, k3) : 0u;
        entries          = t2 ? (entries << 5) | ent(o2, k2) : entries;
        entries          = t1 ? (entries << 5) | ent(o1, k1) : entries;
        entries          = t0 ? (entries << 5) | ent(o0, k0) : entries;
        const int n      = (t0 ? 1 : 0) + (t1 ? 1 : 0) + (t2 ? 1 : 0) + (t3 ? 1 : 0);

        if (n > 0) {
            /* pop the first pending entry now (octree_fsh.c:336-367) */
            const int foct = (int) (entries & 7u);
            st.pw[level * st.stride] = (entries << 8) | (uint32_t) n | (1u << 3);
            st.ns[level * st.stride] = t.ns;
            if (DUAL) st.nd[level * st.stride] = t.nd;
            t.pend |= (n > 1 ? 1u : 0u) << level;
            t.entry = pick_entry((int) ((entries >> 3) & 3u), t.entry, az, ax, ay);
            t.ns    = sb.child(foct);
            t.nd    = DUAL ? db.child(foct) : 0;
            t.ix    = (t.ix << 1) | (foct & 1);
            t.iy    = (t.iy << 1) | ((foct >> 1) & 1);
            t.iz    = (t.iz << 1) | (foct >> 2);
            t.level = level + 1;
            return t.level == s.maxlevel ? ST_HIT : ST_CONT;
        }
    }

    return trace_pop_direct<DUAL, SEM, GRID>(s, r, st, t);
}

/*
 * One step: expand the node just entered and descend into its nearest
 * pending child, or backtrack and descend into the next pending child of an
 * ancestor. Returns ST_CONT, ST_HIT (t.level == maxlevel; the leaf is
 * t.ns / t.nd with entry point t.entry), ST_MISS or ST_ABORT.
 */
template <bool CMP, bool DUAL, int SEM, bool GRID>
__device__ __forceinline__ int trace_step(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t)
{
    if constexpr (CMP && DUAL) return trace_step_c2<SEM, GRID>(s, r, st, t);
    else if constexpr (CMP) return trace_step_c1<SEM, GRID>(s, r, st, t);
    else return trace_step_direct<DUAL, SEM, GRID>(s, r, st, t);
}

/* backtrack only: the next pending entry of the deepest level below t.level
 * that has one */
template <bool CMP, bool DUAL, int SEM, bool GRID>
__device__ __forceinline__ int trace_pop(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t)
{
    if constexpr (CMP && DUAL) return trace_pop_c2<SEM, GRID>(s, r, st, t);
    else if constexpr (CMP) return trace_pop_c1<SEM, GRID>(s, r, st, t);
    else return trace_pop_direct<DUAL, SEM, GRID>(s, r, st, t);
}

/* The iteration cap: a ray whose trace takes more than iter_cap steps is
 * aborted, whatever its last step came to. The direct layout's step counts
 * itself; that of the compact ones is counted by its callers, a run of steps
 * at a time. Only lanes far enough from the cap for a whole run take one
 * (near_cap: all lanes of the wave then go one step at a time), so the count
 * of a lane that may be over is its own. */
template <bool CMP>
__device__ __forceinline__ bool near_cap(const SceneDev& s, const TraceState& t, int run)
{
    return CMP && t.it > s.iter_cap - run;
}

/* counts the `steps` of the run just taken; whether the ray is over the cap */
template <bool CMP, bool DUAL>
__device__ __forceinline__ bool count_steps(const SceneDev& s, TraceState& t, int steps)
{
    if constexpr (CMP) {
        t.it += steps;
        return t.it > s.iter_cap;
    }
    return false; /* trace_step reports the abort */
}

/*
 * Trace one ray to the end. Returns ST_HIT / ST_MISS / ST_DISCARD / ST_ABORT.
 * DUAL: the dynamic tree takes part. SEM: kSemCpu for octree.c plane-test
 * returns and root acceptance, kSemParticle for the particle shader's (both
 * single tree; callers pass DUAL = false).
 */
template <bool CMP, bool DUAL, int SEM, bool GRID>
__device__ int trace(const SceneDev& s, const Ray& r, const Stack& st, Hit& out)
{
    TraceState t;
    Ray        rr  = r;
    int        stt = trace_begin<SEM>(s, rr, t);
    while (stt == ST_CONT) {
        stt = trace_step<CMP, DUAL, SEM, GRID>(s, rr, st, t);
        if (count_steps<CMP, DUAL>(s, t, 1)) stt = ST_ABORT;
    }
    out.exps = t.exps;
    if (stt == ST_HIT) {
        out.isp = t.entry;
        out.ns  = t.ns;
        out.nd  = t.nd;
        out.ix  = t.ix;
        out.iy  = t.iy;
        out.iz  = t.iz;
    }
    return stt;
}

} // namespace qbt
