// Scene access on the device: BVH traversal (closest hit and occlusion), hit records,
// rehydration of packed interactions, the GGX BSDF and emitter sampling.
//
// Traversal replaces optixTrace over the triangle GAS/IAS (include/graph/trace.h:25-88).
// The result of a query is a pure function of the ray and the triangle set:
//   closest hit  = the minimum (t, primitive) over all triangles whose watertight test
//                  (Woop, Benthin, Wald, JCGT 2013) reports t in [tmin, tmax];
//   occlusion    = whether any such triangle exists.
// Node boxes are padded outward at build time and the box test carries a relative slack,
// so traversal only ever visits more nodes than needed; which BVH is used, and in which
// order children are visited, cannot change a result.
#pragma once

#include "cx_dev.h"

namespace cx {

static constexpr uint32_t INVALID_PRIM = 0xFFFFFFFFu;
static constexpr float PI_F = 3.14159265358979323846264f;   // shader/brdf.cu:12

// Binary BVH node, 64 bytes:
//   a = (c0.lo.x, c0.hi.x, c0.lo.y, c0.hi.y)   b = (c1.lo.x, c1.hi.x, c1.lo.y, c1.hi.y)
//   c = (c0.lo.z, c0.hi.z, c1.lo.z, c1.hi.z)   d = (ref0, ref1, -, -)
// ref >= 0: inner node index; ref < 0: leaf, ~ref = (first triangle slot << 4) | count.
// Triangle slots hold 3 float4: (v0.xyz, primitive index bits), (v1.xyz, skip bits), (v2.xyz, 0);
// the skip bits are the complement of the triangle's CX_VIS_* mask: bit 0 hides it from
// closest-hit rays, bit 1 from occlusion rays.
struct DMaterial {
    float4 diffRough;   // diffuse rgb, roughness
    float4 spec;        // specF0 rgb, -
    float4 emissive;    // emissive rgb, -
    int4 tex;           // diffuse, specular, roughness texture (-1: none), specular usage
};

static constexpr int32_t SPEC_USAGE_OCC_ROUGH_METAL = 1;   // SpecTexUsage::OccRoughMetal

// Wide BVH node (width N = 4 or 8), N/4 groups of 7 float4, padded to 8 float4 per group:
//   lo.x[4], hi.x[4], lo.y[4], hi.y[4], lo.z[4], hi.z[4], ref[4]
// with refs as in the binary node; an empty slot has ref WIDE_EMPTY (never a leaf code, since
// a leaf's first slot plus its count stays below 2^27) and a point box at WIDE_EMPTY_COORD,
// which no ray with tmax <= 1e30 can reach.
static constexpr int32_t WIDE_EMPTY = (int32_t)0x80000000;
static constexpr float WIDE_EMPTY_COORD = 3.0e38f;

struct DScene {
    const float4* __restrict__ nodes;
    const float4* __restrict__ wnodes;    // wide nodes (width 4 or 8), or null
    const float4* __restrict__ tris;
    const float* __restrict__ pos;        // [V][3]
    const float* __restrict__ nrm;        // [V][3]
    const uint32_t* __restrict__ idx;     // [T][3]
    const uint32_t* __restrict__ triMat;  // [T]
    const DMaterial* __restrict__ mats;
    const float* __restrict__ emitFaces;  // [F][9]
    const uint32_t* __restrict__ emitOff; // [E+1]
    const float* __restrict__ emitColor;  // [E][3]
    uint32_t numTris;
    uint32_t numEmitters;
    int32_t root;         // root of `nodes` (binary)
    int32_t wroot;        // root of `wnodes`
    uint32_t width;       // 2: traverse `nodes`; 4 or 8: traverse `wnodes`
    uint32_t numTextures;
    float reach;          // largest coordinate of any vertex, by magnitude
    uint32_t pad;
    const float* __restrict__ uv;         // [V][2], or null (all zero)
    const uint32_t* __restrict__ texels;  // RGBA8 texels of every texture, one word each
    const uint4* __restrict__ texInfo;    // [textures]: first texel, width, height, -
};

static constexpr int STACK_DEPTH = 64;

struct RayPre {
    int kx, ky, kz;
    float Sx, Sy, Sz;
};

CX_HD RayPre ray_pre(V3 d) {
    const float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    RayPre r;
    r.kz = (ax >= ay) ? ((ax >= az) ? 0 : 2) : ((ay >= az) ? 1 : 2);
    r.kx = r.kz == 2 ? 0 : r.kz + 1;
    r.ky = r.kx == 2 ? 0 : r.kx + 1;
    if (comp(d, r.kz) < 0.0f) {
        const int t = r.kx;
        r.kx = r.ky;
        r.ky = t;
    }
    const float dz = comp(d, r.kz);
    r.Sx = comp(d, r.kx) / dz;
    r.Sy = comp(d, r.ky) / dz;
    r.Sz = 1.0f / dz;
    return r;
}

// Watertight ray/triangle test.  u weights v1 and v weights v2 (optixGetTriangleBarycentrics).
CX_HD bool tri_hit(V3 o, const RayPre& r, V3 v0, V3 v1, V3 v2, float tmin, float tmax,
                                        float& t, float& u, float& v) {
    const V3 A = v0 - o, B = v1 - o, C = v2 - o;
    const float Akx = comp(A, r.kx), Aky = comp(A, r.ky), Akz = comp(A, r.kz);
    const float Bkx = comp(B, r.kx), Bky = comp(B, r.ky), Bkz = comp(B, r.kz);
    const float Ckx = comp(C, r.kx), Cky = comp(C, r.ky), Ckz = comp(C, r.kz);
    const float Ax = Akx - r.Sx * Akz, Ay = Aky - r.Sy * Akz;
    const float Bx = Bkx - r.Sx * Bkz, By = Bky - r.Sy * Bkz;
    const float Cx = Ckx - r.Sx * Ckz, Cy = Cky - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
        V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
        W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    const float det = U + V + W;
    if (det == 0.0f) return false;
    const float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
    const float T = U * Az + V * Bz + W * Cz;
    const float tt = T / det;
    if (!(tt >= tmin && tt <= tmax)) return false;
    t = tt;
    u = V / det;
    v = W / det;
    return true;
}

struct Hit {
    uint32_t prim;
    float t, u, v;
};

// The slab tests of a ray: the plane x_i = c is crossed at fma(c, inv_i, -o_i inv_i), one operation
// per plane.  The rounding of the product o_i inv_i is an absolute error in t, so it is kept as an
// interval: nn_i (used for the near planes) lies below it, nf_i (far planes) above it, and the one
// rounding of the fma is relative and covered by the far plane's slack; every box the ray enters
// is so reported as entered.  A ray with d_i = 0 never changes x_i: its inv_i is a large power of
// two (the product is then exact) and its interval is widened by 2^-40 in x_i, so that a box
// whose face holds the origin is entered.
//
// Where an interval is not finite (a reciprocal or a product overflows: a subnormal component, an
// origin of 1e30, a direction of 1e-37) it would constrain nothing, for fmaxf / fminf pass over it, and
// the ray would visit most of the tree: 100 k rays on 1.06 M triangles took 59 ms with one component of
// 1e-40 and 1.3 s with directions of 1e-37, 0.13 and 0.37 ms as it is.  In the caller's ray arrays (ODD:
// rays of any floats) such a ray is `odd`: a node's planes are moved to its origin first, so that its
// intervals are those of o = 0.  A frame's rays, of unit length from points of the scene, do without:
// asking for odd rays in their steps took 2.7 % of the 1080p frame.
struct RaySlab {
    V3 inv, nn, nf;
    bool odd;
};

CX_HD void slab_axis(float o, float d, float big, float& inv, float& nn, float& nf) {
    inv = d == 0.0f ? copysignf(big, d) : 1.0f / d;
    const float noi = -(o * inv);
    const float e = (fabsf(noi) * 1.1920929e-7f + 1e-30f) + (d == 0.0f ? big * 9.094947e-13f : 0.0f);
    nn = noi - e;
    nf = noi + e;
}

// An axis of an odd ray.  An infinite reciprocal (d = 0 or below 3e-39) is taken as the largest
// number, and its interval is widened by `cover`, a time that no hit lies beyond.
CX_HD void slab_axis_odd(float d, float cover, float& inv, float& nn, float& nf) {
    const float most = 3.4028235e38f, q = 1.0f / d;
    const bool beyond = fabsf(q) > most;
    inv = beyond ? copysignf(most, d) : q;
    nf = beyond ? cover : 1e-30f;
    nn = -nf;
}

template <bool ODD>
CX_HD RaySlab slab_init(const DScene& S, V3 o, V3 d) {
    const float m = fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
    // 2^96 over the power of two at or below the largest component (0 and denormals as they are)
    const float p = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, m) & 0x7f800000u);
    const float big = 7.9228163e28f / (p > 0.0f ? p : 1.0f);
    RaySlab r;
    r.odd = false;
    slab_axis(o.x, d.x, big, r.inv.x, r.nn.x, r.nf.x);
    slab_axis(o.y, d.y, big, r.inv.y, r.nn.y, r.nf.y);
    slab_axis(o.z, d.z, big, r.inv.z, r.nn.z, r.nf.z);
    // 2^96 over a subnormal p says nothing of the ray's times, so such a ray is odd as well
    if (ODD && !(p > 0.0f && fabsf(r.nn.x) < INFINITY && fabsf(r.nf.x) < INFINITY && fabsf(r.nn.y) < INFINITY &&
                 fabsf(r.nf.y) < INFINITY && fabsf(r.nn.z) < INFINITY && fabsf(r.nf.z) < INFINITY)) {
        if (!(fabsf(o.x) < INFINITY && fabsf(o.y) < INFINITY && fabsf(o.z) < INFINITY) || d.x != d.x || d.y != d.y ||
            d.z != d.z || m == 0.0f) {
            // every triangle's t is a NaN (tri_hit): no box is entered
            r.inv.x = 1.0f;
            r.nn.x = INFINITY;
            r.nf.x = -INFINITY;
        } else {
            // along the largest component no vertex is farther than the origin and the scene reach
            const float far = fabsf(o.x) + fabsf(o.y) + fabsf(o.z) + S.reach;
            const float cover = fminf(4.0f * far / p, 3.4028235e38f);
            r.odd = true;
            slab_axis_odd(d.x, cover, r.inv.x, r.nn.x, r.nf.x);
            slab_axis_odd(d.y, cover, r.inv.y, r.nn.y, r.nf.y);
            slab_axis_odd(d.z, cover, r.inv.z, r.nn.z, r.nf.z);
        }
    }
    return r;
}

// Whether any lane that asks has an odd ray, and what a plane of this lane's ray is moved by.
CX_HD bool slab_any_odd(const RaySlab& r) {
#ifdef __HIP_DEVICE_COMPILE__
    return __ballot(r.odd) != 0ull;
#else
    return r.odd;
#endif
}

CX_HD V3 slab_shift(V3 o, const RaySlab& r) { return r.odd ? o : V3{0.0f, 0.0f, 0.0f}; }

// Entry distance of a box whose near and far planes (by the signs of inv) are given, and whether
// the ray enters it in [tmin, tcap].  The far plane carries a relative slack so that a triangle
// whose computed t equals the current best is never pruned.
CX_HD float slab_box(float nx, float fx, float ny, float fy, float nz, float fz, const RaySlab& r, float tmin,
                     float tcap, bool& hit) {
    const float n = fmaxf(fmaxf(fmaf(nx, r.inv.x, r.nn.x), fmaf(ny, r.inv.y, r.nn.y)),
                          fmaxf(fmaf(nz, r.inv.z, r.nn.z), tmin));
    const float f = fminf(fminf(fmaf(fx, r.inv.x, r.nf.x), fmaf(fy, r.inv.y, r.nf.y)),
                          fminf(fmaf(fz, r.inv.z, r.nf.z), tcap));
    hit = n <= fmaf(fabsf(f), 2e-5f, f);
    return n;
}

__device__ __forceinline__ V3 load_v3(const float* p, uint32_t i) { return V3{p[3 * i], p[3 * i + 1], p[3 * i + 2]}; }

// Traversal stack: the first SHORT entries in a per-thread LDS column (lds[i * STRIDE]), deeper
// entries in a per-lane private array that the caller declares beside it (STACK_OVF entries; an
// array inside this struct would pin the whole struct in private memory).
template <int SHORT>
static constexpr int STACK_OVF = STACK_DEPTH - SHORT > 0 ? STACK_DEPTH - SHORT : 1;

template <int SHORT, int STRIDE>
struct TravStack {
    int* lds;
    int* ovf;
    CX_HD void put(int i, int v) {
        if (SHORT >= STACK_DEPTH || i < SHORT) lds[i * STRIDE] = v;
        else ovf[i - SHORT] = v;
    }
    // The entry below depth sp, read ahead of its use (any value when sp is 0 or the entry lies in
    // private memory), and the pop of it.
    CX_HD int peek(int sp) const { return lds[(sp > 0 && (SHORT >= STACK_DEPTH || sp <= SHORT) ? sp - 1 : 0) * STRIDE]; }
    CX_HD int pop(int& sp, int peeked) const {
        --sp;
        int v = peeked;
        if (SHORT < STACK_DEPTH && sp >= SHORT) v = ovf[sp - SHORT];
        return v;
    }
    // Pushes c3, c2, c1 in this order, of which only the first n entries of (c1, c2, c3) are
    // valid; sp becomes sp + n.  While all three fit in LDS they are stored without branches, the
    // invalid ones above the new top.
    CX_HD void push3(int& sp, int c1, int c2, int c3, bool h1, bool h2, bool h3) {
        if (sp + 3 <= SHORT) {
            int* const b = lds + sp * STRIDE;
            const int a2 = h2 ? 1 : 0, a3 = h3 ? 1 : 0;
            b[(a2 + a3) * STRIDE] = c1;
            b[h2 && !h3 ? 0 : STRIDE] = c2;
            b[h3 ? 0 : 2 * STRIDE] = c3;
            sp += (h1 ? 1 : 0) + a2 + a3;
        } else {
            if (h3) put(sp++, c3);
            if (h2) put(sp++, c2);
            if (h1) put(sp++, c1);
        }
    }
};

// Closest-hit / any-hit leaf loop shared by the binary and wide traversals.  Returns true when
// an any-hit query is answered.  Triangles whose skip bits hide them from the ray kind (closest
// hit: bit 0, any hit: bit 1) are passed over, as OptiX passes over an instance whose
// visibilityMask shares no bit with the ray's.  The interval tested is [tmin, best.t]: best.t
// starts at the ray's tmax and only falls, so a triangle behind the current closest hit is
// rejected before its barycentric divisions, and one at exactly best.t still reaches the
// (t, primitive) tie-break.
CX_HD bool leaf_hits_rt(const DScene& S, int32_t ref, V3 o, const RayPre& rp, float tmin, Hit& best, bool any) {
    const uint32_t code = ~(uint32_t)ref;
    const uint32_t first = code >> 4, cnt = code & 15u;
    // the next triangle's vertices are fetched before the current one is tested, so a leaf's
    // fetches overlap instead of queueing behind each test (a leaf holds at least one triangle)
    const float4* tv = S.tris + 3 * (size_t)first;
    float4 n0 = tv[0], n1 = tv[1], n2 = tv[2];
    for (uint32_t i = 0; i < cnt; i++) {
        const float4 p0 = n0, p1 = n1, p2 = n2;
        if (i + 1 < cnt) {
            const float4* nv = tv + 3 * (size_t)(i + 1);
            n0 = nv[0];
            n1 = nv[1];
            n2 = nv[2];
        }
        if (__builtin_bit_cast(uint32_t, p1.w) & (any ? 2u : 1u)) continue;   // invisible to this ray kind
        float t, u, v;
        if (!tri_hit(o, rp, V3{p0.x, p0.y, p0.z}, V3{p1.x, p1.y, p1.z}, V3{p2.x, p2.y, p2.z}, tmin, best.t, t, u, v))
            continue;
        const uint32_t prim = __builtin_bit_cast(uint32_t, p0.w);
        if (any) {
            best.prim = prim;
            best.t = t;
            return true;
        }
        if (t < best.t || (t == best.t && prim < best.prim)) {
            best.prim = prim;
            best.t = t;
            best.u = u;
            best.v = v;
        }
    }
    return false;
}

template <bool ANY>
CX_HD bool leaf_hits(const DScene& S, int32_t ref, V3 o, const RayPre& rp, float tmin, Hit& best) {
    return leaf_hits_rt(S, ref, o, rp, tmin, best, ANY);
}

// One triangle of a leaf, its slot already loaded in q0..q2: leaf_hits' test of that triangle.
// Returns true when an any-hit query is answered.
typedef float f32x4 __attribute__((ext_vector_type(4)));

// The bits of a value.  By value: __builtin_bit_cast applied directly to an element of a vector
// reads the vector's first element.
CX_HD uint32_t bits_of(float x) { return __builtin_bit_cast(uint32_t, x); }

CX_HD bool tri_hits_q(f32x4 q0, f32x4 q1, f32x4 q2, V3 o, const RayPre& rp, float tmin, Hit& best, bool any) {
    if (bits_of(q1[3]) & (any ? 2u : 1u)) return false;   // invisible to this ray kind
    float t, u, v;
    if (!tri_hit(o, rp, V3{q0[0], q0[1], q0[2]}, V3{q1[0], q1[1], q1[2]}, V3{q2[0], q2[1], q2[2]}, tmin, best.t, t, u,
                 v))
        return false;
    const uint32_t prim = bits_of(q0[3]);
    if (any) {
        best.prim = prim;
        best.t = t;
        return true;
    }
    if (t < best.t || (t == best.t && prim < best.prim)) {
        best.prim = prim;
        best.t = t;
        best.u = u;
        best.v = v;
    }
    return false;
}

// A child box's entry distance and reference as one double, the distance's bits in the high word:
// for the distances of hit boxes (any float but NaN, +inf marking a miss) the order of the doubles
// is the order of the distances, so a compare-exchange is a minimum and a maximum (v_min_f64 and
// v_max_f64 issue at the rate of the 32-bit operations on gfx950) instead of a comparison and four
// selects.  The low word only breaks ties.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

CX_HD double hit_key(float t, int ref) {
    return __builtin_bit_cast(double, u32x2{(uint32_t)ref, __builtin_bit_cast(uint32_t, t)});
}

CX_HD int key_ref(double k) {
    const u32x2 b = __builtin_bit_cast(u32x2, k);
    return (int)b.x;
}
CX_HD bool key_miss(double k) {
    const u32x2 b = __builtin_bit_cast(u32x2, k);
    return b.y == 0x7f800000u;
}

// The instructions themselves on the device: fmin and fmax would quiet their operands first.
CX_HD double key_min(double a, double b) {
#ifdef __HIP_DEVICE_COMPILE__
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return b < a ? b : a;
#endif
}

CX_HD double key_max(double a, double b) {
#ifdef __HIP_DEVICE_COMPILE__
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
#else
    return b < a ? a : b;
#endif
}

CX_HD void key_cswap(double& a, double& b) {
    const double lo = key_min(a, b), hi = key_max(a, b);
    a = lo;
    b = hi;
}

// One wide node (2 N float4 per node, the 8th of each group of 4 children unused): test the N
// child boxes, sort the hit ones by entry distance (a fixed compare-exchange network on
// registers, misses last), push all but the nearest, farthest first, and return the nearest in
// ref; false (ref unchanged) when no child box is hit.  The near and far planes of an axis are
// chosen by address, from the sign of the ray's direction, so no minimum or maximum is needed per
// plane pair: a node's offset is a 32-bit number of bytes (cx_scene_build keeps the array below
// 4 GiB), and a far plane lies 16 bytes from its near plane.
#ifdef __HIP_DEVICE_COMPILE__
typedef const f32x4 __attribute__((address_space(1)))* gf32x4;   // a global-memory address
#else
typedef const f32x4* gf32x4;
#endif

struct WideLoads {
    f32x4 nx, fx, ny, fy, nz, fz, ref;
};

CX_HD f32x4 load_at(const float4* base, uint32_t bytes) { return *(const f32x4*)((const char*)base + bytes); }

CX_HD WideLoads wide_load(const float4* nodes, uint32_t off, const RaySlab& r) {
    const uint32_t ax = off + ((__builtin_bit_cast(uint32_t, r.inv.x) >> 27) & 16u);
    const uint32_t ay = off + ((__builtin_bit_cast(uint32_t, r.inv.y) >> 27) & 16u);
    const uint32_t az = off + ((__builtin_bit_cast(uint32_t, r.inv.z) >> 27) & 16u);
    WideLoads w;
    w.nx = load_at(nodes, ax);
    w.fx = load_at(nodes, ax ^ 16u);
    w.ny = load_at(nodes + 2, ay);
    w.fy = load_at(nodes + 2, ay ^ 16u);
    w.nz = load_at(nodes + 4, az);
    w.fz = load_at(nodes + 4, az ^ 16u);
    w.ref = load_at(nodes + 6, off);
    return w;
}

// Moves a node's planes to the origin of an odd ray.
CX_HD void wide_shift(WideLoads& w, V3 by) {
    w.nx -= by.x;
    w.fx -= by.x;
    w.ny -= by.y;
    w.fy -= by.y;
    w.nz -= by.z;
    w.fz -= by.z;
}

CX_HD void wide_keys(const WideLoads& w, const RaySlab& r, float tmin, float tcap, double* k) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
        bool h;
        const float t = slab_box(w.nx[j], w.fx[j], w.ny[j], w.fy[j], w.nz[j], w.fz[j], r, tmin, tcap, h);
        const int ref = (int)bits_of(w.ref[j]);
        k[j] = hit_key(h && ref != WIDE_EMPTY ? t : INFINITY, ref);
    }
}

// wide_visit of a 4-wide node whose float4 are loaded.
template <bool ODD, typename Stack>
CX_HD bool wide_visit4(WideLoads& w, int& ref, V3 o, const RaySlab& r, float tmin, float tcap, Stack& st, int& sp) {
    if (ODD && slab_any_odd(r)) wide_shift(w, slab_shift(o, r));
    double k[4];
    wide_keys(w, r, tmin, tcap, k);
    key_cswap(k[0], k[1]);
    key_cswap(k[2], k[3]);
    key_cswap(k[0], k[2]);
    key_cswap(k[1], k[3]);
    key_cswap(k[1], k[2]);
    if (key_miss(k[0])) return false;
    st.push3(sp, key_ref(k[1]), key_ref(k[2]), key_ref(k[3]), !key_miss(k[1]), !key_miss(k[2]), !key_miss(k[3]));
    ref = key_ref(k[0]);
    return true;
}

template <int N, bool ODD, typename Stack>
CX_HD bool wide_visit(const DScene& S, int& ref, V3 o, const RaySlab& r, float tmin, float tcap, Stack& st, int& sp) {
    if constexpr (N == 4) {
        WideLoads w = wide_load(S.wnodes, (uint32_t)ref * 128u, r);
        return wide_visit4<ODD>(w, ref, o, r, tmin, tcap, st, sp);
    } else {
        double k[8];
        WideLoads w0 = wide_load(S.wnodes, (uint32_t)ref * 256u, r);
        WideLoads w1 = wide_load(S.wnodes, (uint32_t)ref * 256u + 128u, r);
        if (ODD && slab_any_odd(r)) {
            wide_shift(w0, slab_shift(o, r));
            wide_shift(w1, slab_shift(o, r));
        }
        wide_keys(w0, r, tmin, tcap, k);
        wide_keys(w1, r, tmin, tcap, k + 4);
        // Batcher's odd-even merge sort of 8 keys (19 compare-exchanges).
#define CX_CS(a, b) key_cswap(k[a], k[b])
        CX_CS(0, 1); CX_CS(2, 3); CX_CS(4, 5); CX_CS(6, 7);
        CX_CS(0, 2); CX_CS(1, 3); CX_CS(4, 6); CX_CS(5, 7);
        CX_CS(1, 2); CX_CS(5, 6);
        CX_CS(0, 4); CX_CS(1, 5); CX_CS(2, 6); CX_CS(3, 7);
        CX_CS(2, 4); CX_CS(3, 5);
        CX_CS(1, 2); CX_CS(3, 4); CX_CS(5, 6);
#undef CX_CS
        if (key_miss(k[0])) return false;
#pragma unroll
        for (int i = 7; i >= 1; i--)
            if (!key_miss(k[i])) st.put(sp++, key_ref(k[i]));
        ref = key_ref(k[0]);
        return true;
    }
}

// One binary node: the nearer hit child in ref (the farther one pushed); false when neither
// child box is hit.
template <bool ODD, typename Stack>
CX_HD bool bin_visit(const DScene& S, int& ref, V3 o, const RaySlab& r, float tmin, float tcap, Stack& st, int& sp) {
    const float4* n = S.nodes + 4 * (size_t)ref;
    float4 a = n[0], b = n[1], c = n[2];
    const int4 dd = __builtin_bit_cast(int4, n[3]);
    if (ODD && slab_any_odd(r)) {
        const V3 by = slab_shift(o, r);
        a = make_float4(a.x - by.x, a.y - by.x, a.z - by.y, a.w - by.y);
        b = make_float4(b.x - by.x, b.y - by.x, b.z - by.y, b.w - by.y);
        c = make_float4(c.x - by.z, c.y - by.z, c.z - by.z, c.w - by.z);
    }
    const bool sx = __builtin_signbitf(r.inv.x), sy = __builtin_signbitf(r.inv.y), sz = __builtin_signbitf(r.inv.z);
    bool h0, h1;
    const float t0 = slab_box(sx ? a.y : a.x, sx ? a.x : a.y, sy ? a.w : a.z, sy ? a.z : a.w, sz ? c.y : c.x,
                              sz ? c.x : c.y, r, tmin, tcap, h0);
    const float t1 = slab_box(sx ? b.y : b.x, sx ? b.x : b.y, sy ? b.w : b.z, sy ? b.z : b.w, sz ? c.w : c.z,
                              sz ? c.z : c.w, r, tmin, tcap, h1);
    if (h0 && h1) {
        const bool first0 = t0 <= t1;
        st.put(sp, first0 ? dd.y : dd.x);
        ++sp;
        ref = first0 ? dd.x : dd.y;
        return true;
    }
    if (h0) { ref = dd.x; return true; }
    if (h1) { ref = dd.y; return true; }
    return false;
}

template <bool ANY, int N, bool ODD, typename Stack>
CX_HD bool traverse_wide(const DScene& S, V3 o, V3 d, float tmin, float tmax, Hit& best,
                                              Stack& st) {
    const RayPre rp = ray_pre(d);
    const RaySlab sl = slab_init<ODD>(S, o, d);
    int sp = 0;
    int ref = S.wroot;
    while (true) {
        if (ref >= 0) {
            if (wide_visit<N, ODD>(S, ref, o, sl, tmin, best.t, st, sp)) continue;
        } else {
            if (leaf_hits<ANY>(S, ref, o, rp, tmin, best)) return true;
        }
        if (sp == 0) break;
        ref = st.pop(sp, st.peek(sp));
    }
    return best.prim != INVALID_PRIM;
}

template <bool ANY, bool ODD, typename Stack>
CX_HD bool traverse_bin(const DScene& S, V3 o, V3 d, float tmin, float tmax, Hit& best,
                                             Stack& st) {
    best.prim = INVALID_PRIM;
    best.t = tmax;
    best.u = 0.0f;
    best.v = 0.0f;
    if (S.numTris == 0) return false;
    const RayPre rp = ray_pre(d);
    const RaySlab sl = slab_init<ODD>(S, o, d);
    int sp = 0;
    int ref = S.root;
    while (true) {
        if (ref >= 0) {
            if (bin_visit<ODD>(S, ref, o, sl, tmin, best.t, st, sp)) continue;
        } else {
            if (leaf_hits<ANY>(S, ref, o, rp, tmin, best)) return true;
        }
        if (sp == 0) break;
        ref = st.pop(sp, st.peek(sp));
    }
    return best.prim != INVALID_PRIM;
}

// The traversal loop above as a resumable state, advanced one node or one leaf per step, for
// kernels that interleave several rays per lane (a lane whose ray ends takes the next one
// without waiting for the rest of its wavefront).  The answer is the loop's: the same nodes in
// the same order.
struct TravRay {
    V3 o;
    RaySlab sl;
    RayPre rp;
    float tmin;
    Hit best;   // best.t: the ray's tmax until a hit lowers it
    int ref;
    int sp;
};


template <int WIDTH, bool ODD>
CX_HD void trav_init(const DScene& S, TravRay& r, V3 o, V3 d, float tmin, float tmax) {
    r.o = o;
    r.sl = slab_init<ODD>(S, o, d);
    r.rp = ray_pre(d);
    r.tmin = tmin;
    r.best = Hit{INVALID_PRIM, tmax, 0.0f, 0.0f};
    r.ref = WIDTH == 2 ? S.root : S.wroot;
    r.sp = 0;
}

// One step; true when the ray is answered: closest hit in r.best (prim INVALID_PRIM: a miss),
// occlusion as r.best.prim != INVALID_PRIM.  A scene without triangles answers at once.
//
// The stack's top entry is read at the start of the step, with the node or triangle fetch, so a
// pop at its end finds it in a register.  At width 4 the lanes at inner nodes and the lanes at
// leaves issue their fetches (7 and 3 float4) before either kind is processed, so a wavefront
// split between the two waits once per step; a leaf step tests one triangle and leaves the lane
// on the rest of the leaf, so the leaf branch costs one triangle test per step.
template <int WIDTH, bool ODD, typename Stack>
CX_HD bool trav_step_rt(const DScene& S, TravRay& r, Stack& st, bool any) {
    if (S.numTris == 0) return true;
    const int top = st.peek(r.sp);
    if constexpr (WIDTH == 4) {
        const bool inner = r.ref >= 0;
        const uint32_t code = ~(uint32_t)r.ref;
        gf32x4 tv = (gf32x4)S.tris + 3 * (size_t)(code >> 4);
        int kind = inner ? 1 : 0;
#ifdef __HIP_DEVICE_COMPILE__
        // the triangle's address is formed ahead of the node's loads, so that both kinds of lane
        // load into the same registers without a wait between them
        asm("" : "+v"(tv));
        asm("" : "+v"(kind));
#endif
        WideLoads w;
        if (inner) w = wide_load(S.wnodes, (uint32_t)r.ref * 128u, r.sl);
        if (!kind) {
            w.nx = tv[0];
            w.fx = tv[1];
            w.ny = tv[2];
        }
#ifdef __HIP_DEVICE_COMPILE__
        // one wait for the loads of both kinds, here
        asm("" : "+v"(w.nx), "+v"(w.fx), "+v"(w.ny), "+v"(w.fy), "+v"(w.nz), "+v"(w.fz), "+v"(w.ref));
#endif
        if (inner) {
            if (wide_visit4<ODD>(w, r.ref, r.o, r.sl, r.tmin, r.best.t, st, r.sp)) return false;
        } else {
            if (tri_hits_q(w.nx, w.fx, w.ny, r.o, r.rp, r.tmin, r.best, any)) return true;
            if ((code & 15u) > 1u) {
                r.ref = (int32_t)~(code + 15u);   // the rest of the leaf, from its next slot
                return false;
            }
        }
    } else if (r.ref >= 0) {
        if constexpr (WIDTH == 2) {
            if (bin_visit<ODD>(S, r.ref, r.o, r.sl, r.tmin, r.best.t, st, r.sp)) return false;
        } else {
            if (wide_visit<WIDTH, ODD>(S, r.ref, r.o, r.sl, r.tmin, r.best.t, st, r.sp)) return false;
        }
    } else {
        if (leaf_hits_rt(S, r.ref, r.o, r.rp, r.tmin, r.best, any)) return true;
    }
    if (r.sp == 0) return true;
    r.ref = st.pop(r.sp, top);
    return false;
}

// ---- four lanes per ray ----
//
// Where there are fewer rays than lanes, a ray's time is its chain of steps: a fetch, then the
// step's instructions one after another.  Four neighbouring lanes (a quad) then share one 4-wide
// ray: each tests one child box of a node, or one triangle of a leaf, so a node step is about 60
// instructions instead of 110 and its fetch 7 loads of one float per lane from one 128-byte node.
// The quad's state is the same in its four lanes, and they stay together.  The nodes are visited
// nearest child first as above (ties and the last two bits of a distance aside), so the answers
// are the same.
template <int CTRL>
__device__ __forceinline__ uint32_t quad_swap(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, CTRL, 0xF, 0xF, true);
}
static constexpr int QUAD_1 = 0xB1, QUAD_2 = 0x4E, QUAD_3 = 0x1B;   // the lane 1, 2 or 3 away (xor) in the quad

__device__ __forceinline__ uint32_t quad_or(uint32_t x) {
    x |= quad_swap<QUAD_1>(x);
    return x | quad_swap<QUAD_2>(x);
}

// The lesser of this lane's and the other lane's hit by (t, primitive), u and v with it.
template <int CTRL>
__device__ __forceinline__ void quad_best(Hit& h) {
    Hit o;
    o.t = __builtin_bit_cast(float, quad_swap<CTRL>(__builtin_bit_cast(uint32_t, h.t)));
    o.u = __builtin_bit_cast(float, quad_swap<CTRL>(__builtin_bit_cast(uint32_t, h.u)));
    o.v = __builtin_bit_cast(float, quad_swap<CTRL>(__builtin_bit_cast(uint32_t, h.v)));
    o.prim = quad_swap<CTRL>(h.prim);
    if (o.t < h.t || (o.t == h.t && o.prim < h.prim)) h = o;
}

// Traces one ray per quad to its end; `col` is the quad's stack column in LDS (STACK_DEPTH entries,
// `stride` apart).  The whole quad calls it with the same ray.  Closest hit in best (prim
// INVALID_PRIM: a miss), occlusion as best.prim != INVALID_PRIM.
template <bool ODD>
__device__ __forceinline__ void quad_trace(const DScene& S, V3 o, V3 d, float tmin, float tmax, bool any, Hit& best,
                                           int* col, int stride) {
    best = Hit{INVALID_PRIM, tmax, 0.0f, 0.0f};
    if (S.numTris == 0) return;
    const RayPre rp = ray_pre(d);
    const RaySlab r = slab_init<ODD>(S, o, d);
    const bool anyOdd = ODD && slab_any_odd(r);
    const uint32_t j = threadIdx.x & 3u;
    const uint32_t ax = 4u * j + ((__builtin_bit_cast(uint32_t, r.inv.x) >> 27) & 16u);
    const uint32_t ay = 4u * j + ((__builtin_bit_cast(uint32_t, r.inv.y) >> 27) & 16u) + 32u;
    const uint32_t az = 4u * j + ((__builtin_bit_cast(uint32_t, r.inv.z) >> 27) & 16u) + 64u;
    const char* const nodes = (const char*)S.wnodes;
    int ref = S.wroot, sp = 0;
    while (true) {
        const int top = col[(sp > 0 ? sp - 1 : 0) * stride];
        if (ref >= 0) {
            const uint32_t off = (uint32_t)ref * 128u;
            float nx = *(const float*)(nodes + (off | ax)), fx = *(const float*)(nodes + ((off | ax) ^ 16u));
            float ny = *(const float*)(nodes + (off | ay)), fy = *(const float*)(nodes + ((off | ay) ^ 16u));
            float nz = *(const float*)(nodes + (off | az)), fz = *(const float*)(nodes + ((off | az) ^ 16u));
            const int child = *(const int*)(nodes + (off | (96u + 4u * j)));
            if (anyOdd) {
                const V3 by = slab_shift(o, r);
                nx -= by.x;
                fx -= by.x;
                ny -= by.y;
                fy -= by.y;
                nz -= by.z;
                fz -= by.z;
            }
            bool h;
            const float t = slab_box(nx, fx, ny, fy, nz, fz, r, tmin, best.t, h);
            h = h && child != WIDE_EMPTY;
            // distance with the lane in its last two bits, as a signed number; misses above all
            const int miss = 0x7fffffff;
            const int k = h ? (int)((__builtin_bit_cast(uint32_t, t) & ~3u) | j) : miss;
            const int k1 = (int)quad_swap<QUAD_1>((uint32_t)k), k2 = (int)quad_swap<QUAD_2>((uint32_t)k),
                      k3 = (int)quad_swap<QUAD_3>((uint32_t)k);
            const int first = min(min(k, k1), min(k2, k3));
            if (first != miss) {
                const int nearer = (k1 < k ? 1 : 0) + (k2 < k ? 1 : 0) + (k3 < k ? 1 : 0);
                const int more = (k != miss ? 1 : 0) + (k1 != miss ? 1 : 0) + (k2 != miss ? 1 : 0) +
                                 (k3 != miss ? 1 : 0) - 1;   // entries to push
                if (h && nearer > 0) col[(sp + more - nearer) * stride] = child;
                // the quad's other lanes read the entries: LDS answers a wavefront in order, so this
                // only keeps the compiler from moving those reads ahead of the writes
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                sp += more;
                ref = (int)quad_or(k == first ? (uint32_t)child : 0u);
                continue;
            }
        } else {
            const uint32_t code = ~(uint32_t)ref;
            const uint32_t slot0 = code >> 4, cnt = code & 15u;
            for (uint32_t b = 0; b < cnt; b += 4u) {
                Hit h = Hit{INVALID_PRIM, INFINITY, 0.0f, 0.0f};
                bool ok = false;
                if (b + j < cnt) {
                    const f32x4* tv = (const f32x4*)S.tris + 3 * (size_t)(slot0 + b + j);
                    const f32x4 q0 = tv[0], q1 = tv[1], q2 = tv[2];
                    float t, u, v;
                    if (!(bits_of(q1[3]) & (any ? 2u : 1u)) &&
                        tri_hit(o, rp, V3{q0[0], q0[1], q0[2]}, V3{q1[0], q1[1], q1[2]}, V3{q2[0], q2[1], q2[2]}, tmin,
                                best.t, t, u, v)) {
                        ok = true;
                        h = Hit{bits_of(q0[3]), t, u, v};
                    }
                }
                if (!quad_or(ok ? 1u : 0u)) continue;
                if (any) {
                    best.prim = 0u;
                    return;
                }
                quad_best<QUAD_1>(h);
                quad_best<QUAD_2>(h);
                if (h.t < best.t || (h.t == best.t && h.prim < best.prim)) best = h;
            }
        }
        if (sp == 0) return;
        --sp;
        ref = top;
    }
}

template <bool ANY, int WIDTH, bool ODD, typename Stack>
CX_HD bool trav_step(const DScene& S, TravRay& r, Stack& st) {
    return trav_step_rt<WIDTH, ODD>(S, r, st, ANY);
}

// Traversal at a BVH width fixed at compile time (WIDTH = S.width; the caller dispatches).
template <bool ANY, int WIDTH, bool ODD, typename Stack>
CX_HD bool traverse_w(const DScene& S, V3 o, V3 d, float tmin, float tmax, Hit& best, Stack& st) {
    best.prim = INVALID_PRIM;
    best.t = tmax;
    best.u = 0.0f;
    best.v = 0.0f;
    if (S.numTris == 0) return false;
    if constexpr (WIDTH == 2) return traverse_bin<ANY, ODD>(S, o, d, tmin, tmax, best, st);
    else return traverse_wide<ANY, WIDTH, ODD>(S, o, d, tmin, tmax, best, st);
}

// Dispatch on the scene's BVH width (uniform across a launch).
template <bool ANY, typename Stack>
CX_HD bool traverse_s(const DScene& S, V3 o, V3 d, float tmin, float tmax, Hit& best, Stack& st) {
    if (S.width == 4) return traverse_w<ANY, 4, false>(S, o, d, tmin, tmax, best, st);
    if (S.width == 8) return traverse_w<ANY, 8, false>(S, o, d, tmin, tmax, best, st);
    return traverse_w<ANY, 2, false>(S, o, d, tmin, tmax, best, st);
}

// Traversal with the whole stack in a per-thread LDS column (stack[i * TRACE_BLOCK]).
static constexpr int TRACE_BLOCK = 128;   // threads per block (the column stride) of the kernels that use it

template <bool ANY>
__device__ __forceinline__ bool traverse(const DScene& S, V3 o, V3 d, float tmin, float tmax, Hit& best,
                                         int* stack) {
    TravStack<STACK_DEPTH, TRACE_BLOCK> st{stack, nullptr};
    return traverse_s<ANY>(S, o, d, tmin, tmax, best, st);
}

// ---- interactions (include/graph/Interaction.h) ----

// PackedInteraction, one flattened mesh (instance 0): prim == INVALID_PRIM means !valid.
struct Packed {
    uint32_t prim;
    float bu, bv;
    V3 dir;
};

CX_HD Packed packed_invalid() { return Packed{INVALID_PRIM, 0.0f, 0.0f, V3{0.0f, 0.0f, 0.0f}}; }

struct Inter {
    uint32_t prim;
    float bu, bv;
    V3 pos, dir, nrm;
    bool valid;
    CX_HD Packed pack() const {
        Packed p;
        p.prim = valid ? prim : INVALID_PRIM;
        p.bu = bu;
        p.bv = bv;
        p.dir = dir;
        return p;
    }
};

// InterpolateBary (Interaction.h:18-25)
CX_HD V3 interp(float u, float v, V3 a, V3 b, V3 c) { return ((1.0f - u - v) * a + u * b) + v * c; }

// Rehydration (Interaction.h:115-172): normals are interpolated and not normalised.
__device__ __forceinline__ Inter rehydrate(const DScene& S, const Packed& p) {
    Inter r;
    r.prim = p.prim;
    r.bu = p.bu;
    r.bv = p.bv;
    r.dir = p.dir;
    r.valid = p.prim != INVALID_PRIM && p.prim < S.numTris;
    r.pos = v3(0.0f);
    r.nrm = v3(0.0f);
    if (!r.valid) return r;
    const uint32_t i0 = S.idx[3 * p.prim], i1 = S.idx[3 * p.prim + 1], i2 = S.idx[3 * p.prim + 2];
    r.pos = interp(p.bu, p.bv, load_v3(S.pos, i0), load_v3(S.pos, i1), load_v3(S.pos, i2));
    r.nrm = interp(p.bu, p.bv, load_v3(S.nrm, i0), load_v3(S.nrm, i1), load_v3(S.nrm, i2));
    return r;
}

// Per-thread traversal context and ray counters.
struct TraceCtx {
    int* stack;
    int stride;
    uint32_t closest;
    uint32_t shadow;
};

// TraceWithDataPointer<Interaction> + __closesthit__mesh / __miss__main
// (trace.h:25-45, mesh_hit.cu:17-69, miss.cu:11-19): a miss keeps every other field.
__device__ __forceinline__ void trace_surface(const DScene& S, TraceCtx& tc, V3 o, V3 d, float tmin, float tmax,
                                              Inter& io) {
    Hit h;
    tc.closest++;
    traverse<false>(S, o, d, tmin, tmax, h, tc.stack);
    io.dir = d;
    if (h.prim == INVALID_PRIM) {
        io.valid = false;
        return;
    }
    io.valid = true;
    io.prim = h.prim;
    io.bu = h.u;
    io.bv = h.v;
    const uint32_t i0 = S.idx[3 * h.prim], i1 = S.idx[3 * h.prim + 1], i2 = S.idx[3 * h.prim + 2];
    io.pos = interp(h.u, h.v, load_v3(S.pos, i0), load_v3(S.pos, i1), load_v3(S.pos, i2));
    io.nrm = normalize(interp(h.u, h.v, load_v3(S.nrm, i0), load_v3(S.nrm, i1), load_v3(S.nrm, i2)));
}

// TraceOcclusion (trace.h:63-88)
__device__ __forceinline__ bool trace_occluded(const DScene& S, TraceCtx& tc, V3 o, V3 d, float tmin, float tmax) {
    Hit h;
    tc.shadow++;
    return traverse<true>(S, o, d, tmin, tmax, h, tc.stack);
}

// ---- BSDF (shader/brdf.cu) ----

struct BrdfEval {
    V3 brdf;
    float pdf;
    V3 emission;
    float roughness;
};

struct BrdfSample {
    V3 outDir, brdf;
    float pdf;
    float roughness;
};

CX_HD float d_ggx(float NdotH, float roughness) {   // brdf.cu:99-104
    const float a2 = roughness * roughness;
    const float d = (NdotH * a2 - NdotH) * NdotH + 1.0f;
    return a2 / (PI_F * d * d);
}

CX_HD float v_smith(float NdotL, float NdotV, float roughness) {   // brdf.cu:106-112
    const float a2 = roughness * roughness;
    const float lv = NdotL * sqrtf(NdotV * NdotV * (1 - a2) + a2);
    const float ll = NdotV * sqrtf(NdotL * NdotL * (1 - a2) + a2);
    return 0.5f / (lv + ll);
}

struct Mat {
    V3 diff, spec, emis;
    float rough;
    float metal;
    bool diffParam;    // diff is the material's constant (not a texture value)
    bool roughParam;   // rough is the material's constant
};

// tex2D<float4> of an RGBA8 texture created as in src/Texture.cpp:44-76 (wrap addressing,
// linear filtering, normalized coordinates, normalized-float reads), channels r, g, b.
// Canonical filter: x = frac(u) * width - 0.5, texels floor(x) and floor(x) + 1 wrapped,
// weight alpha = frac(x) rounded to a multiple of 1/256 (likewise y); the exact integer sum of
// weight * texel is rounded once, sum / (65536 * 255).  frac(u) = u - floor(u) lies in [0, 1],
// so floor(x) lies in [-1, width - 1] for width <= 65536; a non-finite coordinate reads as 0.
__device__ __forceinline__ V3 tex_fetch(const DScene& S, int32_t t, float u, float v) {
    const uint4 ti = S.texInfo[t];
    if (!(fabsf(u) <= 3.0e38f)) u = 0.0f;
    if (!(fabsf(v) <= 3.0e38f)) v = 0.0f;
    const float x = (u - floorf(u)) * (float)ti.y - 0.5f;
    const float y = (v - floorf(v)) * (float)ti.z - 0.5f;
    const float xf = floorf(x), yf = floorf(y);
    const uint32_t a = (uint32_t)rintf((x - xf) * 256.0f), b = (uint32_t)rintf((y - yf) * 256.0f);
    const uint32_t i0 = xf < 0.0f ? ti.y - 1u : (uint32_t)xf, j0 = yf < 0.0f ? ti.z - 1u : (uint32_t)yf;
    const uint32_t i1 = i0 + 1u == ti.y ? 0u : i0 + 1u, j1 = j0 + 1u == ti.z ? 0u : j0 + 1u;
    const uint32_t* row0 = S.texels + ti.x + (size_t)j0 * ti.y;
    const uint32_t* row1 = S.texels + ti.x + (size_t)j1 * ti.y;
    const uint32_t t00 = row0[i0], t10 = row0[i1], t01 = row1[i0], t11 = row1[i1];
    const uint32_t w00 = (256u - a) * (256u - b), w10 = a * (256u - b), w01 = (256u - a) * b, w11 = a * b;
    float c[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const uint32_t sh = 8u * (uint32_t)k;
        const uint32_t sum = w00 * ((t00 >> sh) & 255u) + w10 * ((t10 >> sh) & 255u) + w01 * ((t01 >> sh) & 255u) +
                             w11 * ((t11 >> sh) & 255u);
        c[k] = (float)sum / 16711680.0f;
    }
    return V3{c[0], c[1], c[2]};
}

// The material of a hit: GetFromTexIfPossible for diffuse colour, specular value and roughness
// at the interaction's uv (InterpolateBary of the vertex uvs, Interaction.h:171), the
// OccRoughMetal channel mapping, then specF0 = mix(diffColor, specF0, metal) (brdf.cu:121-138).
__device__ __forceinline__ Mat resolve_mat(const DScene& S, const DMaterial& m, uint32_t prim, float bu, float bv) {
    Mat r;
    r.diff = V3{m.diffRough.x, m.diffRough.y, m.diffRough.z};
    r.rough = m.diffRough.w;
    V3 spec = V3{m.spec.x, m.spec.y, m.spec.z};
    r.emis = V3{m.emissive.x, m.emissive.y, m.emissive.z};
    r.diffParam = true;
    r.roughParam = true;
    float metal = 0.0f;
    const int4 t = m.tex;
    if ((t.x & t.y & t.z) != -1 || t.w == SPEC_USAGE_OCC_ROUGH_METAL) {
        float tu = 0.0f, tv = 0.0f;
        if ((t.x & t.y & t.z) != -1 && S.uv != nullptr) {
            const uint32_t i0 = S.idx[3 * prim], i1 = S.idx[3 * prim + 1], i2 = S.idx[3 * prim + 2];
            const float w = 1.0f - bu - bv;
            tu = (w * S.uv[2 * i0] + bu * S.uv[2 * i1]) + bv * S.uv[2 * i2];
            tv = (w * S.uv[2 * i0 + 1] + bu * S.uv[2 * i1 + 1]) + bv * S.uv[2 * i2 + 1];
        }
        if (t.x >= 0) {
            r.diff = tex_fetch(S, t.x, tu, tv);
            r.diffParam = false;
        }
        if (t.y >= 0) spec = tex_fetch(S, t.y, tu, tv);
        if (t.z >= 0) {
            r.rough = tex_fetch(S, t.z, tu, tv).x;
            r.roughParam = false;
        }
        if (t.w == SPEC_USAGE_OCC_ROUGH_METAL) {
            r.rough = spec.y;
            metal = spec.z;
            spec = v3(1.0f);
            r.roughParam = false;
        }
    }
    r.spec = r.diff * (1.0f - metal) + spec * metal;
    r.metal = metal;
    return r;
}

__device__ __forceinline__ Mat load_mat(const DScene& S, const Inter& it) {
    return resolve_mat(S, S.mats[S.triMat[it.prim]], it.prim, it.bu, it.bv);
}

__device__ __forceinline__ V3 spec_term(const Mat& m, float nDotH, float nDotL, float nDotV, float lDotH) {
    V3 specBrdf = v3(0.0f);
    if ((double)dot(m.spec, m.spec) > 1e-6) {
        const float d = d_ggx(nDotH, m.rough);
        const float v = v_smith(nDotL, nDotV, m.rough);
        const float p = pow5(gmax(0.0f, 1.0f - lDotH));
        const V3 f = m.spec + (v3(1.0f) - m.spec) * p;
        specBrdf = d * v * f;
    }
    return specBrdf;
}

// __direct_callable__ggx_eval (brdf.cu:115-190)
__device__ __forceinline__ BrdfEval ggx_eval(const DScene& S, const Inter& it, V3 outDir) {
    const Mat m = load_mat(S, it);
    BrdfEval r;
    const V3 lightDir = outDir;
    const V3 viewDir = -it.dir;
    const V3 normal = it.nrm;
    const float nDotV = dot(normal, viewDir);
    const float nDotL = dot(normal, lightDir);
    if (nDotV <= 0.0f || nDotL < 0.0f) {
        r.brdf = v3(0.0f);
        r.emission = v3(0.0f);
        r.pdf = 0.0f;
        r.roughness = 0.0f;
        return r;
    }
    const V3 diffBrdf = m.diff / PI_F;
    const float diffProb = dot(m.diff, v3(1.0f)) / (dot(m.diff, v3(1.0f)) + dot(m.spec, v3(1.0f)));
    const V3 halfway = normalize(lightDir + viewDir);
    const float nDotH = dot(halfway, normal);
    const float lDotH = dot(halfway, lightDir);
    const V3 specBrdf = spec_term(m, nDotH, nDotL, nDotV, lDotH);
    r.brdf = (diffBrdf + specBrdf) * nDotL;
    r.pdf = diffProb * nDotL / PI_F + (1.0f - diffProb) * d_ggx(nDotH, m.rough) * nDotH / (4.0f * lDotH);
    r.emission = m.emis;
    r.roughness = m.rough;
    return r;
}

// ComputeLocalFrame (brdf.cu:192-212) applied to a local vector: mat3 columns (X, Y, Z).
CX_HD V3 frame_mul(V3 n, V3 l) {
    const float x = n.x, y = n.y, z = n.z;
    const float sz = (z >= 0) ? 1.0f : -1.0f;
    const float a = 1 / (sz + z);
    const float ya = y * a;
    const float b = x * ya;
    const float c = x * sz;
    const V3 X = V3{c * x * a - 1, sz * b, c};
    const V3 Y = V3{b, y * ya - sz, y};
    return V3{X.x * l.x + Y.x * l.y + n.x * l.z, X.y * l.x + Y.y * l.y + n.y * l.z, X.z * l.x + Y.z * l.y + n.z * l.z};
}

// __direct_callable__ggx_sample (brdf.cu:214-338)
__device__ __forceinline__ BrdfSample ggx_sample(const DScene& S, const Inter& it, Rng& rng) {
    const Mat m = load_mat(S, it);
    const V3 normal = it.nrm;
    const V3 viewDir = -it.dir;
    BrdfSample r;
    r.roughness = m.rough;
    const float nDotV = dot(normal, viewDir);
    if (nDotV <= 0) {
        r.outDir = v3(0.0f);
        r.brdf = v3(0.0f);
        r.pdf = 0.0f;
        return r;
    }
    const float diffProb = dot(m.diff, v3(1.0f)) / (dot(m.diff, v3(1.0f)) + dot(m.spec, v3(1.0f)));
    if (rng.f() < diffProb) {
        const float phi = rng.f() * 2.0f * PI_F;
        const float rr = sqrtf(rng.f());
        float sp, cp;
        sincos_cw(phi, &sp, &cp);
        const float x = rr * cp;
        const float y = rr * sp;
        const float z = sqrtf(gclamp(1.0f - x * x - y * y, 0.0f, 1.0f));
        r.outDir = frame_mul(normal, V3{x, y, z});
    } else {
        const float u = rng.f();
        const float mz = sqrtf(gclamp((1 - u) / (1 + (m.rough * m.rough - 1) * u), 0.0f, 1.0f));
        const float mr = sqrtf(gclamp(1 - mz * mz, 0.0f, 1.0f));
        const float phi = rng.f() * 2.0f * PI_F;
        float sp, cp;
        sincos_cw(phi, &sp, &cp);
        r.outDir = reflect(it.dir, frame_mul(normal, V3{mr * cp, mr * sp, mz}));
        if (dot(r.outDir, normal) < 0.0f) {
            r.outDir = v3(0.0f);
            r.brdf = v3(0.0f);
            r.pdf = 0.0f;
            return r;
        }
    }
    const V3 diffBrdf = m.diff / PI_F;
    const V3 lightDir = r.outDir;
    const float nDotL = dot(normal, lightDir);
    const V3 halfway = normalize(lightDir + viewDir);
    const float nDotH = dot(halfway, normal);
    const float lDotH = dot(halfway, lightDir);
    const V3 specBrdf = spec_term(m, nDotH, nDotL, nDotV, lDotH);
    r.pdf = diffProb * nDotL / PI_F + (1.0f - diffProb) * d_ggx(nDotH, m.rough) * nDotH / (4.0f * lDotH);
    r.brdf = (diffBrdf + specBrdf) * nDotL;
    return r;
}

// ---- emitters (include/graph/sample_emitter.h:3-12, include/model/Emitter.h:21-54) ----

struct EmitterSample {
    V3 pos, color;
};

__device__ __forceinline__ EmitterSample sample_emitter(const DScene& S, Rng& rng) {
    const uint64_t ei = rng.u64() % (uint64_t)S.numEmitters;
    const uint32_t f0 = S.emitOff[ei], f1 = S.emitOff[ei + 1];
    const uint64_t face = f0 + rng.u64() % (uint64_t)(f1 - f0);
    const float* fv = S.emitFaces + 9 * face;
    const V3 v0 = V3{fv[0], fv[1], fv[2]}, v1 = V3{fv[3], fv[4], fv[5]}, v2 = V3{fv[6], fv[7], fv[8]};
    float r0 = rng.f();
    float r1 = rng.f();
    float r2 = rng.f();
    const float rSum = r0 + r1 + r2;
    r0 /= rSum;
    r1 /= rSum;
    r2 /= rSum;
    EmitterSample e;
    e.pos = r0 * v0 + r1 * v1 + r2 * v2;
    e.color = V3{S.emitColor[3 * ei], S.emitColor[3 * ei + 1], S.emitColor[3 * ei + 2]};
    return e;
}

}  // namespace cx
