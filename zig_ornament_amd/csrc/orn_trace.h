// orn_trace.h -- device-side scene view, BVH traversal and shading for the
// gfx950 path-tracing kernels.
//
// Semantics follow the reference's WGSL megakernel
// (src/wgpu_backend/shaders/*.wgsl) operation for operation, so that the
// closest hit, every RNG draw and every accumulated value are reproduced
// bit for bit. The layout work is the MI355X part: nodes are fetched as four
// 16-byte vector loads, the traversal stack lives in LDS (one column per
// lane, stride = block size, so the 64 lanes of a wave hit 64 different
// banks), and materials are two 16-byte loads.
#pragma once

#include "orn_common.h"

namespace orn {

constexpr uint32_t kFinishedTraverseBlas = 0xffffffffu;  // pathtracer.wgsl:19
constexpr uint32_t kInTlas = 0xffffffffu;
constexpr float kTMaxInit = 3.40282e+38f;                 // bvh.wgsl:23
// The ordered search's distance culls (cull_spheres, blas_slack)
constexpr float kUnit = 5.9604645e-8f;            // unit roundoff
constexpr float kCullOffset = 4.0f * kUnit;       // of |o * inv|: the slab distances' rounding
constexpr float kCullRel = 1.0f + 16.0f * kUnit;  // of t
constexpr float kLeastDir2 = 3.2e-10f;  // |d|^2 from which safe_invdir leaves the largest component alone
constexpr float kEtaNear = 4.5f, kEtaFar = 8.9f, kEtaBall = 8.0f;

// One texture in the texel pool. format: components | (hdr << 8)
struct DevTexture {
    uint64_t offset;  // byte offset in the texel pool
    uint32_t width;
    uint32_t height;
    uint32_t components;
    uint32_t hdr;
};

// BVH4 child references: a BVH4 node index, a BVH2 leaf (kLeafRef | index
// into the BVH2 array of the same level) or an empty slot.
constexpr uint32_t kLeafRef = 0x80000000u;
constexpr uint32_t kEmptyRef = 0xfffffffeu;

// How far in front of its box rounding can put a sphere's distance, over every
// sphere of a scene without meshes (SearchTree::sphere_cull, cull_spheres).
struct SphereCull {
    float fixed, origin, dist, dist2;  // of 1, the ray's origin, and the distance and its square
    float least_dir2;                  // |d|^2 below which squares underflow
};

// The bound buffers of pathtracer.wgsl:7-17, resident in HBM, plus the
// derived BVH4 arrays (8 float4 = 128 B per node: children's min x, y, z,
// max x, y, z as float4 lanes, then the 4 child references).
struct DevScene {
    const float4 *__restrict__ tlas4;       // BVH4 of the TLAS
    const float4 *__restrict__ blas4;       // BVH4 of every BLAS
    const float4 *__restrict__ tlas_leaves; // TLAS copy whose mesh leaves point at BLAS BVH4 roots
    // The BVH2 of TLAS and BLASes in one array (4 float4 per node; BLAS nodes
    // follow the TLAS's), child indices and mesh leaves' BLAS roots carrying
    // kLeafRef for leaves: a node visit needs no choice of array (with the
    // object-space ray kept apart from the world's: Cornell box 1.69 -> 1.52
    // ms, random spheres 25.3 -> 24.1, instanced icospheres 22.6 -> 21.4).
    const float4 *__restrict__ nodes2;
    const float4 *__restrict__ blas2;       // where the BLAS nodes begin in it (BVH4 leaf references)
    const float4 *__restrict__ normals;     // 1 float4 per normal
    const uint32_t *__restrict__ normal_indices;
    const float2 *__restrict__ uvs;
    const uint32_t *__restrict__ uv_indices;
    const float4 *__restrict__ transforms;  // 4 float4 (columns) per matrix
    const uint4 *__restrict__ materials;    // 2 uint4 per material
    const DevTexture *__restrict__ textures;
    const uint8_t *__restrict__ texels;
    uint32_t tlas_len;
    uint32_t textures_len;
    uint32_t stack_slots;  // LDS stack entries per lane
    uint32_t tlas4_root;   // reference of the TLAS root in the BVH4
    uint32_t tlas2_root;   // index of the TLAS root, kLeafRef set when it is a leaf
    // The internal nodes of the search tree over the same leaves (orn_sah.h), in
    // the format of bvh2_format(); null: there is none, and rays take the
    // reference's order.
    const char *__restrict__ search;
    uint32_t search_root;  // as the search tree's references go
    uint32_t plain_spheres;  // every sphere is scaled along the axes and moved (see sphere_leaf)
    SphereCull cull;
};

// An internal node of the search tree of a scene without meshes: per axis the
// children's planes as left min, right min, left max, right max, left min,
// right min, so that one 16-byte load at an offset of 0 or 8, by the sign of
// the ray's direction, gives both near planes and then both far planes: 12
// minima and maxima of a node visit less. (The nearer of fma(min, inv, ox) and
// fma(max, inv, ox) is the min plane's for inv > 0 and the max plane's for
// inv < 0, whatever the rounding: fma is monotone.)
// References of a search tree: a leaf's index in nodes2 with kLeafRef, or an
// internal node's place in units of 16 bytes.
struct alignas(8) SearchQuad {
    float a, b, c, d;
};
struct SearchNode {
    float plane[3][6];
    uint32_t left, right;
};
static_assert(sizeof(SearchNode) == 80, "a search node is five 16-byte units");

struct Hit {
    float t;
    uint32_t material;
    uint32_t node_type;
    uint32_t inv_tid;  // 2 * transform_id
    uint32_t tri_id;   // 3 * triangle index
    float u, v;
};

struct Ray {
    f3 o, d;
};

// bvh.wgsl:139-174
__device__ __forceinline__ float copysign_ref(float a, float b) { return (b < 0.0f) ? -a : a; }

__device__ __forceinline__ f3 safe_invdir(f3 d)
{
    const float eps = 1e-5f;
    const float x = (fabsf(d.x) > eps) ? d.x : copysign_ref(eps, d.x);
    const float y = (fabsf(d.y) > eps) ? d.y : copysign_ref(eps, d.y);
    const float z = (fabsf(d.z) > eps) ? d.z : copysign_ref(eps, d.z);
    return f3{1.0f / x, 1.0f / y, 1.0f / z};
}

// bvh.wgsl:184-192: slab test with fused multiply-adds
__device__ __forceinline__ bool aabb_hit(float3 mn, float3 mx, f3 inv, f3 ox, float t_min,
                                         float t_max, float &near_t)
{
    const float fx = fmaf(mx.x, inv.x, ox.x), fy = fmaf(mx.y, inv.y, ox.y),
                fz = fmaf(mx.z, inv.z, ox.z);
    const float nx = fmaf(mn.x, inv.x, ox.x), ny = fmaf(mn.y, inv.y, ox.y),
                nz = fmaf(mn.z, inv.z, ox.z);
    const float far_t = fminf(fminf(fminf(fmaxf(fx, nx), fmaxf(fy, ny)), fmaxf(fz, nz)), t_max);
    near_t = fmaxf(fmaxf(fmaxf(fminf(fx, nx), fminf(fy, ny)), fminf(fz, nz)), t_min);
    return near_t <= far_t;
}
__device__ __forceinline__ bool aabb_hit(float3 mn, float3 mx, f3 inv, f3 ox, float t_min, float t_max)
{
    float near_t;
    return aabb_hit(mn, mx, inv, ox, t_min, t_max, near_t);
}

// bvh.wgsl:194-226: Moller-Trumbore as the reference writes it (no
// determinant test; NaN falls through the comparisons). Returns t_max and
// `ok` false for a miss.
__device__ __forceinline__ float triangle_hit(const Ray &r, f3 v1, f3 v2, f3 v3, float t_min,
                                              float t_max, float &hu, float &hv, bool &ok)
{
    ok = false;
    const f3 e1 = v2 - v1;
    const f3 e2 = v3 - v1;
    const f3 s1 = cross(r.d, e2);
    const float invd = 1.0f / dot(s1, e1);
    const f3 d = r.o - v1;
    const float u = dot(d, s1) * invd;
    if (u < 0.0f || u > 1.0f) return t_max;
    const f3 s2 = cross(d, e1);
    const float v = dot(r.d, s2) * invd;
    if (v < 0.0f || u + v > 1.0f) return t_max;
    const float t = dot(e2, s2) * invd;
    if (t < t_min || t > t_max) return t_max;
    hu = u;
    hv = v;
    ok = true;
    return t;
}

// bvh.wgsl:228-249: unit sphere at the origin of object space (`ok` as above)
__device__ __forceinline__ float sphere_hit(const Ray &r, float t_min, float t_max, bool &ok)
{
    ok = false;
    const float a = r.d.x * r.d.x + r.d.y * r.d.y + r.d.z * r.d.z;
    const float half_b = dot(r.o, r.d);
    const float c = (r.o.x * r.o.x + r.o.y * r.o.y + r.o.z * r.o.z) - 1.0f;
    const float disc = half_b * half_b - a * c;
    if (disc < 0.0f) return t_max;
    const float sq = sqrtf(disc);
    float t = (-half_b - sq) / a;
    if (t < t_min || t_max < t) {
        t = (-half_b + sq) / a;
        if (t < t_min || t_max < t) return t_max;
    }
    ok = true;
    return t;
}

// transform.wgsl: the 16 floats are read column-major; c0..c3 are columns
__device__ __forceinline__ f3 xform_point(const float4 *m, f3 p)
{
    const float4 c0 = m[0], c1 = m[1], c2 = m[2], c3 = m[3];
    return f3{c0.x * p.x + c1.x * p.y + c2.x * p.z + c3.x * 1.0f,
              c0.y * p.x + c1.y * p.y + c2.y * p.z + c3.y * 1.0f,
              c0.z * p.x + c1.z * p.y + c2.z * p.z + c3.z * 1.0f};
}

__device__ __forceinline__ Ray xform_ray(const float4 *m, const Ray &r)
{
    const float4 c0 = m[0], c1 = m[1], c2 = m[2], c3 = m[3];
    Ray o;
    o.o = f3{c0.x * r.o.x + c1.x * r.o.y + c2.x * r.o.z + c3.x * 1.0f,
             c0.y * r.o.x + c1.y * r.o.y + c2.y * r.o.z + c3.y * 1.0f,
             c0.z * r.o.x + c1.z * r.o.y + c2.z * r.o.z + c3.z * 1.0f};
    o.d = f3{c0.x * r.d.x + c1.x * r.d.y + c2.x * r.d.z + c3.x * 0.0f,
             c0.y * r.d.x + c1.y * r.d.y + c2.y * r.d.z + c3.y * 0.0f,
             c0.z * r.d.x + c1.z * r.d.y + c2.z * r.d.z + c3.z * 0.0f};
    return o;
}

// transform.wgsl:16-19: transpose(M) * (n, 0), i.e. dot(column_i, (n, 0))
__device__ __forceinline__ f3 xform_normal(const float4 *m, f3 n)
{
    const float4 c0 = m[0], c1 = m[1], c2 = m[2];
    return f3{c0.x * n.x + c0.y * n.y + c0.z * n.z + c0.w * 0.0f,
              c1.x * n.x + c1.y * n.y + c1.z * n.z + c1.w * 0.0f,
              c2.x * n.x + c2.y * n.y + c2.z * n.z + c2.w * 0.0f};
}

// A sphere leaf's test: n2 and n3 are the last two quarters of its node.
// Spheres made by the scene's factories are unit spheres scaled and moved, so
// off the diagonal their inverse transforms are zero; then (plain_spheres) the
// leaf holds the diagonal and the translation itself, and the ray reaches
// object space in 9 operations instead of 39, without a second load that
// waits for the first. The products left out are zeros: they can change the
// sign of a zero only, which the distance can show only for t_min <= 0 (a ray
// from the surface along it: t = -0 or +0), where the whole matrix is used.
// Infinite coordinates miss in both forms (NaN distance). With the centre
// below: random spheres 1080p 64 spp 28.4 -> 25.9 ms.
__device__ __forceinline__ float sphere_leaf(const DevScene &sc, float4 n2, float4 n3, uint32_t inv_tid,
                                             const Ray &r, float t_min, float limit, bool &ok)
{
    Ray o;
    if (sc.plain_spheres != 0u && t_min > 0.0f) {
        o.o = xyz(n2) * r.o + xyz(n3);
        o.d = xyz(n2) * r.d;
    } else {
        o = xform_ray(sc.transforms + 4u * inv_tid, r);
    }
    return sphere_hit(o, t_min, limit, ok);
}

// The centre of a sphere, M * (0, 0, 0, 1): the model matrix's translation
// where the leaf is plain (checked at upload: finite columns, no -0 in the
// translation, so that the zero products leave it as it is).
__device__ __forceinline__ f3 sphere_centre(const DevScene &sc, uint32_t inv_tid)
{
    const float4 *m = sc.transforms + 4u * (inv_tid + 1u);
    const float4 c3 = m[3];
    if (sc.plain_spheres != 0u) return xyz(c3);
    const float4 c0 = m[0], c1 = m[1], c2 = m[2];
    return f3{c0.x * 0.0f + c1.x * 0.0f + c2.x * 0.0f + c3.x * 1.0f,
              c0.y * 0.0f + c1.y * 0.0f + c2.y * 0.0f + c3.y * 1.0f,
              c0.z * 0.0f + c1.z * 0.0f + c2.z * 0.0f + c3.z * 1.0f};
}

// Scene content known at launch: kernels are instantiated without the code
// (and registers) of primitive kinds a scene does not contain.
enum SceneFeatures : uint32_t {
    kHasSpheres = 1u,
    kHasMeshes = 2u,
    kHasTextures = 4u,
    kNoSearchTree = 8u,  // BVH2 launches take the reference's order
};
// Node format of a BVH2 launch (the W of the traversal below). The wider nodes
// of format 2 take a quarter more of the caches for their shorter test: random
// spheres 1920x1080, 64 spp, 23.8 -> 23.3 ms with them and 500x500, 1 spp, 0.25 ->
// 0.235 ms, but 1,024 instanced icospheres 20.4 -> 20.9 ms (cost-ordered, 32 spp,
// with fewer visits, by a cull at every box; a stride of 96 bytes 21.1, of 128
// bytes 22.1). So the trees of a mesh scene,
// which are the large ones, keep the 64-byte boxes.
constexpr uint32_t bvh2_format(uint32_t f) { return (f & kNoSearchTree) ? 1u : (f & kHasMeshes) ? 3u : 2u; }
constexpr bool is_search_format(uint32_t w) { return w == 2u || w == 3u; }

// bvh.wgsl:14-137 as a resumable state machine: trav_begin() sets up one ray,
// trav_internal()/trav_leaf() visit one node and return false once the ray is
// finished. The node taken next is kept in a register: only nodes left for
// later go to the lane's LDS column (`stack`, stride = block size).
//
// The searches share the code, by the node format W. With W = 1 the order is
// the reference's (left pushed before right, so the right child is taken
// first), with the same strict `t < t_max` update; W = 4 is the BVH4 below.
// With W = 2 (SearchNode) and W = 3 (the BVH2's own node) the ray searches
// the scene's SAH tree, the nearer child first, and finds the same
// closest hit with far fewer node visits:
//  * A primitive is in reach of a ray when the ray passes the slab test of
//    its own leaf box without a distance limit. Every box above contains that
//    box and the slab arithmetic is monotone (fma, min, max), so the boxes
//    above then pass too, in either tree, and no other primitive is visited
//    by either search.
//  * The reference returns the smallest t over the primitives in reach, the
//    first visited among equal ones, unless that t lies in front of the
//    primitive's own boxes (rounding: half of all hits on a flat,
//    axis-aligned wall) and another hit lies between the two: the other one,
//    met first, culls the boxes. The ordered search sees both cases, a tie
//    with the best t and another hit in front of the best one's boxes: they
//    set `redo`, and the ray is searched again in the reference's order
//    (trav_redo).
//  * That holds as long as every primitive in reach is visited whose t is no
//    larger than the best one's, or than where the best one's boxes begin
//    (`near_best`). So a box is culled only beyond t_cull, which lies past
//    both by as much as rounding can put a primitive's t in front of its
//    box. For spheres that is bounded by the scene (cull_spheres).
//    For triangles it is bounded only where the ray is not nearly in the
//    triangle's plane: there the determinant, which the reference does not
//    test, is rounding noise, and so is t. A BLAS is culled where its mesh's
//    core rules such triangles out (blas_slack), and searched whole where not;
//    between BLASes, whose meshes a ray has not yet been compared with,
//    nothing is culled.
// The search is bound by the vector instructions of its node visits, so fewer
// visits are time: random spheres 1920x1080, 64 spp, 52 -> 33 ms with it. The
// kernels of mesh scenes in the reference's order and in this one: 1,024 instanced
// icospheres 1080p, 32 spp, 33.7 -> 22.8 ms, textured, metal and glass icospheres
// 700x700, 8 spp, 6.5 -> 3.75, 16 images of such scenes 9.5 -> 6.9, the Cornell
// box 256x256, 16 spp, 1.52 -> 1.47, a radiance-cache frame over the icospheres
// 1.25 -> 0.92. (A cull by distance at every box would take the icospheres 18.5 ms
// and miss hits; the instances behind the hit cost 2.1, the slack's arithmetic 0.9
// and rays that pass by the core 1.4.) Scenes whose arrays do not have nested
// boxes, or which would not gain (SearchTree::build), have no search tree.
struct Traversal {
    Ray ray;        // the ray in object space, inside a BLAS
    f3 inv, ox;     // safe_invdir(d) and -o * inv of the ray in the current space
    f3 winv, wox;   // the same of the world-space ray, restored on leaving a BLAS
    uint32_t sx, sy, sz;  // W = 2: plane offsets of a SearchNode by the signs of inv
    float t_max;
    float t_cull;     // search tree: boxes and hits beyond it are skipped
    float near_best;  // search tree: where the boxes of the closest hit begin
    float mesh_near;  // search tree: where the ray enters the box of the instance it is in
    float slack;      // search tree: how far past the best hit the BLAS it is in is searched
    uint32_t addr;  // next node to visit
    uint32_t top;   // pending entries in the LDS column
    uint32_t material_index, inv_tid;  // of the mesh being traversed
    uint32_t blas_top;  // `top` when the ray entered the BLAS it is in (kInTlas: none)
    bool hit;
    bool redo;   // search tree: the closest hit needs the reference's order (see above)
    Hit h;
};

// Where a ray finds its near planes in a SearchNode's three axes.
__device__ __forceinline__ void trav_signs(Traversal &tr)
{
    tr.sx = (as_u32(tr.inv.x) >> 31) * 8u;
    tr.sy = (as_u32(tr.inv.y) >> 31) * 8u + 24u;
    tr.sz = (as_u32(tr.inv.z) >> 31) * 8u + 48u;
}

// `root`: the TLAS root reference in the traversed format (BVH2, its search
// tree, or BVH4).
__device__ __forceinline__ void trav_begin(uint32_t root, const Ray &world, Traversal &tr)
{
    tr.inv = safe_invdir(world.d);
    tr.ox = (-world.o) * tr.inv;
    trav_signs(tr);
    tr.winv = tr.inv;
    tr.wox = tr.ox;
    tr.t_max = kTMaxInit;
    tr.t_cull = kTMaxInit;
    tr.near_best = 0.0f;
    tr.mesh_near = 0.0f;
    tr.slack = 0.0f;
    tr.redo = false;
    tr.addr = root;
    tr.top = 0u;
    tr.material_index = 0u;
    tr.inv_tid = 0u;
    tr.blas_top = kInTlas;
    tr.hit = false;
}

// An empty asm statement that reads and "writes" one register of each of a
// node's four 16-byte loads: the compiler must have all four loaded at this
// point and cannot sink any of them into a branch. No instruction is emitted.
__device__ __forceinline__ void pin_node(float4 &a, float4 &b, float4 &c, float4 &d)
{
    asm volatile("" : "+v"(a.x), "+v"(b.x), "+v"(c.x), "+v"(d.x));
}

// Takes the next pending node off the lane's stack; false when none is left.
// A BLAS is done when the stack is down to where it was on entering it (the
// reference pushes a marker instead, bvh.wgsl:88-95).
template <uint32_t F>
__device__ __forceinline__ bool trav_pop(uint32_t *stack, uint32_t stride, Traversal &tr)
{
    if (tr.top == 0u) return false;
    if ((F & kHasMeshes) && tr.top == tr.blas_top) {
        // back in the TLAS: the world-space ray's reciprocal, kept from
        // trav_begin
        tr.blas_top = kInTlas;
        tr.t_cull = kTMaxInit;
        tr.inv = tr.winv;
        tr.ox = tr.wox;
    }
    tr.addr = stack[(--tr.top) * stride];
    return true;
}

// One BVH4 node: the hit children are pushed in slot order and the last hit
// one is taken next, so they come off the stack last slot first -- the
// reference's right-before-left order, two levels at a time.
__device__ __forceinline__ bool bvh4_node(const float4 *nd, uint32_t *stack, uint32_t stride,
                                          uint32_t cap, float t_min, Traversal &tr)
{
    const float4 lx = nd[0], ly = nd[1], lz = nd[2], hx = nd[3], hy = nd[4], hz = nd[5];
    const uint4 c = *reinterpret_cast<const uint4 *>(nd + 6);
    const bool h0 = c.x != kEmptyRef &&
                    aabb_hit(make_float3(lx.x, ly.x, lz.x), make_float3(hx.x, hy.x, hz.x), tr.inv, tr.ox, t_min, tr.t_max);
    const bool h1 = c.y != kEmptyRef &&
                    aabb_hit(make_float3(lx.y, ly.y, lz.y), make_float3(hx.y, hy.y, hz.y), tr.inv, tr.ox, t_min, tr.t_max);
    const bool h2 = c.z != kEmptyRef &&
                    aabb_hit(make_float3(lx.z, ly.z, lz.z), make_float3(hx.z, hy.z, hz.z), tr.inv, tr.ox, t_min, tr.t_max);
    const bool h3 = c.w != kEmptyRef &&
                    aabb_hit(make_float3(lx.w, ly.w, lz.w), make_float3(hx.w, hy.w, hz.w), tr.inv, tr.ox, t_min, tr.t_max);
    uint32_t next = kEmptyRef;
    if (h0) next = c.x;
    if (h1) {
        if (next != kEmptyRef && tr.top < cap) stack[(tr.top++) * stride] = next;
        next = c.y;
    }
    if (h2) {
        if (next != kEmptyRef && tr.top < cap) stack[(tr.top++) * stride] = next;
        next = c.z;
    }
    if (h3) {
        if (next != kEmptyRef && tr.top < cap) stack[(tr.top++) * stride] = next;
        next = c.w;
    }
    if (next == kEmptyRef) return false;
    tr.addr = next;
    return true;
}

__device__ __forceinline__ float max_abs(f3 a) { return fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fabsf(a.z)); }

// sqrt to within an ulp, for bounds that have room for it
ORN_HD float sqrt_near(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_sqrtf(x);
#else
    return sqrtf(x);
#endif
}

// What t_cull is measured from: the best hit, where its boxes begin, and the
// size of any distance in front of those.
__device__ __forceinline__ float cull_from(const Traversal &tr, float t_min)
{
    return fmaxf(fmaxf(tr.t_max, tr.near_best), fabsf(t_min));
}

// t_cull in a scene of spheres alone. With o, d the ray in a sphere's object
// space and q = |o|, the terms of sphere_hit's discriminant are off by at most
// u (17 q^2 + 6) |d|^2 (u: unit roundoff), and the root taken from them puts
// the point o + t d outside of the unit sphere by at most X / 2 with
// X = 28 u (q^2 + 1), near-tangent hits included: there t is off along the
// surface, not away from it. q itself is at most 1.002 (|t d| + 1.01). In
// world space that, the rounding of the transform and what the sphere's box
// leaves out of the sphere bound how far the point lies outside of the box
// (SphereCull, by SearchTree::sphere_cull), and the slab distance of the box
// is in front of t by no more than that over the direction's smallest
// component. The bound grows with t, so it is taken for the largest t that
// matters.
__device__ __forceinline__ void cull_spheres(const DevScene &sc, const Ray &world, float t_min, Traversal &tr)
{
    const float from = cull_from(tr, t_min), dd = dot(world.d, world.d), y = from * sqrt_near(dd);
    const float out = fmaf(y, fmaf(y, sc.cull.dist2, sc.cull.dist), fmaf(max_abs(world.o), sc.cull.origin, sc.cull.fixed));
    const float slack = fmaf(max_abs(tr.inv), out, kCullOffset * max_abs(tr.ox));
    // (fminf drops a NaN, and infinite coordinates cull nothing)
    tr.t_cull = dd >= sc.cull.least_dir2 ? fminf(fmaf(from, kCullRel, slack), kTMaxInit) : kTMaxInit;
}

// The slack of a BLAS for the object-space ray in `tr`; infinite where the ray
// may lie nearly in the plane of one of the mesh's triangles. n2 and n3 are
// the mesh leaf's words: the core's centre c, its squared radius r2, and eta
// (times kEtaNear, and times kEtaFar and the mesh's size; SearchTree::mesh_core).
// A triangle hit (u, v and t accepted) whose determinant is below kappa |d|
// |e1| |e2| lies nearly in the ray's plane, so the ray passes c at a distance
// of at least the triangle plane's, less what the core leaves for it. A ray
// that comes closer to c meets every triangle at a larger determinant, where
// rounding moves u, v and t by at most eta (1 + |o - v| / |e|), so that the
// slab distance of the triangle's box is in front of t by no more than eta
// (4.5 |o - c| + 8.9 R) over the direction's smallest component, in front of
// which slab distances round by a few units of o * inv.
__device__ __forceinline__ float blas_slack(float4 n2, float4 n3, const Traversal &tr)
{
    const f3 p = tr.ray.o - xyz(n2);
    const float a = dot(p, p), b = dot(p, tr.ray.d), c = dot(tr.ray.d, tr.ray.d), ac = a * c;
    const bool inside = fmaf(ac, n3.y * (1.0f / (kEtaNear * kEtaBall)), ac - b * b) < n3.x * c;
    const float slack = fmaf(max_abs(tr.inv), fmaf(n3.y, sqrt_near(a), n3.z), kCullOffset * max_abs(tr.ox));
    return inside && c >= kLeastDir2 ? slack : __builtin_inff();
}
__device__ __forceinline__ float blas_cull(const Traversal &tr, float t_min)
{
    return fminf(fmaf(cull_from(tr, t_min), kCullRel, tr.slack), kTMaxInit);
}

// A new closest hit (tr.t_max) after one at t_old, its boxes entered at near_t.
__device__ __forceinline__ void trav_nearer(Traversal &tr, float t_old, float near_t)
{
    tr.near_best = near_t;
    tr.redo = near_t > t_old;
}

// A hit at t no closer than the best one.
__device__ __forceinline__ void trav_behind(Traversal &tr, float t)
{
    if (t < tr.near_best || t == tr.t_max) tr.redo = true;
}

// Node references carry kLeafRef when they name a leaf (in the BVH4 by
// construction, in the BVH2 through the flagged copies), so a lane knows
// whether its next step is an internal node or a leaf before loading it.
// trav_internal() visits an internal node, trav_leaf() a leaf; both return
// false once the ray is finished.
template <uint32_t F, uint32_t W>
__device__ __forceinline__ bool trav_internal(const DevScene &sc, float t_min, const Ray &world,
                                              uint32_t *stack, uint32_t stride, Traversal &tr)
{
    const uint32_t cap = sc.stack_slots;
    if (W == 4u) {
        const bool blas = (F & kHasMeshes) && tr.blas_top != kInTlas;
        const float4 *nd = (blas ? sc.blas4 : sc.tlas4) + 8u * tr.addr;
        if (bvh4_node(nd, stack, stride, cap, t_min, tr)) return true;
        return trav_pop<F>(stack, stride, tr);
    }
    bool l, r;
    uint32_t left, right;
    bool left_first;
    if constexpr (W == 2u) {
        const uint32_t off = tr.addr << 4;  // 32 bits from a scalar base: the tree is at most 4 GB
        auto quad = [&](uint32_t o) { return *reinterpret_cast<const SearchQuad *>(sc.search + (off + o)); };
        const SearchQuad x = quad(tr.sx), y = quad(tr.sy), z = quad(tr.sz);
        const uint2 kids = *reinterpret_cast<const uint2 *>(sc.search + off + offsetof(SearchNode, left));
        left = kids.x;
        right = kids.y;
        const float ln = fmaxf(fmaxf(fmaxf(fmaf(x.a, tr.inv.x, tr.ox.x), fmaf(y.a, tr.inv.y, tr.ox.y)),
                                     fmaf(z.a, tr.inv.z, tr.ox.z)), t_min);
        const float rn = fmaxf(fmaxf(fmaxf(fmaf(x.b, tr.inv.x, tr.ox.x), fmaf(y.b, tr.inv.y, tr.ox.y)),
                                     fmaf(z.b, tr.inv.z, tr.ox.z)), t_min);
        const float lf = fminf(fminf(fminf(fmaf(x.c, tr.inv.x, tr.ox.x), fmaf(y.c, tr.inv.y, tr.ox.y)),
                                     fmaf(z.c, tr.inv.z, tr.ox.z)), tr.t_cull);
        const float rf = fminf(fminf(fminf(fmaf(x.d, tr.inv.x, tr.ox.x), fmaf(y.d, tr.inv.y, tr.ox.y)),
                                     fmaf(z.d, tr.inv.z, tr.ox.z)), tr.t_cull);
        l = ln <= lf;
        r = rn <= rf;
        left_first = !r | (l & (ln < rn));  // the nearer child
    } else {
        constexpr bool ORD = W == 3u;
        const float4 *node = ORD ? reinterpret_cast<const float4 *>(sc.search + (tr.addr << 4)) : sc.nodes2 + 4u * tr.addr;
        const float4 n0 = node[0], n1 = node[1], n2 = node[2], n3 = node[3];
        const float limit = ORD ? tr.t_cull : tr.t_max;
        float ln, rn;
        l = aabb_hit(make_float3(n0.x, n0.y, n0.z), make_float3(n1.x, n1.y, n1.z), tr.inv, tr.ox, t_min, limit, ln);
        r = aabb_hit(make_float3(n2.x, n2.y, n2.z), make_float3(n3.x, n3.y, n3.z), tr.inv, tr.ox, t_min, limit, rn);
        left = as_u32(n0.w);
        right = as_u32(n1.w);
        left_first = !r | (ORD & l & (ln < rn));  // the nearer child, or the reference's order: right first
    }
    // both hit: one child is next, the other waits on the stack
    if (l && r && tr.top < cap) stack[(tr.top++) * stride] = left_first ? right : left;
    if (l || r) {
        tr.addr = left_first ? left : right;
        return true;
    }
    return trav_pop<F>(stack, stride, tr);
}

template <uint32_t F, uint32_t W>
__device__ __forceinline__ bool trav_leaf(const DevScene &sc, float t_min, const Ray &world,
                                          uint32_t *stack, uint32_t stride, Traversal &tr)
{
    const uint32_t idx = tr.addr & ~kLeafRef;
    constexpr bool ORD = is_search_format(W);
    const float4 *base = W != 4u ? sc.nodes2 : ((F & kHasMeshes) && tr.blas_top != kInTlas ? sc.blas2 : sc.tlas_leaves);
    const float4 *node = base + 4u * idx;
    float4 n0 = node[0], n1 = node[1], n2 = node[2], n3 = node[3];
    // Keep the four 16-byte loads of the node together ahead of the type
    // branch: left alone, the compiler loads the type word first and the
    // rest inside each branch, two dependent trips to memory per node.
    pin_node(n0, n1, n2, n3);
    const float limit = ORD ? tr.t_cull : tr.t_max;
    const uint32_t type = as_u32(n2.w);
    if ((F & kHasSpheres) && type == 1u) {
        const uint32_t tid = as_u32(n3.w) * 2u;
        bool ok;
        const float t = sphere_leaf(sc, n2, n3, tid, world, t_min, limit, ok);
        if (t < tr.t_max) {
            const float t_old = tr.t_max;
            tr.hit = true;
            tr.t_max = t;
            tr.h.t = t;
            tr.h.material = as_u32(n1.w);
            tr.h.node_type = 1u;
            tr.h.inv_tid = tid;
            if constexpr (ORD) {
                float near_t;  // the leaf's own box is kept in the unused words of the leaf
                (void)aabb_hit(make_float3(n0.x, n0.y, n0.z), make_float3(n1.x, n1.y, n1.z), tr.inv, tr.ox, t_min,
                               tr.t_max, near_t);
                trav_nearer(tr, t_old, near_t);
                if constexpr (W == 2u) cull_spheres(sc, world, t_min, tr);
            }
        } else if (ORD && ok) {
            trav_behind(tr, t);
        }
    } else if ((F & kHasMeshes) && type == 2u) {
        if constexpr (ORD)
            (void)aabb_hit(make_float3(n0.x, n0.y, n0.z), make_float3(n1.x, n1.y, n1.z), tr.inv, tr.ox, t_min,
                           tr.t_max, tr.mesh_near);
        tr.blas_top = tr.top;
        tr.inv_tid = as_u32(n3.w) * 2u;
        tr.material_index = as_u32(n1.w);
        tr.ray = xform_ray(sc.transforms + 4u * tr.inv_tid, world);
        tr.inv = safe_invdir(tr.ray.d);
        tr.ox = (-tr.ray.o) * tr.inv;
        if constexpr (ORD) {
            tr.slack = blas_slack(n2, n3, tr);
            tr.t_cull = blas_cull(tr, t_min);
        }
        tr.addr = as_u32(n0.w);
        return true;
    } else if ((F & kHasMeshes) && type == 3u) {
        float u = 0.0f, v = 0.0f;
        bool ok;
        const float t = triangle_hit(tr.ray, xyz(n0), xyz(n1), xyz(n2), t_min, limit, u, v, ok);
        if (t < tr.t_max) {
            const float t_old = tr.t_max;
            tr.hit = true;
            tr.t_max = t;
            tr.h.t = t;
            tr.h.material = tr.material_index;
            tr.h.node_type = 2u;
            tr.h.inv_tid = tr.inv_tid;
            tr.h.tri_id = as_u32(n0.w) * 3u;
            tr.h.u = u;
            tr.h.v = v;
            if constexpr (ORD) {
                float near_t;  // a triangle's box spans its vertices (checked at upload)
                (void)aabb_hit(make_float3(fminf(fminf(n0.x, n1.x), n2.x), fminf(fminf(n0.y, n1.y), n2.y),
                                           fminf(fminf(n0.z, n1.z), n2.z)),
                               make_float3(fmaxf(fmaxf(n0.x, n1.x), n2.x), fmaxf(fmaxf(n0.y, n1.y), n2.y),
                                           fmaxf(fmaxf(n0.z, n1.z), n2.z)),
                               tr.inv, tr.ox, t_min, tr.t_max, near_t);
                trav_nearer(tr, t_old, fmaxf(near_t, tr.mesh_near));
                tr.t_cull = blas_cull(tr, t_min);
            }
        } else if (ORD && ok) {
            trav_behind(tr, t);
        }
    }
    return trav_pop<F>(stack, stride, tr);
}

// The ray of a finished ordered search once more, in the reference's order
// from the reference's TLAS root.
template <uint32_t F>
__device__ __forceinline__ void trav_redo(const DevScene &sc, uint32_t root, float t_min, const Ray &world,
                                          uint32_t *stack, uint32_t stride, Traversal &tr)
{
    trav_begin(root, world, tr);
    for (bool on = true; on;)
        on = (tr.addr & kLeafRef) ? trav_leaf<F, 1>(sc, t_min, world, stack, stride, tr)
                                  : trav_internal<F, 1>(sc, t_min, world, stack, stride, tr);
}

// The whole of bvh_hit for one ray. With STEPS > 1 a lane visits up to STEPS
// internal nodes in a row and then, if it stands at one, a leaf: lanes of a
// wave that stand at leaves then test them together instead of each leaf
// visit splitting the wave. Every lane still meets its own nodes in the same
// order, so the result does not depend on STEPS.
template <uint32_t F, uint32_t W, uint32_t STEPS = 1>
__device__ __forceinline__ bool bvh_hit(const DevScene &sc, float t_min, const Ray &world,
                                        uint32_t *stack, uint32_t stride, Hit &h)
{
    constexpr bool ORD = is_search_format(W);
    Traversal tr;
    trav_begin(W == 4u ? sc.tlas4_root : ORD ? sc.search_root : sc.tlas2_root, world, tr);
    bool on = true;
    while (on) {
        for (uint32_t k = 0; k < STEPS && on && !(tr.addr & kLeafRef); k++)
            on = trav_internal<F, W>(sc, t_min, world, stack, stride, tr);
        if (on && (tr.addr & kLeafRef)) on = trav_leaf<F, W>(sc, t_min, world, stack, stride, tr);
    }
    if (ORD && tr.redo) trav_redo<F>(sc, sc.tlas2_root, t_min, world, stack, stride, tr);
    h = tr.h;
    return tr.hit;
}

// bvh_hit for the 64 rays of a wave at once (BVH2). The wave walks the tree
// one node at a time on one stack (entry i held by lane i of three registers:
// the node and the 64-bit mask of the lanes that entered it). At an internal
// node each active lane tests both child boxes with its own ray and t_max;
// the wave goes on with the right child for the lanes whose ray hit it and
// pushes the left child for the lanes whose ray hit that. So a lane is active
// in exactly the nodes its own bvh_hit visits, meets them in the same order
// with the same t_max, and ends with bvh_hit's result bit for bit. For
// coherent rays (a camera tile) the wave visits few more nodes than one ray
// does, with every lane busy and every node load at one address. Every lane
// of the wave calls it (valid = false for a lane without a ray); `cap` is the
// scene's BVH2 stack bound (at most 64).
template <uint32_t F>
__device__ __forceinline__ bool bvh_hit_packet(const DevScene &sc, float t_min, const Ray &world, bool valid,
                                               uint32_t cap, Hit &h)
{
    Traversal tr;
    trav_begin(sc.tlas2_root, world, tr);
    const uint32_t lane = __lane_id();
    uint64_t active = lanes_where(valid);
    uint32_t addr = sc.tlas2_root;
    uint32_t top = 0;
    uint32_t s_node = 0, s_lo = 0, s_hi = 0;  // the wave's stack, entry i in lane i
    auto push = [&](uint32_t node, uint64_t mask) {
        if (top >= cap) return;
        const bool mine = lane == top;  // lane `top` holds the new entry
        s_node = mine ? node : s_node;
        s_lo = mine ? static_cast<uint32_t>(mask) : s_lo;
        s_hi = mine ? static_cast<uint32_t>(mask >> 32) : s_hi;
        top++;
    };
    while (active) {
        const bool me = (active >> lane) & 1ull;
        if (!(addr & kLeafRef)) {
            const float4 *node = sc.nodes2 + 4u * addr;
            const float4 n0 = node[0], n1 = node[1], n2 = node[2], n3 = node[3];
            const bool l = me && aabb_hit(make_float3(n0.x, n0.y, n0.z), make_float3(n1.x, n1.y, n1.z), tr.inv,
                                          tr.ox, t_min, tr.t_max);
            const bool r = me && aabb_hit(make_float3(n2.x, n2.y, n2.z), make_float3(n3.x, n3.y, n3.z), tr.inv,
                                          tr.ox, t_min, tr.t_max);
            const uint64_t ml = lanes_where(l), mr = lanes_where(r);
            const uint32_t left = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(as_u32(n0.w))));
            const uint32_t right = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(as_u32(n1.w))));
            if (mr) {
                if (ml) push(left, ml);
                addr = right;
                active = mr;
                continue;
            }
            if (ml) {
                addr = left;
                active = ml;
                continue;
            }
        } else {
            const uint32_t idx = addr & ~kLeafRef;
            const float4 *node = sc.nodes2 + 4u * idx;
            const float4 n0 = node[0], n1 = node[1], n2 = node[2], n3 = node[3];
            const uint32_t type = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(as_u32(n2.w))));
            if ((F & kHasSpheres) && type == 1u) {
                if (me) {
                    const uint32_t tid = as_u32(n3.w) * 2u;
                    bool ok;
                    const float t = sphere_leaf(sc, n2, n3, tid, world, t_min, tr.t_max, ok);
                    if (t < tr.t_max) {
                        tr.hit = true;
                        tr.t_max = t;
                        tr.h.t = t;
                        tr.h.material = as_u32(n1.w);
                        tr.h.node_type = 1u;
                        tr.h.inv_tid = tid;
                    }
                }
            } else if ((F & kHasMeshes) && type == 2u) {
                if (me) {
                    tr.inv_tid = as_u32(n3.w) * 2u;
                    tr.material_index = as_u32(n1.w);
                    tr.ray = xform_ray(sc.transforms + 4u * tr.inv_tid, world);
                    tr.inv = safe_invdir(tr.ray.d);
                    tr.ox = (-tr.ray.o) * tr.inv;
                }
                push(kFinishedTraverseBlas, 0ull);
                addr = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(as_u32(n0.w))));
                continue;  // the same lanes go on into the BLAS
            } else if ((F & kHasMeshes) && type == 3u) {
                if (me) {
                    float u = 0.0f, v = 0.0f;
                    bool ok;
                    const float t = triangle_hit(tr.ray, xyz(n0), xyz(n1), xyz(n2), t_min, tr.t_max, u, v, ok);
                    if (t < tr.t_max) {
                        tr.hit = true;
                        tr.t_max = t;
                        tr.h.t = t;
                        tr.h.material = tr.material_index;
                        tr.h.node_type = 2u;
                        tr.h.inv_tid = tr.inv_tid;
                        tr.h.tri_id = as_u32(n0.w) * 3u;
                        tr.h.u = u;
                        tr.h.v = v;
                    }
                }
            }
        }
        // next pending entry; leaving a BLAS restores every lane's world ray
        // (a no-op for the lanes that did not enter it)
        active = 0ull;
        while (top) {
            --top;
            const uint32_t a = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(s_node),
                                                                               static_cast<int>(top)));
            if ((F & kHasMeshes) && a == kFinishedTraverseBlas) {
                tr.inv = tr.winv;
                tr.ox = tr.wox;
                continue;
            }
            addr = a;
            active = (uint64_t(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(s_hi),
                                                                               static_cast<int>(top))))
                      << 32) |
                     static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(s_lo), static_cast<int>(top)));
            break;
        }
    }
    h = tr.h;
    return tr.hit;
}


// ---------------------------------------------------------------------------
// Shading: material.wgsl, hitrecord.wgsl, pathtracer.wgsl:95-161
// ---------------------------------------------------------------------------

struct Material {
    f3 albedo;
    uint32_t texture;
    float fuzz;
    float ior;
    uint32_t type;
};

__device__ __forceinline__ Material load_material(const DevScene &sc, uint32_t i)
{
    const uint4 a = sc.materials[2u * i], b = sc.materials[2u * i + 1u];
    Material m;
    m.albedo = f3{as_f32(a.x), as_f32(a.y), as_f32(a.z)};
    m.texture = a.w;
    m.fuzz = as_f32(b.x);
    m.ior = as_f32(b.y);
    m.type = b.z;
    return m;
}

__device__ __forceinline__ float half_to_float(uint32_t h)
{
    const uint32_t sign = (h >> 15) << 31;
    const uint32_t e = (h >> 10) & 0x1fu, man = h & 0x3ffu;
    if (e == 0u) {
        const float f = static_cast<float>(man) * 5.9604644775390625e-08f;
        return sign ? -f : f;
    }
    if (e == 31u) return as_f32(sign | 0x7f800000u | (man << 13));
    return as_f32(sign | ((e + 112u) << 23) | (man << 13));
}

// textureSampleLevel with the default WebGPU sampler: nearest, clamp to edge,
// level 0 (webgpu.zig:812-825); rgba8unorm reads as byte / 255.
__device__ __forceinline__ f3 sample_texture(const DevScene &sc, uint32_t id, float u, float v)
{
    const DevTexture tx = sc.textures[id];
    float fx = floorf(u * static_cast<float>(tx.width));
    float fy = floorf(v * static_cast<float>(tx.height));
    fx = fminf(fmaxf(fx, 0.0f), static_cast<float>(tx.width - 1u));
    fy = fminf(fmaxf(fy, 0.0f), static_cast<float>(tx.height - 1u));
    const uint64_t texel = static_cast<uint64_t>(static_cast<uint32_t>(fy)) * tx.width +
                           static_cast<uint32_t>(fx);
    float c[3] = {0.0f, 0.0f, 0.0f};
    if (tx.hdr) {
        const uint16_t *d =
            reinterpret_cast<const uint16_t *>(sc.texels + tx.offset) + texel * tx.components;
        if (tx.components == 4u) {
            const uint2 q = *reinterpret_cast<const uint2 *>(d);
            c[0] = half_to_float(q.x & 0xffffu);
            c[1] = half_to_float(q.x >> 16);
            c[2] = half_to_float(q.y & 0xffffu);
        } else {
            for (uint32_t k = 0; k < tx.components; k++) c[k] = half_to_float(d[k]);
        }
    } else {
        const uint8_t *d = sc.texels + tx.offset + texel * tx.components;
        if (tx.components == 4u) {
            const uint32_t q = *reinterpret_cast<const uint32_t *>(d);
            c[0] = static_cast<float>(q & 0xffu) / 255.0f;
            c[1] = static_cast<float>((q >> 8) & 0xffu) / 255.0f;
            c[2] = static_cast<float>((q >> 16) & 0xffu) / 255.0f;
        } else {
            for (uint32_t k = 0; k < tx.components; k++) c[k] = static_cast<float>(d[k]) / 255.0f;
        }
    }
    return f3{c[0], c[1], c[2]};
}

__device__ __forceinline__ bool near_zero(f3 e)
{
    return fabsf(e.x) < 1e-8f && fabsf(e.y) < 1e-8f && fabsf(e.z) < 1e-8f;
}

// WGSL reflect / refract
__device__ __forceinline__ f3 reflect_dir(f3 v, f3 n) { return v - (2.0f * dot(n, v)) * n; }

__device__ __forceinline__ f3 refract_dir(f3 e1, f3 e2, float eta)
{
    const float d = dot(e2, e1);
    const float k = 1.0f - eta * eta * (1.0f - d * d);
    if (k < 0.0f) return f3{0.0f, 0.0f, 0.0f};
    return eta * e1 - (eta * d + sqrtf(k)) * e2;
}

// The shading point of a closest hit (pathtracer.wgsl:114-135,
// hitrecord.wgsl:10-18): position, front-facing shading normal, material and
// texture coordinates (uv is only computed when a texture will be read).
struct Surface {
    f3 p;
    f3 normal;
    bool front;
    bool textured;
    float tu, tv;
    Material m;
};

// The same operations as the first half of shade() (which keeps its own
// copy: sharing this function changed the hot kernel's register allocation).
template <uint32_t F>
__device__ __forceinline__ Surface surface(const DevScene &sc, uint32_t textures_count, uint32_t tex_base,
                                           const Ray &ray, const Hit &h)
{
    Surface s;
    s.p = ray.o + h.t * ray.d;
    s.m = load_material(sc, h.material);
    const Material &m = s.m;
    s.textured =
        (F & kHasTextures) && m.texture - tex_base < textures_count && m.texture < sc.textures_len;
    s.tu = 0.0f;
    s.tv = 0.0f;
    f3 outward;
    if ((F & kHasSpheres) && (!(F & kHasMeshes) || h.node_type == 1u)) {
        // sphere: outward = normalize(p - M * (0,0,0,1))
        outward = normalize(s.p - sphere_centre(sc, h.inv_tid));
        if (s.textured) {  // uv only reaches the result through a texture fetch
            const float theta = acos_f(-outward.y);
            const float phi = atan2_f(-outward.z, outward.x) + kPi;
            s.tu = phi / (2.0f * kPi);
            s.tv = theta / kPi;
        }
    } else {
        // mesh: barycentric shading normal and uv, normal by transpose(inverse)
        const uint32_t i0 = sc.normal_indices[h.tri_id], i1 = sc.normal_indices[h.tri_id + 1u],
                       i2 = sc.normal_indices[h.tri_id + 2u];
        const f3 n0 = xyz(sc.normals[i0]), n1 = xyz(sc.normals[i1]), n2 = xyz(sc.normals[i2]);
        const float w = 1.0f - h.u - h.v;
        const f3 nrm = (w * n0 + h.u * n1) + h.v * n2;
        if (s.textured) {
            const float2 uv0 = sc.uvs[sc.uv_indices[h.tri_id]];
            const float2 uv1 = sc.uvs[sc.uv_indices[h.tri_id + 1u]];
            const float2 uv2 = sc.uvs[sc.uv_indices[h.tri_id + 2u]];
            s.tu = w * uv0.x + h.u * uv1.x + h.v * uv2.x;
            s.tv = w * uv0.y + h.u * uv1.y + h.v * uv2.y;
        }
        outward = normalize(xform_normal(sc.transforms + 4u * h.inv_tid, nrm));
    }
    // hitrecord.wgsl:10-18
    if (dot(ray.d, outward) > 0.0f) {
        s.normal = -outward;
        s.front = false;
    } else {
        s.normal = outward;
        s.front = true;
    }
    return s;
}

// Shading of one closest hit: fills the next ray and the attenuation, or the
// emitted radiance when the path ends (pathtracer.wgsl:114-157).
// Returns true when the path continues.
// Texture lookup (material.wgsl:91-99): a material's texture is sampled when
// its index, counted from `tex_base`, is below `textures_count`. tex_base is
// the scene's first texture in the shared texture table (non-zero when
// several scenes share one device scene; their materials then hold indices
// into the shared table, and 0xffffffff for "none"). Textures beyond what was
// uploaded read as "no texture" (the reference would index its binding array
// out of range there).
// `ud` is normalize(ray.d), computed by the caller once for every kind of lane
// (sky, metal and dielectric lanes of a wave would each run their own).
template <uint32_t F>
__device__ __forceinline__ bool shade(const DevScene &sc, uint32_t textures_count, uint32_t tex_base,
                                      const Ray &ray, f3 ud, const Hit &h, uint32_t &rng, Ray &next, f3 &weight)
{
    const f3 p = ray.o + h.t * ray.d;
    const Material m = load_material(sc, h.material);
    const bool textured =
        (F & kHasTextures) && m.texture - tex_base < textures_count && m.texture < sc.textures_len;
    f3 normal;
    bool front;
    float tu = 0.0f, tv = 0.0f;
    f3 outward;
    if ((F & kHasSpheres) && (!(F & kHasMeshes) || h.node_type == 1u)) {
        // sphere: outward = normalize(p - M * (0,0,0,1))
        outward = normalize(p - sphere_centre(sc, h.inv_tid));
        if (textured) {  // uv only reaches the result through a texture fetch
            const float theta = acos_f(-outward.y);
            const float phi = atan2_f(-outward.z, outward.x) + kPi;
            tu = phi / (2.0f * kPi);
            tv = theta / kPi;
        }
    } else {
        // mesh: barycentric shading normal and uv, normal by transpose(inverse)
        const uint32_t i0 = sc.normal_indices[h.tri_id], i1 = sc.normal_indices[h.tri_id + 1u],
                       i2 = sc.normal_indices[h.tri_id + 2u];
        const f3 n0 = xyz(sc.normals[i0]), n1 = xyz(sc.normals[i1]), n2 = xyz(sc.normals[i2]);
        const float w = 1.0f - h.u - h.v;
        const f3 nrm = (w * n0 + h.u * n1) + h.v * n2;
        if (textured) {
            const float2 uv0 = sc.uvs[sc.uv_indices[h.tri_id]];
            const float2 uv1 = sc.uvs[sc.uv_indices[h.tri_id + 1u]];
            const float2 uv2 = sc.uvs[sc.uv_indices[h.tri_id + 2u]];
            tu = w * uv0.x + h.u * uv1.x + h.v * uv2.x;
            tv = w * uv0.y + h.u * uv1.y + h.v * uv2.y;
        }
        outward = normalize(xform_normal(sc.transforms + 4u * h.inv_tid, nrm));
    }
    // hitrecord.wgsl:10-18
    if (dot(ray.d, outward) > 0.0f) {
        normal = -outward;
        front = false;
    } else {
        normal = outward;
        front = true;
    }
    if (m.type <= 1u) {
        // Lambertian (material.wgsl:9-20) and metal (:22-27) draw the same
        // three numbers for random_in_unit_sphere; one code path serves both
        // kinds of lanes in a wave.
        const f3 s = random_in_unit_sphere(rng);
        f3 dir;
        bool cont;
        if (m.type == 0u) {
            dir = normal + normalize_draw(s);
            if (near_zero(dir)) dir = normal;
            cont = true;
        } else {
            dir = reflect_dir(ud, normal) + m.fuzz * s;
            cont = dot(dir, normal) > 0.0f;  // absorbed below the surface
        }
        next.o = p;
        next.d = dir;
        if (cont) {
            weight = textured ? sample_texture(sc, m.texture, tu, tv) : m.albedo;
            return true;
        }
        weight = f3{0.0f, 0.0f, 0.0f};  // material_emit of a metal
        return false;
    }
    switch (m.type) {
    case 2u: {  // material.wgsl:36-59
        const float ratio = front ? (1.0f / m.ior) : m.ior;
        const float cos_theta = fminf(dot(-ud, normal), 1.0f);
        const float sin_theta = sqrt_tame(1.0f - cos_theta * cos_theta);
        const bool cannot_refract = ratio * sin_theta > 1.0f;
        bool reflect = cannot_refract;
        if (!reflect) {  // the draw happens only when refraction is possible
            float r0 = (1.0f - ratio) / (1.0f + ratio);
            r0 = r0 * r0;
            const float refl = r0 + (1.0f - r0) * pow_draw(1.0f - cos_theta, 5.0f);
            reflect = refl > rng_f32(rng);
        }
        next.o = p;
        next.d = reflect ? reflect_dir(ud, normal) : refract_dir(ud, normal, ratio);
        weight = f3{1.0f, 1.0f, 1.0f};
        return true;
    }
    default:  // diffuse light (3) emits; anything else emits black
        weight = (m.type == 3u) ? (textured ? sample_texture(sc, m.texture, tu, tv) : m.albedo)
                                : f3{0.0f, 0.0f, 0.0f};
        return false;
    }
}


// The material part of shade() (material.wgsl:9-89) at a shading point from
// surface(): the same operations, for callers that need the shading point's
// data before scattering.
template <uint32_t F>
__device__ __forceinline__ bool scatter(const DevScene &sc, const Surface &srf, const Ray &ray, uint32_t &rng,
                                        Ray &next, f3 &weight)
{
    const Material &m = srf.m;
    const f3 &p = srf.p;
    const f3 &normal = srf.normal;
    const bool front = srf.front;
    const bool textured = srf.textured;
    const float tu = srf.tu, tv = srf.tv;
    if (m.type <= 1u) {
        // Lambertian (material.wgsl:9-20) and metal (:22-27) draw the same
        // three numbers for random_in_unit_sphere; one code path serves both
        // kinds of lanes in a wave.
        const f3 s = random_in_unit_sphere(rng);
        f3 dir;
        bool cont;
        if (m.type == 0u) {
            dir = normal + normalize_draw(s);
            if (near_zero(dir)) dir = normal;
            cont = true;
        } else {
            dir = reflect_dir(normalize(ray.d), normal) + m.fuzz * s;
            cont = dot(dir, normal) > 0.0f;  // absorbed below the surface
        }
        next.o = p;
        next.d = dir;
        if (cont) {
            weight = textured ? sample_texture(sc, m.texture, tu, tv) : m.albedo;
            return true;
        }
        weight = f3{0.0f, 0.0f, 0.0f};  // material_emit of a metal
        return false;
    }
    switch (m.type) {
    case 2u: {  // material.wgsl:36-59
        const float ratio = front ? (1.0f / m.ior) : m.ior;
        const f3 ud = normalize(ray.d);
        const float cos_theta = fminf(dot(-ud, normal), 1.0f);
        const float sin_theta = sqrt_tame(1.0f - cos_theta * cos_theta);
        const bool cannot_refract = ratio * sin_theta > 1.0f;
        bool reflect = cannot_refract;
        if (!reflect) {  // the draw happens only when refraction is possible
            float r0 = (1.0f - ratio) / (1.0f + ratio);
            r0 = r0 * r0;
            const float refl = r0 + (1.0f - r0) * pow_draw(1.0f - cos_theta, 5.0f);
            reflect = refl > rng_f32(rng);
        }
        next.o = p;
        next.d = reflect ? reflect_dir(ud, normal) : refract_dir(ud, normal, ratio);
        weight = f3{1.0f, 1.0f, 1.0f};
        return true;
    }
    default:  // diffuse light (3) emits; anything else emits black
        weight = (m.type == 3u) ? (textured ? sample_texture(sc, m.texture, tu, tv) : m.albedo)
                                : f3{0.0f, 0.0f, 0.0f};
        return false;
    }
}

// Two floats to packed bf16 (first in the low half) with gfx950's
// v_cvt_pk_bf16_f32, which rounds to nearest even. For every non-NaN input
// that is the software rounding (u + 0x7fff + ((u >> 16) & 1)) >> 16 of the
// radiance cache's numerics; a NaN input may come out with another NaN
// payload. orn_eval_math op 5 evaluates it for the tests.
__device__ __forceinline__ uint32_t pack_bf16_rne(float a, float b)
{
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    const bf16x2_t v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
    return __builtin_bit_cast(uint32_t, v);
}

// Low 32 bits of the device's constant 100 MHz clock (wave-uniform).
__device__ __forceinline__ uint32_t device_ticks() { return static_cast<uint32_t>(__builtin_amdgcn_s_memrealtime()); }

// Quarter-octave class of a cost (queues ordered by cost): 4 * floor(log2(c +
// 1)) plus the two bits below the leading one of c + 1; non-decreasing in c,
// below 128.
constexpr uint32_t kCostClasses = 128;
__device__ __forceinline__ uint32_t cost_class(uint32_t c)
{
    const uint32_t v = c == 0xffffffffu ? c : c + 1u;
    const uint32_t e = 31u - static_cast<uint32_t>(__clz(v));
    const uint32_t f = e >= 2u ? (v >> (e - 2u)) & 3u : (v << (2u - e)) & 3u;
    return 4u * e + f;
}
// The least cost of a class.
__device__ __forceinline__ float cost_of_class(uint32_t c)
{
    return ldexpf(1.0f + 0.25f * static_cast<float>(c & 3u), static_cast<int>(c >> 2)) - 1.0f;
}

}  // namespace orn
