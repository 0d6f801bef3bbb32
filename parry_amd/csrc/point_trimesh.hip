// point_trimesh.hip -- batched point projections onto a TriMesh through its Bvh (gfx950).
//
// TriMesh::project_local_point (src/query/point/point_composite_shape.rs:164-168
// -> CompositeShapeRef::project_local_point, :59-80): parry's best-first
// Bvh::find_best (bvh_traverse.rs:335-417) from max cost Real::MAX, with the
// point's distance to a child's AABB as node cost (Aabb::distance_to_local_point,
// solid = true, point_aabb.rs:135-146) and the distance to the point's
// projection on the triangle as leaf cost (Triangle::project_local_point,
// point_triangle.rs:54-291).  The chosen triangle and the projection are
// bit-identical to parry3d's.
//
// Two mappings.  One lane per point with the ray kernel's node fetches (four
// 16-byte loads of the 64-byte wide record) and LDS stack, over points sorted by
// grid cell so that a wave's lanes walk similar paths.  And one wave per point for
// small calls and for the points whose walk is long: a point near the middle of a
// closed mesh has most of the surface at nearly the same distance, and on an
// 81,920-triangle sphere one of 262,147 points visits 8,100 nodes where the mean
// is 134, so that the call lasted as long as that one lane's chain of fetches
// (3.1 ms).  A lane leaves its point to a wave after some nodes, later where the point
// is outside the mesh's box; if too many points are left for waves to be the faster
// way, lanes walk them again.
#include <cfloat>

#include "contact_gjk.h"
#include "pq_internal.h"

namespace pq {
namespace {

constexpr int kPtBlock = 256;

// |max(mins - p, p - maxs, 0)| (nalgebra sup and norm).
__device__ __forceinline__ float aabb_point_dist(float mnx, float mny, float mnz, float mxx, float mxy, float mxz,
                                                 f3 p) {
    const float sx = fmaxf(fmaxf(mnx - p.x, p.x - mxx), 0.0f);
    const float sy = fmaxf(fmaxf(mny - p.y, p.y - mxy), 0.0f);
    const float sz = fmaxf(fmaxf(mnz - p.z, p.z - mxz), 0.0f);
    return sqrtf((sx * sx + sy * sy) + sz * sz);
}

struct PtBest {
    float cost;
    f3 p;
    uint32_t leaf;
    bool have;
};

// Triangle::project_local_point's point (tri_project's, bit for bit).  The regions
// are selected, not branched to: the lanes of a wave project onto triangles in
// every region, and took all of tri_project's branches with a division each.
__device__ __forceinline__ f3 tri_point(f3 a, f3 b, f3 c, f3 pt, bool solid) {
    const f3 ab = sub3(b, a), ac = sub3(c, a), bc = sub3(c, b);
    const f3 ap = sub3(pt, a), bp = sub3(pt, b), cp = sub3(pt, c);
    const float ab_ap = dot3(ab, ap), ac_ap = dot3(ac, ap);
    const float ab_bp = dot3(ab, bp), ac_bp = dot3(ac, bp);
    const float ab_cp = dot3(ab, cp), ac_cp = dot3(ac, cp);
    const f3 n = cross3(ab, ac);
    const float vc = dot3(n, cross3(ab, ap)), vb = -dot3(n, cross3(ac, cp)), va = dot3(n, cross3(bc, bp));
    const bool at_a = (ab_ap <= 0.0f) & (ac_ap <= 0.0f);
    const bool at_b = !at_a & (ab_bp >= 0.0f) & (ac_bp <= ab_bp);
    const bool at_c = !at_a & !at_b & (ac_cp >= 0.0f) & (ab_cp <= ac_cp);
    const bool vertex = at_a | at_b | at_c;
    const bool on_ab = !vertex & (vc < 0.0f) & (ab_ap >= 0.0f) & (ab_bp <= 0.0f);
    const bool on_ac = !vertex & !on_ab & (vb < 0.0f) & (ac_ap >= 0.0f) & (ac_cp <= 0.0f);
    const bool on_bc =
        !vertex & !on_ab & !on_ac & (va < 0.0f) & (ac_bp - ab_bp >= 0.0f) & (ab_cp - ac_cp >= 0.0f);
    const bool edge = on_ab | on_ac | on_bc;
    const float sum = va + vb + vc;
    const f3 base = sel2(at_b | on_bc, b, sel2(at_c, c, a));
    const f3 dir = sel2(on_ab, ab, sel2(on_ac, ac, bc));
    const float t = (on_ab ? ab_ap : (on_ac ? ac_ap : dot3(bc, bp))) / norm_sq3(dir);
    const float denom = 1.0f / sum;
    const f3 face = add3(add3(a, mul3(ab, vb * denom)), mul3(ac, vc * denom));
    f3 r = sel2(vertex, base, sel2(edge, add3(base, mul3(dir, t)), face));
    if (!(vertex | edge) && !(sum != 0.0f)) {  // a degenerate triangle
        bool inside;
        r = tri_project(a, b, c, pt, solid, inside);
    }
    return r;
}

// A leaf's projection and its cost (na::distance).
__device__ __forceinline__ f3 leaf_point(const float4 *tri4, uint32_t leaf, f3 pt, bool solid, float &cost) {
    const float4 q0 = tri4[3 * (size_t)leaf], q1 = tri4[3 * (size_t)leaf + 1], q2 = tri4[3 * (size_t)leaf + 2];
    const f3 p = tri_point(f3{q0.x, q0.y, q0.z}, f3{q0.w, q1.x, q1.y}, f3{q1.z, q1.w, q2.x}, pt, solid);
    cost = sqrtf(norm_sq3(sub3(pt, p)));
    return p;
}

// A leaf of find_best: replaces the best only if strictly closer.
__device__ __forceinline__ void visit_leaf(const float4 *tri4, uint32_t leaf, f3 pt, bool solid, PtBest &b) {
    float cost;
    const f3 p = leaf_point(tri4, leaf, pt, solid, cost);
    const bool closer = cost < b.cost;
    b.cost = closer ? cost : b.cost;
    b.p = sel2(closer, p, b.p);
    b.leaf = closer ? leaf : b.leaf;
    b.have = b.have | closer;
}

// find_best from the root, by one lane; `stk` with stride `stride`.
template <bool COUNT>
__device__ __forceinline__ void walk(const float4 *node4, const float4 *tri4, f3 pt, bool solid, uint32_t *stk,
                                     uint32_t stride, PtBest &b, uint32_t &n_wide, uint32_t &n_tri) {
    const float4 root3 = node4[3];
    if ((__float_as_uint(root3.w) & 0x3fffffffu) == 0u) {  // partial root, bvh_traverse.rs:348-359
        const float4 q0 = node4[0], q1 = node4[1];
        n_wide = 1;
        if (aabb_point_dist(q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, pt) < FLT_MAX) {
            ++n_tri;
            visit_leaf(tri4, __float_as_uint(q0.w), pt, solid, b);
        }
        return;
    }
    uint32_t curr = 0, sp = 0;
    for (;;) {
        if (COUNT) ++n_wide;
        const float4 q0 = node4[4 * curr + 0];  // left mins, left children
        const float4 q1 = node4[4 * curr + 1];  // left maxs, left data
        const float4 q2 = node4[4 * curr + 2];  // right mins, right children
        const float4 q3 = node4[4 * curr + 3];  // right maxs, right data
        float ls = aabb_point_dist(q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, pt);
        float rs = aabb_point_dist(q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, pt);
        uint32_t lc = __float_as_uint(q0.w), ld = __float_as_uint(q1.w);
        uint32_t rc = __float_as_uint(q2.w), rd = __float_as_uint(q3.w);
        if (ls > rs) {
            const float tf = ls;
            ls = rs;
            rs = tf;
            const uint32_t tc = lc;
            lc = rc;
            rc = tc;
            const uint32_t td = ld;
            ld = rd;
            rd = td;
        }
        // one latch: into a child, or back to the stack's top, by selects
        const uint32_t below = stk[(sp != 0u ? sp - 1u : 0u) * stride];
        const bool near_leaf = (ld & 0x3fffffffu) == 1u, far_leaf = (rd & 0x3fffffffu) == 1u;
        const bool near_in = ls < b.cost && ls != FLT_MAX;
        if (near_in && near_leaf) {
            if (COUNT) ++n_tri;
            visit_leaf(tri4, lc, pt, solid, b);
        }
        const bool far_in = rs < b.cost && rs != FLT_MAX;
        if (far_in && far_leaf) {
            if (COUNT) ++n_tri;
            visit_leaf(tri4, rc, pt, solid, b);
        }
        const bool go_near = near_in && !near_leaf, go_far = far_in && !far_leaf;
        if (go_near && go_far) stk[sp * stride] = rc;
        const bool pop = !go_near && !go_far;
        if (pop && sp == 0u) return;
        curr = go_near ? lc : (go_far ? rc : below);
        sp = go_near && go_far ? sp + 1u : (pop ? sp - 1u : sp);
    }
}

__device__ __forceinline__ bool in_box(f3 a, f3 b, f3 c, f3 p) {
    const f3 mn = min3(min3(a, b), c), mx = max3(max3(a, b), c);
    return (p.x >= mn.x) & (p.y >= mn.y) & (p.z >= mn.z) & (p.x <= mx.x) & (p.y <= mx.y) & (p.z <= mx.z);
}
// Whether the projection on a triangle lies in the triangle's box.  Costs are then
// monotone down the tree: box cost and leaf cost are sums of squares of the same
// form, and float subtraction, product, sum and root are monotone, so the leaf
// costs no less than its box, and no less than any box above it (where the boxes
// are nested, MeshBounds).
__device__ __forceinline__ bool point_in_box(const float4 *tri4, uint32_t leaf, f3 p) {
    const float4 q0 = tri4[3 * (size_t)leaf], q1 = tri4[3 * (size_t)leaf + 1], q2 = tri4[3 * (size_t)leaf + 2];
    return in_box(f3{q0.x, q0.y, q0.z}, f3{q0.w, q1.x, q1.y}, f3{q1.z, q1.w, q2.x}, p);
}

// find_best by one lane, with the leaves put aside: a lane reaches a leaf at one
// node in ten, so some lane of a wave did at nearly every node, and each node cost
// the wave two projections (2.2 us per node, two thirds of it for them).  Up to four
// leaves wait in registers, and the wave projects the first of every lane when one
// lane has more than two.  After `limit` nodes a lane that may leaves its point to the
// wave kernel: `leave` puts it in the list (and returns its argument).  Where `far` it
// does so only once `few` lanes of its wave or less still walk, or after four times
// `limit`.
//
// The nodes are taken in find_best's order with a best cost that is late, so this
// walk sees find_best's leaves and a few more, in its order, as long as the
// projection of every leaf it takes as the best lies in that leaf's box (a leaf
// find_best prunes does not then cost less than its best).  So does find_best take
// the first leaf W of smallest cost: each leaf before it costs more than W, so no box
// above W costs as much as the best cost find_best has there, and nothing after W
// costs less.
enum : uint32_t { WALK_DONE, WALK_UNKNOWN, WALK_LEFT };  // unknown: the answer may not be find_best's
template <class Leave>
__device__ __forceinline__ uint32_t walk_deferred(const float4 *node4, const float4 *tri4, f3 pt, bool solid,
                                                  uint32_t *stk, uint32_t stride, uint32_t limit, int few, bool may,
                                                  bool far, const Leave &leave, PtBest &b) {
    uint32_t curr = 0, sp = 0, n = 0, steps = 0, check = limit;
    uint32_t l0 = 0, l1 = 0, l2 = 0, l3 = 0;
    bool walking = true, known = true;
    auto put = [&](bool add, uint32_t leaf) {
        l0 = add && n == 0u ? leaf : l0;
        l1 = add && n == 1u ? leaf : l1;
        l2 = add && n == 2u ? leaf : l2;
        l3 = add && n == 3u ? leaf : l3;
        n += add ? 1u : 0u;
    };
    for (;;) {
        // A node adds two leaves at most: wave-uniform, so that the lanes keep step.
        const bool leaves = __any(n > 2u) || !__any(walking);
        if (!leaves && steps == check) {  // all walking lanes at once: they keep step
            check += limit / 2u;
            const bool late = __popcll(__ballot(walking)) <= few || steps >= 4u * limit;
            if (leave(walking && may && (!far || late))) return WALK_LEFT;
        }
        steps += leaves ? 0u : 1u;
        if (!leaves && walking) {
            const float4 q0 = node4[4 * (size_t)curr + 0];  // left mins, left children
            const float4 q1 = node4[4 * (size_t)curr + 1];  // left maxs, left data
            const float4 q2 = node4[4 * (size_t)curr + 2];  // right mins, right children
            const float4 q3 = node4[4 * (size_t)curr + 3];  // right maxs, right data
            const uint32_t below = stk[(sp != 0u ? sp - 1u : 0u) * stride];
            const float cl = aabb_point_dist(q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, pt);
            const float cr = aabb_point_dist(q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, pt);
            const bool swap = cl > cr;
            const float ls = swap ? cr : cl, rs = swap ? cl : cr;
            const uint32_t lc = __float_as_uint(swap ? q2.w : q0.w), rc = __float_as_uint(swap ? q0.w : q2.w);
            const uint32_t ld = __float_as_uint(swap ? q3.w : q1.w), rd = __float_as_uint(swap ? q1.w : q3.w);
            const bool near_leaf = (ld & 0x3fffffffu) == 1u, far_leaf = (rd & 0x3fffffffu) == 1u;
            const bool near_in = (ls < b.cost) & (ls != FLT_MAX), far_in = (rs < b.cost) & (rs != FLT_MAX);
            put(near_in & near_leaf, lc);
            put(far_in & far_leaf, rc);
            const bool go_near = near_in & !near_leaf, go_far = far_in & !far_leaf;
            if (go_near & go_far) stk[sp * stride] = rc;
            const bool pop = !go_near & !go_far;
            walking = !(pop & (sp == 0u));
            curr = go_near ? lc : (go_far ? rc : below);
            sp = (go_near & go_far) ? sp + 1u : (pop ? sp - 1u : sp);
        }
        if (leaves) {
            if (n != 0u) {
                const float4 q0 = tri4[3 * (size_t)l0], q1 = tri4[3 * (size_t)l0 + 1], q2 = tri4[3 * (size_t)l0 + 2];
                const f3 ta{q0.x, q0.y, q0.z}, tb{q0.w, q1.x, q1.y}, tc{q1.z, q1.w, q2.x};
                const f3 p = tri_point(ta, tb, tc, pt, solid);
                const float cost = sqrtf(norm_sq3(sub3(pt, p)));
                const bool closer = cost < b.cost;
                known = known & (!closer | in_box(ta, tb, tc, p));
                b.cost = closer ? cost : b.cost;
                b.leaf = closer ? l0 : b.leaf;
                b.have = b.have | closer;
                l0 = l1;
                l1 = l2;
                l2 = l3;
                --n;
            }
            if (!walking && n == 0u) break;
        }
    }
    return known ? WALK_DONE : WALK_UNKNOWN;
}

// is_inside comes from the winner's triangle, projected again.
__device__ __forceinline__ void write_projection(pq_point_projection *out, uint64_t i, const float4 *tri4, f3 pt,
                                                 bool solid, const PtBest &b) {
    pq_point_projection o;
    if (b.have) {
        const float4 q0 = tri4[3 * (size_t)b.leaf], q1 = tri4[3 * (size_t)b.leaf + 1], q2 = tri4[3 * (size_t)b.leaf + 2];
        bool inside = false;
        const f3 p = tri_project(f3{q0.x, q0.y, q0.z}, f3{q0.w, q1.x, q1.y}, f3{q1.z, q1.w, q2.x}, pt, solid, inside);
        o.point[0] = p.x;
        o.point[1] = p.y;
        o.point[2] = p.z;
        o.is_inside = inside ? 1u : 0u;
        o.triangle = __float_as_uint(q2.y);
    } else {
        o.point[0] = o.point[1] = o.point[2] = 0.0f;
        o.is_inside = 0u;
        o.triangle = PQ_NO_HIT;
    }
    out[i] = o;
}
__device__ __forceinline__ f3 load_point(const float *points, uint64_t i) {
    return f3{points[3 * i], points[3 * i + 1], points[3 * i + 2]};
}

// No leaf has a cost for a point with a NaN (find_best visits the whole tree to no end).
__device__ __forceinline__ bool any_nan(f3 p) { return p.x != p.x || p.y != p.y || p.z != p.z; }
__device__ __forceinline__ float bound_dist(const MeshBounds &bounds, f3 p) {  // MeshBounds' |p|_1 + 3 * extent
    return fabsf(p.x) + fabsf(p.y) + fabsf(p.z) + 3.0f * bounds.extent;
}
__device__ __forceinline__ bool in_root_box(const float4 *node4, f3 p) {
    const float4 a = node4[0], b = node4[1], c = node4[2], d = node4[3];
    const auto in = [](float l0, float l1, float h0, float h1, float v) {
        return v >= fminf(l0, l1) && v <= fmaxf(h0, h1);
    };
    return in(a.x, c.x, b.x, d.x, p.x) && in(a.y, c.y, b.y, d.y, p.y) && in(a.z, c.z, b.z, d.z, p.z);
}

// The points that lanes leave to waves: a long walk ends sooner there, but takes 16 to
// 240 ns of the whole GPU.  Beyond kHeavyMax of them lanes walk them again, without a
// limit.  Measured with all points in a ball of radius 0.02 / 0.1 / 0.3 at the middle of
// the 81,920-triangle unit sphere, ms a call: 130,000 points by waves 32 / 11.5 / 6.4, by
// lanes 34 / 16.2 / 10.9; 260,000 by waves 63 / 22.4 / 12.3, by lanes 34.6 / 16.3 / 11.4; 10^6
// 244 / 86 / 47 and 94 / 39 / 22.
constexpr uint32_t kHeavyMax = 131072;
// Farther out than this share of the bound's reach the slack keeps a wave from pruning:
// 260,000 points at 120 radii of that sphere 1,830 us, 720 if they stay with their lanes.
constexpr float kWaveReach = 0.25f;
struct HeavyList {
    uint32_t *at;
    uint32_t *count;
};

// COUNT = true also writes, per point, the wide-node records fetched and the
// triangles tested (the traffic model of the roofline figure).  With LIMIT, long walks
// go to `heavy` (walk_deferred), and so do points whose answer is not known to be
// find_best's; without it, a list is walked plainly if it is too long for waves.
template <bool COUNT, bool LIMIT>
__global__ __launch_bounds__(kPtBlock) void project_points_kernel(const pq_bvh_node_wide *__restrict__ nodes,
                                                                  const TriRecord *__restrict__ tris,
                                                                  const float *__restrict__ points, uint64_t n,
                                                                  int solid_flag,
                                                                  pq_point_projection *__restrict__ out,
                                                                  uint32_t *__restrict__ counts,
                                                                  const uint32_t *order, uint32_t limit,
                                                                  int few, MeshBounds bounds, HeavyList heavy) {
    extern __shared__ uint32_t lds_stack[];
    const uint64_t j = (uint64_t)blockIdx.x * kPtBlock + threadIdx.x;
    if (!LIMIT && heavy.at) {
        n = *heavy.count;
        if (n <= kHeavyMax) return;  // the wave kernel's
        order = heavy.at;
    }
    if (j >= n) return;
    const uint64_t i = order ? (uint64_t)order[j] : j;
    const float4 *node4 = reinterpret_cast<const float4 *>(nodes);
    const float4 *tri4 = reinterpret_cast<const float4 *>(tris);
    PtBest b{FLT_MAX, f3{0.0f, 0.0f, 0.0f}, 0u, false};
    uint32_t n_wide = 0, n_tri = 0;
    const f3 pt = load_point(points, i);
    const bool solid = solid_flag != 0;
    uint32_t *const stk = lds_stack + threadIdx.x;
    if constexpr (LIMIT) {
        if (!any_nan(pt)) {
            const auto leave = [&](bool left) {  // one atomic per wave, by the first lane that leaves
                const uint64_t mask = __ballot(left);
                if (mask == 0ull) return false;
                const uint32_t leader = (uint32_t)__builtin_ctzll(mask);
                uint32_t base = 0;
                if (__lane_id() == leader) base = atomicAdd(heavy.count, (uint32_t)__popcll(mask));
                base = (uint32_t)__builtin_amdgcn_readlane((int)base, (int)leader);
                if (left)
                    heavy.at[base + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] =
                        (uint32_t)i;
                return left;
            };
            const bool may = bound_dist(bounds, pt) <= kWaveReach * bounds.reach;
            const uint32_t r = walk_deferred(node4, tri4, pt, solid, stk, kPtBlock, limit, few, may,
                                             !in_root_box(node4, pt), leave, b);
            if (r == WALK_LEFT || leave(r == WALK_UNKNOWN)) return;
        }
    } else {
        walk<COUNT>(node4, tri4, pt, solid, stk, kPtBlock, b, n_wide, n_tri);
    }
    if (COUNT) {
        counts[2 * i] = n_wide;
        counts[2 * i + 1] = n_tri;
    }
    write_projection(out, i, tri4, pt, solid, b);
}

// ---------------------------------------------------------------------------
// One wave per point.  The wave takes up to 64 pending nodes at a time, one per
// lane, and keeps every child whose box is within the best cost so far plus
// `slack`.  Let W be, of the leaves of smallest cost, the one find_best reaches
// first.  If W's projection lies in W's box, find_best's answer is W (as for
// walk_deferred).  The wave finds W if it sees every leaf that can cost so little:
// those it does not see lie in a box costing more than best + slack, and cost less
// than that box by at most their projection's distance outside it, which `slack`
// bounds (MeshBounds).
// find_best reaches leaves in the order of a path key: at each node a child leaf
// before a child node, otherwise the nearer child (the left on ties) first.  The
// key holds one bit per level from the top, then a marker bit.  A winner whose
// projection is outside its box or a full stack falls back to find_best by lane 0,
// and so does a point out of the bound's reach unless `shared` is set: then the first
// blocks take `shared` points each and walk those out of reach, a lane for each.
// ---------------------------------------------------------------------------
constexpr uint32_t kDescentNodes = 8;
constexpr uint32_t kWaveStack = 1024;
constexpr uint32_t kWaveMaxDepth = 62;  // path key: levels and a marker in 64 bits

template <int CTRL> __device__ __forceinline__ float min_dpp(float v) {
    return fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float wave_min(float v) {  // no NaN
    v = min_dpp<0x140>(min_dpp<0x141>(min_dpp<0x4E>(min_dpp<0xB1>(v))));  // the rows of 16
    const float r[4] = {__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0)),
                        __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16)),
                        __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32)),
                        __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48))};
    return fminf(fminf(r[0], r[1]), fminf(r[2], r[3]));
}
__device__ __forceinline__ uint64_t wave_min(uint64_t v) {
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t o = (uint64_t)__shfl_xor((long long)v, d);
        v = o < v ? o : v;
    }
    return v;
}
__device__ __forceinline__ uint32_t rank_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__global__ __launch_bounds__(64) void project_points_wave_kernel(const pq_bvh_node_wide *__restrict__ nodes,
                                                                 const TriRecord *__restrict__ tris,
                                                                 const float *__restrict__ points, uint32_t n,
                                                                 HeavyList list, uint32_t shared, int solid_flag,
                                                                 MeshBounds bounds,
                                                                 pq_point_projection *__restrict__ out) {
    __shared__ alignas(8) uint32_t lds[4 * kWaveStack];
    uint32_t *const s_node = lds;
    float *const s_cost = reinterpret_cast<float *>(lds + kWaveStack);
    uint64_t *const s_key = reinterpret_cast<uint64_t *>(lds + 2 * kWaveStack);
    const float4 *node4 = reinterpret_cast<const float4 *>(nodes);
    const float4 *tri4 = reinterpret_cast<const float4 *>(tris);
    const bool solid = solid_flag != 0;
    const uint32_t lane = __lane_id();
    const auto plain = [&](uint32_t i, f3 pt, uint32_t lanes) {  // by one of `lanes` lanes
        PtBest s{FLT_MAX, f3{0.0f, 0.0f, 0.0f}, 0u, false};
        uint32_t n_wide = 0, n_tri = 0;
        walk<false>(node4, tri4, pt, solid, lds + (lanes > 1u ? lane : 0u), lanes, s, n_wide, n_tri);
        write_projection(out, i, tri4, pt, solid, s);
    };
    uint32_t first = blockIdx.x;
    if (list.at) {
        n = *list.count;
        if (n > kHeavyMax) return;  // project_points_kernel's
    } else if (shared != 0u) {
        const uint32_t blocks = (n + shared - 1u) / shared;
        if (first < blocks) {
            const uint32_t i = first * shared + lane;
            if (lane < shared && i < n) {
                const f3 pt = load_point(points, i);
                if (!any_nan(pt) && !(bound_dist(bounds, pt) <= bounds.reach)) plain(i, pt, shared);
            }
            return;
        }
        first -= blocks;
    }
    for (uint32_t q = first; q < n; q += gridDim.x) {
        const uint32_t i = list.at ? list.at[q] : q;
        const f3 pt = load_point(points, i);
        const float d = bound_dist(bounds, pt);
        const float slack = bounds.foot * d;
        if (any_nan(pt)) {
            if (lane == 0) write_projection(out, i, tri4, pt, solid, PtBest{FLT_MAX, f3{0.0f, 0.0f, 0.0f}, 0u, false});
            continue;
        }
        if (shared != 0u && !(d <= bounds.reach)) continue;
        PtBest b{FLT_MAX, f3{0.0f, 0.0f, 0.0f}, 0u, false};  // the lane's best
        uint64_t key = ~0ull;
        uint32_t sp = 1;
        float bound = FLT_MAX;
        bool fits = d <= bounds.reach;
        if (lane == 0) {
            s_node[0] = 0u;
            s_cost[0] = 0.0f;
            s_key[0] = 1ull << 63;
        }
        __syncthreads();  // one wave: orders the LDS accesses below
        while (fits && sp != 0u) {
            // each node taken leaves at most two
            const uint32_t room = kWaveStack - sp;
            // few nodes at a time until a leaf gives a bound to prune by
            const uint32_t wide = bound < FLT_MAX ? 64u : kDescentNodes;
            uint32_t take = sp < wide ? sp : wide;
            take = take < room ? take : room;
            if (take == 0u) {
                fits = false;
                break;
            }
            sp -= take;
            bool active = lane < take;
            const uint32_t at = sp + (active ? lane : 0u);
            const uint32_t node = s_node[at];
            const uint64_t path = s_key[at];
            active = active && s_cost[at] <= bound;
            __syncthreads();
            bool push_near = false, push_far = false;
            float ls = FLT_MAX, rs = FLT_MAX;
            uint32_t lc = 0, rc = 0;
            uint64_t lk = 0, rk = 0;
            if (active) {
                const float4 q0 = node4[4 * (size_t)node + 0], q1 = node4[4 * (size_t)node + 1];
                const float4 q2 = node4[4 * (size_t)node + 2], q3 = node4[4 * (size_t)node + 3];
                ls = aabb_point_dist(q0.x, q0.y, q0.z, q1.x, q1.y, q1.z, pt);
                rs = aabb_point_dist(q2.x, q2.y, q2.z, q3.x, q3.y, q3.z, pt);
                lc = __float_as_uint(q0.w);
                rc = __float_as_uint(q2.w);
                uint32_t ld = __float_as_uint(q1.w) & 0x3fffffffu, rd = __float_as_uint(q3.w) & 0x3fffffffu;
                const bool swap = ls > rs;
                if (swap) {
                    const float tf = ls;
                    ls = rs;
                    rs = tf;
                    const uint32_t tc = lc;
                    lc = rc;
                    rc = tc;
                    const uint32_t td = ld;
                    ld = rd;
                    rd = td;
                }
                const bool near_leaf = ld == 1u, far_leaf = rd == 1u;
                const bool far_first = far_leaf && !near_leaf;
                const uint64_t mark = path & (0ull - path), first = (path ^ mark) | (mark >> 1), second = first | mark;
                lk = far_first ? second : first;
                rk = far_first ? first : second;
                const bool near_in = ls <= bound && ls < FLT_MAX, far_in = rs <= bound && rs < FLT_MAX;
                push_near = near_in && !near_leaf;
                push_far = far_in && !far_leaf;
#pragma unroll
                for (int side = 0; side < 2; ++side) {
                    if (side == 0 ? !(near_in && near_leaf) : !(far_in && far_leaf)) continue;
                    const uint32_t leaf = side == 0 ? lc : rc;
                    const uint64_t lkey = side == 0 ? lk : rk;
                    float cost;
                    const f3 p = leaf_point(tri4, leaf, pt, solid, cost);
                    if (cost < b.cost || (cost == b.cost && b.have && lkey < key)) {
                        b = PtBest{cost, p, leaf, true};
                        key = lkey;
                    }
                }
            }
            // far children below near ones, so that near ones are taken first
            const uint64_t fm = __ballot(push_far), nm = __ballot(push_near);
            if (push_far) {
                const uint32_t o = sp + rank_below(fm);
                s_node[o] = rc;
                s_cost[o] = rs;
                s_key[o] = rk;
            }
            sp += (uint32_t)__popcll(fm);
            if (push_near) {
                const uint32_t o = sp + rank_below(nm);
                s_node[o] = lc;
                s_cost[o] = ls;
                s_key[o] = lk;
            }
            sp += (uint32_t)__popcll(nm);
            if (__any(b.cost + slack < bound)) bound = wave_min(b.cost) + slack;
            __syncthreads();
        }
        if (fits) {
            const float cost = wave_min(b.cost);
            const uint64_t none = ~(uint64_t)0;
            const uint64_t win = wave_min(b.have && b.cost == cost ? key : none);
            bool ok = true;
            if (b.have && key == win) {  // the winner's lane (none if no leaf has a cost)
                ok = point_in_box(tri4, b.leaf, b.p);
                if (ok) write_projection(out, i, tri4, pt, solid, b);
            } else if (win == none && lane == 0) {
                write_projection(out, i, tri4, pt, solid, b);  // none
            }
            fits = __ballot(!ok) == 0ull;
        }
        if (!fits && lane == 0) plain(i, pt, 1u);
        __syncthreads();
    }
}

// Up to this many points a call is waves only: they fill the GPU, and lanes would
// wait for the longest walk and for the sort.  Measured on the 81,920-triangle
// sphere, us a call (lanes with their waves / waves only): 1,000 points 376 / 76,
// 8,000 488 / 205, 16,000 433 / 288, 32,000 479 / 540, 65,536 580 / 1,100.
constexpr uint64_t kWavePoints = 16384;
// Nodes a lane walks before it leaves its point to a wave.  A wave spends about
// 16 ns of the whole GPU on a point; a lane's chain costs 1.2 to 1.7 us per node, which
// the larger calls hide better.  Measured (limit 192 / 256 / 384): 32,000 points
// 480 / 553 / 736 us, 65,536 534 / 587 / 763, 262,147 815 / 801 / 936, 2^20
// 2,553 / 2,203 / 1,927.
uint32_t lane_nodes(uint64_t n) { return n < 49152 ? 192u : (n < 524288 ? 256u : 384u); }
// Points outside the mesh's box often have walks of even lengths, which no wave needs to
// cut short (463 nodes at most on that sphere, from any distance): they leave when this
// many lanes of their wave or less still walk.  Measured, us a call, with no such points
// kept back / with 8 / 24 / 40 / only after four times the limit: 260,000 points at 3
// radii 1,158 / 596 / 909 / 1,141 / 507, at 20 6,250 / 931 / 997 / 1,731 / 702, up to ten widths
// above rough ground 576 / 562 / 559 / 559 / 745; 20,000 at 3 radii 579 / 425 / 417 / 454 / 387,
// up to ten widths high 356 / 400 / 357 / 351 / 531, up to one 390 / 692 / 497 / 478 / 696.
int few_lanes(uint64_t n) { return n <= 131072 ? 24 : 8; }
constexpr uint32_t kWaveGrid = 256 * 10;  // resident waves (LDS: ten per CU)
// Points out of reach that share a wave in a small call (0: a wave each; so many fit the
// GPU at once).  16,000 points at 200 radii: 1,376 us with a wave each, 657 with eight to
// a wave; 1,209 before there were waves.
uint32_t shared_lanes(uint32_t n) {
    if (n <= kWaveGrid) return 0u;
    return n <= 2 * kWaveGrid ? 2u : (n <= 4 * kWaveGrid ? 4u : 8u);
}
static_assert(8 * kWaveMaxDepth <= 4 * kWaveStack, "the shared walks' stacks");

}  // namespace

hipError_t launch_project_points(const DeviceMesh &m, const float *points, uint64_t n, int solid,
                                 pq_point_projection *out, uint32_t *counts, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    // The traversal stack never holds more than depth - 1 entries (as for rays).
    const size_t lds = (size_t)ray_stack_entries(m.depth) * kPtBlock * sizeof(uint32_t);
    const auto grid = [](uint64_t k) { return dim3((uint32_t)((k + kPtBlock - 1) / kPtBlock)); };
    const uint32_t *const none = nullptr;
    const HeavyList no_list{nullptr, nullptr};
    if (counts) {
        hipLaunchKernelGGL((project_points_kernel<true, false>), grid(n), dim3(kPtBlock), lds, stream, m.nodes, m.tris,
                           points, n, solid, out, counts, none, 0u, 0, m.bounds, no_list);
        return hipGetLastError();
    }
    // Waves need the mesh's bound on projections, a tree their keys can hold and two leaves.
    const bool waves = m.bounds.reach >= 0.0f && m.depth <= kWaveMaxDepth && m.num_triangles > 1;
    if (waves && n <= kWavePoints) {
        const uint32_t shared = shared_lanes((uint32_t)n);
        const uint32_t blocks = (uint32_t)n + (shared ? ((uint32_t)n + shared - 1u) / shared : 0u);
        hipLaunchKernelGGL(project_points_wave_kernel, dim3(blocks), dim3(64), 0, stream, m.nodes, m.tris, points,
                           (uint32_t)n, no_list, shared, solid, m.bounds, out);
        return hipGetLastError();
    }
    // The sort's buffers may have to grow, which a capture does not allow, and a
    // per-thread stream is another stream in each thread.
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(stream, &capture);
    if (e != hipSuccess) return e;
    const bool sorted = waves && capture == hipStreamCaptureStatusNone && stream != hipStreamPerThread;
    for (uint64_t at = 0; at < n; at += kPointSortMax) {
        const uint64_t part = sorted && n - at > kPointSortMax ? kPointSortMax : n - at;
        const float *const pts = points + 3 * at;
        PointBinSpace ws{};
        if (sorted && point_bin_workspace(stream, part, point_bin_blocks(part), &ws) == hipSuccess) {
            if ((e = launch_point_bins(m, pts, part, stream, ws)) != hipSuccess) return e;
            const HeavyList heavy{ws.keyrank, ws.count};  // keyrank: the sort's last kernel has read it
            hipLaunchKernelGGL((project_points_kernel<false, true>), grid(part), dim3(kPtBlock), lds, stream, m.nodes,
                               m.tris, pts, part, solid, out + at, nullptr, ws.order, lane_nodes(part),
                               few_lanes(part), m.bounds, heavy);
            hipLaunchKernelGGL(project_points_wave_kernel, dim3(kWaveGrid), dim3(64), 0, stream, m.nodes, m.tris, pts,
                               0u, heavy, 0u, solid, m.bounds, out + at);
            if (part > kHeavyMax)
                hipLaunchKernelGGL((project_points_kernel<false, false>), grid(part), dim3(kPtBlock), lds, stream,
                                   m.nodes, m.tris, pts, 0ull, solid, out + at, nullptr, none, 0u, 0, m.bounds, heavy);
        } else {
            if (sorted) (void)hipGetLastError();  // no room for the buffers: the plain walk needs none
            hipLaunchKernelGGL((project_points_kernel<false, false>), grid(part), dim3(kPtBlock), lds, stream, m.nodes,
                               m.tris, pts, part, solid, out + at, nullptr, none, 0u, 0, m.bounds, no_list);
        }
        if ((e = hipGetLastError()) != hipSuccess) return e;
        if (!sorted) break;
    }
    return hipSuccess;
}

}  // namespace pq
