// contact.hip -- batched query::contact on shape pairs (gfx950).
//
// Stage 1 (one lane per pair): pos12 = pos1.inv_mul(pos2), the dispatch of
// DefaultQueryDispatcher::contact (src/query/default_query_dispatcher.rs:302-356)
// for the shapes held here, then
//   * Ball-Ball: the closed form of contact_ball_ball.rs:9-42;
//   * Ball with a Cuboid, Capsule or Cone: the closed-form projection of the
//     ball centre (point_aabb.rs, point_capsule.rs, point_cone.rs) and
//     contact_ball_convex_polyhedron.rs:12-63; with a ConvexPolyhedron, GJK
//     of the shape against ConstantOrigin (point_support_map.rs:17-51), the
//     centre inside going to the EPA queue like an intersecting pair;
//   * support-map pairs: contact_support_map_support_map_with_params
//     (src/query/contact/contact_support_map_support_map.rs:40-77) -- seed
//     direction (caller-supplied or parry's normalize(pos12.t) / +x), then GJK
//     in registers.  Pairs GJK finds intersecting are appended, with their
//     final simplex, to an EPA queue (one atomic per wave: ballot + masked
//     popcount give each lane its slot).
// Stage 2 (a group of lanes per queued pair): EPA (src/query/epa/epa3.rs:428-651)
//   with the polytope in LDS, in three tiers: eight lanes per pair and 60 faces,
//   sixteen lanes and 132 faces, a wave and 760 faces (more lanes in small calls).  A pair that outgrows a
//   tier's buffers goes on in the next one where it stopped.  The group's lanes
//   share the support scans, pick the next face, test every face's visibility
//   and build the new faces in parallel; the silhouette walk is serial.
// Stage 3 (one wave per pair): the same with parry's heap of faces (the binary
//   heap algorithm of Rust's BinaryHeap), 2048 faces in LDS, then 8192 in global
//   memory, for the few pairs beyond 760 faces or with non-finite face distances.
// Every contact is finished as contact_support_map_support_map (dist, point2,
// normal2 in shape 2's frame) and Contact::transform_by_mut (contact.rs:171-176).
#include <cstring>
#include <type_traits>

#include "contact_gjk.h"

namespace pq {
namespace {

constexpr int kBlock = 256;
constexpr uint32_t kUnsupportedPair = 0xffffffffu;

struct DevContact {
    float p1[3], p2[3], n1[3], n2[3], dist;
    uint32_t has;
};
static_assert(sizeof(DevContact) == sizeof(pq_contact), "pq_contact layout");

// Queued EPA work item: pair index, what the EPA solves and GJK's final simplex.
enum : uint32_t {
    kPairSupportMaps = 0,  // contact_support_map_support_map on (shape 1, shape 2)
    kBallSecond = 1,       // (ConvexPolyhedron, Ball): project the ball centre
    kBallFirst = 2,        // (Ball, ConvexPolyhedron): the same, flipped
    kPairSupportMapsLocal = 3,  // contact_support_map_support_map on any pair, Ball included,
                                // results left in the shapes' local frames (the shape cast's
                                // impact geometry, shape_cast_support_map_support_map.rs:42-46)
    kPairFeatureMaps = 4,       // the same on the pair's polygonal feature maps (a Capsule is its
                                // segment), for contact manifolds (contact_manifolds_pfm_pfm.rs:66-74)
};
__device__ __forceinline__ bool is_ball_mode(uint32_t mode) { return mode == kBallFirst || mode == kBallSecond; }
__device__ __forceinline__ bool is_local_mode(uint32_t mode) {
    return mode == kPairSupportMapsLocal || mode == kPairFeatureMaps;
}
// A shape's polygonal feature map and border radius (shape.rs as_polygonal_feature_map):
// Cuboid, Cone and Triangle are their own, a Capsule is its segment with the radius as
// border, a ConvexPolyhedron is its own when it has faces (its face count, as uint32
// bits in param[1], is not zero).  False for shapes without one here (Ball).
__device__ __forceinline__ bool feature_map(ShapeRef &g, float &border) {
    border = 0.0f;
    if (g.type == PQ_SHAPE_CUBOID || g.type == PQ_SHAPE_CONE || g.type == PQ_SHAPE_TRIANGLE) return true;
    if (g.type == PQ_SHAPE_CONVEX_POLYHEDRON) return __float_as_uint(g.p1) != 0u;
    if (g.type == PQ_SHAPE_CAPSULE) {
        g.type = kShapeSegment;
        border = g.p1;
        return true;
    }
    return false;
}
struct alignas(16) EpaItem {
    uint32_t pair;
    uint32_t dim_mode;  // simplex dimension | mode << 8
    uint32_t i, j;      // the pair's shapes
    float v[4][9];      // point, orig1, orig2
};
__device__ __forceinline__ uint32_t item_mode(const EpaItem *it) { return it->dim_mode >> 8; }

// Writes a contact record straight to its output slot (a local record copied
// out afterwards would be kept in scratch memory).
__device__ __forceinline__ void store_contact(DevContact *c, f3 w1, f3 w2, f3 m1, f3 m2, float dist) {
    c->p1[0] = w1.x; c->p1[1] = w1.y; c->p1[2] = w1.z;
    c->p2[0] = w2.x; c->p2[1] = w2.y; c->p2[2] = w2.z;
    c->n1[0] = m1.x; c->n1[1] = m1.y; c->n1[2] = m1.z;
    c->n2[0] = m2.x; c->n2[1] = m2.y; c->n2[2] = m2.z;
    c->dist = dist;
    c->has = 1;
}

__device__ __forceinline__ DevContact no_contact(uint32_t has) {
    DevContact c;
    for (int k = 0; k < 3; ++k) c.p1[k] = c.p2[k] = c.n1[k] = c.n2[k] = 0.0f;
    c.dist = 0.0f;
    c.has = has;
    return c;
}

__device__ __forceinline__ void finish_contact(const iso &pos1, const iso &pos2, const iso &pos12, f3 p1, f3 p2_1,
                                               f3 n1, bool local, DevContact *o) {
    // contact_support_map_support_map (contact_support_map_support_map.rs:18-26)
    const float dist = dot3(sub3(p2_1, p1), n1);
    const f3 p2 = qrot_inv(pos12.q, sub3(p2_1, pos12.t));
    const f3 n2 = qrot_inv(pos12.q, neg3(n1));
    if (local) {
        store_contact(o, p1, p2, n1, n2, dist);
        return;
    }
    // Contact::transform_by_mut
    store_contact(o, iso_point(pos1, p1), iso_point(pos2, p2), qrot(pos1.q, n1), qrot(pos2.q, n2), dist);
}

// Builds the Ball-vs-convex contact (contact_ball_convex_polyhedron.rs:27-63)
// and maps it to world space; pb = pose of the ball in the convex shape's frame.
__device__ __forceinline__ void finish_ball_contact(const iso &pos1, const iso &pos2, const iso &pb, float radius,
                                                    float prediction, const PointProj &proj, bool has_fn, f3 fnrm,
                                                    uint32_t mode, DevContact *o) {
    f3 p1, p2, n1, n2;
    float dist;
    if (!convex_ball_contact(pb, radius, prediction, proj, has_fn, fnrm, p1, p2, n1, n2, dist)) {
        *o = no_contact(0);
        return;
    }
    const bool flip = mode == kBallFirst;  // Contact::flipped (contact.rs:156-166)
    const f3 q1 = sel2(flip, p2, p1), q2 = sel2(flip, p1, p2), m1 = sel2(flip, n2, n1), m2 = sel2(flip, n1, n2);
    store_contact(o, iso_point(pos1, q1), iso_point(pos2, q2), qrot(pos1.q, m1), qrot(pos2.q, m2), dist);
}

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// counters[0..4]: EPA queue length and the four overflow-list lengths;
// counters[5..9]: the next list entry each EPA tier hands out;
// counters[10..11]: continuation records taken by the first and second tier.
constexpr uint32_t kNumCounters = 12;
constexpr uint32_t kTiers = 5;

// ---------------------------------------------------------------------------
// The order the pairs are taken in
// ---------------------------------------------------------------------------
// A wave of mixed pairs runs the union of its pairs' support functions, vertex
// scans and iteration counts.  Where it pays (takes_order), a counting sort by
// the pair's two shape classes (below) puts like pairs side by side for GJK, and
// so for the EPA queue GJK appends to; the shapes whose EPA runs longest (curved
// ones) come first, so the tiers do not end on them.  Results go to the pair's own
// slot, and no result depends on the order.
constexpr uint32_t kShapeClasses = 16;
constexpr uint32_t kPairClasses = 2 * kShapeClasses * kShapeClasses;
constexpr uint32_t kOrderBlock = 256, kOrderRange = 2048;  // lanes and pairs per workgroup
__device__ __forceinline__ uint32_t shape_class(const ShapeRecord *rec, uint32_t i) {
    const uint4 r = *reinterpret_cast<const uint4 *>(rec + i);  // type, first vertex, vertices
    if (r.x == PQ_SHAPE_CAPSULE) return 0;
    if (r.x == PQ_SHAPE_CONE) return 1;
    if (r.x == PQ_SHAPE_CONVEX_POLYHEDRON) return 9u - (r.z >= 64u ? 7u : r.z / 8u);  // 2 to 9 by vertex count
    if (r.x == PQ_SHAPE_CUBOID) return 10;
    if (r.x == PQ_SHAPE_TRIANGLE) return 11;
    return 12;
}
// The two classes, the earlier one first, and which of the shapes has it.
__device__ __forceinline__ uint32_t pair_class(const ShapeRecord *rec, uint32_t i, uint32_t j) {
    const uint32_t a = shape_class(rec, i), b = shape_class(rec, j);
    const uint32_t lo = a < b ? a : b, hi = a < b ? b : a;
    return (lo * kShapeClasses + hi) * 2u + (a > b ? 1u : 0u);
}
__device__ __forceinline__ uint64_t pair_count(uint64_t m, const unsigned long long *m_dev) {
    if (m_dev && *m_dev < m) m = *m_dev;
    return m;
}
// Pairs per class, and every pair's class.
__global__ __launch_bounds__(kOrderBlock) void order_count_kernel(const ShapeRecord *__restrict__ rec,
                                                                  const uint32_t *__restrict__ pairs, uint64_t m,
                                                                  const unsigned long long *__restrict__ m_dev,
                                                                  uint16_t *__restrict__ cls,
                                                                  uint32_t *__restrict__ totals) {
    __shared__ uint32_t hist[kPairClasses];
    for (uint32_t c = threadIdx.x; c < kPairClasses; c += kOrderBlock) hist[c] = 0u;
    __syncthreads();
    m = pair_count(m, m_dev);
    const uint64_t first = (uint64_t)blockIdx.x * kOrderRange;
#pragma unroll 4
    for (uint32_t q = threadIdx.x; q < kOrderRange; q += kOrderBlock) {
        const uint64_t k = first + q;
        if (k < m) {
            const uint32_t c = pair_class(rec, pairs[2 * k], pairs[2 * k + 1]);
            cls[k] = (uint16_t)c;
            atomicAdd(&hist[c], 1u);
        }
    }
    __syncthreads();
    for (uint32_t c = threadIdx.x; c < kPairClasses; c += kOrderBlock)
        if (hist[c]) atomicAdd(&totals[c], hist[c]);
}
// order[]: the pairs class by class.  A workgroup reserves its part of each class
// with one atomic; taken[] starts at zero.
__global__ __launch_bounds__(kOrderBlock) void order_scatter_kernel(uint64_t m,
                                                                    const unsigned long long *__restrict__ m_dev,
                                                                    const uint16_t *__restrict__ cls,
                                                                    const uint32_t *__restrict__ totals,
                                                                    uint32_t *__restrict__ taken,
                                                                    uint32_t *__restrict__ order) {
    static_assert(kPairClasses == 2 * kOrderBlock, "two classes per lane");
    __shared__ uint32_t hist[kPairClasses], base[kPairClasses], scan[kOrderBlock];
    const uint32_t l = threadIdx.x;
    hist[2 * l] = hist[2 * l + 1] = 0u;
    const uint32_t t0 = totals[2 * l], t1 = totals[2 * l + 1];
    scan[l] = t0 + t1;
    __syncthreads();
    for (uint32_t d = 1; d < kOrderBlock; d *= 2) {
        const uint32_t v = l >= d ? scan[l - d] : 0u;
        __syncthreads();
        scan[l] += v;
        __syncthreads();
    }
    m = pair_count(m, m_dev);
    const uint64_t first = (uint64_t)blockIdx.x * kOrderRange;
    uint32_t key[kOrderRange / kOrderBlock], rank[kOrderRange / kOrderBlock];
#pragma unroll
    for (uint32_t u = 0; u < kOrderRange / kOrderBlock; ++u) {
        const uint64_t k = first + u * kOrderBlock + l;
        key[u] = k < m ? cls[k] : 0u;
        rank[u] = k < m ? atomicAdd(&hist[key[u]], 1u) : 0u;
    }
    __syncthreads();
    const uint32_t before = scan[l] - t0 - t1, h0 = hist[2 * l], h1 = hist[2 * l + 1];
    base[2 * l] = before + (h0 ? atomicAdd(&taken[2 * l], h0) : 0u);
    base[2 * l + 1] = before + t0 + (h1 ? atomicAdd(&taken[2 * l + 1], h1) : 0u);
    __syncthreads();
#pragma unroll
    for (uint32_t u = 0; u < kOrderRange / kOrderBlock; ++u) {
        const uint64_t k = first + u * kOrderBlock + l;
        if (k < m) order[base[key[u]] + rank[u]] = (uint32_t)k;
    }
}

__global__ void reset_counters_kernel(uint32_t *counters, uint32_t n) {
    for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) counters[k] = 0u;
}

// ---------------------------------------------------------------------------
// Stage 1
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void contact_gjk_kernel(
    const ShapeRecord *__restrict__ rec, const float4 *__restrict__ verts, const float *__restrict__ poses,
    const uint32_t *__restrict__ pairs, uint64_t m, const unsigned long long *__restrict__ m_dev, float prediction,
    const float *__restrict__ seeds, DevContact *__restrict__ out, uint32_t *__restrict__ iters,
    EpaItem *__restrict__ queue, uint32_t *__restrict__ counters, uint32_t flags,
    const uint32_t *__restrict__ order) {
    uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (m_dev) {
        const uint64_t md = *m_dev;
        if (md < m) m = md;
    }
    if (order && k < m) k = order[k];
    bool need_epa = false;
    uint32_t ball_mode = kPairSupportMaps;
    Simplex s;
    uint32_t pair_id = 0, shape_i = 0, shape_j = 0;
    if (k < m) {
        pair_id = (uint32_t)k;
        const uint32_t i = pairs[2 * k], j = pairs[2 * k + 1];
        shape_i = i;
        shape_j = j;
        const iso pos1 = load_iso(poses + 7 * (size_t)i), pos2 = load_iso(poses + 7 * (size_t)j);
        const iso pos12 = iso_inv_mul(pos1, pos2);
        ShapeRef g1 = load_shape(rec, verts, i), g2 = load_shape(rec, verts, j);
        DevContact *const c = out + k;
        uint32_t gi = 0;
        const bool pfm = (flags & kContactFeatureMaps) != 0u;
        bool unsupported = false;
        float total_prediction = prediction;
        if (pfm) {  // total_prediction = prediction + border1 + border2 (contact_manifolds_pfm_pfm.rs:65)
            float br1 = 0.0f, br2 = 0.0f;
            unsupported = !feature_map(g1, br1) || !feature_map(g2, br2);
            total_prediction = prediction + br1 + br2;
        }
        // What GJK runs on, if anything: a support-map pair, or a ConvexPolyhedron
        // against ConstantOrigin (the ball-centre projection).  One call site below.
        bool run_gjk = false;
        iso gjk_pos{}, seed_pos{};
        ShapeRef ga{}, gb{};
        float max_dist = prediction;
        f3 dir{1.0f, 0.0f, 0.0f}, dflt{1.0f, 0.0f, 0.0f};
        bool seeded = false;
        // Ball pairs: the pose of the ball in the convex shape's frame, the shape, the radius.
        iso pb{};
        ShapeRef cv{};
        float radius = 0.0f;
        const bool local = (flags & (kContactLocalSupportMaps | kContactFeatureMaps)) != 0u;
        if (unsupported) {
            *c = no_contact(kUnsupportedPair);
        } else if (!local && g1.type == PQ_SHAPE_BALL && g2.type == PQ_SHAPE_BALL) {
            // contact_ball_ball
            const float r1 = g1.p0, r2 = g2.p0;
            const f3 c21 = pos12.t;
            const float d2 = norm_sq3(c21);
            const float sum = r1 + r2;
            const float sum_err = sum + prediction;
            if (d2 < sum_err * sum_err) {
                const f3 n1 = d2 != 0.0f ? div3(c21, sqrtf(norm_sq3(c21))) : f3{1.0f, 0.0f, 0.0f};
                const f3 n2 = neg3(qrot_inv(pos12.q, n1));
                const f3 a = mul3(n1, r1), b = mul3(n2, r2);
                store_contact(c, iso_point(pos1, a), iso_point(pos2, b), qrot(pos1.q, n1), qrot(pos2.q, n2),
                              sqrtf(d2) - sum);
            } else {
                *c = no_contact(0);
            }
        } else if (!local && (g1.type == PQ_SHAPE_BALL || g2.type == PQ_SHAPE_BALL)) {
            // contact_ball_convex_polyhedron / contact_convex_polyhedron_ball
            // (default_query_dispatcher.rs:326-335): a Ball first is the flipped
            // contact of (shape 2, ball) under pos12^-1.
            if (g1.type == PQ_SHAPE_BALL) {
                ball_mode = kBallFirst;
                pb = iso_inverse(pos12);
                cv = g2;
                radius = g1.p0;
            } else {
                ball_mode = kBallSecond;
                pb = pos12;
                cv = g1;
                radius = g2.p0;
            }
            const f3 ctr = pb.t;
            PointProj proj{false, f3{0.0f, 0.0f, 0.0f}};
            uint32_t fk = CF_UNKNOWN, fid = 0;
            if (cv.type == PQ_SHAPE_CONVEX_POLYHEDRON) {
                // local_point_projection_on_support_map (point_support_map.rs:17-51)
                run_gjk = true;
                ga = cv;
                gb = origin_shape();
                seed_pos = point_proj_seed_iso(ctr);
                gjk_pos = point_proj_iso(ctr);
                max_dist = kFltMax;
                float l;
                if (!try_unit(ctr, dir, l)) dir = f3{1.0f, 0.0f, 0.0f};
            } else {
                bool has_fn = false;
                f3 fnrm{0.0f, 0.0f, 0.0f};
                if (cv.type == PQ_SHAPE_CUBOID) {
                    proj = cuboid_point_feature(cv, ctr, fk, fid);
                    has_fn = cuboid_feature_normal(fk, fid, fnrm);
                } else if (cv.type == PQ_SHAPE_TRIANGLE) {
                    proj = triangle_point(cv, ctr);
                    has_fn = triangle_normal(cv, fnrm);  // any feature (shape.rs:919-928)
                } else if (cv.type == PQ_SHAPE_CAPSULE) {
                    proj = capsule_point(cv, ctr);
                } else {
                    proj = cone_point(cv, ctr);
                }
                finish_ball_contact(pos1, pos2, pb, radius, prediction, proj, has_fn, fnrm, ball_mode, c);
            }
        } else {
            run_gjk = true;
            ball_mode = pfm ? kPairFeatureMaps : (local ? kPairSupportMapsLocal : kPairSupportMaps);
            max_dist = total_prediction;
            ga = g1;
            gb = g2;
            seed_pos = gjk_pos = pos12;
            // parry's default seed: normalize(pos12.t), else +x (contact_support_map_support_map.rs:52-60)
            const float tsq = norm_sq3(pos12.t);
            dflt = tsq > kEps * kEps ? div3(pos12.t, sqrtf(tsq)) : f3{1.0f, 0.0f, 0.0f};
            dir = dflt;
            if (seeds) {
                const f3 sd = f3{seeds[3 * k], seeds[3 * k + 1], seeds[3 * k + 2]};
                seeded = norm_sq3(sd) > kEps * kEps;  // a zero (or NaN) seed means the default
                if (seeded) dir = sd;
            }
        }
        if (run_gjk) {
            GjkOut r;
            for (int attempt = 0;; ++attempt) {
                sx_reset(s, cso_from_shapes(seed_pos, ga, gb, dir));
                r = gjk_closest_points(gjk_pos, ga, gb, max_dist, s);
                gi += r.iters;
                // a seeded run that reaches the cap falls back to the unseeded GJK,
                // except for a manifold's cached normal, which parry takes as is
                if (!(seeded && !pfm && attempt == 0 && r.iters == kGjkMaxIters)) break;
                dir = dflt;
            }
            if (is_ball_mode(ball_mode)) {
                if (r.kind == GJK_CLOSEST) {
                    finish_ball_contact(pos1, pos2, pb, radius, prediction, PointProj{false, r.p1}, false,
                                        f3{0.0f, 0.0f, 0.0f}, ball_mode, c);
                } else if (r.kind == GJK_INTERSECTION) {
                    need_epa = true;
                } else {
                    *c = no_contact(kUnsupportedPair);  // parry: unreachable!() in gjk::project_origin
                }
            } else if (r.kind == GJK_CLOSEST) {
                finish_contact(pos1, pos2, pos12, r.p1, r.p2, r.n, is_local_mode(ball_mode), c);
            } else if (r.kind == GJK_NO_INTERSECTION) {
                *c = no_contact(0);
                if (pfm) {  // the manifold caches GJK's separating direction (contact_manifolds_pfm_pfm.rs:148-151)
                    c->n1[0] = r.n.x;
                    c->n1[1] = r.n.y;
                    c->n1[2] = r.n.z;
                }
            } else {
                need_epa = true;
            }
        }
        if (iters) {
            iters[2 * k] = gi;
            iters[2 * k + 1] = 0;
        }
    }
    // Wave-aggregated append to the EPA queue.
    const uint64_t mask = __ballot(need_epa);
    if (mask) {
        const uint32_t lane = __lane_id();
        const uint32_t leader = (uint32_t)__builtin_ctzll(mask);
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(&counters[0], (uint32_t)__popcll(mask));
        base = __shfl(base, leader);
        if (need_epa) {
            EpaItem &it = queue[base + lanes_below(mask)];
            it.pair = pair_id;
            it.dim_mode = s.dim | (ball_mode << 8);
            it.i = shape_i;
            it.j = shape_j;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const Cso &v = s.v[q];
                it.v[q][0] = v.p.x; it.v[q][1] = v.p.y; it.v[q][2] = v.p.z;
                it.v[q][3] = v.o1.x; it.v[q][4] = v.o1.y; it.v[q][5] = v.o1.z;
                it.v[q][6] = v.o2.x; it.v[q][7] = v.o2.y; it.v[q][8] = v.o2.z;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Stage 2: EPA, a group of G lanes per pair
// ---------------------------------------------------------------------------
// The argmax reduction over a group of G consecutive lanes: largest value, then
// lowest index (a total order, so any pairing of the lanes gives the same
// winner).  Groups of up to 16 lanes exchange through DPP row permutations --
// mirror within 16 lanes, mirror within 8, then the two quad swaps -- which
// reach every lane of the group in log2(G) steps without the LDS crossbar;
// wider groups use shuffles.  A group's lanes are always active together.
template <int CTRL> __device__ __forceinline__ uint32_t dpp_get(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false);
}
template <int CTRL> __device__ __forceinline__ void argmax_dpp(float &best, uint32_t &bi, f3 &bp) {
    const float ob = __uint_as_float(dpp_get<CTRL>(__float_as_uint(best)));
    const uint32_t oi = dpp_get<CTRL>(bi);
    const float ox = __uint_as_float(dpp_get<CTRL>(__float_as_uint(bp.x)));
    const float oy = __uint_as_float(dpp_get<CTRL>(__float_as_uint(bp.y)));
    const float oz = __uint_as_float(dpp_get<CTRL>(__float_as_uint(bp.z)));
    if (ob > best || (ob == best && oi < bi)) {
        best = ob;
        bi = oi;
        bp = f3{ox, oy, oz};
    }
}
constexpr int kDppRowMirror = 0x140, kDppRowHalfMirror = 0x141, kDppQuadXor2 = 0x4E, kDppQuadXor1 = 0xB1;
template <int G> __device__ __forceinline__ void group_argmax(float &best, uint32_t &bi, f3 &bp) {
    if constexpr (G <= 16) {
        if constexpr (G == 16) argmax_dpp<kDppRowMirror>(best, bi, bp);
        if constexpr (G >= 8) argmax_dpp<kDppRowHalfMirror>(best, bi, bp);
        if constexpr (G >= 4) {
            argmax_dpp<kDppQuadXor2>(best, bi, bp);
            argmax_dpp<kDppQuadXor1>(best, bi, bp);
        }
    } else {
        for (int off = G / 2; off >= 1; off >>= 1) {
            const float ob = __shfl_xor(best, off, G);
            const uint32_t oi = __shfl_xor(bi, off, G);
            const float ox = __shfl_xor(bp.x, off, G), oy = __shfl_xor(bp.y, off, G), oz = __shfl_xor(bp.z, off, G);
            if (ob > best || (ob == best && oi < bi)) {
                best = ob;
                bi = oi;
                bp = f3{ox, oy, oz};
            }
        }
    }
}

// The bits of a wave ballot that belong to the caller's group.
template <int G> __device__ __forceinline__ uint64_t group_ballot(bool p) {
    const uint32_t gbase = __lane_id() & ~(uint32_t)(G - 1);
    return (__ballot(p) >> gbase) & (G >= 64 ? ~0ull : ((1ull << (G & 63)) - 1ull));
}

// ConvexPolyhedron support points computed by a group of G consecutive lanes:
// parry takes the first strict maximum of p.d over the vertex list; if vertex
// 0's product is NaN nothing ever beats it, otherwise the result is the lowest
// index among the largest non-NaN products, which is what the group reduction
// (largest value, then lowest index) returns.  Each lane scans vertices sub,
// sub + G, ... in order; the coordinates of the best one travel with it.
struct Scan {
    float best;
    uint32_t bi;
    f3 bp;
    bool nan0;  // vertex 0's product is NaN (lane 0 of the group)
};
constexpr uint32_t kNoVertex = 0xffffffffu;
__device__ __forceinline__ void scan_step(Scan &s, float4 p, uint32_t k, bool valid, f3 d) {
    const f3 q = f3{p.x, p.y, p.z};
    const float dd = dot3(q, d);
    const bool take = valid && dd == dd && (s.bi == kNoVertex || dd > s.best);
    s.nan0 = (valid && k == 0u) ? dd != dd : s.nan0;
    s.best = take ? dd : s.best;
    s.bi = take ? k : s.bi;
    s.bp = sel2(take, q, s.bp);
}
// Two scans side by side, four vertices of each in flight: one memory latency per
// 4 G vertices of the longer list (a list of length 0 repeats loads of the
// other's first vertex and is ignored).  Vertex 0's product is taken from the
// scan itself, without a load of its own before it.
template <int G>
__device__ __forceinline__ void group_scan2(const float4 *v1, uint32_t n1, f3 d1, const float4 *v2, uint32_t n2, f3 d2,
                                            f3 &r1, f3 &r2) {
    const uint32_t sub = __lane_id() % G;
    Scan a{-INFINITY, kNoVertex, f3{0.0f, 0.0f, 0.0f}, false}, b = a;
    const uint32_t n = n1 > n2 ? n1 : n2;
    const uint32_t last1 = n1 ? n1 - 1u : 0u, last2 = n2 ? n2 - 1u : 0u;
    for (uint32_t k0 = 0; k0 < n; k0 += 4 * G) {
        float4 p[4], q[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t k = k0 + j * G + sub;
            p[j] = v1[k < last1 ? k : last1];
            q[j] = v2[k < last2 ? k : last2];
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t k = k0 + j * G + sub;
            scan_step(a, p[j], k, k < n1, d1);
            scan_step(b, q[j], k, k < n2, d2);
        }
    }
    const bool nan1 = group_ballot<G>(a.nan0) != 0ull, nan2 = group_ballot<G>(b.nan0) != 0ull;
    if (nan1 || nan2) {  // vertex 0, whatever the others are
        if (nan1) a = Scan{0.0f, 0u, f3{v1[0].x, v1[0].y, v1[0].z}, true};
        if (nan2) b = Scan{0.0f, 0u, f3{v2[0].x, v2[0].y, v2[0].z}, true};
    }
    group_argmax<G>(a.best, a.bi, a.bp);
    group_argmax<G>(b.best, b.bi, b.bp);
    r1 = a.bp;
    r2 = b.bp;
}

// One scan over vertices staged in LDS.
template <int G> __device__ __forceinline__ f3 group_scan_staged(const float (*sv)[3], uint32_t n, f3 d) {
    const uint32_t sub = __lane_id() % G;
    Scan a{-INFINITY, kNoVertex, f3{0.0f, 0.0f, 0.0f}, false};
    for (uint32_t k = sub; k < n; k += G)
        scan_step(a, make_float4(sv[k][0], sv[k][1], sv[k][2], 0.0f), k, true, d);
    if (group_ballot<G>(a.nan0) != 0ull) return f3{sv[0][0], sv[0][1], sv[0][2]};
    group_argmax<G>(a.best, a.bi, a.bp);
    return a.bp;
}

struct Staged {
    const float (*s1)[3];  // null: not staged
    const float (*s2)[3];
};

// CSOPoint::from_shapes (see cso_from_shapes) by a group; STAGED: the
// ConvexPolyhedra may be staged in LDS.
template <int G, bool STAGED>
__device__ __forceinline__ Cso group_cso(const iso &pos12, const ShapeRef &g1, const ShapeRef &g2, const Staged &st,
                                         f3 dir) {
    const f3 d2 = qrot_inv(pos12.q, neg3(dir));
    const bool poly1 = g1.type == PQ_SHAPE_CONVEX_POLYHEDRON, poly2 = g2.type == PQ_SHAPE_CONVEX_POLYHEDRON;
    f3 a{0.0f, 0.0f, 0.0f}, b{0.0f, 0.0f, 0.0f};
    const bool scan1 = poly1 && !(STAGED && st.s1), scan2 = poly2 && !(STAGED && st.s2);
    if (scan1 || scan2)
        group_scan2<G>(scan1 ? g1.v : g2.v, scan1 ? g1.n : 0u, dir, scan2 ? g2.v : g1.v, scan2 ? g2.n : 0u, d2, a, b);
    if (STAGED && poly1 && st.s1) a = group_scan_staged<G>(st.s1, g1.n, dir);
    if (STAGED && poly2 && st.s2) b = group_scan_staged<G>(st.s2, g2.n, d2);
    if (!poly1) a = local_support(g1, dir);
    if (!poly2) b = local_support(g2, d2);
    b = g2.type == kShapeOrigin ? pos12.t : iso_point(pos12, b);
    return Cso{sub3(a, b), a, b};
}

// Copies a ConvexPolyhedron's vertices into LDS (group-cooperative); returns
// the staged array or nullptr if the shape is not staged.
template <int G, class W> __device__ const float (*stage_shape(W *w, int slot, const ShapeRef &s))[3] {
    if (W::kSV == 0 || s.type != PQ_SHAPE_CONVEX_POLYHEDRON || s.n > (uint32_t)W::kSV) return nullptr;
    const uint32_t sub = __lane_id() % G;
    for (uint32_t k = sub; k < s.n; k += G) {
        const float4 p = s.v[k];
        w->sv[slot][k][0] = p.x;
        w->sv[slot][k][1] = p.y;
        w->sv[slot][k][2] = p.z;
    }
    return w->sv[slot];
}

constexpr uint32_t kOrigFloats = 6;  // orig1, orig2 per CSO vertex
template <class W> __device__ __forceinline__ f3 vpt(const W *w, uint32_t i) {
    return f3{w->vp[i][0], w->vp[i][1], w->vp[i][2]};
}
template <class W> __device__ __forceinline__ void vset(W *w, float *orig, uint32_t i, const Cso &c) {
    w->vp[i][0] = c.p.x;
    w->vp[i][1] = c.p.y;
    w->vp[i][2] = c.p.z;
    float *o = orig + kOrigFloats * i;
    o[0] = c.o1.x; o[1] = c.o1.y; o[2] = c.o1.z;
    o[3] = c.o2.x; o[4] = c.o2.y; o[5] = c.o2.z;
}

enum : uint32_t { EPA_OK = 0, EPA_NONE = 1, EPA_OVERFLOW = 2, EPA_RUNNING = 3, EPA_POINT = 4, EPA_RESTART = 5 };

// Barycentric coordinates of Face::new's projection (epa3.rs:96-118,
// TrianglePointLocation::barycentric_coordinates); returns proj_inside.
__device__ __forceinline__ bool face_bcoords(f3 pa, f3 pb, f3 pc, float bc[3]) {
    Loc l;
    bool inside;
    const f3 proj = tri_origin(pa, pb, pc, l, inside);
    bc[0] = bc[1] = bc[2] = 0.0f;
    const float e = kEps * 100.0f;
    if (l.kind == LOC_VERTEX) {
        bc[0] = l.id == 0 ? 1.0f : 0.0f;
        bc[1] = l.id == 1 ? 1.0f : 0.0f;
        bc[2] = l.id == 2 ? 1.0f : 0.0f;
        return inside || norm_sq3(proj) < e * e;
    }
    if (l.kind == LOC_EDGE) {  // edges (0,1), (1,2), (0,2)
        bc[0] = l.id == 1 ? 0.0f : l.b0;
        bc[1] = l.id == 0 ? l.b1 : (l.id == 1 ? l.b0 : 0.0f);
        bc[2] = l.id == 0 ? 0.0f : l.b1;
        return inside || norm_sq3(proj) < e * e;
    }
    if (l.kind == LOC_FACE) {
        bc[0] = l.b0;
        bc[1] = l.b1;
        bc[2] = l.b2;
        return true;
    }
    return false;
}

// ccw_face_normal (utils/ccw_face_normal.rs:19-27), zero if degenerate.
__device__ __forceinline__ f3 ccw_normal(f3 pa, f3 pb, f3 pc) {
    const f3 r = cross3(sub3(pb, pa), sub3(pc, pa));
    const float sq = norm_sq3(r);
    f3 n = f3{0.0f, 0.0f, 0.0f};
    if (sq > kEps * kEps) n = div3(r, sqrtf(sq));
    return n;
}

// The polytope of one pair in LDS.  A face is three vertex ids (8 bits each) with
// its visibility bits and, where kMask is false, its deleted flag in one word,
// and its three neighbours in another, so a step of the silhouette walk reads
// one face with two loads.  The shape-space points orig1/orig2 of a CSO vertex
// are only needed for the final witness points: they go to a per-group global
// buffer, and the face's barycentric coordinates are recomputed there (the same
// projection as Face::new).
//
// There is no heap.  parry's BinaryHeap pops the live face of largest key
// (-distance); which one only depends on the heap's layout when two live faces
// share the largest key.  So the next face is the maximum of key[] over the live
// faces, taken by the group's lanes in parallel, and the heap itself is only
// rebuilt when that maximum is not unique (lazy_replay): every push and pop so
// far is known from the face ids, pops[] and nfs[].  On 20,695 mixed pairs the
// maximum was shared in 0.1% of the iterations.
//
// The scans of an iteration (the maximum, can_be_seen_by) go over live[], a list of
// the faces not deleted, in any order: a new face takes the list place of a face
// the iteration deleted.  Of a polytope's faces half are deleted after eight
// iterations and four fifths after sixty.  Scanning them all, 2^20 mixed pairs took
// 3.31 ms (3.14 with the list) and 300 pairs 405 us (368).  Normals are kept by list
// place too, not by face, which a deleted face does not need: three waves per CU more
// in the third tier, 2^20 mixed pairs 3.14 -> 3.07 ms.
template <int V, int F, int S, int K, class I, int SV, int L> struct LazyState {
    static constexpr int kV = V, kF = F, kS = S, kK = K, kSV = SV, kL = L;
    static constexpr bool kMask = F <= 64;  // deleted flags in a 64-bit register mask
    static constexpr uint32_t kShift = sizeof(I) == 1 ? 8u : 16u;
    using Idx = I;
    using Entry = std::conditional_t<sizeof(I) == 1, uint16_t, uint32_t>;
    struct alignas(sizeof(I) == 1 ? 8 : 4) Face {
        uint32_t px;  // vertices; bits 24-26: can_be_seen_by the newest vertex per opposite vertex; 27: deleted
        I adj[4];     // the three neighbours, and the face's place in live[]
    };
    alignas(16) float nk[L][4];  // by place in live[]: normal, then FaceId's neg_dist (-inf for a face that was
                                 // not pushed, or a place whose face was deleted)
    float key[F];                // neg_dist of every face, for the rebuilt heap
    float vp[V][4];
    Face face[F];
    float sv[SV > 0 ? 2 : 1][SV > 0 ? SV : 1][3];  // both ConvexPolyhedra's vertices (local frames), if SV > 0
    Entry sil[S + 1];          // face | opp << kShift, and a slot for what is not kept
    Entry stk[K + 1];          // face | point << kShift, likewise
    I dl[S + 2];               // places in live[] of the faces the current iteration deleted, and a spare
    I live[L];                 // the faces not deleted
    I hid[F];                  // the heap's face ids, when it is rebuilt
    I pops[V], nfs[V];         // per iteration: the face it popped, and the number of faces before it
};
constexpr uint32_t kDeadBit = 1u << 27;


// With a wave per pair every value of the pair is the same in all lanes: saying so
// makes the branches on shape types and counts scalar (support points 3,700 ->
// 2,600 cycles, the next face 3,900 -> 3,100; the walk got slower, 3,600 -> 4,900, and
// keeps its vector form).
template <int G> __device__ __forceinline__ uint32_t uni(uint32_t v) {
    if constexpr (G == 64) return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
    return v;
}
template <int G> __device__ __forceinline__ float uni(float v) {
    if constexpr (G == 64) return __uint_as_float(uni<G>(__float_as_uint(v)));
    return v;
}
template <int G> __device__ __forceinline__ f3 uni(f3 v) { return f3{uni<G>(v.x), uni<G>(v.y), uni<G>(v.z)}; }
template <int G> __device__ __forceinline__ ShapeRef uni(ShapeRef g) {
    g.type = uni<G>(g.type);
    g.n = uni<G>(g.n);
    return g;
}

struct LazyRegs {
    uint32_t nv, nf, best_id, niter;
    float max_dist, old_dist;
    uint64_t dead;  // kMask: the deleted faces
    // the rebuilt heap: its length, the iterations and faces it has taken in
    uint32_t hlen, hiter, hnf;
    uint32_t nl;  // length of live[]
};

template <class W> __device__ __forceinline__ bool face_dead(const W *w, const LazyRegs &r, uint32_t f, uint32_t x) {
    if constexpr (W::kMask) return ((r.dead >> f) & 1ull) != 0ull;
    return (x & kDeadBit) != 0u;
}
// The three neighbours of a face, kShift bits each.
template <class F> __device__ __forceinline__ auto face_adj(const F &f) {
    if constexpr (sizeof(f.adj[0]) == 1)
        return __builtin_bit_cast(uint32_t, f.adj);
    else
        return (uint64_t)f.adj[0] | ((uint64_t)f.adj[1] << 16) | ((uint64_t)f.adj[2] << 32);
}
template <class W> __device__ __forceinline__ float face_key(const W *w, uint32_t f) { return w->key[f]; }
template <class W> __device__ __forceinline__ f3 place_normal(const W *w, uint32_t place) {
    return f3{w->nk[place][0], w->nk[place][1], w->nk[place][2]};
}
template <class W, class A> __device__ __forceinline__ uint32_t adj_at(A a, uint32_t k) {
    return (uint32_t)(a >> (W::kShift * k)) & ((1u << W::kShift) - 1u);
}
__device__ __forceinline__ uint32_t pt_at(uint32_t x, uint32_t k) { return (x >> (8u * k)) & 0xffu; }
// Entry of the silhouette walk: neighbour k of a face and the face's point k.
template <class W> __device__ __forceinline__ uint32_t walk_entry(const typename W::Face &f, uint32_t k) {
    if constexpr (sizeof(typename W::Idx) == 1)  // bytes k of adj and px
        return __builtin_amdgcn_perm(f.px, face_adj(f), 0x0c0c0400u + k * 0x0101u);
    else
        return adj_at<W>(face_adj(f), k) | (pt_at(f.px, k) << W::kShift);
}

__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The largest value of a group's lanes (no NaN), in every lane of the group.
template <int CTRL> __device__ __forceinline__ float max_dpp(float v) {
    return fmaxf(v, __uint_as_float(dpp_get<CTRL>(__float_as_uint(v))));
}
template <int G> __device__ __forceinline__ float group_max(float v) {
    if constexpr (G >= 16) v = max_dpp<kDppRowMirror>(v);
    if constexpr (G >= 8) v = max_dpp<kDppRowHalfMirror>(v);
    v = max_dpp<kDppQuadXor2>(v);
    v = max_dpp<kDppQuadXor1>(v);
    if constexpr (G >= 32) v = fmaxf(v, __shfl_xor(v, 16, 64));
    if constexpr (G >= 64) v = fmaxf(v, __shfl_xor(v, 32, 64));
    return v;
}
// proj_inside of Face::new (epa3.rs:96-118): whether the origin projects inside
// the triangle, or onto a vertex or edge within 100 EPS of the origin.  The
// comparisons are those of Triangle::project_local_point_and_get_location
// (point_triangle.rs:54-291) in its order, but the regions are selected instead
// of branched to: the lanes of a wave build faces of every region, and took all
// six branches with a division each.
__device__ __forceinline__ bool face_inside(f3 a, f3 b, f3 c) {
    const f3 ab = sub3(b, a), ac = sub3(c, a), bc = sub3(c, b);
    const f3 ap = neg3(a), bp = neg3(b), cp = neg3(c);
    const float ab_ap = dot3(ab, ap), ac_ap = dot3(ac, ap);
    const float ab_bp = dot3(ab, bp), ac_bp = dot3(ac, bp);
    const float ab_cp = dot3(ab, cp), ac_cp = dot3(ac, cp);
    const f3 n = cross3(ab, ac);
    const float vc = dot3(n, cross3(ab, ap)), vb = -dot3(n, cross3(ac, cp)), va = dot3(n, cross3(bc, bp));
    const bool va_ = (ab_ap <= 0.0f) & (ac_ap <= 0.0f);
    const bool vb_ = !va_ & (ab_bp >= 0.0f) & (ac_bp <= ab_bp);
    const bool vc_ = !va_ & !vb_ & (ac_cp >= 0.0f) & (ab_cp <= ac_cp);
    const bool vertex = va_ | vb_ | vc_;
    const bool eab = !vertex & (vc < 0.0f) & (ab_ap >= 0.0f) & (ab_bp <= 0.0f);
    const bool eac = !vertex & !eab & (vb < 0.0f) & (ac_ap >= 0.0f) & (ac_cp <= 0.0f);
    const bool ebc = !vertex & !eab & !eac & (va < 0.0f) & (ac_bp - ab_bp >= 0.0f) & (ab_cp - ac_cp >= 0.0f);
    const f3 base = sel2(vb_ | ebc, b, sel2(vc_, c, a));
    const f3 dir = sel2(eab, ab, sel2(eac, ac, bc));
    const float t = (eab ? ab_ap : (eac ? ac_ap : dot3(bc, bp))) / norm_sq3(dir);
    const f3 r = sel2(vertex, base, add3(base, mul3(dir, t)));
    const float e = kEps * 100.0f;
    const bool near = near_origin(r) || norm_sq3(r) < e * e;
    return (vertex | eab | eac | ebc) ? near : va + vb + vc != 0.0f;
}

// Face::new (epa3.rs:96-118) by one lane; returns proj_inside.
template <class W>
__device__ __forceinline__ bool lazy_face(W *w, uint32_t f, uint32_t a, uint32_t b, uint32_t c, uint32_t j0,
                                          uint32_t j1, uint32_t j2, uint32_t place, f3 &n, f3 &pa) {
    using I = typename W::Idx;
    w->face[f] = typename W::Face{a | (b << 8) | (c << 16), {(I)j0, (I)j1, (I)j2, (I)place}};
    w->live[place] = (I)f;
    pa = vpt(w, a);
    const f3 pb = vpt(w, b), pc = vpt(w, c);
    n = ccw_normal(pa, pb, pc);
    return face_inside(pa, pb, pc);
}
template <class W> __device__ __forceinline__ void set_normal(W *w, uint32_t f, uint32_t place, f3 n, float key) {
    *reinterpret_cast<float4 *>(w->nk[place]) = make_float4(n.x, n.y, n.z, key);
    w->key[f] = key;
}

// Face::closest_points (epa3.rs:120-130).
template <class W> __device__ void lazy_points(const W *w, const float *orig, uint32_t f, f3 &p1, f3 &p2, f3 &n) {
    const uint32_t x = w->face[f].px;
    const f3 a = vpt(w, pt_at(x, 0)), b = vpt(w, pt_at(x, 1)), c = vpt(w, pt_at(x, 2));
    float bc[3];
    face_bcoords(a, b, c, bc);
    f3 o1[3], o2[3];
    for (int q = 0; q < 3; ++q) {
        const float *o = orig + kOrigFloats * pt_at(x, q);
        o1[q] = f3{o[0], o[1], o[2]};
        o2[q] = f3{o[3], o[4], o[5]};
    }
    p1 = add3(add3(mul3(o1[0], bc[0]), mul3(o1[1], bc[1])), mul3(o1[2], bc[2]));
    p2 = add3(add3(mul3(o2[0], bc[0]), mul3(o2[1], bc[1])), mul3(o2[2], bc[2]));
    n = ccw_normal(a, b, c);  // as lazy_face computed it
}

// BinaryHeap<FaceId> over face ids (max-heap on key[]; equal keys compare Equal),
// with std's sift_up / sift_down_to_bottom so equal keys pop in parry's order.
template <class W> __device__ __forceinline__ void heap_sift_up(W *w, uint32_t pos) {
    const uint32_t id = w->hid[pos];
    const float nd = face_key(w, id);
    while (pos > 0) {
        const uint32_t parent = (pos - 1) / 2, pid = w->hid[parent];
        if (nd <= face_key(w, pid)) break;
        w->hid[pos] = (typename W::Idx)pid;
        pos = parent;
    }
    w->hid[pos] = (typename W::Idx)id;
}
template <class W> __device__ __forceinline__ void heap_pop(W *w, uint32_t &len) {
    --len;
    if (len == 0) return;
    const uint32_t id = w->hid[len];
    uint32_t pos = 0, child = 1;
    while (child + 2 <= len) {
        uint32_t cid = w->hid[child];
        const uint32_t rid = w->hid[child + 1];
        if (face_key(w, cid) <= face_key(w, rid)) {
            ++child;
            cid = rid;
        }
        w->hid[pos] = (typename W::Idx)cid;
        pos = child;
        child = 2 * pos + 1;
    }
    if (child == len - 1) {
        w->hid[pos] = w->hid[child];
        pos = child;
    }
    w->hid[pos] = (typename W::Idx)id;
    heap_sift_up(w, pos);
}
// The face parry's heap pops next when several live faces share the largest key:
// brings the heap up to date with every push and pop so far, in parry's order
// (each iteration pops until its face, deleted faces included, then pushes its
// new faces by id), then pops the deleted faces at the top.  Run by all lanes of
// the group with the same values.  Every push and pop is replayed once per pair.
constexpr uint32_t kNoFace = 0xffffffffu;
template <class W> __device__ uint32_t lazy_replay(W *w, LazyRegs &r) {
    for (;;) {
        const bool now = r.hiter == r.niter;
        const uint32_t upto = now ? r.nf : w->nfs[r.hiter];
        for (; r.hnf < upto; ++r.hnf)
            if (face_key(w, r.hnf) != -INFINITY) {
                w->hid[r.hlen] = (typename W::Idx)r.hnf;
                heap_sift_up(w, r.hlen++);
            }
        if (now) break;
        const uint32_t until = w->pops[r.hiter];
        uint32_t id = kNoFace;
        while (r.hlen != 0 && id != until) {
            id = w->hid[0];
            heap_pop(w, r.hlen);
        }
        ++r.hiter;
    }
    while (r.hlen != 0) {
        const uint32_t id = w->hid[0];
        if (!face_dead(w, r, id, w->face[id].px)) return id;
        heap_pop(w, r.hlen);
    }
    return kNoFace;  // not reached: a live pushed face is in the heap
}

// A polytope at the start of an iteration, handed to the next tier so that the
// pair continues where it stopped instead of starting over.
template <int V, int F> struct EpaRec {
    uint32_t nv, nf, best_id, niter;
    float max_dist, old_dist;
    uint32_t pad[2];
    float vp[V][3];
    float orig[V][6];
    uint32_t px[F];   // with kDeadBit
    uint32_t adj[F];  // 8 bits each
    float key[F];
    uint8_t pops[V], nfs[V];
};
constexpr uint32_t kNoCont = 0xffffffffu;
// Where a tier writes the polytopes it hands on.
template <class R> struct RecSink {
    R *recs;
    uint32_t *count;
    uint32_t cap;
};

template <int G, class W, class R>
__device__ uint32_t lazy_export(const W *w, const float *orig, const RecSink<R> &sink, const LazyRegs &r) {
    static_assert(sizeof(typename W::Idx) == 1, "records hold byte ids");
    const uint32_t sub = __lane_id() % G;
    uint32_t ci = 0;
    if (sub == 0) ci = atomicAdd(sink.count, 1u);
    ci = (uint32_t)__shfl((int)ci, 0, G);
    if (ci >= sink.cap) return kNoCont;
    // orig rows were written to global memory by this wave; the group's lanes
    // read each other's rows below
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
    R *o = sink.recs + ci;
    if (sub == 0) {
        o->nv = r.nv;
        o->nf = r.nf;
        o->best_id = r.best_id;
        o->niter = r.niter;
        o->max_dist = r.max_dist;
        o->old_dist = r.old_dist;
    }
    for (uint32_t k = sub; k < r.nv; k += G) {
        for (int q = 0; q < 3; ++q) o->vp[k][q] = w->vp[k][q];
        for (int q = 0; q < 6; ++q) o->orig[k][q] = orig[kOrigFloats * k + q];
    }
    for (uint32_t k = sub; k < r.nf; k += G) {
        const typename W::Face f = w->face[k];
        o->px[k] = (f.px & 0x00ffffffu) | (face_dead(w, r, k, f.px) ? kDeadBit : 0u);
        o->adj[k] = face_adj(f);
        o->key[k] = w->key[k];
    }
    for (uint32_t k = sub; k < r.niter; k += G) {
        o->pops[k] = (uint8_t)w->pops[k];
        o->nfs[k] = (uint8_t)w->nfs[k];
    }
    return ci;
}

// Loads a record into the group's polytope; face normals are recomputed from the
// vertices exactly as Face::new computed them.
template <int G, class W, class R> __device__ void lazy_import(W *w, float *orig, const R *o, LazyRegs &r) {
    static_assert(!W::kMask, "a tier that continues keeps its deleted flags in LDS");
    using I = typename W::Idx;
    const uint32_t sub = __lane_id() % G;
    r.nv = o->nv;
    r.nf = o->nf;
    r.best_id = o->best_id;
    r.niter = o->niter;
    r.max_dist = o->max_dist;
    r.old_dist = o->old_dist;
    for (uint32_t k = sub; k < r.nv; k += G) {
        for (int q = 0; q < 3; ++q) w->vp[k][q] = o->vp[k][q];
        for (int q = 0; q < 6; ++q) orig[kOrigFloats * k + q] = o->orig[k][q];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    __builtin_amdgcn_wave_barrier();
    r.nl = 0;
    for (uint32_t k0 = 0; k0 < r.nf; k0 += G) {
        const uint32_t k = k0 + sub;
        const uint32_t x = k < r.nf ? o->px[k] : kDeadBit;
        const uint64_t alive = group_ballot<G>((x & kDeadBit) == 0u);
        const uint32_t place = r.nl + (uint32_t)__popcll(alive & ((1ull << sub) - 1ull));
        r.nl += (uint32_t)__popcll(alive);
        if (k < r.nf) {
            const uint32_t a = o->adj[k];
            w->face[k] = typename W::Face{x, {(I)(a & 0xffu), (I)((a >> 8) & 0xffu), (I)((a >> 16) & 0xffu), (I)place}};
            if ((x & kDeadBit) == 0u) {
                w->live[place] = (I)k;
                const f3 n = ccw_normal(vpt(w, pt_at(x, 0)), vpt(w, pt_at(x, 1)), vpt(w, pt_at(x, 2)));
                set_normal(w, k, place, n, o->key[k]);
            } else {
                w->key[k] = o->key[k];
            }
        }
    }
    for (uint32_t k = sub; k < r.niter; k += G) {
        w->pops[k] = (I)o->pops[k];
        w->nfs[k] = (I)o->nfs[k];
    }
    lds_order();
}

// The EPA problem of a queued pair (contact_support_map_support_map.rs:60-76):
// its two shapes (their feature maps in kPairFeatureMaps mode) and relative pose,
// or, for a Ball, the other shape against the ball centre
// (point_support_map.rs:39-49).
struct EpaProblem {
    iso pos;
    ShapeRef a, b;
};

__device__ EpaProblem epa_problem(const ShapeRecord *rec, const float4 *verts, const float *poses, const EpaItem *it) {
    const uint32_t i = it->i, j = it->j;
    const iso pos1 = load_iso(poses + 7 * (size_t)i), pos2 = load_iso(poses + 7 * (size_t)j);
    const iso pos12 = iso_inv_mul(pos1, pos2);
    ShapeRef g1 = load_shape(rec, verts, i), g2 = load_shape(rec, verts, j);
    const uint32_t mode = item_mode(it);
    if (mode == kPairFeatureMaps) {
        float br;
        (void)feature_map(g1, br);
        (void)feature_map(g2, br);
    }
    if (is_ball_mode(mode)) {
        if (mode == kBallFirst) return EpaProblem{point_proj_iso(iso_inverse(pos12).t), g2, origin_shape()};
        return EpaProblem{point_proj_iso(pos12.t), g1, origin_shape()};
    }
    return EpaProblem{pos12, g1, g2};
}

// EPA::closest_points (epa3.rs:428-651) for one pair by a group of G lanes, one
// iteration at a time: lazy_begin, then lazy_step until it returns a result.
// Results: EPA_OK (the answer is face r.best_id), EPA_POINT (a simplex of
// dimension 0), EPA_NONE, EPA_OVERFLOW (the polytope outgrew this tier's buffers
// and is as it was at the start of the iteration), EPA_RESTART (a face key the
// maximum cannot order -- NaN or -inf -- which the heap tiers handle).
template <int G, class W, class R>
__device__ uint32_t lazy_begin(W *w, float *orig, const EpaProblem &pr, const EpaItem *it, const R *resume, Staged &st,
                               LazyRegs &r) {
    st = Staged{stage_shape<G>(w, 0, pr.a), stage_shape<G>(w, 1, pr.b)};
    lds_order();  // the staged vertices, before any lane reads another lane's entries
    r = LazyRegs{0, 0, 0, 0, kFltMax, 0.0f, 0ull, 0, 0, 0};
    if constexpr (!W::kMask) {
        if (resume) {
            lazy_import<G>(w, orig, resume, r);
            return EPA_RUNNING;
        }
    }
    const uint32_t dim = it->dim_mode & 0xffu;
    if (dim == 0) return EPA_POINT;
    f3 pv[4];
    for (int i = 0; i < 4; ++i) pv[i] = f3{it->v[i][0], it->v[i][1], it->v[i][2]};
    // a tetrahedron of the wrong orientation swaps its vertices 1 and 2
    const bool swap = dim == 3 && dot3(cross3(sub3(pv[1], pv[0]), sub3(pv[2], pv[0])), sub3(pv[3], pv[0])) > 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        if (i > dim) break;
        const uint32_t from = swap && i == 1 ? 2u : (swap && i == 2 ? 1u : i);
        for (int q = 0; q < 3; ++q) w->vp[i][q] = it->v[from][q];
        for (int q = 0; q < 6; ++q) orig[kOrigFloats * i + q] = it->v[from][3 + q];
    }
    r.nv = dim + 1;
    const uint32_t sub = __lane_id() % G;
    if (dim == 1) {
        // orthonormal_subspace_basis([dpt]): first vector a x dpt
        const f3 dpt = sub3(pv[1], pv[0]);
        f3 a = fabsf(dpt.x) > fabsf(dpt.y) ? f3{dpt.z, 0.0f, -dpt.x} : f3{0.0f, -dpt.z, dpt.y};
        a = div3(a, sqrtf(norm_sq3(a)));
        vset(w, orig, 2, group_cso<G, (W::kSV > 0)>(pr.pos, pr.a, pr.b, st, cross3(a, dpt)));
        r.nv = 3;
    }
    lds_order();
    // The first faces, one per lane: (0,1,2) (1,3,2) (0,2,3) (0,3,1) of a
    // tetrahedron (epa3.rs:459-500), both sides of a triangle otherwise.
    r.nf = dim == 3 ? 4u : 2u;
    r.nl = r.nf;
    bool in = false, bad = false, weird = false;
    if (sub < r.nf) {
        uint32_t pts, adj;
        if (dim == 3) {
            pts = sub == 0 ? 0x020100u : (sub == 1 ? 0x020301u : (sub == 2 ? 0x030200u : 0x010300u));
            adj = sub == 0 ? 0x020103u : (sub == 1 ? 0x000203u : (sub == 2 ? 0x030100u : 0x000102u));
        } else {
            pts = sub == 0 ? 0x020100u : 0x010200u;
            adj = sub == 0 ? 0x010101u : 0x000000u;
        }
        f3 n, pa;
        in = lazy_face(w, sub, pt_at(pts, 0), pt_at(pts, 1), pt_at(pts, 2), pt_at(adj, 0), pt_at(adj, 1),
                       pt_at(adj, 2), sub, n, pa);
        float k = 0.0f;
        if (dim == 3) {
            const float dist = dot3(n, vpt(w, sub));  // vertex `sub`, as parry takes it
            bad = in && -dist > kEpsTol;              // FaceId::new -> None
            weird = in && !(fabsf(dist) <= kFltMax);
            k = in ? -dist : -INFINITY;
        }
        set_normal(w, sub, sub, n, k);
    }
    lds_order();
    if (dim == 3) {
        if (group_ballot<G>(bad) != 0ull || group_ballot<G>(in) == 0ull) return EPA_NONE;
        if (group_ballot<G>(weird) != 0ull) return EPA_RESTART;
    }
    return EPA_RUNNING;
}

// One EPA iteration (the body of the loop of epa3.rs:499-647).
template <int G, class W>
__device__ uint32_t lazy_step(W *w, float *orig, const EpaProblem &pr, const Staged &st, LazyRegs &r) {
    using I = typename W::Idx;
    using E = typename W::Entry;
    constexpr uint32_t kIdMask = (1u << W::kShift) - 1u;
    const float eps_tol = kEps * 100.0f;
    const uint32_t sub = __lane_id() % G;
    r.nv = uni<G>(r.nv);
    r.nf = uni<G>(r.nf);
    r.niter = uni<G>(r.niter);
    r.nl = uni<G>(r.nl);
    const ShapeRef ga = uni<G>(pr.a), gb = uni<G>(pr.b);
    // The live face of largest key.
    uint32_t fid, fplace;
    float fkey;
    {
        float kb = -INFINITY;
        uint32_t ib = 0;
        bool dup = false;
        for (uint32_t i0 = sub; i0 < r.nl; i0 += 4 * G) {  // four keys' loads in flight
            float k[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) k[u] = w->nk[i0 + u * G < r.nl ? i0 + u * G : i0][3];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const float kk = i0 + u * G < r.nl ? k[u] : -INFINITY;
                dup = kk > kb ? false : (kk == kb ? true : dup);
                ib = kk > kb ? i0 + u * G : ib;
                kb = fmaxf(kk, kb);
            }
        }
        fkey = uni<G>(group_max<G>(kb));
        if (fkey == -INFINITY) return EPA_OK;  // parry's heap is empty
        const uint64_t top = group_ballot<G>(kb == fkey);
        const uint64_t twice = group_ballot<G>(kb == fkey && dup);
        fplace = (uint32_t)__shfl((int)ib, __builtin_ctzll(top), G);
        if (twice != 0ull || (top & (top - 1ull)) != 0ull) {
            fid = lazy_replay(w, r);
            if (fid == kNoFace) return EPA_RESTART;
            fplace = w->face[fid].adj[3];
        }
        fplace = uni<G>(fplace);
        fid = uni<G>((uint32_t)w->live[fplace]);
    }
    const typename W::Face face = w->face[fid];
    const uint32_t fx = face.px;
    const f3 fn = place_normal(w, fplace);
    const Cso c = group_cso<G, (W::kSV > 0)>(pr.pos, ga, gb, st, fn);
    const float cand = dot3(c.p, fn);
    uint32_t best_t = r.niter == 0 ? fid : r.best_id;  // the heap's first top is parry's first best face
    float max_t = r.max_dist;
    if (cand < max_t) {
        best_t = fid;
        max_t = cand;
    }
    const float curr_dist = -fkey;
    if (max_t - curr_dist < eps_tol || (fabsf(curr_dist - r.old_dist) < kEps && cand < max_t)) {
        r.best_id = best_t;
        return EPA_OK;
    }
    if (r.nv >= (uint32_t)W::kV) return EPA_OVERFLOW;
    const uint32_t sp = r.nv;  // counted when the iteration commits
    vset(w, orig, sp, c);
    const uint64_t dead0 = r.dead;
    if constexpr (W::kMask)
        r.dead |= 1ull << fid;
    else
        w->face[fid].px = fx | kDeadBit;
    lds_order();
    // Face::can_be_seen_by (epa3.rs:153-166) of every face from the new vertex,
    // for each of the three opposite vertices, by the group's lanes in parallel;
    // the depth-first walk below only reads the bits.  With no branch in the body the
    // loads of consecutive faces overlap.
    {
        const float E2 = kEps * 100.0f;
        for (uint32_t i0 = sub; i0 < r.nl; i0 += 2 * G) {  // two faces' loads in flight
            const uint32_t f[2] = {w->live[i0], w->live[i0 + G < r.nl ? i0 + G : i0]};
            uint32_t x[2];
            f3 fnn[2], qs[2][3];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                x[u] = w->face[f[u]].px;
                fnn[u] = place_normal(w, u == 0 || i0 + G >= r.nl ? i0 : i0 + G);
            }
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int q = 0; q < 3; ++q) qs[u][q] = vpt(w, pt_at(x[u], q));
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                uint32_t bits = 0;
#pragma unroll
                for (int opp = 0; opp < 3; ++opp) {
                    const f3 p0 = qs[u][opp], p1 = qs[u][(opp + 1) % 3], p2 = qs[u][(opp + 2) % 3];
                    const bool front = dot3(sub3(c.p, p0), fnn[u]) >= -kEpsTol;
                    const bool flat = norm_sq3(cross3(sub3(p2, p1), sub3(c.p, p1))) <= E2 * E2;  // is_affinely_dependent
                    bits |= (uint32_t)(front | flat) << opp;
                }
                reinterpret_cast<uint8_t *>(&w->face[f[u]].px)[3] =
                    (uint8_t)(bits | ((x[u] >> 24) & (kDeadBit >> 24)));
            }
        }
    }
    lds_order();
    // compute_silhouette (epa3.rs:653-675) for the three neighbours in order
    // adj[0], adj[1], adj[2]; a visible face recurses into adj[(opp + 2) % 3],
    // then adj[opp].  The recursion is an explicit stack of (face, the point its
    // opposite vertex follows) with its top entry kept in a register as well.  A
    // step is one read of the visited face and no branch: what a step does not do
    // (record an edge, push) is written to a spare slot, and running out of a
    // buffer ends the loop.  With branches a step took the wave about 550 cycles.
    uint32_t ns = 0, ndel = 1, depth = 2;
    w->dl[0] = (I)fplace;
    uint32_t cur = walk_entry<W>(face, 0), top = walk_entry<W>(face, 1);
    w->stk[0] = (E)walk_entry<W>(face, 2);
    w->stk[1] = (E)top;
    bool ended;
    for (;;) {
        const uint32_t id = cur & kIdMask, pt = cur >> W::kShift;
        const typename W::Face f = w->face[id];
        const uint32_t below = w->stk[depth > 2u ? depth - 2u : 0u];
        const bool at0 = pt_at(f.px, 0) == pt, at1 = pt_at(f.px, 1) == pt;
        const uint32_t opp = at0 ? 1u : (at1 ? 2u : 0u);  // next_ccw_pt_id
        const uint32_t k1 = at0 ? 0u : (at1 ? 1u : 2u);   // (opp + 2) % 3
        const bool live = !face_dead(w, r, id, f.px);
        const bool vis = ((f.px >> (24u + opp)) & 1u) != 0u;
        const bool del = live & vis, edge = live & !vis;
        w->sil[edge ? ns : (uint32_t)W::kS] = (E)(id | (opp << W::kShift));
        ns += edge ? 1u : 0u;
        w->dl[del ? ndel : (uint32_t)W::kS + 1u] = f.adj[3];
        ndel += del ? 1u : 0u;
        if constexpr (W::kMask) {
            r.dead |= (uint64_t)(del ? 1u : 0u) << id;
        } else {
            reinterpret_cast<uint8_t *>(&w->face[id].px)[3] =
                (uint8_t)((f.px >> 24) | (del ? kDeadBit >> 24 : 0u));
        }
        ended = !del & (depth == 0u);
        const uint32_t pushed = walk_entry<W>(f, opp);
        w->stk[del ? depth : (uint32_t)W::kK] = (E)pushed;
        cur = del ? walk_entry<W>(f, k1) : top;
        top = del ? pushed : below;
        depth += del ? 1u : ~0u;
        if (ended | (ns >= (uint32_t)W::kS) | (del & (depth >= (uint32_t)W::kK)) |
            (ndel > (uint32_t)W::kS))
            break;
    }
    const bool room = ended;  // not out of a buffer
    if (room && ns == 0) return EPA_NONE;
    // Room for the new faces: at most one per silhouette edge.
    const uint32_t first_new = r.nf;
    if (!room || first_new + ns > (uint32_t)W::kF || r.nl + ns > (uint32_t)W::kL + ndel) {
        if constexpr (W::kMask) {
            r.dead = dead0;
        } else {
            for (uint32_t k = 0; k < ndel; ++k) w->face[w->live[w->dl[k]]].px &= ~kDeadBit;
            lds_order();
        }
        return EPA_OVERFLOW;
    }
    w->pops[r.niter] = (I)fid;
    w->nfs[r.niter] = (I)first_new;
    ++r.nv;
    r.best_id = best_t;
    r.max_dist = max_t;
    r.old_dist = curr_dist;
    lds_order();
    // The new faces (epa3.rs:598-626), G silhouette edges at a time, one per
    // lane.  The edges whose face is still live get consecutive ids in
    // silhouette order (a ballot gives each its rank), and each lane builds its
    // edge's face (Face::new reads vertex positions only, and each edge rewrites
    // its own adjacency slot).  Parry's loop returns at the first new face that
    // ends EPA, whose heap pushes before that would be discarded anyway.
    const uint64_t lower = (1ull << sub) - 1ull;
    uint32_t n_alive = 0;
    for (uint32_t c0 = 0; c0 < ns; c0 += G) {
        const uint32_t q = c0 + sub;
        uint32_t e = 0, ex = 0;
        bool alive = false;
        if (q < ns) {
            e = w->sil[q];
            ex = w->face[e & kIdMask].px;
            alive = !face_dead(w, r, e & kIdMask, ex);
        }
        const uint64_t am = group_ballot<G>(alive);
        const uint32_t new_id = first_new + n_alive + (uint32_t)__popcll(am & lower);
        bool in = false;
        float dist = 0.0f;
        if (alive) {
            const uint32_t ef = e & kIdMask, opp = e >> W::kShift;
            const uint32_t k1 = opp == 0u ? 2u : opp - 1u, k2 = opp == 2u ? 0u : opp + 1u;
            const uint32_t nth = new_id - first_new;
            const uint32_t place = nth < ndel ? (uint32_t)w->dl[nth] : r.nl + (nth - ndel);
            f3 n, pa;
            in = lazy_face(w, new_id, pt_at(ex, k1), pt_at(ex, k2), sp, ef, new_id + 1, new_id - 1, place, n, pa);
            w->face[ef].adj[k2] = (I)new_id;
            if (in) dist = dot3(n, pa);
            set_normal(w, new_id, place, n, in ? -dist : -INFINITY);
        }
        n_alive += (uint32_t)__popcll(am);
        const bool closer = in && dist < curr_dist;
        const uint64_t stop_m = group_ballot<G>(closer || (in && -dist > kEpsTol));
        if (stop_m != 0ull) {
            if ((group_ballot<G>(closer) >> __builtin_ctzll(stop_m)) & 1ull) {
                r.best_id = fid;  // the popped face is the answer
                return EPA_OK;
            }
            return EPA_NONE;  // FaceId::new -> None
        }
        if (group_ballot<G>(in && !(fabsf(dist) <= kFltMax)) != 0ull) return EPA_RESTART;
    }
    lds_order();
    r.nf = first_new + n_alive;
    r.nl += n_alive > ndel ? n_alive - ndel : 0u;
    for (uint32_t k = n_alive; k < ndel; ++k) w->nk[w->dl[k]][3] = -INFINITY;  // places no new face took
    if (first_new == r.nf) return EPA_NONE;
    w->face[first_new].adj[2] = (I)(r.nf - 1);
    w->face[r.nf - 1].adj[1] = (I)first_new;
    lds_order();
    ++r.niter;
    return r.niter > 100 ? EPA_OK : EPA_RUNNING;  // parry's iteration cap
}

// Writes the result of a queued pair's EPA (one lane per pair): the contact, or
// the pair's entry in the next tier's list if it moves on.
__device__ void epa_finish(const ShapeRecord *rec, const float4 *verts, const float *poses, float prediction,
                           const EpaItem *it, uint32_t st, f3 p1, f3 p2, f3 n, uint32_t ei, uint32_t cont,
                           DevContact *out, uint32_t *iters, uint32_t *overflow_list, uint32_t *overflow_cont,
                           uint32_t *overflow_count, uint32_t slot) {
    const uint32_t k = it->pair;
    if (st == EPA_OVERFLOW) {
        if (overflow_list) {
            const uint32_t pos = atomicAdd(overflow_count, 1u);
            overflow_list[pos] = slot;
            if (overflow_cont) overflow_cont[pos] = cont;
        } else {
            out[k] = no_contact(kUnsupportedPair);  // cannot happen with the large buffers
        }
        return;
    }
    const uint32_t i = it->i, j = it->j;
    const iso pos1 = load_iso(poses + 7 * (size_t)i), pos2 = load_iso(poses + 7 * (size_t)j);
    const iso pos12 = iso_inv_mul(pos1, pos2);
    const uint32_t mode = item_mode(it);
    if (is_ball_mode(mode)) {
        // the Ball-vs-convex contact from the projection of the ball centre
        const iso pb = mode == kBallFirst ? iso_inverse(pos12) : pos12;
        const float radius = rec[mode == kBallFirst ? i : j].param[0];
        const PointProj proj{true, st == EPA_OK ? p1 : pb.t};
        finish_ball_contact(pos1, pos2, pb, radius, prediction, proj, false, f3{0.0f, 0.0f, 0.0f}, mode, out + k);
    } else if (st == EPA_OK) {
        finish_contact(pos1, pos2, pos12, p1, p2, n, is_local_mode(mode), out + k);
    } else {
        out[k] = no_contact(0);  // EPA failed: NoIntersection (contact_support_map_support_map.rs:75-76)
        if (mode == kPairFeatureMaps) out[k].n1[0] = 1.0f;  // ... of Vector::x_axis()
    }
    if (iters) iters[2 * k + 1] = ei;
}

// One EPA tier: what it reads and where it sends the pairs that outgrow it.
struct TierArgs {
    const ShapeRecord *rec;
    const float4 *verts;
    const float *poses;
    float prediction;
    const EpaItem *queue;
    const uint32_t *in_list;  // null: the queue itself
    const uint32_t *in_count;
    uint32_t *next;
    const uint32_t *in_cont;
    DevContact *out;
    uint32_t *iters;
    uint32_t *out_list;
    uint32_t *out_cont;
    uint32_t *out_count;
    float *orig;
};

// Each trip through the loop is one EPA iteration of every running group.  Groups
// that are done wait until half of the wave's groups are (or none runs): then the
// wave writes their contacts and sets up their next pairs together, so the
// memory latency of both (about 14,000 cycles, a third of an iteration's trip
// when it was paid whenever one group finished) is paid once for all of them.
// Measured on 2^20 mixed pairs, whole call, with 8 groups per wave: a turn-over
// at 2 waiting groups 3.82 ms, 3 3.78, 4 3.77, 6 3.81, 8 3.80.  A wave reserves
// list entries from the tier's counter in chunks (one atomic's latency per chunk)
// and hands them to the
// waiting groups by rank; the turn-over is wave-uniform, so the ballot, lane 0's
// atomic and the readfirstlane run converged.  Everything else is group-uniform,
// and the cross-lane operations of the EPA code stay within a group.
//
// The first tier is bound by instruction issue (counters on 2^20 mixed pairs: VALU
// busy 80% of the kernel's SIMD cycles, half of the lanes enabled, ten waves per CU; the
// second 53%), the third by its longest pairs' chains of about 17,000
// cycles per iteration (12%).  4 lanes per pair in the first tier measured 4.18 ms on
// the mixed pairs against 3.37 with 8 and 3.9 with 16 (the lanes of a wave take
// the longest walk of its pairs); the second tier with 8 lanes 3.56 against 3.32
// with 16.
template <int G, class W, class RI, class RO, int MINW>
__global__ __launch_bounds__(64, MINW) void epa_lazy_kernel(TierArgs t, const RI *recs, RecSink<RO> sink) {
    constexpr uint32_t kGroups = 64 / G;
    constexpr uint32_t kTurnover = kGroups > 2 ? kGroups / 2 : 1;
    __shared__ W w[kGroups];
    const uint32_t group = threadIdx.x / G;
    const uint32_t sub = __lane_id() % G;
    W *const wg = &w[group];
    float *orig = t.orig + (size_t)(blockIdx.x * kGroups + group) * W::kV * kOrigFloats;
    const uint32_t count = __hip_atomic_load(t.in_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // As many waves as pairs are enough; the others, and an empty tier, would wait for an
    // atomic: updates of 60 manifolds without an overlap 46.5 us (42 without this wait).
    if (blockIdx.x >= count) return;
    uint32_t chunk = count / (gridDim.x * 8u);  // the last chunks are an eighth of a wave's share at most
    chunk = chunk < 1u ? 1u : (chunk > 32u ? 32u : chunk);
    uint32_t at = 0, end = 0;  // the wave's reserved entries
    bool busy = false, drained = false;
    uint32_t slot = 0, status = EPA_OK;
    EpaProblem pr{};
    Staged st{nullptr, nullptr};
    LazyRegs r{};
    for (;;) {
        // group-uniform: running a pair, or waiting for the next turn-over
        const bool running = status == EPA_RUNNING;
        const uint64_t wait = __ballot(!running && !drained && sub == 0);
        const uint32_t n = (uint32_t)__popcll(wait);
        if (n >= kTurnover || __ballot(running) == 0ull) {  // wave-uniform
            if (!running && !drained && busy) {
                uint32_t cont = kNoCont, ei = 0;
                f3 p1{0.0f, 0.0f, 0.0f}, p2{0.0f, 0.0f, 0.0f}, nn{0.0f, 1.0f, 0.0f};
                if constexpr (sizeof(typename W::Idx) == 1) {
                    if (status == EPA_OVERFLOW) cont = lazy_export<G>(wg, orig, sink, r);
                }
                if (sub == 0) {
                    if (status == EPA_OK) {
                        lazy_points(wg, orig, r.best_id, p1, p2, nn);
                        ei = r.niter + 1;
                    }
                    const uint32_t done = status == EPA_POINT ? EPA_OK : (status == EPA_RESTART ? EPA_OVERFLOW : status);
                    epa_finish(t.rec, t.verts, t.poses, t.prediction, t.queue + slot, done, p1, p2, nn, ei, cont, t.out,
                               t.iters, t.out_list, t.out_cont, t.out_count, slot);
                }
            }
            if (n == 0) break;  // nothing runs and every group has seen the end of the list
            const uint32_t left = end - at;
            uint32_t more = 0;
            if (left < n) {
                const uint32_t take = chunk > n - left ? chunk : n - left;
                if (__lane_id() == 0) more = atomicAdd(t.next, take);
                more = __builtin_amdgcn_readfirstlane(more);
                end = more + take;
            }
            const uint32_t rank = (uint32_t)__popcll(wait & ((1ull << (group * G)) - 1ull));
            const uint32_t q = rank < left ? at + rank : more + (rank - left);
            at = left < n ? more + (n - left) : at + n;
            if (!running && !drained) {
                if (q >= count) {
                    drained = true;
                } else {
                    slot = t.in_list ? t.in_list[q] : q;
                    const uint32_t ci = t.in_cont ? t.in_cont[q] : kNoCont;
                    const EpaItem *it = t.queue + slot;
                    pr = epa_problem(t.rec, t.verts, t.poses, it);
                    status = lazy_begin<G>(wg, orig, pr, it, ci != kNoCont ? recs + ci : nullptr, st, r);
                    busy = true;
                }
            }
        }
        if (status == EPA_RUNNING) status = lazy_step<G>(wg, orig, pr, st, r);
    }
}

// First tier: LDS for ten waves per CU, deleted flags in registers.  1,888 bytes per
// polytope: an odd multiple of 32 puts a wave's eight polytopes on different LDS banks
// (with 1,920 bytes 2^20 mixed pairs took 3.07 ms, with 1,888 3.05).  Its polytopes move on to the second tier (four pairs per wave,
// eight waves per CU: kWideGroups), those to the third (one wave per pair, seven waves per CU, room
// for parry's 100 iterations).  A closed polytope of V vertices has 2 V - 4 faces:
// that many places and a few more; one that needs more moves on as well.
using LazySmall = LazyState<20, 60, 16, 20, uint8_t, 0, 37>;
using LazyWide = LazyState<36, 132, 36, 64, uint8_t, 0, 70>;
using LazyWave = LazyState<112, 760, 128, 256, uint16_t, 64, 208>;
using SmallRec = EpaRec<LazySmall::kV, LazySmall::kF>;
using WideRec = EpaRec<LazyWide::kV, LazyWide::kF>;

// ---------------------------------------------------------------------------
// Stage 3: EPA with parry's heap, one wave per pair
// ---------------------------------------------------------------------------
// For the pairs whose polytope outgrows the third tier (more than 760 faces) and
// those with a NaN or infinite face key: the heap itself, 2048 faces in LDS, then
// 8192 in global memory.
template <class I> struct EpaFaceT {
    I pts[3];
    I adj[3];
    uint8_t deleted;
    float n[3];
};

template <int V, int F, int H, int S, int K, class I, int SV> struct EpaState {
    static constexpr int kV = V, kF = F, kH = H, kS = S, kK = K, kSV = SV;
    using Idx = I;
    using Face = EpaFaceT<I>;
    float vp[V][3];
    Face face[F];
    I heap_id[H];
    float heap_nd[H];
    uint32_t sil[S];  // face | opp << 16
    uint32_t stk[K];  // face | opp << 16
    uint8_t vis[F];   // per face: can_be_seen_by the newest vertex, one bit per opposite vertex
    float sv[2][SV > 0 ? SV : 1][3];  // both ConvexPolyhedra's vertices (local frames), if SV > 0
};
using EpaBig = EpaState<112, 2048, 2048, 128, 2048, uint16_t, 64>;
using EpaLarge = EpaState<112, 8192, 8192, 2048, 8192, uint16_t, 0>;

// BinaryHeap<FaceId> (max-heap on neg_dist; equal keys compare Equal), with
// std's sift_up / sift_down_to_bottom so equal keys pop in parry's order.
template <class W> struct Heap {
    W *w;
    uint32_t len;
    __device__ int cmp(float a, float b) const { return a < b ? -1 : (a > b ? 1 : 0); }
    __device__ uint32_t sift_up(uint32_t start, uint32_t pos) {
        const uint32_t eid = w->heap_id[pos];
        const float end = w->heap_nd[pos];
        while (pos > start) {
            const uint32_t parent = (pos - 1) / 2;
            if (cmp(end, w->heap_nd[parent]) <= 0) break;
            w->heap_id[pos] = w->heap_id[parent];
            w->heap_nd[pos] = w->heap_nd[parent];
            pos = parent;
        }
        w->heap_id[pos] = (typename W::Idx)eid;
        w->heap_nd[pos] = end;
        return pos;
    }
    // Places an element at position pos (the heap's current end plus the pushes
    // before it) and sifts it up; the caller advances len.
    __device__ void insert_at(uint32_t pos, uint32_t id, float nd) {
        w->heap_id[pos] = (typename W::Idx)id;
        w->heap_nd[pos] = nd;
        sift_up(0, pos);
    }
    __device__ bool push(uint32_t id, float nd) {
        if (len >= (uint32_t)W::kH) return false;
        w->heap_id[len] = (typename W::Idx)id;
        w->heap_nd[len] = nd;
        ++len;
        sift_up(0, len - 1);
        return true;
    }
    __device__ void sift_down_to_bottom(uint32_t pos) {
        const uint32_t end = len, start = pos;
        const uint32_t eid = w->heap_id[pos];
        const float end_nd = w->heap_nd[pos];
        uint32_t child = 2 * pos + 1;
        while (child + 2 <= end) {
            if (cmp(w->heap_nd[child], w->heap_nd[child + 1]) <= 0) child += 1;
            w->heap_id[pos] = w->heap_id[child];
            w->heap_nd[pos] = w->heap_nd[child];
            pos = child;
            child = 2 * pos + 1;
        }
        if (child == end - 1) {
            w->heap_id[pos] = w->heap_id[child];
            w->heap_nd[pos] = w->heap_nd[child];
            pos = child;
        }
        w->heap_id[pos] = (typename W::Idx)eid;
        w->heap_nd[pos] = end_nd;
        sift_up(start, pos);
    }
    __device__ bool pop(uint32_t &id, float &nd) {
        if (len == 0) return false;
        --len;
        uint32_t iid = w->heap_id[len];
        float ind = w->heap_nd[len];
        if (len > 0) {
            const uint32_t t_id = w->heap_id[0];
            const float t_nd = w->heap_nd[0];
            w->heap_id[0] = (typename W::Idx)iid;
            w->heap_nd[0] = ind;
            iid = t_id;
            ind = t_nd;
            sift_down_to_bottom(0);
        }
        id = iid;
        nd = ind;
        return true;
    }
};

// Face::new: fills face f; returns proj_inside.
template <class W>
__device__ bool face_new(W *w, uint32_t f, uint32_t a, uint32_t b, uint32_t c, uint32_t j0, uint32_t j1, uint32_t j2) {
    using I = typename W::Idx;
    typename W::Face &F = w->face[f];
    F.pts[0] = (I)a; F.pts[1] = (I)b; F.pts[2] = (I)c;
    F.adj[0] = (I)j0; F.adj[1] = (I)j1; F.adj[2] = (I)j2;
    F.deleted = 0;
    const f3 pa = vpt(w, a), pb = vpt(w, b), pc = vpt(w, c);
    float bc[3];
    const bool in = face_bcoords(pa, pb, pc, bc);
    const f3 n = ccw_normal(pa, pb, pc);
    F.n[0] = n.x; F.n[1] = n.y; F.n[2] = n.z;
    return in;
}

template <class W> __device__ __forceinline__ f3 fnormal(const W *w, uint32_t f) {
    return f3{w->face[f].n[0], w->face[f].n[1], w->face[f].n[2]};
}

// Face::closest_points (epa3.rs:120-130).
template <class W> __device__ void face_points(const W *w, const float *orig, uint32_t f, f3 &p1, f3 &p2) {
    const typename W::Face &F = w->face[f];
    float bc[3];
    face_bcoords(vpt(w, F.pts[0]), vpt(w, F.pts[1]), vpt(w, F.pts[2]), bc);
    f3 o1[3], o2[3];
    for (int q = 0; q < 3; ++q) {
        const float *o = orig + kOrigFloats * F.pts[q];
        o1[q] = f3{o[0], o[1], o[2]};
        o2[q] = f3{o[3], o[4], o[5]};
    }
    p1 = add3(add3(mul3(o1[0], bc[0]), mul3(o1[1], bc[1])), mul3(o1[2], bc[2]));
    p2 = add3(add3(mul3(o2[0], bc[0]), mul3(o2[1], bc[1])), mul3(o2[2], bc[2]));
}

// Element k (0, 1 or 2) of three values, by selects rather than an indexed array.
__device__ __forceinline__ uint32_t pick3(uint32_t k, uint32_t a, uint32_t b, uint32_t c) {
    return k == 0 ? a : (k == 1 ? b : c);
}

// Face::next_ccw_pt_id (epa3.rs:135-151) on a face record held in registers.
template <class Fc> __device__ __forceinline__ uint32_t ccw_index(const Fc &f, uint32_t id) {
    if (f.pts[0] == id) return 1;
    if (f.pts[1] == id) return 2;
    return 0;
}

template <class W> __device__ __forceinline__ uint32_t next_ccw(const W *w, uint32_t f, uint32_t id) {
    if (w->face[f].pts[0] == id) return 1;
    if (w->face[f].pts[1] == id) return 2;
    return 0;
}

template <class W> struct EpaRegs {
    Heap<W> heap;  // the polytope's face heap (LDS) and its length
    uint32_t nv, nf, best_id, niter;
    float max_dist, old_dist;
};

// The set-up before EPA's first iteration: the polytope from the GJK simplex.
// Returns EPA_RUNNING, or the result if EPA ends here.
template <int G, class W>
__device__ uint32_t epa_begin(W *w, float *orig, const iso &pos12, const ShapeRef &g1, const ShapeRef &g2,
                              const EpaItem *it, Staged &st, EpaRegs<W> &r, f3 &p1, f3 &p2, f3 &n,
                              uint32_t &epa_iters) {
    st = Staged{stage_shape<G>(w, 0, g1), stage_shape<G>(w, 1, g2)};
    // The group's lanes wrote the staged vertices; make them visible to the
    // whole wave before any lane reads another lane's entries.
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    r = EpaRegs<W>{Heap<W>{w, 0}, 0, 0, 0, 0, kFltMax, 0.0f};
    Heap<W> &heap = r.heap;
    uint32_t &nv = r.nv, &nf = r.nf, &best_id = r.best_id;
    epa_iters = 0;
    {
        const uint32_t dim = it->dim_mode & 0xffu;
        for (uint32_t i = 0; i <= dim; ++i) {
            w->vp[i][0] = it->v[i][0];
            w->vp[i][1] = it->v[i][1];
            w->vp[i][2] = it->v[i][2];
            for (int q = 0; q < 6; ++q) orig[kOrigFloats * i + q] = it->v[i][3 + q];
        }
        nv = dim + 1;
        if (dim == 0) {
            p1 = p2 = f3{0.0f, 0.0f, 0.0f};
            n = f3{0.0f, 1.0f, 0.0f};
            return EPA_OK;
        } else if (dim == 3) {
            const f3 dp1 = sub3(vpt(w, 1), vpt(w, 0));
            const f3 dp2 = sub3(vpt(w, 2), vpt(w, 0));
            const f3 dp3 = sub3(vpt(w, 3), vpt(w, 0));
            if (dot3(cross3(dp1, dp2), dp3) > 0.0f) {
                for (int q = 0; q < 3; ++q) {
                    const float t = w->vp[1][q];
                    w->vp[1][q] = w->vp[2][q];
                    w->vp[2][q] = t;
                }
                for (int q = 0; q < 6; ++q) {
                    const float t = orig[kOrigFloats * 1 + q];
                    orig[kOrigFloats * 1 + q] = orig[kOrigFloats * 2 + q];
                    orig[kOrigFloats * 2 + q] = t;
                }
            }
            const bool in0 = face_new(w, 0, 0, 1, 2, 3, 1, 2);
            const bool in1 = face_new(w, 1, 1, 3, 2, 3, 2, 0);
            const bool in2 = face_new(w, 2, 0, 2, 3, 0, 1, 3);
            const bool in3 = face_new(w, 3, 0, 3, 1, 2, 1, 0);
            nf = 4;
            const bool ins[4] = {in0, in1, in2, in3};
    #pragma unroll
            for (uint32_t f = 0; f < 4; ++f) {
                if (ins[f]) {
                    const float dist = dot3(fnormal(w, f), vpt(w, f));
                    if (-dist > kEpsTol) return EPA_NONE;  // FaceId::new -> None
                    heap.push(f, -dist);
                }
            }
            if (!(in0 || in1 || in2 || in3)) return EPA_NONE;
        } else {
            if (dim == 1) {
                // orthonormal_subspace_basis([dpt]): first vector a x dpt
                const f3 dpt = sub3(vpt(w, 1), vpt(w, 0));
                f3 a = fabsf(dpt.x) > fabsf(dpt.y) ? f3{dpt.z, 0.0f, -dpt.x} : f3{0.0f, -dpt.z, dpt.y};
                a = div3(a, sqrtf(norm_sq3(a)));
                vset(w, orig, 2, group_cso<G, (W::kSV > 0)>(pos12, g1, g2, st, cross3(a, dpt)));
                nv = 3;
            }
            face_new(w, 0, 0, 1, 2, 1, 1, 1);
            face_new(w, 1, 0, 2, 1, 0, 0, 0);
            nf = 2;
            heap.push(0, 0.0f);
            heap.push(1, 0.0f);
        }
        if (heap.len == 0) return EPA_NONE;
        best_id = w->heap_id[0];
    }
    return EPA_RUNNING;
}

// One EPA iteration (the body of the loop of epa3.rs:499-647).  Returns
// EPA_RUNNING while EPA goes on, else the result.
template <int G, class W>
__device__ uint32_t epa_step(W *w, float *orig, const iso &pos12, const ShapeRef &g1, const ShapeRef &g2,
                             const Staged &st, EpaRegs<W> &r, f3 &p1, f3 &p2, f3 &n, uint32_t &epa_iters) {
    const float eps_tol = kEps * 100.0f;
    Heap<W> &heap = r.heap;
    uint32_t &nv = r.nv, &nf = r.nf, &best_id = r.best_id, &niter = r.niter;
    float &max_dist = r.max_dist, &old_dist = r.old_dist;
    // parry's loop ends when the heap is empty or after 100 iterations
    auto done = [&]() -> uint32_t {
        epa_iters = niter + 1;
        face_points(w, orig, best_id, p1, p2);
        n = fnormal(w, best_id);
        return EPA_OK;
    };
    // Faces deleted since they were pushed are popped and skipped here, as
    // parry's loop skips them (`continue`), rather than one per call.
    while (heap.len > 0 && w->face[w->heap_id[0]].deleted) {
        uint32_t pid;
        float pnd;
        heap.pop(pid, pnd);
    }
    if (heap.len == 0) return done();
    {
        const uint32_t fid = w->heap_id[0];
        const float fnd = w->heap_nd[0];
        const typename W::Face face = w->face[fid];
        const f3 fn = f3{face.n[0], face.n[1], face.n[2]};
        const Cso c = group_cso<G, (W::kSV > 0)>(pos12, g1, g2, st, fn);
        if (nv >= (uint32_t)W::kV) return EPA_OVERFLOW;
        const uint32_t sp = nv;  // counted when the iteration commits
        vset(w, orig, sp, c);
        const float cand = dot3(c.p, fn);
        uint32_t best_t = best_id;
        float max_t = max_dist;
        if (cand < max_t) {
            best_t = fid;
            max_t = cand;
        }
        const float curr_dist = -fnd;
        if (max_t - curr_dist < eps_tol || (fabsf(curr_dist - old_dist) < kEps && cand < max_t)) {
            face_points(w, orig, best_t, p1, p2);
            n = fnormal(w, best_t);
            epa_iters = niter + 1;
            return EPA_OK;
        }
        w->face[fid].deleted = 1;
        // Face::can_be_seen_by (epa3.rs:153-166) of every live face from the new
        // vertex, for each of the three opposite vertices, by the group's lanes in
        // parallel; the depth-first walk below only reads the bits.
        {
            const uint32_t sub = __lane_id() % G;
            const f3 pt = vpt(w, sp);
            const float E = kEps * 100.0f;
            // Deleted faces get bits too (the walk never reads them): with no
            // branch in the body, the loads of consecutive faces overlap.
#pragma unroll 2
            for (uint32_t f = sub; f < nf; f += G) {
                const typename W::Face F = w->face[f];
                const f3 q0 = vpt(w, F.pts[0]), q1 = vpt(w, F.pts[1]), q2 = vpt(w, F.pts[2]);
                const f3 fnn = f3{F.n[0], F.n[1], F.n[2]};
                const f3 qs[3] = {q0, q1, q2};
                uint32_t bits = 0;
#pragma unroll
                for (int opp = 0; opp < 3; ++opp) {
                    const f3 p0 = qs[opp], p1 = qs[(opp + 1) % 3], p2 = qs[(opp + 2) % 3];
                    const bool front = dot3(sub3(pt, p0), fnn) >= -kEpsTol;
                    const bool flat = norm_sq3(cross3(sub3(p2, p1), sub3(pt, p1))) <= E * E;  // is_affinely_dependent
                    bits |= (uint32_t)(front | flat) << opp;
                }
                w->vis[f] = (uint8_t)bits;
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        // compute_silhouette (epa3.rs:653-675) for the three neighbours in order
        // adj[0], adj[1], adj[2]; a visible face recurses into adj[(opp + 2) % 3],
        // then adj[opp].  The recursion is an explicit stack of face | opp << 16
        // whose top entry lives in a register.  After a visible face, the face
        // visited next (its first far neighbour) is loaded together with the
        // second one's points and carried in registers, so a step costs one
        // round trip to LDS. 
        uint32_t ns = 0, sk = 0, depth = 0, top = 0;
        typename W::Face cf = w->face[face.adj[0]];
        uint32_t cvis = w->vis[face.adj[0]];
        uint32_t cur = face.adj[0] | (ccw_index(cf, face.pts[0]) << 16);
        {
            const uint32_t o2 = next_ccw(w, face.adj[2], face.pts[2]);
            const uint32_t o1 = next_ccw(w, face.adj[1], face.pts[1]);
            w->stk[0] = face.adj[2] | (o2 << 16);
            top = face.adj[1] | (o1 << 16);
            sk = 1;
            depth = 2;
        }
        // One latch: both ways on (into a deleted face's first far neighbour, or
        // back to the stack's top) end in the same read of the next face.  With
        // the stack path as a separate branch the compiler split the walk into
        // nested loops, and a wave's groups that had to pop waited for the others.
        for (;;) {
            const uint32_t id = cur & 0xffffu, opp = cur >> 16;
            const bool del = !cf.deleted && ((cvis >> opp) & 1u);
            if (!cf.deleted && !del) {
                if (ns >= (uint32_t)W::kS) return EPA_OVERFLOW;
                w->sil[ns++] = cur;
            }
            if (!del && depth == 0) break;
            uint32_t nid, pt1 = 0, popped = 0;
            if (del) {
                w->face[id].deleted = 1;
                // a1 = (opp + 2) % 3 and a2 = opp, selected by value so the
                // record stays in registers
                const uint32_t adj1 = pick3(opp, cf.adj[2], cf.adj[0], cf.adj[1]);
                const uint32_t adj2 = pick3(opp, cf.adj[0], cf.adj[1], cf.adj[2]);
                pt1 = pick3(opp, cf.pts[2], cf.pts[0], cf.pts[1]);
                const uint32_t pt2 = pick3(opp, cf.pts[0], cf.pts[1], cf.pts[2]);
                const uint32_t o2 = next_ccw(w, adj2, pt2);
                if (depth > 0) {
                    if (sk >= (uint32_t)W::kK) return EPA_OVERFLOW;
                    w->stk[sk++] = top;
                }
                top = adj2 | (o2 << 16);
                ++depth;
                nid = adj1;
            } else {
                popped = top;
                nid = top & 0xffffu;
                --depth;
                const uint32_t below = w->stk[sk != 0u ? sk - 1u : 0u];  // slot 0 always exists
                if (depth > 0) {
                    top = below;
                    --sk;
                }
            }
            const typename W::Face f = w->face[nid];
            cvis = w->vis[nid];
            cur = del ? (nid | (ccw_index(f, pt1) << 16)) : popped;
            cf = f;
            if (del && nid == id) cf.deleted = 1;  // a face adjacent to itself (degenerate ring)
        }
        const uint32_t first_new = nf;
        if (ns == 0) return EPA_NONE;
        const uint32_t sub = __lane_id() % G;
        const uint32_t gbase = __lane_id() - sub;
        const uint64_t gmask = G >= 64 ? ~0ull : ((1ull << (G & 63)) - 1ull);
        const uint64_t below = (1ull << sub) - 1ull;
        // Room for the new faces and their heap entries (at most one per live
        // silhouette edge), checked before anything is committed.
        uint32_t n_live = 0;
        for (uint32_t c0 = 0; c0 < ns; c0 += G) {
            const uint32_t q = c0 + sub;
            const bool alive = q < ns && !w->face[w->sil[q] & 0xffffu].deleted;
            n_live += (uint32_t)__popcll((__ballot(alive) >> gbase) & gmask);
        }
        if (first_new + n_live > (uint32_t)W::kF || heap.len - 1 + n_live > (uint32_t)W::kH)
            return EPA_OVERFLOW;
        // Commit: parry popped this face before all of the above.
        {
            uint32_t pid;
            float pnd;
            heap.pop(pid, pnd);
        }
        ++nv;
        best_id = best_t;
        max_dist = max_t;
        old_dist = curr_dist;
        // The new faces (epa3.rs:598-626), G silhouette edges at a time, one per
        // lane.  The edges whose face is still live get consecutive ids in
        // silhouette order (a ballot gives each its rank), and each lane builds
        // its edge's face (Face::new reads vertex positions only, and each edge
        // rewrites its own adjacency slot).  Parry's loop then either returns at
        // the first new face that ends EPA -- its heap pushes before that would
        // be discarded anyway -- or pushes every new face in silhouette order;
        // the lane holding an edge's face does that edge's push.
        uint32_t n_alive = 0;
        for (uint32_t c0 = 0; c0 < ns; c0 += G) {
            const uint32_t q = c0 + sub;
            uint32_t e = 0;
            bool alive = false;
            if (q < ns) {
                e = w->sil[q];
                alive = !w->face[e & 0xffffu].deleted;
            }
            const uint64_t am = (__ballot(alive) >> gbase) & gmask;
            const uint32_t new_id = first_new + n_alive + (uint32_t)__popcll(am & below);
            bool in = false;
            float dist = 0.0f;
            if (alive) {
                const uint32_t ef = e & 0xffffu, opp = e >> 16;
                const uint32_t pt1 = w->face[ef].pts[(opp + 2) % 3];
                const uint32_t pt2 = w->face[ef].pts[(opp + 1) % 3];
                in = face_new(w, new_id, pt1, pt2, sp, ef, new_id + 1, new_id - 1);
                w->face[ef].adj[(opp + 1) % 3] = (typename W::Idx)new_id;
                if (in) dist = dot3(fnormal(w, new_id), vpt(w, pt1));
            }
            n_alive += (uint32_t)__popcll(am);
            const bool pushed = alive && in;
            const bool closer = pushed && dist < curr_dist;
            const bool stop = closer || (pushed && -dist > kEpsTol);
            const uint64_t stop_m = (__ballot(stop) >> gbase) & gmask;
            const uint64_t closer_m = (__ballot(closer) >> gbase) & gmask;
            if (stop_m != 0) {
                if ((closer_m >> __builtin_ctzll(stop_m)) & 1ull) {
                    face_points(w, orig, fid, p1, p2);  // the popped face: its points are unchanged
                    n = fn;
                    epa_iters = niter + 1;
                    return EPA_OK;
                }
                return EPA_NONE;  // FaceId::new -> None
            }
            const uint64_t push_m = (__ballot(pushed) >> gbase) & gmask;
            for (uint64_t m = push_m; m != 0; m &= m - 1) {
                if (sub == (uint32_t)__builtin_ctzll(m))
                    heap.insert_at(heap.len + (uint32_t)__popcll(push_m & below), new_id, -dist);
            }
            heap.len += (uint32_t)__popcll(push_m);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        nf = first_new + n_alive;
        if (first_new == nf) return EPA_NONE;
        w->face[first_new].adj[2] = (typename W::Idx)(nf - 1);
        w->face[nf - 1].adj[1] = (typename W::Idx)first_new;
        ++niter;
        if (niter > 100) return done();
    }
    return EPA_RUNNING;
}


// A tier of this stage: a wave per pair, the next pair from the tier's counter.
// P: the wave's polytope, in LDS or global memory.
template <class W>
__device__ void epa_wave_loop(const TierArgs &t, W *w, float *orig) {
    const uint32_t count = __hip_atomic_load(t.in_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (blockIdx.x >= count) return;
    for (;;) {
        uint32_t q = 0;
        if (__lane_id() == 0) q = atomicAdd(t.next, 1u);
        q = __builtin_amdgcn_readfirstlane(q);
        if (q >= count) break;
        const uint32_t slot = t.in_list[q];
        const EpaItem *it = t.queue + slot;
        const EpaProblem pr = epa_problem(t.rec, t.verts, t.poses, it);
        f3 p1, p2, n;
        uint32_t ei = 0;
        Staged st;
        EpaRegs<W> r;
        uint32_t s = epa_begin<64>(w, orig, pr.pos, pr.a, pr.b, it, st, r, p1, p2, n, ei);
        while (s == EPA_RUNNING) s = epa_step<64>(w, orig, pr.pos, pr.a, pr.b, st, r, p1, p2, n, ei);
        if (__lane_id() == 0)
            epa_finish(t.rec, t.verts, t.poses, t.prediction, it, s, p1, p2, n, ei, kNoCont, t.out, t.iters, t.out_list,
                       nullptr, t.out_count, slot);
    }
}
__global__ __launch_bounds__(64) void epa_big_kernel(TierArgs t) {
    __shared__ EpaBig w;
    epa_wave_loop(t, &w, t.orig + (size_t)blockIdx.x * EpaBig::kV * kOrigFloats);
}
__global__ __launch_bounds__(64) void epa_global_kernel(TierArgs t, EpaLarge *scratch) {
    epa_wave_loop(t, scratch + blockIdx.x, t.orig + (size_t)blockIdx.x * EpaLarge::kV * kOrigFloats);
}

// Waves that fill the current device with a kernel of 64-lane workgroups.
hipError_t resident_waves(const void *kernel, uint64_t *waves) {
    hipError_t e;
    int dev = 0, cus = 0, per_cu = 0;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) != hipSuccess) return e;
    if ((e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 64, 0)) != hipSuccess) return e;
    *waves = (uint64_t)cus * (uint64_t)(per_cu < 1 ? 1 : per_cu);
    return hipSuccess;
}

template <int G, class W, class RI, class RO, int MINW>
hipError_t launch_lazy(const TierArgs &t, const RI *recs, const RecSink<RO> &sink, uint64_t max_items,
                       uint64_t max_groups, hipStream_t stream) {
    constexpr uint64_t kGroups = 64 / G;
    uint64_t waves = 0;
    hipError_t e = resident_waves((const void *)epa_lazy_kernel<G, W, RI, RO, MINW>, &waves);
    if (e != hipSuccess) return e;
    const uint64_t need = (max_items + kGroups - 1) / kGroups;
    if (waves > need) waves = need;
    if (waves * kGroups > max_groups) waves = max_groups / kGroups;
    if (waves < 1) waves = 1;
    hipLaunchKernelGGL((epa_lazy_kernel<G, W, RI, RO, MINW>), dim3((uint32_t)waves), dim3(64), 0, stream, t, recs, sink);
    return hipGetLastError();
}

}  // namespace

// Resident EPA groups the workspace provides orig1/orig2 buffers for, per tier.
constexpr uint64_t kSmallGroups = 256ull * 12 * 8;
constexpr uint64_t kWideGroups = 256ull * 8 * 4;
constexpr uint64_t kWaveGroups = 256ull * 8;
constexpr uint64_t kBigWaves = 256ull * 2;

// Calls of at most this many pairs are bound by the longest chain of iterations, not
// by instruction issue: more lanes per pair make an iteration shorter.  First tier
// with 8 lanes and second with 16, against 16 and 64: 100 mixed pairs 205 and 194 us,
// 500 493 and 435, 2,000 602 and 560, 10,000 805 and 775, 20,000 731 and 688, 32,000
// 1,126 and 1,108, 80,000 1,048 and 1,136; polyhedra 500 251 and 233, 10,000 332 and 340,
// 20,000 371 and 368, 32,000 384 and 398, 40,000 431 and 467.
constexpr uint64_t kFewPairs = 16384;

int g_epa_lanes_per_pair = 16;
int g_epa_polytope = 1;
int g_epa_schedule = 0;
bool g_contact_phase_timing = false;
hipEvent_t g_contact_phase_events[kContactPhases + 1] = {};

namespace {
struct ContactWorkspace {
    uint32_t *counters;  // list lengths and the tiers' next entries (reset_counters_kernel)
    uint32_t *bins;  // of the pair order, after the counters
    uint32_t *order;
    uint16_t *cls;
    EpaItem *queue;
    uint32_t *lists[4];
    uint32_t *cont_list[2];  // per entry of lists[0] and lists[1]: its continuation record or kNoCont
    SmallRec *small_recs;
    WideRec *wide_recs;
    uint32_t small_cap, wide_cap;
    EpaLarge *large;
    float *orig_small, *orig_wide, *orig_wave, *orig_big, *orig_large;
    size_t bytes;
};

// Whether the pairs are ordered by class: where there are enough of them to fill
// the GPU several times over (below that a call lasts as long as its longest
// pairs, in any order) and the shapes are of several types.  Measured, ordered
// and not, us a call: mixed types 1,124 and 1,126 at 32,000 pairs, 1,070 and 1,048 at
// 80,000, 1,260 and 1,272 at 128,000, 3,028 and 3,676 at 2^20; polyhedra alone 422 and
// 384 at 32,000, 704 and 648 at 128,000 (the two ordering kernels take 22 us at 131,072
// pairs and 54 at 2^20, and the broadphase's order has its own locality).
constexpr uint64_t kOrderMinPairs = 1u << 17;
bool takes_order(const DeviceShapes &s, uint64_t m) {
    return m >= kOrderMinPairs && (s.types & (s.types - 1u)) != 0u;
}

uint64_t clamp_u64(uint64_t v, uint64_t lo, uint64_t hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Continuation records: the first tier hands on about 3% of mixed-shape pairs,
// the second 0.3%.  A pair that finds them all taken restarts in the next tier.
ContactWorkspace carve_workspace(void *base, uint64_t m) {
    const size_t align = 256;
    auto up = [&](size_t b) { return (b + align - 1) / align * align; };
    char *ws = (char *)base;
    ContactWorkspace w{};
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char *p = ws ? ws + off : nullptr;
        off += up(bytes);
        return p;
    };
    w.counters = (uint32_t *)take((kNumCounters + kPairOrderBins) * sizeof(uint32_t));
    w.bins = w.counters + kNumCounters;
    const uint64_t ordered = m >= kOrderMinPairs ? m : 0;  // whatever the types: the size depends on m alone
    w.order = (uint32_t *)take(ordered * sizeof(uint32_t));
    w.cls = (uint16_t *)take(ordered * sizeof(uint16_t));
    w.queue = (EpaItem *)take(m * sizeof(EpaItem));
    for (uint32_t *&l : w.lists) l = (uint32_t *)take(m * sizeof(uint32_t));
    for (uint32_t *&l : w.cont_list) l = (uint32_t *)take(m * sizeof(uint32_t));
    w.small_cap = (uint32_t)clamp_u64(m / 16, 256, 131072);
    w.wide_cap = (uint32_t)clamp_u64(m / 128, 256, 16384);
    w.small_recs = (SmallRec *)take((size_t)w.small_cap * sizeof(SmallRec));
    w.wide_recs = (WideRec *)take((size_t)w.wide_cap * sizeof(WideRec));
    w.large = (EpaLarge *)take(kEpaGlobalWaves * sizeof(EpaLarge));
    auto orig = [&](uint64_t groups, uint64_t verts) { return (float *)take(groups * verts * kOrigFloats * sizeof(float)); };
    w.orig_small = orig(kSmallGroups, LazySmall::kV);
    w.orig_wide = orig(kWideGroups, LazyWide::kV);
    w.orig_wave = orig(kWaveGroups, LazyWave::kV);
    w.orig_big = orig(kBigWaves, EpaBig::kV);
    w.orig_large = orig(kEpaGlobalWaves, EpaLarge::kV);
    w.bytes = off;
    return w;
}

// order_count_kernel and order_scatter_kernel; `bins` zeroed.
static_assert(kPairOrderBins == 2 * kPairClasses, "totals and positions per class");
hipError_t order_pairs(const DeviceShapes &s, const uint32_t *pairs, uint64_t m, const uint64_t *m_dev, uint16_t *cls,
                       uint32_t *bins, uint32_t *order, hipStream_t stream) {
    const dim3 grid((uint32_t)((m + kOrderRange - 1) / kOrderRange));
    hipLaunchKernelGGL(order_count_kernel, grid, dim3(kOrderBlock), 0, stream, s.rec, pairs, m,
                       (const unsigned long long *)m_dev, cls, bins);
    hipLaunchKernelGGL(order_scatter_kernel, grid, dim3(kOrderBlock), 0, stream, m, (const unsigned long long *)m_dev,
                       cls, bins, bins + kPairClasses, order);
    return hipGetLastError();
}

template <int G>
hipError_t launch_small(const TierArgs &t, const RecSink<SmallRec> &sink, uint64_t m, hipStream_t stream) {
    return launch_lazy<G, LazySmall, SmallRec, SmallRec, 3>(t, nullptr, sink, m, kSmallGroups, stream);
}
}  // namespace

hipError_t launch_pair_order(const DeviceShapes &s, const uint32_t *pairs, uint64_t m, const uint64_t *m_dev,
                             uint16_t *cls, uint32_t *bins, uint32_t *order, hipStream_t stream) {
    hipLaunchKernelGGL(reset_counters_kernel, dim3(1), dim3(256), 0, stream, bins, kPairOrderBins);
    return order_pairs(s, pairs, m, m_dev, cls, bins, order, stream);
}

size_t contact_workspace_bytes(uint64_t num_pairs) { return carve_workspace(nullptr, num_pairs).bytes; }

hipError_t launch_contacts(const DeviceShapes &s, const float *poses, const uint32_t *pairs, uint64_t m,
                           const uint64_t *m_dev, float prediction, const float *seeds, pq_contact *out,
                           uint32_t *iters, void *workspace, hipStream_t stream, uint32_t flags) {
    if (m == 0) return hipSuccess;
    const ContactWorkspace w = carve_workspace(workspace, m);
    DevContact *o = (DevContact *)out;
    const bool timed = g_contact_phase_timing;
    auto mark = [&](int k) { return timed ? hipEventRecord(g_contact_phase_events[k], stream) : hipSuccess; };
    const bool ordered = !(flags & kContactInOrder) && takes_order(s, m);
    hipLaunchKernelGGL(reset_counters_kernel, dim3(1), dim3(256), 0, stream, w.counters,
                       kNumCounters + (ordered ? kPairOrderBins : 0u));
    hipError_t e = mark(0);
    if (e != hipSuccess) return e;
    if (ordered && (e = order_pairs(s, pairs, m, m_dev, w.cls, w.bins, w.order, stream)) != hipSuccess) return e;
    hipLaunchKernelGGL(contact_gjk_kernel, dim3((uint32_t)((m + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream,
                       s.rec, s.verts, poses, pairs, m, (const unsigned long long *)m_dev, prediction, seeds, o, iters,
                       w.queue, w.counters, flags, ordered ? w.order : nullptr);
    e = hipGetLastError();
    if (e == hipSuccess) e = mark(1);
    if (e != hipSuccess) return e;
    uint32_t *const c = w.counters;
    // Tier k reads list k - 1 (the queue for the first) and sends the pairs that outgrow it to list k.
    auto tier = [&](uint32_t k, float *orig) {
        return TierArgs{s.rec, s.verts, poses, prediction, w.queue, k ? w.lists[k - 1] : nullptr, c + k, c + kTiers + k,
                        k == 1 ? w.cont_list[0] : (k == 2 ? w.cont_list[1] : nullptr), o, iters,
                        k < 4 ? w.lists[k] : nullptr, k < 2 ? w.cont_list[k] : nullptr, c + k + 1, orig};
    };
    const TierArgs t0 = tier(0, w.orig_small);
    const RecSink<SmallRec> small_sink{w.small_recs, c + 10, w.small_cap};
    const bool few = m <= kFewPairs;
    // 16 lanes with schedule 0, the default, is automatic; any other setting is the caller's
    const bool automatic = g_epa_schedule == 0 && g_epa_lanes_per_pair == 16;
    const int lanes = automatic ? (few ? 16 : 8) : g_epa_lanes_per_pair;
    switch (lanes) {
        case 4: e = launch_small<4>(t0, small_sink, m, stream); break;
        case 8: e = launch_small<8>(t0, small_sink, m, stream); break;
        case 16: e = launch_small<16>(t0, small_sink, m, stream); break;
        case 32: e = launch_small<32>(t0, small_sink, m, stream); break;
        default: e = launch_small<64>(t0, small_sink, m, stream); break;
    }
    if (e != hipSuccess) return e;
    const RecSink<WideRec> wide_sink{w.wide_recs, c + 11, w.wide_cap};
    if (few)
        e = launch_lazy<64, LazyWide, SmallRec, WideRec, 3>(tier(1, w.orig_wide), w.small_recs, wide_sink, m,
                                                            kWideGroups, stream);
    else
        e = launch_lazy<16, LazyWide, SmallRec, WideRec, 3>(tier(1, w.orig_wide), w.small_recs, wide_sink, m,
                                                            kWideGroups, stream);
    if (e == hipSuccess) e = mark(2);
    if (e != hipSuccess) return e;
    e = launch_lazy<64, LazyWave, WideRec, WideRec, 1>(tier(2, w.orig_wave), w.wide_recs,
                                                       RecSink<WideRec>{nullptr, nullptr, 0}, m, kWaveGroups, stream);
    if (e == hipSuccess) e = mark(3);
    if (e != hipSuccess) return e;
    uint64_t waves = 0;
    if ((e = resident_waves((const void *)epa_big_kernel, &waves)) != hipSuccess) return e;
    waves = clamp_u64(waves, 1, kBigWaves < m ? kBigWaves : m);
    hipLaunchKernelGGL(epa_big_kernel, dim3((uint32_t)waves), dim3(64), 0, stream, tier(3, w.orig_big));
    e = hipGetLastError();
    if (e == hipSuccess) e = mark(4);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(epa_global_kernel, dim3(kEpaGlobalWaves), dim3(64), 0, stream, tier(4, w.orig_large), w.large);
    e = hipGetLastError();
    if (e == hipSuccess) e = mark(5);
    return e;
}

}  // namespace pq
