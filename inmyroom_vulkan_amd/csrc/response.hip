// Response: shooting the uncollide rays and splitting the delta
// (ShootUncollideRays::ExecuteShootUncollideRays,
//  inMyRoom_vulkan/src/CollisionDetection/ShootUncollideRays.cpp:14-179;
//  Ray::IntersectOBBtree, Ray.cpp:13-236; CollisionDetection.cpp:70-99, 143-150).
//
//  k_shoot    two lanes per uncollide ray, or four where a call's rays fill no
//             more than 16 to a wavefront (shootshape.hpp).  Pass 1 shoots the ray at the
//             other entity's tree (closest hit, even lane); it succeeds when
//             that hit is a back face reached before the ray re-enters its own
//             tree (odd lane; the Hermann pass, :129-158).  On success the ray is reflected (origin
//             moved by the response, direction minus the hit's normal,
//             :104-110) and pass 2 shoots it the other way.  Each pass's force
//             response and push-out vector are kept per ray.
//  k_respond  one wavefront per entity pair: the force responses summed,
//             FindResponse (:160-169) over the push-out vectors, the
//             world-space delta, and its split by how far each entity's
//             average contact point moved since the previous frame.
//
// The closest-hit traversal keeps an explicit stack in LDS.  At an internal
// node both children's entry/exit distances are computed, the farther child
// is pushed below the nearer, and a child is entered only if its exit
// distance is not negative and, when it is popped, its entry distance is
// below the best hit so far: the nodes visited, and the order in which equal
// distances are met, are those of the reference's recursion.
#include "rayattr.hpp"

namespace cdk {

namespace {

constexpr float FLT_EPS = 1.1920928955078125e-07f;  // std::numeric_limits<float>::epsilon()

__device__ __forceinline__ float max_std(float a, float b) { return (a < b) ? b : a; }  // std::max
__device__ __forceinline__ float min_std(float a, float b) { return (b < a) ? b : a; }  // std::min

// glm::intersectRayTriangle from the origin (glm 0.9.9's Möller-Trumbore
// form); back = the negative-determinant branch, the backface output of the
// reference's glm fork.
__device__ __forceinline__ bool ray_triangle(f3 dir, f3 v0, f3 v1, f3 v2, float& bx, float& by, float& dist,
                                             bool& back) {
    const f3 e1 = sub(v1, v0), e2 = sub(v2, v0);
    const f3 p = cross(dir, e2);
    const float det = dot(e1, p);
    const f3 d0 = sub(mk(0.f, 0.f, 0.f), v0);
    f3 perp;
    if (det > FLT_EPS) {
        bx = dot(d0, p);
        if (bx < 0.f || bx > det) return false;
        perp = cross(d0, e1);
        by = dot(dir, perp);
        if (by < 0.f || bx + by > det) return false;
        back = false;
    } else if (det < -FLT_EPS) {
        bx = dot(d0, p);
        if (bx > 0.f || bx < det) return false;
        perp = cross(d0, e1);
        by = dot(dir, perp);
        if (by > 0.f || bx + by < det) return false;
        back = true;
    } else {
        return false;
    }
    const float inv = 1.f / det;
    dist = dot(e2, perp) * inv;
    bx = bx * inv;
    by = by * inv;
    return true;
}

// The ray in a tree's own frame.  C maps the mesh's coordinates to the
// ray's frame (origin at the ray's origin), so the mesh-frame ray
// x(t) = o + t d with o = -A^-1 c, d = A^-1 dir (A, c: C's linear part and
// translation) is mapped onto t dir: a slab crossing has the same parameter t
// in both frames.  The boxes are then tested where they are stored, with no
// transform and no normalised normal per test.
struct LocalRay {
    f3 o, d;
    float on;       // |o|_1
    float kappa;    // relative rounding margin of the box tests, grown with A's condition number
    float dk;       // 4 kappa |d|_1
    bool ok;        // A invertible: else every box is entered
};
__device__ __forceinline__ float norm1f(f3 v) { return (fabsf(v.x) + fabsf(v.y)) + fabsf(v.z); }
__device__ __forceinline__ LocalRay local_ray(const M4& C, f3 dir) {
    const f3 a0 = mk(C.m[0], C.m[1], C.m[2]), a1 = mk(C.m[4], C.m[5], C.m[6]), a2 = mk(C.m[8], C.m[9], C.m[10]);
    const f3 r0 = cross(a1, a2), r1 = cross(a2, a0), r2 = cross(a0, a1);  // rows of det(A) A^-1
    const float det = dot(a0, r0);
    const float inv = 1.f / det;
    const f3 c = mk(C.m[12], C.m[13], C.m[14]);
    LocalRay L;
    L.o = mk(-dot(r0, c) * inv, -dot(r1, c) * inv, -dot(r2, c) * inv);
    L.d = mk(dot(r0, dir) * inv, dot(r1, dir) * inv, dot(r2, dir) * inv);
    L.on = norm1f(L.o);
    const float dn = norm1f(L.d);
    // |A|_F |A^-1|_F is 3 for a rotation times a uniform scale
    const float fa = sqrtf((dot(a0, a0) + dot(a1, a1)) + dot(a2, a2));
    const float fi = sqrtf((dot(r0, r0) + dot(r1, r1)) + dot(r2, r2)) * fabsf(inv);
    const float cond = fa * fi * (1.f / 3.f);
    L.kappa = 0x1p-16f * (cond > 1.f ? cond : 1.f);
    L.dk = 4.f * L.kappa * dn;
    L.ok = det != 0.f && __builtin_isfinite(inv) && __builtin_isfinite(L.kappa) && L.kappa < 0x1p-4f &&
           __builtin_isfinite(L.on) && __builtin_isfinite(dn);
    return L;
}
// Ray::IntersectParalgram from the origin (Ray.cpp:36-133): the three slabs
// of the box, normals v x w, w x u, u x v.
__device__ __forceinline__ bool ray_box(f3 dir, const Box& b, float& tmin, float& tmax) {
    tmin = -__builtin_huge_valf();
    tmax = __builtin_huge_valf();
    const f3 ro = sub(mk(0.f, 0.f, 0.f), b.c);
    const f3 side[3] = {b.u, b.v, b.w};
    const f3 pa[3] = {b.v, b.w, b.u}, pb[3] = {b.w, b.u, b.v};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const f3 n = normalize(cross(pa[k], pb[k]));
        const float d = -fabsf(dot(n, side[k]));
        const float hc = dot(n, ro);
        const float vn1 = hc + d;
        const float vn2 = -hc + d;
        const float vd = dot(n, dir);
        if (fabsf(vd) >= FLT_EPS) {
            const float inv = 1.f / vd;
            float t1 = -vn1 * inv;
            float t2 = vn2 * inv;
            if (t1 > t2) {
                const float t = t1;
                t1 = t2;
                t2 = t;
            }
            tmin = max_std(t1, tmin);
            tmax = min_std(t2, tmax);
            if (tmin > tmax || tmax < 0.f) return false;
        } else if (vn1 > 0.f || vn2 > 0.f) {
            return false;
        }
    }
    return true;
}

// What a walk reads of a stored box (RaySlab), computed once per box.
__device__ __forceinline__ RaySlab make_slab(const ChildRec& r) {
    const float* bx = r.box;
    const f3 u = mk(bx[3], bx[4], bx[5]), v = mk(bx[6], bx[7], bx[8]), w = mk(bx[9], bx[10], bx[11]);
    const f3 nrm[3] = {cross(v, w), cross(w, u), cross(u, v)};
    RaySlab s;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const f3 n = nrm[k];
        s.n[3 * k] = n.x;
        s.n[3 * k + 1] = n.y;
        s.n[3 * k + 2] = n.z;
        s.h[k] = (fabsf(dot(n, u)) + fabsf(dot(n, v))) + fabsf(dot(n, w));
        s.c[k] = bx[k];
    }
    s.entry = r.link | (child_cnt(r) << RAY_LINK_BITS);
    return s;
}

// The mesh-frame test of a stored box (centre c, half-sides u, v, w): the
// three slabs of Ray::IntersectParalgram (Ray.cpp:36-133), normals v x w,
// w x u, u x v, each slab's half-width the box's projection radius on its
// normal.  Every slab and crossing parameter is computed once and bounded by
// its rounding (kappa, and the relative error rho of the crossing's
// denominator), giving a widened and a shrunk interval.  BOX_OUT: even the
// widened interval misses, so the exact ray misses and so does the
// reference's float test, whose rounding is far inside these bounds.
// BOX_IN: even the shrunk interval meets the ray ahead of its origin.
// BOX_NEAR: the decision is within rounding (a box the ray grazes, one ending
// at the ray's origin, a flat box, a slab the ray runs along); the caller
// then runs the reference's own test.  tmin/tmax: the unwidened parameters,
// for the order of the children and the pruning against the best hit.
// The crossings of a slab widened by e lie e |r| further out, and rho of
// their own size beyond that, so both intervals differ from the crossing t by
// at most e |r| (1 + rho) + rho |t|.  e is bounded by the 1-norms of the
// normal, the centre and the half-sides; the latter's from the record: the
// sides are orthogonal, so |u|_1 <= sqrt(3) |u| <= 3 h / |n|_1 (0.1 more for
// the rounding; tests/test_box_margin.py).  Written without branches: a
// node's two tests are most of a step's instructions, with about one
// wavefront per SIMD, and the exec-mask turns of the branches cost as much as
// the arithmetic.
enum : int { BOX_OUT = 0, BOX_IN = 1, BOX_NEAR = 2 };
__device__ __forceinline__ int box_local(const LocalRay& R, const RaySlab& sl, float& tmin, float& tmax) {
    const float inf = __builtin_huge_valf();
    tmin = -inf;
    tmax = inf;
    const f3 c = mk(sl.c[0], sl.c[1], sl.c[2]);
    const f3 q = sub(R.o, c);
    float nn[3], sides = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        nn[k] = norm1f(mk(sl.n[3 * k], sl.n[3 * k + 1], sl.n[3 * k + 2]));
        sides = __builtin_fmaf(sl.h[k], __builtin_amdgcn_rcpf(nn[k]), sides);
    }
    const float reach = __builtin_fmaf(3.1f, sides, (norm1f(q) + R.on) + norm1f(c));  // infinite or NaN without a normal
    const float kr = R.kappa * reach;
    float lo_w = -inf, hi_w = inf, lo_s = -inf, hi_s = inf;
    bool decided = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const f3 n = mk(sl.n[3 * k], sl.n[3 * k + 1], sl.n[3 * k + 2]);
        const float h = sl.h[k];
        const float e = kr * nn[k];     // bound on the rounding of h and num
        const float d4 = R.dk * nn[k];  // four times the bound on den's rounding
        const float num = dot(n, q);
        const float den = dot(n, R.d);
        const bool cuts = fabsf(den) > fmaxf(d4, 0x1p-100f);  // else the ray runs along the slab
        const float r = __builtin_amdgcn_rcpf(cuts ? den : 1.f);  // within an ulp, far inside rho
        const float ar = fabsf(r);
        const float rho = __builtin_fmaf(0.5f * d4, ar, R.kappa);  // relative error of a crossing parameter
        const float t1 = (-h - num) * r, t2 = (h - num) * r;
        const float a = fminf(t1, t2), b = fmaxf(t1, t2);
        const float m0 = e * ar, m = __builtin_fmaf(rho, m0, m0);
        const float ma = __builtin_fmaf(rho, fabsf(a), m), mb = __builtin_fmaf(rho, fabsf(b), m);
        tmin = fmaxf(cuts ? a : -inf, tmin);
        tmax = fminf(cuts ? b : inf, tmax);
        lo_w = fmaxf(cuts ? a - ma : -inf, lo_w);
        hi_w = fminf(cuts ? b + mb : inf, hi_w);
        lo_s = fmaxf(cuts ? a + ma : -inf, lo_s);
        hi_s = fminf(cuts ? b - mb : inf, hi_s);
        // a slab thinner than its rounding, or one the ray runs along and is not clearly inside
        decided &= cuts ? h > e : fabsf(num) + e < h;
    }
    const bool usable = R.ok & (reach < 0x1p100f);
    const bool out = !((lo_w <= hi_w) & (hi_w >= 0.f));
    const bool in = decided & (lo_s <= hi_s) & (hi_s >= 0.f);
    return !usable ? BOX_NEAR : out ? BOX_OUT : in ? BOX_IN : BOX_NEAR;
}

struct Hit {
    bool hit, back;
    float dist, bx, by;
    uint32_t tri;  // mesh-local tree-order slot
};

// Per-lane traversal stack in LDS, entry-major (entry e of lane l at
// e * 64 + l, so a wavefront's accesses fall in distinct banks).  An entry
// is a child still to visit: cnt 0 for internal node `link`, else a leaf of
// cnt triangles from `link`; t0 its entry distance.  A child whose exit
// distance is negative is never pushed (that check does not depend on the
// best hit, so making it at push time is the reference's check).
// link and cnt share one word (link < 2^RAY_LINK_BITS, cnt <= 64; the host
// checks the meshes): 8 bytes an entry, so six wavefronts fit a CU's LDS
// where 12-byte entries allowed four.
struct RayStack {
    uint32_t* lc;
    float* t0;
    int lane;
    int cap;  // entries per lane
    __device__ __forceinline__ void put(int i, uint32_t entry, float t) {
        lc[i * 64 + lane] = entry;
        t0[i * 64 + lane] = t;
    }
};

// The lanes' published best hits (LDS, one word per lane): relaxed atomic
// accesses, so that a lane reads its partner's latest value each time and the
// accesses stay LDS operations.
__device__ __forceinline__ void publish(float* sbest, int lane, float v) {
    __hip_atomic_store(&sbest[lane], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
__device__ __forceinline__ float partner(float* sbest, int lane) {
    return __hip_atomic_load(&sbest[lane ^ 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Closest hit of the ray (o, dir) on mesh m moved by M (Ray.cpp:135-236).
// A stack that would overflow (the host sizes it from the tree depths, so
// this is unreachable unless that sizing is wrong) sets bit 0 of *err and
// ends the traversal; the host then fails the call with CD_E_STACK.
// sbest: per lane of the wavefront, the best hit distance so far of its walk,
// and when the walk is over its hit distance if that is a back face, else -1.
// bounded (the own-tree pass of a Hermann pair): the walk only decides
// whether p2.dist <= p3.dist + eps holds, with p2 the partner lane's closest
// hit, so an entry whose entry distance lies beyond the partner's best so far
// (never below its final one) plus eps, widened by BOUND_SLACK for rounding,
// is skipped, and the walk stops once the partner ends without a back-face
// hit (the pass fails whatever this walk finds).
constexpr float BOUND_SLACK = 1.f + 0x1p-12f;

// What a wavefront's walks share in LDS.
struct WalkShared {
    float best[64];     // the lanes' published best hits
    float ray[15][64];  // each lane's walk: its mesh-to-ray matrix (columns' x, y, z) and direction
    uint32_t tri[64], own[64];  // the leaf tests of a step: triangle, and the lane whose walk it belongs to
};
__device__ __forceinline__ void wave_order() { __builtin_amdgcn_wave_barrier(); }
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_addu(uint32_t v) {
    return v + uint32_t(__builtin_amdgcn_update_dpp(0, int(v), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t v) {  // inclusive
    v = dpp_addu<0x111, 0xf>(v);
    v = dpp_addu<0x112, 0xf>(v);
    v = dpp_addu<0x114, 0xf>(v);
    v = dpp_addu<0x118, 0xf>(v);
    v = dpp_addu<0x142, 0xa>(v);  // lane 15 of a row into the next row (rows 1 and 3)
    v = dpp_addu<0x143, 0xc>(v);  // lane 31 into rows 2 and 3
    return v;
}
__device__ __forceinline__ float lane_f32(float v, int src) { return __shfl(v, src, 64); }
// The value of the lane two away in its group of four, and of the group's lane 0 or 1.
__device__ __forceinline__ uint32_t other_half(uint32_t v) {
    return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x4E, 0xf, 0xf, false));
}
__device__ __forceinline__ uint32_t first_half(uint32_t v) {
    return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x44, 0xf, 0xf, false));
}

// The whole wavefront calls this together; lanes without a walk (live false)
// only lend themselves to the others' leaf tests.
// nslab: the slab records of the node arena's children (2 per node),
// rslab: the root's of this lane's mesh.
// A step enters at most one internal node and tests at most one leaf per
// lane, then pops the next entry: the lanes of a wavefront, each at its own
// place in its own walk, all make progress every step.  About one lane in
// ten is at a leaf in a step, so the leaf tests of all lanes are dealt out over
// the wavefront, one triangle a lane, and every owner takes its results in
// the walk's order: a lane testing its own four triangles ran four tests'
// instructions every step for a tenth of the lanes.  A step's node records
// and triangles are loaded together (at clamped addresses, not under their
// conditions), and the two children's near ties run through one copy of the
// reference's test.
// QUAD: four lanes per ray; lanes l and l + 2 of a group keep the same walk
// and test one child each.  Their state stays equal: both see both results,
// and only the first half's leaf tests are dealt out.
template <bool QUAD>
__device__ __forceinline__ Hit ray_tree(bool live, const MeshRec& m, const NodeRec* __restrict__ nodes,
                                        const RaySlab* __restrict__ nslab, const RaySlab& rslab,
                                        const float* __restrict__ tris, M4 C, f3 o, f3 dir, RayStack& S,
                                        unsigned long long* err, uint32_t& nbox, uint32_t& ntri, WalkShared& W,
                                        bool bounded, float eps) {
    const int lane = S.lane;
    constexpr int KIDS = QUAD ? 1 : 2;  // children a lane tests itself
    const uint32_t half = QUAD ? uint32_t(lane >> 1) & 1u : 0u;
    C.m[12] = C.m[12] - o.x;  // centred on the ray origin (Ray.cpp:150-154)
    C.m[13] = C.m[13] - o.y;
    C.m[14] = C.m[14] - o.z;
    C.m[15] = C.m[15] - 0.f;
    Hit best = {false, false, __builtin_huge_valf(), 0.f, 0.f, 0xFFFFFFFFu};
    publish(W.best, lane, __builtin_huge_valf());
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < 3; ++e) W.ray[3 * k + e][lane] = C.m[4 * k + e];
    W.ray[12][lane] = dir.x;
    W.ray[13][lane] = dir.y;
    W.ray[14][lane] = dir.z;
    wave_order();
    const LocalRay R = local_ray(C, dir);
    auto finish = [&]() {  // the walk's end, as the partner lane reads it
        publish(W.best, lane, (best.hit && best.back) ? best.dist : -1.f);
    };
    // the reference's own test of a box whose mesh-frame test is within rounding
    auto reference = [&](const float* bx, float& t0, float& t1) -> bool {
        return ray_box(dir, xform_box(C, box_from12(bx)), t0, t1) && t1 >= 0.f;
    };
    bool active = live;
    {
        float r0, r1;
        const int k = box_local(R, rslab, r0, r1);
        bool in = k == BOX_IN;
        if (live && k == BOX_NEAR) in = reference(m.root.box, r0, r1);
        if (live && half == 0u) ++nbox;
        active = live && in;
    }
    if (live && !active) finish();
    int sp = 0;
    const uint32_t node_base = m.node_base, tri_base = m.tri_base;
    bool at_node = active && m.nnodes != 0;  // the root, entered without a distance check
    uint32_t node = 0;
    uint32_t leaf_link = 0, leaf_cnt = active && m.nnodes == 0 ? m.ntri : 0u;  // the root is a leaf
    while (__ballot(active)) {
        // the step's node records
        const size_t ni = at_node ? size_t(node_base) + node : 0;
        const ChildRec* cr = nodes[ni].c;
        RaySlab sl[KIDS];
        uint32_t entry[2];
#pragma unroll
        for (int k = 0; k < KIDS; ++k) {
            sl[k] = nslab[2 * ni + (QUAD ? half : uint32_t(k))];
            entry[k] = sl[k].entry;
        }
        // the step's leaf tests, 64 at a time
        const bool leaves = __ballot(leaf_cnt != 0u) != 0;
        bool top = false;
        uint32_t top_entry = 0;
        float top_t = 0.f;
        const uint32_t dealt = half == 0u ? leaf_cnt : 0u;
        uint32_t excl = 0, total = 0;  // this walk's first test
        uint32_t own = 0, tri = 0;
        float T[9];
        auto deal = [&](uint32_t base) {
            for (uint32_t k = 0; __ballot(k < dealt); ++k) {
                const uint32_t at = excl + k - base;
                if (k < dealt && at < 64u) {
                    W.tri[at] = tri_base + leaf_link + k;
                    W.own[at] = uint32_t(lane);
                }
            }
            wave_order();
            const bool in = base + uint32_t(lane) < total;
            own = in ? W.own[lane] : uint32_t(lane);
            tri = in ? W.tri[lane] : 0u;
            wave_order();
            const float* p = tris + size_t(tri) * 9;
#pragma unroll
            for (int e = 0; e < 9; ++e) T[e] = p[e];
        };
        if (leaves) {
            const uint32_t incl = wave_scan_u32(dealt);
            total = uint32_t(__builtin_amdgcn_readlane(int(incl), 63));
            excl = QUAD ? first_half(incl - dealt) : incl - dealt;
            deal(0);
        }
        if (__ballot(at_node)) {
            float t0[2], t1;
            bool in[2], near[KIDS];
#pragma unroll
            for (int k = 0; k < KIDS; ++k) {
                const int d = box_local(R, sl[k], t0[k], t1);
                in[k] = d == BOX_IN;
                near[k] = at_node && d == BOX_NEAR;
            }
            if (QUAD) {
                if (near[0]) in[0] = reference(cr[half].box, t0[0], t1);
                const bool i = in[0];
                const float t = t0[0];
                const uint32_t l = entry[0];
                const bool oi = other_half(uint32_t(i)) != 0u;
                const float ot = __uint_as_float(other_half(__float_as_uint(t)));
                const uint32_t ol = other_half(l);
                in[0] = half ? oi : i;
                in[1] = half ? i : oi;
                t0[0] = half ? ot : t;
                t0[1] = half ? t : ot;
                entry[0] = half ? ol : l;
                entry[1] = half ? l : ol;
            } else {
                while (__ballot(near[0] || near[KIDS - 1])) {
                    if (near[0] || near[KIDS - 1]) {
                        const bool second = !near[0];
                        float u0, u1;
                        const bool hit = reference(cr[second ? 1 : 0].box, u0, u1);
                        in[0] = second ? in[0] : hit;
                        in[1] = second ? hit : in[1];
                        t0[0] = second ? t0[0] : u0;
                        t0[1] = second ? u0 : t0[1];
                        near[KIDS - 1] = second ? false : near[KIDS - 1];
                        near[0] = false;
                    }
                }
            }
            if (at_node) {
                nbox += half == 0u ? 2u : 0u;
                if (sp + 2 > S.cap) {  // deeper than the host allows (it sizes the stack from the tree depths)
                    atomicOr(err, 1ull);
                    best.hit = false;
                    active = false;
                    sp = 0;
                } else {
                    const bool lh = in[0], rh = in[1];
                    // the farther below the nearer (Ray.cpp:175-199); order set by the entry distances alone
                    const bool left_first = !(lh && rh) || t0[0] < t0[1];
                    // the nearer waits in registers: it is the next entry to pop
                    const bool l = lh && left_first;
                    if (lh && rh) S.put(sp++, l ? entry[1] : entry[0], l ? t0[1] : t0[0]);
                    top = lh || rh;
                    top_entry = l ? entry[0] : entry[1];
                    top_t = l ? t0[0] : t0[1];
                }
                at_node = false;
            }
        }
        if (leaves) {
            for (uint32_t base = 0;;) {
                M4 D;
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int e = 0; e < 3; ++e) D.m[4 * k + e] = W.ray[3 * k + e][own];
                const f3 rd = mk(W.ray[12][own], W.ray[13][own], W.ray[14][own]);
                float hx = 0.f, hy = 0.f, hd = __builtin_huge_valf();
                bool hb = false;
                const bool hit = ray_triangle(rd, mul4(D, mk(T[0], T[1], T[2]), 1.f), mul4(D, mk(T[3], T[4], T[5]), 1.f),
                                              mul4(D, mk(T[6], T[7], T[8]), 1.f), hx, hy, hd, hb);
                if (!(hit && hd > 0.f)) hd = __builtin_huge_valf();
                // every owner takes its triangles in order
                const uint32_t at0 = excl - base;
                int win = -1;
                for (uint32_t k0 = 0; __ballot(k0 < leaf_cnt); k0 += 4) {
                    float d[4];
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) d[k] = lane_f32(hd, int((at0 + k0 + k) & 63u));
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k)
                        if (k0 + k < leaf_cnt && at0 + k0 + k < 64u && d[k] < best.dist) {
                            best.dist = d[k];
                            best.tri = leaf_link + k0 + k;
                            win = int(at0 + k0 + k);
                        }
                }
                if (__ballot(win >= 0)) {
                    const float wx = lane_f32(hx, win & 63), wy = lane_f32(hy, win & 63);
                    const int wb = __shfl(int(hb), win & 63, 64);
                    if (win >= 0) {
                        best.hit = true;
                        best.back = wb != 0;
                        best.bx = wx;
                        best.by = wy;
                    }
                }
                base += 64;
                if (base >= total) break;
                deal(base);
            }
            if (leaf_cnt) {
                ntri += dealt;
                leaf_cnt = 0;
                publish(W.best, lane, best.dist);
            }
        }
        // the next entry the best hit so far does not prune
        bool more = false;
        const float pb = bounded ? partner(W.best, lane) : __builtin_huge_valf();
        if (pb < 0.f) {  // the partner ended without a back-face hit
            sp = 0;
            top = false;
        }
        const float bound = (pb + eps) * BOUND_SLACK;
        // an entry is skipped when the best hit prunes it, or when no hit in it can make the pass fail
        auto take = [&](uint32_t entry, float et) {
            if (!(et < best.dist) || et > bound) return;
            more = true;
            const uint32_t el = entry & ((1u << RAY_LINK_BITS) - 1u), ec = entry >> RAY_LINK_BITS;
            if (ec == 0u) {
                node = el;
                at_node = true;
            } else {
                leaf_link = el;
                leaf_cnt = ec;
            }
        };
        if (top) take(top_entry, top_t);
        while (sp > 0 && !more) {  // four entries a look: their LDS reads overlap
            uint32_t ew[4];
            float et[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int i = max(sp - 1 - k, 0);
                ew[k] = S.lc[i * 64 + lane];
                et[k] = S.t0[i * 64 + lane];
            }
            const int n = min(sp, 4);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (k < n && !more) {
                    --sp;
                    take(ew[k], et[k]);
                }
        }
        if (!more) {
            if (live) finish();  // a walk already over publishes the same again
            active = false;
        }
    }
    return best;
}

// Ray::MoveOriginEpsilonTowardsDirection (Ray.cpp:13-21).
__device__ __forceinline__ f3 move_eps(f3 o, f3 d, float factor) {
    float big = fabsf(o.x);
    if (big < fabsf(o.y)) big = fabsf(o.y);
    if (big < fabsf(o.z)) big = fabsf(o.z);
    const float e = big * FLT_EPS;
    return add(o, scale(d, factor * e));
}

struct Pass {
    bool ok;
    f3 response, normal;
};

struct MeshView {
    const MeshRec* meshes;
    const NodeRec* nodes;
    const RaySlab* slabs;  // 2 per node, node arena order
    const RaySlab* roots;  // per mesh
    const float* tris;
    const uint2* attrs;
    const uint32_t* vid;
    const float* nrm;
    const uint32_t* perm;
};

// HermannPass (ShootUncollideRays.cpp:129-158), on two lanes: the even lane
// shoots the ray at the other entity's tree (p2), the odd lane shoots the
// ray moved 4 epsilon along itself at the entity's own tree (p3), which does
// not depend on p2; both lanes then hold both hits and decide the same way.
// The reference skips p3 when p2 fails; computing it anyway changes nothing.
__device__ __forceinline__ Hit shfl_hit(const Hit& h, int src) {
    Hit r;
    r.hit = __shfl(int(h.hit), src, 64) != 0;
    r.back = __shfl(int(h.back), src, 64) != 0;
    r.dist = __shfl(h.dist, src, 64);
    r.bx = __shfl(h.bx, src, 64);
    r.by = __shfl(h.by, src, 64);
    r.tri = uint32_t(__shfl(int(h.tri), src, 64));
    return r;
}

// The whole wavefront calls it; live: this lane's ray is shot in this pass.
template <bool QUAD>
__device__ __forceinline__ Pass hermann(bool live, const MeshView& V, uint32_t meshA, const M4& Amat, uint32_t meshB,
                                        const M4& Bmat, const M3& Bn, f3 o, f3 d, RayStack& S, unsigned long long* err,
                                        uint32_t& nbox, uint32_t& ntri, WalkShared& W) {
    Pass r = {false, mk(0.f, 0.f, 0.f), mk(0.f, 0.f, 0.f)};
    const bool own = (threadIdx.x & 1u) != 0;
    const f3 o2 = move_eps(o, d, 4.f);
    M4 C;  // one call with lane-selected arguments, so the two traversals run as one instruction stream
#pragma unroll
    for (int e = 0; e < 16; ++e) C.m[e] = own ? Amat.m[e] : Bmat.m[e];
    const float eps = vlength(sub(o2, o));
    const uint32_t mesh = own ? meshA : meshB;
    const Hit h = ray_tree<QUAD>(live, V.meshes[mesh], V.nodes, V.slabs, V.roots[mesh], V.tris, C, own ? o2 : o, d, S, err,
                           nbox, ntri, W, own, eps);
    const int even = int(threadIdx.x & ~1u);
    const Hit p2 = shfl_hit(h, even), p3 = shfl_hit(h, even + 1);
    if (live && p2.hit && p2.back && p2.dist <= p3.dist + eps) {
        const MeshRec mb = V.meshes[meshB];
        r.ok = true;
        r.response = scale(d, p2.dist);
        const uint2 attr = V.attrs[meshB];
        const float* t9 = V.tris + (size_t(mb.tri_base) + p2.tri) * 9;
        f3 nk[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) nk[k] = corner_normal(attr, V.nrm, vertex_id(mb, attr, V.vid, V.perm, p2.tri, k), t9);
        const f3 ni = add(add(scale(nk[0], (1.f - p2.bx) - p2.by), scale(nk[1], p2.bx)), scale(nk[2], p2.by));
        r.normal = normalize(mul3(Bn, ni));
    }
    return r;
}

// CalcForceResponse (:118-127).
__device__ __forceinline__ f3 force_response(const Pass& p) {
    const f3 dir = normalize(p.response);
    const float len = vlength(p.response);
    const float c = dot(p.normal, dir);
    const float c2 = c * c;
    return scale(dir, c2 * len);
}

__device__ __forceinline__ f3 neg(f3 v) { return mk(-v.x, -v.y, -v.z); }  // glm's unary minus
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ void put3(float* o, f3 v) {
    o[0] = v.x;
    o[1] = v.y;
    o[2] = v.z;
}
__device__ __forceinline__ f3 get3(const float* o) { return mk(o[0], o[1], o[2]); }

}  // namespace

// The rays [r0, r0 + per_wave) of one wavefront, both passes.
template <bool QUAD>
__device__ __forceinline__ void shoot_rays(const cd_ray* __restrict__ rays, uint32_t nrays, uint32_t base1,
                                           const uint32_t* __restrict__ pbegin, uint32_t nq, uint32_t stride,
                                           const QueryRec* __restrict__ qs, const MeshView& V,
                                           RayShot* __restrict__ out, uint32_t r0, uint32_t per_wave, RayStack& S,
                                           unsigned long long* err, uint32_t& nbox, uint32_t& ntri, WalkShared& W) {
    const uint32_t at = threadIdx.x >> (QUAD ? 2 : 1);  // two or four lanes per ray
    const uint32_t r = min(r0 + at, nrays - 1);
    const bool have = at < per_wave && r0 + at < nrays;
    const int side = r >= base1 ? 1 : 0;
    const uint32_t local = r - (side ? base1 : 0u);
    const uint32_t* begin = pbegin + size_t(stride) * side;
    // the pair: the last one whose rays begin at or before this ray (of equal
    // begins only the last can hold rays)
    uint32_t lo = 0, hi = nq;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (begin[mid] <= local) lo = mid;
        else hi = mid;
    }
    const QueryRec q = qs[lo];
    const M3 Mn = adjoint_transpose(q.rel);
    RayShot s = {};
    f3 o = get3(rays[r].origin), d = get3(rays[r].direction);
    bool live = have;
    // side 0: first-to-second, then the reflected ray second-to-first; side 1 the other way round
#pragma unroll 1
    for (int pass = 0; pass < 2 && __ballot(live); ++pass) {
        const bool f2s = (pass == 0) == (side == 0);
        // from the first entity (the identity) at the second (rel), or the other way round
        M4 A, B;
        M3 Bn;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float id = (e % 5 == 0) ? 1.f : 0.f;
            A.m[e] = f2s ? id : q.rel[e];
            B.m[e] = f2s ? q.rel[e] : id;
        }
#pragma unroll
        for (int e = 0; e < 9; ++e) Bn.m[e] = f2s ? Mn.m[e] : ((e % 4 == 0) ? 1.f : 0.f);
        const Pass p = hermann<QUAD>(live, V, f2s ? q.mesh_a : q.mesh_b, A, f2s ? q.mesh_b : q.mesh_a, B, Bn, o, d, S, err,
                               nbox, ntri, W);
        live = live && p.ok;
        if (live) {
            const f3 F = force_response(p);
            put3(s.force[pass], f2s ? neg(F) : F);  // sum - F == sum + (-F) exactly
            put3(s.push[pass], f2s ? neg(p.response) : p.response);
            s.ok |= 1u << pass;
            o = add(o, p.response);  // ReflectHermannResult (:104-110)
            d = neg(p.normal);
        }
    }
    s.pair = lo;
    if (have && (threadIdx.x & (QUAD ? 3u : 1u)) == 0) out[r] = s;
}

// Per-ray result: for each of the two passes, the contribution to the summed
// force response and the push-out vector, as the reference accumulates them
// (a first-to-second pass subtracts its force and pushes -response, a
// second-to-first pass adds and pushes +response).
// pbegin: per side (at + stride), the first ray of every pair
// (non-decreasing; a pair without rays has the next pair's begin)
// dc: the step's count block, when the ray and pair counts are read on the
// device (nrays, nq then the capacities of the launch)
// DEEP: the stacks live in HBM, a block's 2 stack_entries 64 words at
// gstack + 2 b stack_entries 64 (link words, then entry distances), for
// trees deeper than the LDS stack holds; the walk is the same.
template <bool DEEP>
__global__ __launch_bounds__(64) void k_shoot(const cd_ray* __restrict__ rays, uint32_t nrays, uint32_t base1,
                                              const uint32_t* __restrict__ pbegin, uint32_t nq, uint32_t stride,
                                              const uint32_t* __restrict__ dc,
                                              const QueryRec* __restrict__ qs, MeshView V,
                                              RayShot* __restrict__ out, int stack_entries,
                                              RunCounters* __restrict__ ctr, uint32_t* __restrict__ gstack) {
    unsigned long long* err = &ctr->err;
    // the stacks are sized by the launch: the deepest tree of the call + 2
    // entries per lane, so shallow trees leave LDS for more wavefronts
    extern __shared__ uint32_t s_stack[];
    __shared__ WalkShared W;
    uint32_t* base = DEEP ? gstack + size_t(blockIdx.x) * 2 * size_t(stack_entries) * 64 : s_stack;
    RayStack S = {base, reinterpret_cast<float*>(base + stack_entries * 64), int(threadIdx.x), stack_entries};
    uint32_t nbox = 0, ntri = 0;  // boxes tested, ray-triangle tests: the work counted in ctr->sat, ctr->tritests
    if (dc) {
        base1 = dc[DC_RAYS0];
        nrays = min(nrays, dc[DC_RAYS0] + dc[DC_RAYS1]);
        nq = min(nq, dc[DC_NQ]);
    }
    const uint32_t per_wave = rays_per_wave(nrays, gridDim.x);
    const uint32_t r0 = blockIdx.x * per_wave;
    if (r0 >= nrays) return;
    if (per_wave <= 16)
        shoot_rays<true>(rays, nrays, base1, pbegin, nq, stride, qs, V, out, r0, per_wave, S, err, nbox, ntri, W);
    else
        shoot_rays<false>(rays, nrays, base1, pbegin, nq, stride, qs, V, out, r0, per_wave, S, err, nbox, ntri, W);
    // per wavefront, one atomic each
    const unsigned long long bsum = wave_sum_u64(nbox), tsum = wave_sum_u64(ntri);
    if ((threadIdx.x & 63u) == 0) {
        atomicAdd(&ctr->sat, bsum);
        atomicAdd(&ctr->tritests, tsum);
    }
}

__device__ __forceinline__ float smoother_step(float a, float b, float x) {  // :171-175
    float t = (x - a) / (b - a);
    t = (t < 0.f) ? 0.f : ((1.f < t) ? 1.f : t);
    return t * t * t * (t * (t * 6.f - 15.f) + 10.f);
}
__device__ __forceinline__ bool same_matrix(const float* a, const float* b) {
    for (int i = 0; i < 16; ++i)
        if (!(a[i] == b[i])) return false;
    return true;
}

__device__ __forceinline__ f3 shfl_down3(f3 v, int off) {
    return mk(__shfl_down(v.x, off, 64), __shfl_down(v.y, off, 64), __shfl_down(v.z, off, 64));
}
// One wavefront per pair.  The force responses are summed lane-strided
// (each shot's first pass, then its second) and then over a fixed shuffle
// tree: a sum that is the same on every run.  The reference sums them in its
// ray order, which follows an unordered_map walk no GPU reproduces.  The
// maximum of FindResponse does not depend on the order.
// qw: per side (at + 2 stride) the pairs' ray counts, then (at + stride)
// their first rays; avg: per side (at + 3 stride) the average origins; dc as
// for k_shoot; nshots: the shots there are (a pair whose rays would lie
// beyond them, which only a step over its ray capacity can give, is left
// unshot for the step to run again).
__global__ __launch_bounds__(64) void k_respond(const RayShot* __restrict__ shots, uint32_t base1,
                                                const uint32_t* __restrict__ qw, uint32_t nq, uint32_t stride,
                                                const uint32_t* __restrict__ dc, uint64_t nshots,
                                                const float* __restrict__ avg, const QueryRec* __restrict__ qs,
                                                const uint2* __restrict__ pair_ids, const cd_entity* __restrict__ ents,
                                                float cos_start, float cos_finish, float bias,
                                                cd_pair_response* __restrict__ out) {
    const uint32_t q = blockIdx.x;
    const int lane = threadIdx.x;
    if (dc) {
        base1 = dc[DC_RAYS0];
        nq = min(nq, dc[DC_NQ]);
    }
    if (q >= nq) return;
    const uint2 ids = pair_ids[q];
    cd_pair_response res = {};
    res.first = ids.x;
    res.second = ids.y;
    const float* c1 = ents[ids.x].current;
    const float* c2 = ents[ids.y].current;
    const float* p1 = ents[ids.x].previous;
    const float* p2 = ents[ids.y].previous;
    const uint32_t n0 = qw[q], b0 = qw[stride + q];
    const uint32_t n1 = qw[2 * size_t(stride) + q], b1 = base1 + qw[3 * size_t(stride) + q];
    const bool beyond = (n0 && uint64_t(b0) + n0 > nshots) || (n1 && uint64_t(b1) + n1 > nshots);
    if ((n0 == 0 && n1 == 0) || beyond || (same_matrix(c1, p1) && same_matrix(c2, p2))) {  // :63, :80-81
        if (lane == 0) out[q] = res;
        return;
    }
    res.shot = 1;
    const uint32_t n = n0 + n1;
    f3 sum = mk(0.f, 0.f, 0.f);
    for (uint32_t i = uint32_t(lane); i < n; i += 64) {
        const RayShot& s = shots[i < n0 ? b0 + i : b1 + (i - n0)];
        for (int pass = 0; pass < 2; ++pass)
            if (s.ok & (1u << pass)) sum = add(sum, get3(s.force[pass]));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum = add(sum, shfl_down3(sum, off));
    sum = mk(__shfl(sum.x, 0, 64), __shfl(sum.y, 0, 64), __shfl(sum.z, 0, 64));
    f3 delta = mk(0.f, 0.f, 0.f);
    if (!(sum.x == 0.f && sum.y == 0.f && sum.z == 0.f)) {  // :87
        const f3 nf = normalize(sum);
        float max_len = 0.f;  // FindResponse (:160-169)
        for (uint32_t i = uint32_t(lane); i < n; i += 64) {
            const RayShot& s = shots[i < n0 ? b0 + i : b1 + (i - n0)];
            for (int pass = 0; pass < 2; ++pass) {
                if (!(s.ok & (1u << pass))) continue;
                const f3 r = get3(s.push[pass]);
                const float c = dot(normalize(r), nf);
                const float need = vlength(r) / c;
                max_len = max_std(max_len, smoother_step(cos_finish, cos_start, c) * need);
            }
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) max_len = max_std(max_len, __shfl_down(max_len, off, 64));
        M4 F;
        for (int e = 0; e < 16; ++e) F.m[e] = c1[e];
        delta = mul4(F, scale(scale(nf, max_len), bias), 0.f);
    }
    if (lane != 0) return;
    // the split by each entity's movement (CollisionDetection.cpp:86-97, 143-150)
    M4 C1, P1, C2, P2;
    for (int e = 0; e < 16; ++e) {
        C1.m[e] = c1[e];
        P1.m[e] = p1[e];
        C2.m[e] = c2[e];
        P2.m[e] = p2[e];
    }
    const f3 a1 = get3(avg + 3 * size_t(q)), a2 = get3(avg + 3 * (size_t(stride) + q));
    const float m1 = vlength(sub(mul4(C1, a1, 1.f), mul4(P1, a1, 1.f)));
    const float m2 = vlength(sub(mul4(C2, a2, 1.f), mul4(P2, a2, 1.f)));
    const float total = m1 + m2;
    put3(res.delta, delta);
    put3(res.delta_first, scale(neg(delta), m1 / total));
    put3(res.delta_second, scale(delta, m2 / total));
    out[q] = res;
}

// Slab records: one thread per child of count nodes, and one for mesh m's root.
__global__ void k_ray_slabs(const NodeRec* __restrict__ nodes, uint32_t count, RaySlab* __restrict__ out,
                            const MeshRec* __restrict__ meshes, uint32_t m, RaySlab* __restrict__ root_out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 2 * count) out[i] = make_slab(nodes[i >> 1].c[i & 1u]);
    if (i == 0) *root_out = make_slab(meshes[m].root);
}
hipError_t launch_ray_slabs(const NodeRec* nodes, uint32_t count, RaySlab* out, const MeshRec* meshes, uint32_t m,
                            RaySlab* root_out, hipStream_t st) {
    hipLaunchKernelGGL(k_ray_slabs, dim3((2 * count + 255) / 256 + 1), dim3(256), 0, st, nodes, count, out, meshes, m,
                       root_out);
    return hipGetLastError();
}
hipError_t launch_shoot(const cd_ray* rays, uint32_t nrays, uint32_t base1, const uint32_t* pbegin, uint32_t nq,
                        const QueryRec* qs, const MeshRec* meshes, const NodeRec* nodes, const RaySlab* slabs,
                        const RaySlab* roots, const float* tris,
                        const uint2* attrs, const uint32_t* vid, const float* nrm, const uint32_t* perm, RayShot* shots,
                        uint32_t stack_entries, RunCounters* ctr, hipStream_t st, uint32_t* gstack, uint32_t stride,
                        const uint32_t* dc) {
    if (!nrays) return hipSuccess;
    if (stack_entries < 2) return hipErrorInvalidValue;
    if (!stride) stride = nq;
    const MeshView V = {meshes, nodes, slabs, roots, tris, attrs, vid, nrm, perm};
    const bool deep = shoot_deep(stack_entries);
    const dim3 grid(shoot_blocks(nrays, stack_entries, deep));
    if (!deep) {
        const size_t lds = size_t(stack_entries) * 64 * (sizeof(uint32_t) + sizeof(float));
        hipLaunchKernelGGL(k_shoot<false>, grid, dim3(64), lds, st, rays, nrays, base1, pbegin, nq, stride, dc, qs, V,
                           shots, int(stack_entries), ctr, (uint32_t*)nullptr);
    } else {
        if (!gstack) return hipErrorInvalidValue;
        hipLaunchKernelGGL(k_shoot<true>, grid, dim3(64), 0, st, rays, nrays, base1, pbegin, nq, stride, dc, qs, V,
                           shots, int(stack_entries), ctr, gstack);
    }
    return hipGetLastError();
}
hipError_t launch_respond(const RayShot* shots, uint32_t base1, const uint32_t* qw, uint32_t nq, const float* avg,
                          const QueryRec* qs, const uint2* pair_ids, const cd_entity* ents, float cos_start,
                          float cos_finish, float bias, cd_pair_response* out, hipStream_t st, uint32_t stride,
                          const uint32_t* dc, uint64_t nshots) {
    if (!nq) return hipSuccess;
    if (!stride) stride = nq;
    hipLaunchKernelGGL(k_respond, dim3(nq), dim3(64), 0, st, shots, base1, qw, nq, stride, dc, nshots, avg, qs, pair_ids,
                       ents, cos_start, cos_finish, bias, out);
    return hipGetLastError();
}

}  // namespace cdk
