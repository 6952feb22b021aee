// OBB-tree build on the GPU, bit-identical to the reference builder.
//
// Reference: inMyRoom_vulkan/src/Geometry/OBB.cpp:33-178 (PCA box),
// inMyRoom_vulkan/src/Geometry/OBBtree.cpp:8-108 (recursive split) and
// :179-233, :321-394 (DFS flatten).
//
// Level-synchronous: the nodes of one depth, across every mesh of the
// batch, are one launch, one 64-lane workgroup per node at a time (levels
// are launched in batches; each launch reads its node range from the
// previous one); nodes of more than BIG_TRIS triangles are spread over the
// chip tile by tile instead (bigbuild.hpp).  Within a node:
//   * the distinct-point check is a wave ballot;
//   * the mean and the six covariance sums are SEQUENTIAL double chains in
//     point order (the reference's std::accumulate / std::inner_product),
//     one lane per chain adding terms the whole wave precomputes per LDS chunk;
//   * eig3 runs in FP64 on one lane;
//   * the three min/max projections are wave reductions whose tie rule
//     reproduces std::min/std::max visiting the points in order;
//   * the split is a stable partition built from ballots, scattering the
//     node's triangles into the next level's buffer.
// Afterwards the tree is flattened to the reference's DFS layout with
// per-level prefix passes (subtree counts bottom-up, preorder top-down).
#include <float.h>
#include <math.h>

#include <algorithm>
#include <cstring>

#include "eig3.hpp"
#include "internal.hpp"

namespace cdk {

struct BNode {
    uint32_t mesh, beg, end, level;
    uint32_t kid[2];
    uint32_t flags;  // bit0 = leaf
    uint32_t icount, tcount, pre, toff;
    float surf;
    float box[12];
};

struct LevelArgs {
    BNode* nodes;
    const float* pos_in;
    const uint32_t* id_in;
    float* pos_out;
    uint32_t* id_out;
    float* pos_fin;
    uint32_t* id_fin;
    unsigned int* mesh_depth;
    unsigned int* slack_bits;   // SLACK_REPS copies per mesh
    unsigned int* radius_bits;  // one per mesh
    uint32_t leaf_max;
    uint32_t big_min;           // nodes of more triangles than this take the tiled passes
};

constexpr int CHUNK = 256;                 // points per step of the sequential chains
constexpr int CHUNK_REGS = CHUNK * 3 / 64;  // floats each lane fetches per chunk
static_assert(CHUNK * 3 % 64 == 0 && CHUNK % 64 == 0, "chunk split over a wave");

// The reference's sequential double sums over a node's points (OBB.cpp:
// 41-73: std::accumulate, then the six inner products), one chain per lane,
// in point order.  Only the final additions form the chain; the terms do
// not depend on it.  So the wave streams the points through LDS a chunk at a
// time: every lane fetches its share of the next chunk, all lanes turn the
// current chunk into its K terms per point (term(p, c, out) for the points
// lane, lane + 64, ...), and the first K lanes add their term of each point
// in order while the fetch is in flight.  The block is one wave.
// k_level's workgroup is one wavefront: its lanes run in lockstep and see
// each other's LDS accesses in program order, so a step between the phases
// of a node only has to keep the compiler from moving LDS accesses across
// it.  (__syncthreads would also wait for the global loads in flight, among
// them the prefetch of the next chunk of points.)
__device__ __forceinline__ void wave_sync() { __builtin_amdgcn_wave_barrier(); }

template <int K, class Term>
__device__ __forceinline__ double stream_chain(const float* __restrict__ P, uint32_t npts, Term term, float* s_raw,
                                               double* s_val) {
    const int lane = threadIdx.x;
    float r[CHUNK_REGS];
    auto fetch = [&](uint32_t base) {
        const uint32_t m3 = 3u * min(uint32_t(CHUNK), npts - base);
#pragma unroll
        for (int j = 0; j < CHUNK_REGS; ++j) {
            const uint32_t t = uint32_t(lane) + 64u * j;
            r[j] = t < m3 ? P[3 * size_t(base) + t] : 0.f;
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int j = 0; j < CHUNK_REGS; ++j) s_raw[lane + 64 * j] = r[j];
    };
    fetch(0);
    store();
    wave_sync();
    double acc = 0.0;
    for (uint32_t base = 0; base < npts; base += CHUNK) {
        const uint32_t next = base + CHUNK;
        const uint32_t m = min(uint32_t(CHUNK), npts - base);
        if (next < npts) fetch(next);
#pragma unroll
        for (int j = 0; j < CHUNK / 64; ++j) {
            const uint32_t k = uint32_t(lane) + 64u * j;
            if (k < m) term(s_raw + 3 * k, s_val + K * k);
        }
        wave_sync();
        if (lane < K) {
            // 16 terms are read from LDS while the previous 16 are added,
            // so the chain waits on its additions only
            const double* q = s_val + lane;
            uint32_t k = 0;
            if (m >= 16) {
                double cur[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) cur[i] = q[K * i];
                for (k = 16; k + 16 <= m; k += 16) {
                    double nxt[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i) nxt[i] = q[K * (k + uint32_t(i))];
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc = acc + cur[i];
#pragma unroll
                    for (int i = 0; i < 16; ++i) cur[i] = nxt[i];
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) acc = acc + cur[i];
            }
            for (; k < m; ++k) acc = acc + q[K * k];
        }
        wave_sync();
        if (next < npts) store();
        wave_sync();
    }
    return acc;
}

__device__ inline void wave_min_last(double& v, int& i) {
    // smaller value wins; equal values (== , so -0 and +0 too): larger index wins
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        double ov = __shfl_xor(v, off, 64);
        int oi = __shfl_xor(i, off, 64);
        if (ov < v || (ov == v && oi > i)) {
            v = ov;
            i = oi;
        }
    }
}
__device__ inline void wave_max_first(double& v, int& i) {
    // larger value wins; equal values: smaller index wins
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        double ov = __shfl_xor(v, off, 64);
        int oi = __shfl_xor(i, off, 64);
        if (ov > v || (ov == v && oi < i)) {
            v = ov;
            i = oi;
        }
    }
}

struct AxisCand {
    float len;
    f3 dir;
};

// std::sort of three (length, axis) pairs, descending (OBBtree.cpp:45-51):
// libstdc++ runs its insertion sort for three elements; reproduced branch
// for branch.
__device__ inline void sort3_desc(AxisCand c[3]) {
#pragma unroll
    for (int i = 1; i < 3; ++i) {
        AxisCand val = c[i];
        if (val.len > c[0].len) {
            for (int k = i; k > 0; --k) c[k] = c[k - 1];
            c[0] = val;
        } else {
            int j = i;
            while (val.len > c[j - 1].len) {
                c[j] = c[j - 1];
                --j;
            }
            c[j] = val;
        }
    }
}

// Triangle::GetMinMaxProjectionToAxis (Triangle.cpp:113-138) then the
// left/right rule of OBBtree.cpp:66-75, on a triangle held in registers.
__device__ inline bool goes_left(const float (&T)[9], f3 axis, float cproj) {
    float lo = INFINITY, hi = -INFINITY;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float q = dot(axis, mk(T[3 * k], T[3 * k + 1], T[3 * k + 2]));
        if (q < lo) lo = q;
        if (q > hi) hi = q;
    }
    float mid = (lo + hi) / 2.f;
    return mid <= cproj;
}

// The node scans below take GROUP wave-wide chunks per step and issue the
// loads of all of them before using any: a node's scans are latency bound
// (one wave per node), and a chunk at a time waits on memory once per chunk.
// Indices past the end are clamped to the last element rather than guarded:
// a guarded load is moved behind the guard of its use, back to one wait per
// chunk.
constexpr int GROUP = 8;

__device__ __forceinline__ void load_tris(const float* __restrict__ P, uint32_t c0, uint32_t n, int lane,
                                          float (&T)[GROUP][9]) {
#pragma unroll
    for (int j = 0; j < GROUP; ++j) {
        const size_t i = min(c0 + 64u * j + uint32_t(lane), n - 1);
#pragma unroll
        for (int t = 0; t < 9; ++t) T[j][t] = P[i * 9 + t];
    }
}

// The box of a node from its axes and the extents along them
// (OBB::CreateAABBfromPoints' tail and OBB.cpp:74-89).
__device__ inline void box_of_extents(const double* ax, const double* lo, const double* hi, float* box12) {
    double cx = 0.0, cy = 0.0, cz = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        double delta = (hi[q] - lo[q]) + 2.0 * double(FLT_EPSILON);
        double mid = (hi[q] + lo[q]) / 2.0;
        cx = cx + mid * ax[3 * q];
        cy = cy + mid * ax[3 * q + 1];
        cz = cz + mid * ax[3 * q + 2];
        double half = delta / 2.0;
        box12[3 + 3 * q] = float(half * ax[3 * q]);
        box12[4 + 3 * q] = float(half * ax[3 * q + 1]);
        box12[5 + 3 * q] = float(half * ax[3 * q + 2]);
    }
    box12[0] = float(cx);
    box12[1] = float(cy);
    box12[2] = float(cz);
}

// OBB::EmptyOBB (OBB.cpp:168-178) at a point.
__device__ inline Box empty_box(f3 c) {
    const float e = FLT_EPSILON;
    Box b;
    b.c = c;
    b.u = mk(e, 0.f, 0.f);
    b.v = mk(0.f, e, 0.f);
    b.w = mk(0.f, 0.f, e);
    return b;
}

// How far a point lies outside a box meant to hold it: its coordinates in the
// side vectors are its offset dotted with the dual basis (v x w, w x u,
// u x v) / det(u, v, w).  A mesh's slack is the largest excess of any point
// over any box above it; it is taken where the node's triangles are read for
// its split anyway, as a pass of its own read every level's triangles again
// (one wavefront per node: 1.8 ms for a level load with a 198,450-triangle
// terrain).
struct Excess {
    double c[3], du[3], dv[3], dw[3], lu, lv, lw;
    bool flat;
    __device__ explicit Excess(const Box& b) {
        const double u[3] = {b.u.x, b.u.y, b.u.z}, v[3] = {b.v.x, b.v.y, b.v.z}, w[3] = {b.w.x, b.w.y, b.w.z};
        auto cross = [](const double* a, const double* q, double* o) {
            o[0] = a[1] * q[2] - a[2] * q[1];
            o[1] = a[2] * q[0] - a[0] * q[2];
            o[2] = a[0] * q[1] - a[1] * q[0];
        };
        c[0] = b.c.x;
        c[1] = b.c.y;
        c[2] = b.c.z;
        cross(v, w, du);
        cross(w, u, dv);
        cross(u, v, dw);
        const double D = u[0] * du[0] + u[1] * du[1] + u[2] * du[2];
        for (int k = 0; k < 3; ++k) {
            du[k] = du[k] / D;
            dv[k] = dv[k] / D;
            dw[k] = dw[k] / D;
        }
        flat = !(fabs(D) > 0.0);
        lu = sqrt(u[0] * u[0] + u[1] * u[1] + u[2] * u[2]);
        lv = sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        lw = sqrt(w[0] * w[0] + w[1] * w[1] + w[2] * w[2]);
    }
    __device__ __forceinline__ double of(const float* p) const {
        if (flat) return INFINITY;
        const double r[3] = {double(p[0]) - c[0], double(p[1]) - c[1], double(p[2]) - c[2]};
        const double al = r[0] * du[0] + r[1] * du[1] + r[2] * du[2];
        const double be = r[0] * dv[0] + r[1] * dv[1] + r[2] * dv[2];
        const double ga = r[0] * dw[0] + r[1] * dw[1] + r[2] * dw[2];
        return fmax(0.0, fabs(al) - 1.0) * lu + fmax(0.0, fabs(be) - 1.0) * lv + fmax(0.0, fabs(ga) - 1.0) * lw;
    }
    // the largest excess and squared norm over a triangle's corners
    __device__ __forceinline__ void take(const float* t9, double& worst, double& rad2) const {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float* p = t9 + 3 * k;
            worst = fmax(worst, of(p));
            rad2 = fmax(rad2, double(p[0]) * double(p[0]) + double(p[1]) * double(p[1]) + double(p[2]) * double(p[2]));
        }
    }
};
__device__ inline float round_up(double x) {  // to float, so that the bound stays an upper bound
    float f = float(x);
    if (double(f) < x) f = nextafterf(f, INFINITY);
    return f;
}
// One of SLACK_REPS copies per mesh, so that a mesh's many nodes do not queue
// on one address; the radius is the root's (sqrt is monotone: the root of
// the largest square is the largest root).
__device__ inline void post_excess(const LevelArgs& a, const BNode& nd, uint32_t rep, double worst, double rad2) {
    atomicMax(&a.slack_bits[size_t(nd.mesh) * SLACK_REPS + (rep % SLACK_REPS)], __float_as_uint(round_up(worst)));
    if (nd.level == 0) atomicMax(&a.radius_bits[nd.mesh], __float_as_uint(round_up(sqrt(rad2))));
}

// The children of a split node, in the next level's slots `slot` and slot + 1.
__device__ inline void place_kids(const LevelArgs& a, BNode* nd, uint32_t nl, uint32_t slot) {
    const uint32_t beg = nd->beg, end = nd->end;
    BNode* k0 = &a.nodes[slot];
    BNode* k1 = &a.nodes[slot + 1];
    k0->mesh = nd->mesh; k0->beg = beg;      k0->end = beg + nl; k0->level = nd->level + 1; k0->flags = 0;
    k1->mesh = nd->mesh; k1->beg = beg + nl; k1->end = end;      k1->level = nd->level + 1; k1->flags = 0;
    nd->kid[0] = slot;
    nd->kid[1] = slot + 1;
    nd->flags = 0;
}
// The same, taking the next two free slots of the level.
__device__ inline uint32_t append_kids(const LevelArgs& a, BNode* nd, uint32_t nl, uint32_t next_first,
                                       unsigned int* next_count) {
    const uint32_t slot = next_first + atomicAdd(next_count, 2u);
    place_kids(a, nd, nl, slot);
    atomicMax(&a.mesh_depth[nd->mesh], nd->level + 1);
    return slot;
}

// The split's three candidates, longest first (OBBtree.cpp:45-51), and their centre projections.
__device__ inline void split_candidates(const Box& box, AxisCand (&cand)[3], float (&cp)[3]) {
    cand[0] = {vlength(box.u), normalize(box.u)};
    cand[1] = {vlength(box.v), normalize(box.v)};
    cand[2] = {vlength(box.w), normalize(box.w)};
    sort3_desc(cand);
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) cp[ch] = dot(box.c, cand[ch].dir);
}
// The first candidate that leaves both sides non-empty, else -1: index halves (OBBtree.cpp:81-93).
__device__ inline int split_pick(const uint32_t (&cnt)[3], uint32_t n) {
    int pick = -1;
#pragma unroll
    for (int ch = 2; ch >= 0; --ch)
        if (cnt[ch] != 0 && cnt[ch] != n) pick = ch;
    return pick;
}

struct LevelShared {
    float raw[CHUNK * 3];
    double val[CHUNK * 6];
    double mean[3];
    double cov[6];
    double ax[9];
    float box[12];
};

// One node of a level: its box (OBB::CreateOBBfromPoints, OBB.cpp:33-89),
// then either its triangles parked as a leaf or its split into two
// children appended to the next level (OBBtreeSplitBuildNode::
// SplitOBBandCreateChildren, OBBtree.cpp:43-108).
__device__ __forceinline__ void level_node(const LevelArgs& a, uint32_t ni, uint32_t next_first,
                                           unsigned int* next_count, LevelShared& S) {
    const int lane = threadIdx.x;
    BNode* nd = &a.nodes[ni];
    const uint32_t beg = nd->beg, end = nd->end;
    const uint32_t n = end - beg, npts = 3 * n;
    const float* P = a.pos_in + size_t(beg) * 9;

    // more than one distinct point?  (the first wave-wide chunk that shows one ends the scan)
    bool multi = false;
    if (npts > 1) {
        const float x0 = P[0], y0 = P[1], z0 = P[2];
        for (uint32_t k0 = 1; k0 < npts && !multi; k0 += 64) {
            const uint32_t k = k0 + lane;
            const bool d = k < npts && !(P[3 * k] == x0 && P[3 * k + 1] == y0 && P[3 * k + 2] == z0);
            multi = __ballot(d) != 0;
        }
    }
    Box box;
    if (npts == 0 || !multi) {
        box = empty_box(npts ? mk(P[0], P[1], P[2]) : mk(0.f, 0.f, 0.f));
    } else {
        const double N = double(npts);
        double acc = stream_chain<3>(
            P, npts,
            [](const float* p, double* o) {
                o[0] = double(p[0]);
                o[1] = double(p[1]);
                o[2] = double(p[2]);
            },
            S.raw, S.val);
        if (lane < 3) S.mean[lane] = acc / N;
        wave_sync();
        // covariance order xx, yy, zz, xy, xz, yz (OBB.cpp:56-73)
        const double mx = S.mean[0], my = S.mean[1], mz = S.mean[2];
        acc = stream_chain<6>(
            P, npts,
            [mx, my, mz](const float* p, double* o) {
                const double dx = double(p[0]) - mx, dy = double(p[1]) - my, dz = double(p[2]) - mz;
                o[0] = dx * dx;
                o[1] = dy * dy;
                o[2] = dz * dz;
                o[3] = dx * dy;
                o[4] = dx * dz;
                o[5] = dy * dz;
            },
            S.raw, S.val);
        if (lane < 6) S.cov[lane] = acc / N;
        wave_sync();
        if (lane == 0) {
            const double xx = S.cov[0], yy = S.cov[1], zz = S.cov[2], xy = S.cov[3], xz = S.cov[4], yz = S.cov[5];
            double A[3][3] = {{xx, xy, xz}, {xy, yy, yz}, {xz, yz, zz}};
            double V[3][3], d[3];
            eig3(A, V, d);
            // OBB.cpp:80-87: the box axes are the ROWS of eig3's V
            for (int r = 0; r < 3; ++r)
                for (int c = 0; c < 3; ++c) S.ax[r * 3 + c] = V[r][c];
        }
        wave_sync();
        double ax[9];
#pragma unroll
        for (int t = 0; t < 9; ++t) ax[t] = S.ax[t];
        // OBB::CreateAABBfromPoints (OBB.cpp:105-166); each lane visits its
        // points in increasing order, as the tie rules below assume
        double lo[3], hi[3];
        int loi[3], hii[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            lo[q] = INFINITY;
            hi[q] = -INFINITY;
            loi[q] = -1;
            hii[q] = -1;
        }
        for (uint32_t k0 = 0; k0 < npts; k0 += 64u * GROUP) {
            float px[GROUP], py[GROUP], pz[GROUP];
#pragma unroll
            for (int j = 0; j < GROUP; ++j) {
                const size_t k = min(k0 + 64u * j + uint32_t(lane), npts - 1);
                px[j] = P[3 * k];
                py[j] = P[3 * k + 1];
                pz[j] = P[3 * k + 2];
            }
#pragma unroll
            for (int j = 0; j < GROUP; ++j) {
                const uint32_t k = k0 + 64u * j + uint32_t(lane);
                if (k < npts) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        double pr = (ax[3 * q] * double(px[j]) + ax[3 * q + 1] * double(py[j])) +
                                    ax[3 * q + 2] * double(pz[j]);
                        if (!(lo[q] < pr)) { lo[q] = pr; loi[q] = int(k); }
                        if (hi[q] < pr) { hi[q] = pr; hii[q] = int(k); }
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            wave_min_last(lo[q], loi[q]);
            wave_max_first(hi[q], hii[q]);
        }
        if (lane == 0) box_of_extents(ax, lo, hi, S.box);
        wave_sync();
        box = box_from12(S.box);
    }
    if (lane == 0) {
        box_to12(box, nd->box);
        nd->surf = surface(box);
    }

    const Excess ex(box);
    double worst = 0.0, rad2 = 0.0;
    auto post = [&]() {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            worst = fmax(worst, __shfl_xor(worst, off, 64));
            rad2 = fmax(rad2, __shfl_xor(rad2, off, 64));
        }
        if (lane == 0) post_excess(a, *nd, ni, worst, rad2);
    };

    // ---- leaf: park the triangles in their final slots ----
    if (n <= a.leaf_max) {
        for (uint32_t t = lane; t < n; t += 64) {
            float T[9];
#pragma unroll
            for (int q = 0; q < 9; ++q) T[q] = P[size_t(t) * 9 + q];
#pragma unroll
            for (int q = 0; q < 9; ++q) a.pos_fin[size_t(beg + t) * 9 + q] = T[q];
            a.id_fin[beg + t] = a.id_in[beg + t];
            ex.take(T, worst, rad2);
        }
        post();
        if (lane == 0) {
            nd->flags = 1u;
            nd->icount = 0;
            nd->tcount = n;
        }
        return;
    }

    // ---- split (OBBtree.cpp:43-108): the longest axis whose centre
    // projection leaves both sides non-empty, else index halves; the three
    // candidates are counted in one scan ----
    AxisCand cand[3];
    float cp[3];
    split_candidates(box, cand, cp);
    uint32_t cnt[3] = {0, 0, 0};
    for (uint32_t c0 = 0; c0 < n; c0 += 64u * GROUP) {
        float T[GROUP][9];
        load_tris(P, c0, n, lane, T);
#pragma unroll
        for (int j = 0; j < GROUP; ++j) {
            const bool valid = c0 + 64u * j + uint32_t(lane) < n;
            if (valid) ex.take(T[j], worst, rad2);
#pragma unroll
            for (int ch = 0; ch < 3; ++ch)
                cnt[ch] += uint32_t(__popcll(__ballot(valid && goes_left(T[j], cand[ch].dir, cp[ch]))));
        }
    }
    post();
    const int pick = split_pick(cnt, n);
    const bool ok = pick >= 0;
    f3 axis = cand[0].dir;
    float cproj = 0.f;
    uint32_t nl = n / 2;  // index halves (OBBtree.cpp:81-93)
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
        if (ch == pick) {
            axis = cand[ch].dir;
            cproj = cp[ch];
            nl = cnt[ch];
        }
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    uint32_t runL = 0, runR = 0;
    for (uint32_t c0 = 0; c0 < n; c0 += 64u * GROUP) {
        float T[GROUP][9];
        load_tris(P, c0, n, lane, T);
        uint32_t idv[GROUP];
#pragma unroll
        for (int j = 0; j < GROUP; ++j) {
            const uint32_t i = c0 + 64u * j + uint32_t(lane);
            idv[j] = a.id_in[beg + min(i, n - 1)];
        }
#pragma unroll
        for (int j = 0; j < GROUP; ++j) {
            const uint32_t i = c0 + 64u * j + uint32_t(lane);
            const bool valid = i < n;
            const bool left = valid && (ok ? goes_left(T[j], axis, cproj) : (i < n / 2));
            const unsigned long long mL = __ballot(left);
            const unsigned long long mR = __ballot(valid && !left);
            if (valid) {
                const uint32_t dst = left ? beg + runL + uint32_t(__popcll(mL & below))
                                          : beg + nl + runR + uint32_t(__popcll(mR & below));
                float* o = a.pos_out + size_t(dst) * 9;
#pragma unroll
                for (int t = 0; t < 9; ++t) o[t] = T[j][t];
                a.id_out[dst] = idv[j];
            }
            runL += uint32_t(__popcll(mL));
            runR += uint32_t(__popcll(mR));
        }
    }
    if (lane == 0) append_kids(a, nd, nl, next_first, next_count);
}

// Nodes of few triangles, one lane each, on levels of at least TINY_LEVEL
// nodes: the deepest levels of a large build hold most of its nodes, and a
// wavefront per node of a few triangles leaves most lanes idle and runs eig3
// on one of them (level load of 13 meshes: levels of 60,000 nodes 250-450 us,
// 60-80 a lane each).  A lane takes about 50 us over its node, so smaller
// levels, whose wavefronts all run at once or nearly so, keep them: 30,000
// nodes 168 us against 163, 15,000 139 against 136, 2,000 to 8,000 33-57
// against 80-100.  Each lane runs the reference's loops as they are written.
constexpr uint32_t TINY_TRIS = 16;
constexpr uint32_t TINY_LEVEL = 32768;

// One triangle's coordinates at a time, TINY_FETCH in flight (indices clamped, as above).
constexpr uint32_t TINY_FETCH = 3;
template <class F>
__device__ __forceinline__ void tiny_tris(const float* __restrict__ P, uint32_t n, F f) {
    for (uint32_t i0 = 0; i0 < n; i0 += TINY_FETCH) {
        float T[TINY_FETCH][9];
#pragma unroll
        for (uint32_t j = 0; j < TINY_FETCH; ++j) {
            const float* p = P + 9 * size_t(min(i0 + j, n - 1));
#pragma unroll
            for (int q = 0; q < 9; ++q) T[j][q] = p[q];
        }
#pragma unroll
        for (uint32_t j = 0; j < TINY_FETCH; ++j)
            if (i0 + j < n) f(i0 + j, T[j]);
    }
}

__global__ __launch_bounds__(64) void k_level_tiny(LevelArgs a, uint4* lv) {
    const uint32_t first = lv[0].x, count = lv[0].y, next_first = first + count;
    if (count < TINY_LEVEL) return;
    const uint32_t lane = threadIdx.x;
    for (uint32_t b0 = blockIdx.x * 64u; b0 < count; b0 += gridDim.x * 64u) {
        const uint32_t ni = first + b0 + lane;
        BNode* nd = nullptr;
        uint32_t beg = 0, n = 0;
        if (b0 + lane < count) {
            nd = &a.nodes[ni];
            beg = nd->beg;
            n = nd->end - beg;
            if (n > TINY_TRIS || n == 0) nd = nullptr;  // the other passes' (an empty mesh's root is the wavefronts')
        }
        if (!nd) n = 0;
        const float* P = a.pos_in + size_t(beg) * 9;
        double worst = 0.0, rad2 = 0.0;
        uint32_t nl = 0;
        bool splits = false;
        if (nd) {
            bool multi = false;
            double m[3] = {0.0, 0.0, 0.0};
            const float x0 = P[0], y0 = P[1], z0 = P[2];
            tiny_tris(P, n, [&](uint32_t, const float (&T)[9]) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    multi |= !(T[3 * k] == x0 && T[3 * k + 1] == y0 && T[3 * k + 2] == z0);
#pragma unroll
                    for (int q = 0; q < 3; ++q) m[q] = m[q] + double(T[3 * k + q]);
                }
            });
            Box box = empty_box(mk(x0, y0, z0));
            if (multi) {
                const double N = double(3 * n);
                m[0] = m[0] / N;
                m[1] = m[1] / N;
                m[2] = m[2] / N;
                double c[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};  // xx, yy, zz, xy, xz, yz (OBB.cpp:56-73)
                tiny_tris(P, n, [&](uint32_t, const float (&T)[9]) {
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const double dx = double(T[3 * k]) - m[0], dy = double(T[3 * k + 1]) - m[1],
                                     dz = double(T[3 * k + 2]) - m[2];
                        c[0] = c[0] + dx * dx;
                        c[1] = c[1] + dy * dy;
                        c[2] = c[2] + dz * dz;
                        c[3] = c[3] + dx * dy;
                        c[4] = c[4] + dx * dz;
                        c[5] = c[5] + dy * dz;
                    }
                });
#pragma unroll
                for (int k = 0; k < 6; ++k) c[k] = c[k] / N;
                double A[3][3] = {{c[0], c[3], c[4]}, {c[3], c[1], c[5]}, {c[4], c[5], c[2]}};
                double V[3][3], d[3], ax[9];
                eig3(A, V, d);
                for (int r = 0; r < 3; ++r)
                    for (int q = 0; q < 3; ++q) ax[r * 3 + q] = V[r][q];
                double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
                tiny_tris(P, n, [&](uint32_t, const float (&T)[9]) {
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int q = 0; q < 3; ++q) {
                            const double pr = (ax[3 * q] * double(T[3 * k]) + ax[3 * q + 1] * double(T[3 * k + 1])) +
                                              ax[3 * q + 2] * double(T[3 * k + 2]);
                            if (!(lo[q] < pr)) lo[q] = pr;
                            if (hi[q] < pr) hi[q] = pr;
                        }
                });
                float bx[12];
                box_of_extents(ax, lo, hi, bx);
                box = box_from12(bx);
            }
            box_to12(box, nd->box);
            nd->surf = surface(box);
            const Excess ex(box);
            if (n <= a.leaf_max) {
                tiny_tris(P, n, [&](uint32_t i, const float (&T)[9]) {
                    ex.take(T, worst, rad2);
                    float* o = a.pos_fin + size_t(beg + i) * 9;
#pragma unroll
                    for (int q = 0; q < 9; ++q) o[q] = T[q];
                    a.id_fin[beg + i] = a.id_in[beg + i];
                });
                nd->flags = 1u;
                nd->icount = 0;
                nd->tcount = n;
            } else {
                splits = true;
                AxisCand cand[3];
                float cp[3];
                split_candidates(box, cand, cp);
                uint32_t cnt[3] = {0, 0, 0};
                tiny_tris(P, n, [&](uint32_t, const float (&T)[9]) {
                    ex.take(T, worst, rad2);
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch) cnt[ch] += goes_left(T, cand[ch].dir, cp[ch]) ? 1u : 0u;
                });
                const int pick = split_pick(cnt, n);
                f3 axis = cand[0].dir;
                float cproj = 0.f;
                nl = n / 2;
#pragma unroll
                for (int ch = 0; ch < 3; ++ch)
                    if (ch == pick) {
                        axis = cand[ch].dir;
                        cproj = cp[ch];
                        nl = cnt[ch];
                    }
                uint32_t l = beg, r = beg + nl;
                tiny_tris(P, n, [&](uint32_t i, const float (&T)[9]) {
                    const bool left = pick >= 0 ? goes_left(T, axis, cproj) : i < n / 2;
                    const uint32_t dst = left ? l++ : r++;
                    float* o = a.pos_out + size_t(dst) * 9;
#pragma unroll
                    for (int q = 0; q < 9; ++q) o[q] = T[q];
                    a.id_out[dst] = a.id_in[beg + i];
                });
            }
        }
        // the wavefront's children take one atomic, and so do its excesses
        // when its nodes are one mesh's below the root
        const unsigned long long live = __ballot(nd != nullptr), kids = __ballot(splits);
        if (!live) continue;
        uint32_t slot = 0;
        if (kids) {
            if (lane == 0) slot = atomicAdd(&lv[1].y, 2u * uint32_t(__popcll(kids)));
            slot = uint32_t(__builtin_amdgcn_readfirstlane(int(slot)));
            slot += next_first + 2u * uint32_t(__popcll(kids & (lane == 0 ? 0ull : (~0ull >> (64 - lane)))));
            if (splits) place_kids(a, nd, nl, slot);
        }
        const int src = __builtin_ctzll(live);
        const uint32_t mesh = nd ? nd->mesh : 0u, level = nd ? nd->level : 0u;
        const uint32_t mesh0 = uint32_t(__shfl(int(mesh), src, 64)), level0 = uint32_t(__shfl(int(level), src, 64));
        if (level0 > 0 && __ballot(nd && mesh != mesh0) == 0) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) worst = fmax(worst, __shfl_xor(worst, off, 64));
            if (int(lane) == src) {
                post_excess(a, *nd, ni, worst, rad2);
                if (kids) atomicMax(&a.mesh_depth[mesh], level + 1);
            }
        } else if (nd) {
            post_excess(a, *nd, ni, worst, rad2);
            if (splits) atomicMax(&a.mesh_depth[mesh], level + 1);
        }
    }
}

// One level of the build: lv[0] = {first node, node count, big nodes, tiles}
// of this level (written by the previous level's launches or by the host);
// the launch writes lv[1] = {first node, count, ..} of the next, its count
// grown by two per split.  A fixed grid strides over the level's nodes, so levels can be
// launched back to back before their sizes are known on the host.
__global__ __launch_bounds__(64) void k_level(LevelArgs a, uint4* lv) {
    __shared__ LevelShared S;
    const uint32_t first = lv[0].x, count = lv[0].y;
    const uint32_t next_first = first + count;
    if (blockIdx.x == 0 && threadIdx.x == 0) lv[1].x = next_first;
    const bool tiny = count >= TINY_LEVEL;  // k_level_tiny takes the nodes of few triangles
    for (uint32_t b = blockIdx.x; b < count; b += gridDim.x) {
        const BNode& nd = a.nodes[first + b];
        const uint32_t n = nd.end - nd.beg;
        if (n > a.big_min || (tiny && n <= TINY_TRIS && n > 0)) continue;
        level_node(a, first + b, next_first, &lv[1].y, S);
        wave_sync();  // the next node reuses the LDS
    }
}

}  // namespace cdk
#include "bigbuild.hpp"
namespace cdk {

// Left child = larger surface (OBBtree.cpp:101-107).
__global__ void k_order_kids(BNode* nodes, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    BNode* nd = &nodes[i];
    if (nd->flags & 1u) return;
    const uint32_t l = nd->kid[0], r = nd->kid[1];
    if (nodes[r].surf > nodes[l].surf) {
        nd->kid[0] = r;
        nd->kid[1] = l;
    }
}

// Subtree sizes, one level at a time from the bottom.
__global__ void k_counts(BNode* nodes, uint32_t first, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    BNode* nd = &nodes[first + i];
    if (nd->flags & 1u) return;
    const BNode& l = nodes[nd->kid[0]];
    const BNode& r = nodes[nd->kid[1]];
    nd->icount = 1 + l.icount + r.icount;
    nd->tcount = l.tcount + r.tcount;
}

// Preorder index and DFS triangle offset, one level at a time from the top
// (OBBtree.cpp:179-233, :385-394).
__global__ void k_preorder(BNode* nodes, uint32_t first, uint32_t count) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const BNode& nd = nodes[first + i];
    if (nd.flags & 1u) return;
    BNode& l = nodes[nd.kid[0]];
    BNode& r = nodes[nd.kid[1]];
    l.pre = nd.pre + 1;
    l.toff = nd.toff;
    r.pre = nd.pre + 1 + l.icount;
    r.toff = nd.toff + l.tcount;
}

// The three passes above in one workgroup, for builds of up to
// FLATTEN_SMALL nodes: one launch instead of one per level and pass.
// lv[l] = {first node, count} of level l.
constexpr uint32_t FLATTEN_SMALL = 1u << 16;
__global__ __launch_bounds__(1024) void k_flatten_small(BNode* nodes, uint32_t total, const uint2* lv, uint32_t nlev) {
    for (uint32_t i = threadIdx.x; i < total; i += blockDim.x) {
        BNode* nd = &nodes[i];
        if (nd->flags & 1u) continue;
        const uint32_t l = nd->kid[0], r = nd->kid[1];
        if (nodes[r].surf > nodes[l].surf) {
            nd->kid[0] = r;
            nd->kid[1] = l;
        }
    }
    __syncthreads();
    for (uint32_t k = nlev; k-- > 0;) {
        for (uint32_t i = threadIdx.x; i < lv[k].y; i += blockDim.x) {
            BNode* nd = &nodes[lv[k].x + i];
            if (nd->flags & 1u) continue;
            const BNode& l = nodes[nd->kid[0]];
            const BNode& r = nodes[nd->kid[1]];
            nd->icount = 1 + l.icount + r.icount;
            nd->tcount = l.tcount + r.tcount;
        }
        __syncthreads();
    }
    for (uint32_t k = 0; k < nlev; ++k) {
        for (uint32_t i = threadIdx.x; i < lv[k].y; i += blockDim.x) {
            const BNode& nd = nodes[lv[k].x + i];
            if (nd.flags & 1u) continue;
            BNode& l = nodes[nd.kid[0]];
            BNode& r = nodes[nd.kid[1]];
            l.pre = nd.pre + 1;
            l.toff = nd.toff;
            r.pre = nd.pre + 1 + l.icount;
            r.toff = nd.toff + l.tcount;
        }
        __syncthreads();
    }
}

__global__ void k_emit_nodes(const BNode* nodes, uint32_t count, const uint32_t* node_base, NodeRec* out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const BNode& nd = nodes[i];
    if (nd.flags & 1u) return;
    NodeRec rec;
    for (int s = 0; s < 2; ++s) {
        const BNode& k = nodes[nd.kid[s]];
        ChildRec& c = rec.c[s];
        for (int t = 0; t < 12; ++t) c.box[t] = k.box[t];
        c.surf = k.surf;
        const bool leaf = (k.flags & 1u) != 0u;
        c.link = leaf ? k.toff : k.pre;
        c.tris = k.tcount | (leaf ? LEAF_BIT : 0u);
        c.toff = k.toff;
    }
    out[node_base[nd.mesh] + nd.pre] = rec;
}

__global__ void k_emit_tris(const BNode* nodes, uint32_t count, const uint32_t* tri_base, const float* pos_fin,
                            const uint32_t* id_fin, float* tris, uint32_t* perm, uint32_t* leafof) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const BNode& nd = nodes[i];
    if (!(nd.flags & 1u)) return;
    const size_t dst0 = size_t(tri_base[nd.mesh]) + nd.toff;
    for (uint32_t t = 0; t < nd.tcount; ++t) {
        const float* s = pos_fin + size_t(nd.beg + t) * 9;
        float* o = tris + (dst0 + t) * 9;
        for (int q = 0; q < 9; ++q) o[q] = s[q];
        perm[dst0 + t] = id_fin[nd.beg + t];
        leafof[dst0 + t] = nd.toff;  // the leaf's first slot names the leaf
    }
}

#define CK(x)                                                        \
    do {                                                             \
        hipError_t e_ = (x);                                         \
        if (e_ != hipSuccess) {                                      \
            res.err = std::string(#x ": ") + hipGetErrorString(e_);  \
            goto fail;                                               \
        }                                                            \
    } while (0)

static inline uint32_t blocks_for(uint64_t n, uint32_t b) { return uint32_t((n + b - 1) / b); }

constexpr uint32_t LEVEL_BATCH = 8;     // level launches per wait of the build
constexpr uint32_t LEVEL_GRID = 8192;  // workgroups of a level launch at most (larger levels are strided)

// Build every soup of the batch and append the trees to the context arenas.
BuildResult build_soups(cd_ctx* ctx, const float* tri9, const uint32_t* counts, uint32_t nmesh, bool tri9_on_device) {
    BuildResult res;
    hipStream_t st = ctx->stream;
    uint64_t T = 0, node_cap = 0;
    std::vector<uint64_t> tri_begin(nmesh);
    for (uint32_t m = 0; m < nmesh; ++m) {
        tri_begin[m] = T;
        T += counts[m];
        node_cap += counts[m] ? 2ull * counts[m] - 1 : 1;
    }
    if (T >= 0xFFFFFFF0ull || node_cap >= 0xFFFFFFF0ull) {
        res.err = "batch too large (triangle or node count exceeds 32-bit indexing)";
        return res;
    }
    // work buffers, kept in the context between builds of up to BUILD_KEEP bytes
    DevBuf* const W = ctx->build_scratch;
    DevBuf* const pos = W;      // pos[0], pos[1]
    DevBuf* const ids = W + 2;  // ids[0], ids[1]
    DevBuf &pos_fin = W[4], &id_fin = W[5], &nodes = W[6], &mesh_depth = W[7], &level_tab = W[8], &base_nodes = W[9],
           &base_tris = W[10], &slack_bits = W[11], &radius_bits = W[12], &level_list = W[13];
    DevBuf& big_work = W[14];  // all of the tiled passes' arrays: one allocation
    std::vector<BNode> roots(nmesh);
    std::vector<std::pair<uint32_t, uint32_t>> levels;
    std::vector<uint32_t> host_ids;
    std::vector<uint32_t> node_base(nmesh), tri_base(nmesh), depth(nmesh), slack(size_t(nmesh) * SLACK_REPS),
        radius(nmesh);
    uint64_t total_internal = 0;
    uint32_t first = 0, count = nmesh, cur = 0;
    // the roots that take the tiled passes; every level's big nodes are
    // disjoint, so their number and their tiles are bounded once
    const uint32_t largest = nmesh ? *std::max_element(counts, counts + nmesh) : 0u;
    uint32_t big_min = largest > BIG_BUILD ? std::max(BIG_TRIS, ctx->leaf_max) : 0xFFFFFFFFu;
    std::vector<BigNode> bigs;
    std::vector<uint2> tiles;
    for (uint32_t m = 0; m < nmesh; ++m) {
        if (counts[m] <= big_min) continue;
        for (uint32_t k = 0; k < big_tiles(counts[m]); ++k) tiles.push_back(make_uint2(uint32_t(bigs.size()), k));
        bigs.push_back({m, uint32_t(tri_begin[m]), counts[m], uint32_t(tiles.size()) - big_tiles(counts[m])});
    }
    uint32_t nbig = uint32_t(bigs.size()), ntiles = uint32_t(tiles.size());
    BigArgs big_args{};
    BigNode* big_list[2] = {};
    uint2* tile_list[2] = {};
    const size_t big_cap = size_t(T / big_min) + 1, tile_cap = size_t(T / TILE_TRIS) + big_cap;
    const size_t posb = std::max<uint64_t>(T, 1) * 9 * sizeof(float), idb = std::max<uint64_t>(T, 1) * sizeof(uint32_t);

    CK(pos[0].ensure(posb));
    CK(pos[1].ensure(posb));
    CK(pos_fin.ensure(posb));
    CK(ids[0].ensure(idb));
    CK(ids[1].ensure(idb));
    CK(id_fin.ensure(idb));
    CK(nodes.ensure(node_cap * sizeof(BNode)));
    CK(mesh_depth.ensure(nmesh * sizeof(uint32_t)));
    CK(slack_bits.ensure(size_t(nmesh) * SLACK_REPS * sizeof(uint32_t)));
    CK(radius_bits.ensure(nmesh * sizeof(uint32_t)));
    CK(level_tab.ensure((LEVEL_BATCH + 1) * sizeof(uint4)));
    if (!bigs.empty()) {
        size_t at = 0;
        auto place = [&at](size_t bytes) {
            const size_t here = at;
            at += (bytes + 255) & ~size_t(255);
            return here;
        };
        const size_t o_state = place(big_cap * sizeof(BigState)), o_sums = place(tile_cap * sizeof(TileSums)),
                     o_ext = place(tile_cap * sizeof(TileExtents)), o_cnt = place(tile_cap * sizeof(uint4)),
                     o_fn = place(tile_cap * 6 * 128 * sizeof(double2));
        size_t o_big[2], o_tiles[2];
        for (int k = 0; k < 2; ++k) {
            o_big[k] = place(big_cap * sizeof(BigNode));
            o_tiles[k] = place(tile_cap * sizeof(uint2));
        }
        if (big_work.ensure(at) != hipSuccess) {  // no room for them: a wavefront per node, which needs none
            (void)hipGetLastError();
            big_min = 0xFFFFFFFFu;
            nbig = ntiles = 0;
        }
        char* const base = big_work.as<char>();
        big_args.state = reinterpret_cast<BigState*>(base + o_state);
        big_args.sums = reinterpret_cast<TileSums*>(base + o_sums);
        big_args.ext = reinterpret_cast<TileExtents*>(base + o_ext);
        big_args.counts = reinterpret_cast<uint4*>(base + o_cnt);
        big_args.fn = reinterpret_cast<double2*>(base + o_fn);
        big_args.tile_cap = uint32_t(tile_cap);
        for (int k = 0; k < 2; ++k) {  // a level's big nodes and their tiles, and the next level's
            big_list[k] = reinterpret_cast<BigNode*>(base + o_big[k]);
            tile_list[k] = reinterpret_cast<uint2*>(base + o_tiles[k]);
        }
        if (nbig) {
            CK(hipMemcpyAsync(big_list[0], bigs.data(), bigs.size() * sizeof(BigNode), hipMemcpyHostToDevice, st));
            CK(hipMemcpyAsync(tile_list[0], tiles.data(), tiles.size() * sizeof(uint2), hipMemcpyHostToDevice, st));
        }
    }
    CK(base_nodes.ensure(nmesh * sizeof(uint32_t)));
    CK(base_tris.ensure(nmesh * sizeof(uint32_t)));

    if (T)
        CK(hipMemcpyAsync(pos[0].p, tri9, T * 9 * sizeof(float),
                          tri9_on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, st));
    host_ids.resize(T);
    for (uint32_t m = 0; m < nmesh; ++m)
        for (uint32_t k = 0; k < counts[m]; ++k) host_ids[tri_begin[m] + k] = k;
    if (T) CK(hipMemcpyAsync(ids[0].p, host_ids.data(), T * sizeof(uint32_t), hipMemcpyHostToDevice, st));
    for (uint32_t m = 0; m < nmesh; ++m) {
        BNode r{};
        r.mesh = m;
        r.beg = uint32_t(tri_begin[m]);
        r.end = uint32_t(tri_begin[m] + counts[m]);
        r.level = 0;
        r.pre = 0;
        r.toff = 0;
        roots[m] = r;
    }
    CK(hipMemcpyAsync(nodes.p, roots.data(), nmesh * sizeof(BNode), hipMemcpyHostToDevice, st));
    CK(hipMemsetAsync(mesh_depth.p, 0, nmesh * sizeof(uint32_t), st));
    CK(hipMemsetAsync(slack_bits.p, 0, size_t(nmesh) * SLACK_REPS * sizeof(uint32_t), st));
    CK(hipMemsetAsync(radius_bits.p, 0, nmesh * sizeof(uint32_t), st));

    // Levels go LEVEL_BATCH launches at a time with one wait per batch: each
    // launch takes its node range from the level table the previous one
    // filled, over a grid sized by an upper bound (a level at most doubles).
    while (count > 0) {
        std::vector<uint4> tab(LEVEL_BATCH + 1, make_uint4(0u, 0u, 0u, 0u));
        tab[0] = make_uint4(first, count, nbig, ntiles);
        CK(hipMemcpyAsync(level_tab.p, tab.data(), tab.size() * sizeof(uint4), hipMemcpyHostToDevice, st));
        uint64_t big_bound = nbig;
        // with big nodes about, as many levels as halving the largest there can be takes to end them
        uint32_t batch = LEVEL_BATCH;
        if (nbig) {
            batch = 1;
            while (batch < LEVEL_BATCH && (uint64_t(ntiles) * TILE_TRIS >> batch) > big_min) ++batch;
        }
        uint64_t bound = count;
        for (uint32_t j = 0; j < batch; ++j) {
            LevelArgs a;
            a.nodes = nodes.as<BNode>();
            a.pos_in = pos[cur].as<float>();
            a.id_in = ids[cur].as<uint32_t>();
            a.pos_out = pos[cur ^ 1].as<float>();
            a.id_out = ids[cur ^ 1].as<uint32_t>();
            a.pos_fin = pos_fin.as<float>();
            a.id_fin = id_fin.as<uint32_t>();
            a.mesh_depth = mesh_depth.as<unsigned int>();
            a.slack_bits = slack_bits.as<unsigned int>();
            a.radius_bits = radius_bits.as<unsigned int>();
            a.leaf_max = ctx->leaf_max;
            a.big_min = big_min;
            uint4* const lv = level_tab.as<uint4>() + j;
            if (big_bound) {
                BigArgs b = big_args;
                b.lv = a;
                b.big = big_list[cur];
                b.tiles = tile_list[cur];
                b.big_out = big_list[cur ^ 1];
                b.tiles_out = tile_list[cur ^ 1];
                // big nodes at most double per level; a tile list holds at most tile_cap entries
                const uint32_t gn = uint32_t(std::min<uint64_t>(big_bound, big_cap));
                const uint32_t gt = uint32_t(std::min<uint64_t>(ntiles + big_bound, tile_cap));
                hipLaunchKernelGGL(k_big_sums, dim3(gt), dim3(256), 0, st, b, lv);
                hipLaunchKernelGGL(k_big_sim<3>, dim3(gt), dim3(192), 0, st, b, lv);
                hipLaunchKernelGGL(k_big_resolve<3>, dim3(3 * gn), dim3(64 * (1 + RESOLVE_TILES)), 0, st, b, lv);
                hipLaunchKernelGGL(k_big_sim<6>, dim3(gt), dim3(384), 0, st, b, lv);
                hipLaunchKernelGGL(k_big_resolve<6>, dim3(6 * gn), dim3(64 * (1 + RESOLVE_TILES)), 0, st, b, lv);
                hipLaunchKernelGGL(k_big_project, dim3(gt), dim3(256), 0, st, b, lv);
                hipLaunchKernelGGL(k_big_count, dim3(gt), dim3(256), 0, st, b, lv);
                hipLaunchKernelGGL(k_big_scatter, dim3(gt), dim3(256), 0, st, b, lv);
                CK(hipGetLastError());
                big_bound *= 2;
            }
            const uint32_t grid = uint32_t(std::min<uint64_t>(bound, LEVEL_GRID));
            hipLaunchKernelGGL(k_level, dim3(grid), dim3(64), 0, st, a, lv);
            if (bound >= TINY_LEVEL) {  // the level's own count decides, on the device
                const uint32_t tiny_grid = std::min<uint32_t>(blocks_for(bound, 64), LEVEL_GRID);
                hipLaunchKernelGGL(k_level_tiny, dim3(tiny_grid), dim3(64), 0, st, a, lv);
                CK(hipGetLastError());
            }
            cur ^= 1;
            bound = std::min<uint64_t>(2 * bound, node_cap);
        }
        CK(hipMemcpyAsync(tab.data(), level_tab.p, tab.size() * sizeof(uint4), hipMemcpyDeviceToHost, st));
        CK(hipStreamSynchronize(st));
        for (uint32_t j = 0; j < batch && tab[j].y > 0; ++j) levels.push_back({tab[j].x, tab[j].y});
        first = tab[batch].x;
        count = tab[batch].y;
        nbig = tab[batch].z;
        ntiles = tab[batch].w;
    }
    {
        const uint32_t total = first;
        std::vector<uint2> lv;  // read by an asynchronous copy until the wait below
        if (total <= FLATTEN_SMALL) {
            lv.resize(levels.size());
            for (size_t l = 0; l < levels.size(); ++l) lv[l] = make_uint2(levels[l].first, levels[l].second);
            CK(level_list.ensure(std::max<size_t>(lv.size(), 1) * sizeof(uint2)));
            CK(hipMemcpyAsync(level_list.p, lv.data(), lv.size() * sizeof(uint2), hipMemcpyHostToDevice, st));
            hipLaunchKernelGGL(k_flatten_small, dim3(1), dim3(1024), 0, st, nodes.as<BNode>(), total,
                               level_list.as<uint2>(), uint32_t(lv.size()));
            CK(hipGetLastError());
        } else {
            hipLaunchKernelGGL(k_order_kids, dim3(blocks_for(total, 256)), dim3(256), 0, st, nodes.as<BNode>(), total);
            CK(hipGetLastError());
            for (size_t l = levels.size(); l-- > 0;) {
                hipLaunchKernelGGL(k_counts, dim3(blocks_for(levels[l].second, 256)), dim3(256), 0, st,
                                   nodes.as<BNode>(), levels[l].first, levels[l].second);
                CK(hipGetLastError());
            }
            for (size_t l = 0; l < levels.size(); ++l) {
                hipLaunchKernelGGL(k_preorder, dim3(blocks_for(levels[l].second, 256)), dim3(256), 0, st,
                                   nodes.as<BNode>(), levels[l].first, levels[l].second);
                CK(hipGetLastError());
            }
        }
        CK(hipMemcpyAsync(roots.data(), nodes.p, nmesh * sizeof(BNode), hipMemcpyDeviceToHost, st));
        CK(hipMemcpyAsync(depth.data(), mesh_depth.p, nmesh * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
        CK(hipStreamSynchronize(st));
        for (uint32_t m = 0; m < nmesh; ++m) {
            node_base[m] = uint32_t(ctx->nodes_used + total_internal);
            total_internal += roots[m].icount;
            tri_base[m] = uint32_t(ctx->tris_used + tri_begin[m]);
        }
        // node indices travel as (node << 1) | side below a flag bit in the batched traversal
        if (ctx->nodes_used + total_internal >= (1ull << 30) || ctx->tris_used + T >= 0xFFFFFFF0ull) {
            res.err = "arena exceeds 32-bit indexing (at most 2^30 internal nodes)";
            goto fail;
        }
        // grow the arenas (keeping what is already registered)
        auto grow = [&](DevBuf& b, size_t need) -> hipError_t {
            if (need <= b.bytes) return hipSuccess;
            size_t want = std::max(need, b.bytes * 2);
            void* np = nullptr;
            hipError_t e = hipMalloc(&np, want);
            if (e != hipSuccess) return e;
            if (b.p) {
                e = hipMemcpyAsync(np, b.p, b.bytes, hipMemcpyDeviceToDevice, st);
                if (e != hipSuccess) return e;
                e = hipStreamSynchronize(st);
                if (e != hipSuccess) return e;
                (void)hipFree(b.p);
            }
            b.p = np;
            b.bytes = want;
            return hipSuccess;
        };
        CK(grow(ctx->d_nodes, (ctx->nodes_used + total_internal + 1) * sizeof(NodeRec)));
        CK(grow(ctx->d_tris, (ctx->tris_used + T + 1) * 9 * sizeof(float)));
        CK(grow(ctx->d_perm, (ctx->tris_used + T + 1) * sizeof(uint32_t)));
        CK(grow(ctx->d_leafof, (ctx->tris_used + T + 1) * sizeof(uint32_t)));
        CK(hipMemcpyAsync(base_nodes.p, node_base.data(), nmesh * sizeof(uint32_t), hipMemcpyHostToDevice, st));
        CK(hipMemcpyAsync(base_tris.p, tri_base.data(), nmesh * sizeof(uint32_t), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_emit_nodes, dim3(blocks_for(total, 256)), dim3(256), 0, st, nodes.as<BNode>(), total,
                           base_nodes.as<uint32_t>(), ctx->d_nodes.as<NodeRec>());
        CK(hipGetLastError());
        hipLaunchKernelGGL(k_emit_tris, dim3(blocks_for(total, 256)), dim3(256), 0, st, nodes.as<BNode>(), total,
                           base_tris.as<uint32_t>(), pos_fin.as<float>(), id_fin.as<uint32_t>(), ctx->d_tris.as<float>(),
                           ctx->d_perm.as<uint32_t>(), ctx->d_leafof.as<uint32_t>());
        CK(hipGetLastError());
        CK(hipMemcpyAsync(slack.data(), slack_bits.p, size_t(nmesh) * SLACK_REPS * sizeof(uint32_t),
                          hipMemcpyDeviceToHost, st));
        CK(hipMemcpyAsync(radius.data(), radius_bits.p, nmesh * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
        CK(hipStreamSynchronize(st));
        res.meshes.resize(nmesh);
        for (uint32_t m = 0; m < nmesh; ++m) {
            MeshRec& r = res.meshes[m];
            r.node_base = node_base[m];
            r.tri_base = tri_base[m];
            r.ntri = counts[m];
            r.nnodes = roots[m].icount;
            r.root = ChildRec{};
            std::memcpy(r.root.box, roots[m].box, sizeof r.root.box);
            r.root.surf = roots[m].surf;
            r.root.link = 0;  // node 0, or triangle 0 of a one-leaf tree
            r.root.tris = counts[m] | (roots[m].icount == 0 ? LEAF_BIT : 0u);
            r.root.toff = 0;
            r.depth = depth[m];
            uint32_t sb = 0;  // the largest of the mesh's copies (positive floats order as their bits)
            for (uint32_t k = 0; k < SLACK_REPS; ++k) sb = std::max(sb, slack[size_t(m) * SLACK_REPS + k]);
            std::memcpy(&r.slack, &sb, sizeof(float));
            std::memcpy(&r.radius, &radius[m], sizeof(float));
        }
        ctx->nodes_used += total_internal;
        ctx->tris_used += T;
    }
fail: {
        // the tiled passes' arrays, an eighth of the rest at most, are kept or freed with it and don't count:
        // what a build keeps does not depend on the passes it takes
        size_t kept = 0;
        for (uint32_t k = 0; k < BUILD_SCRATCH; ++k) kept += &W[k] == &big_work ? 0 : W[k].bytes;
        if (!res.err.empty() || kept > BUILD_KEEP)
            for (uint32_t k = 0; k < BUILD_SCRATCH; ++k) W[k].release();
    }
    return res;
}

}  // namespace cdk
