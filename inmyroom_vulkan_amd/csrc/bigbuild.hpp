// The level passes of the tree build for nodes of many triangles
// (included by build.hip).  A node that one wavefront works through costs a
// chain of two double additions per point; the few nodes of the top levels
// hold the whole level and leave the chip idle.  Here a node is cut into
// tiles of TILE_TRIS triangles, one workgroup each, and the sequential sums
// are replayed rather than run:
//
//   k_big_sums     approximate sums and second moments per tile (any order)
//   k_big_sim<3>   per chunk of CHUNK_PTS points and mean chain: the chain
//                  simulated from a guessed start (see ChunkFn)
//   k_big_resolve<3>  the true chains from the chunks: the mean
//   k_big_sim<6>, k_big_resolve<6>  the same for the covariance
//   k_big_project  eig3, extents per tile
//   k_big_count    the box, its slack, the split's three counts per tile
//   k_big_scatter  the stable partition, and the children
//
// Bound: the resolve's chain of runs and single chunks (the covariance of a
// terrain's row-wise triangles swings through zero every row, so 17% of its
// chunks leave their binade).  A level load of 13 meshes, the largest a
// 198,450-triangle terrain: 42.4 -> 13.1 ms; its root node 17.3 -> 2.2 ms.
#pragma once

namespace cdk {

constexpr uint32_t CHUNK_TRIS = 8, CHUNK_PTS = 3 * CHUNK_TRIS;  // points one lane simulates
constexpr uint32_t TILE_TRIS = 64 * CHUNK_TRIS, TILE_PTS = 3 * TILE_TRIS;
constexpr uint32_t CHUNK_FLOATS = 9 * CHUNK_TRIS;
constexpr uint32_t TILE_LDS = 64 * (CHUNK_FLOATS + 1);

// Nodes of more triangles than this take the tiled passes: their eight
// launches cost about 60 us a level, a wavefront about 90 ns a triangle.
// The level load with 512: 12.7, 1,024: 12.6, 2,048: 13.1 ms.
constexpr uint32_t BIG_TRIS = 1024;
// A build takes them when one of its meshes has more than this: below, the
// one or two levels they would shorten do not pay for their buffers.
constexpr uint32_t BIG_BUILD = 2048;

struct BigNode {
    uint32_t node, beg, n, tile0;
};
struct BigState {  // per big node of the level being built
    double mean[3], cov[6], ax[9];
    uint32_t multi, pad;
};
struct TileSums {
    double s[9];  // x, y, z, xx, yy, zz, xy, xz, yz
    uint32_t multi, pad;
};
struct TileExtents {
    double lo[3], hi[3];
    int loi[3], hii[3];
};
struct BigArgs {
    LevelArgs lv;
    const BigNode* big;   // this level's
    const uint2* tiles;   // this level's: {big node, tile within it}
    BigNode* big_out;     // the next level's
    uint2* tiles_out;
    BigState* state;
    TileSums* sums;
    TileExtents* ext;
    uint4* counts;        // per tile: left counts of the three candidates
    double2* fn;          // chunk functions, [chain][tile][2][64]
    uint32_t tile_cap;
};
__host__ __device__ inline uint32_t big_tiles(uint32_t n) { return (n + TILE_TRIS - 1) / TILE_TRIS; }

// A tile's coordinates in LDS; one word of padding per chunk keeps both the
// lane-per-chunk and the lane-per-triangle reads on distinct banks.
__device__ __forceinline__ uint32_t lds_at(uint32_t t) { return t + t / CHUNK_FLOATS; }
__device__ __forceinline__ void load_tile(const float* __restrict__ src, uint32_t nt, float* s) {
    for (uint32_t t = threadIdx.x; t < 9 * nt; t += blockDim.x) s[lds_at(t)] = src[t];
    __syncthreads();
}
__device__ __forceinline__ void tri_of(const float* s, uint32_t i, float (&T)[9]) {
    const uint32_t at = lds_at(9 * i);
#pragma unroll
    for (int q = 0; q < 9; ++q) T[q] = s[at + q];
}

struct BigTile {
    BigNode b;
    uint32_t slot, tile, nt;  // its big node, place in it, triangles
    const float* src;         // its first triangle
};
__device__ __forceinline__ BigTile big_tile(const BigArgs& a, uint32_t i) {
    BigTile t;
    const uint2 e = a.tiles[i];
    t.slot = e.x;
    t.tile = e.y;
    t.b = a.big[e.x];
    t.nt = min(TILE_TRIS, t.b.n - e.y * TILE_TRIS);
    t.src = a.lv.pos_in + (size_t(t.b.beg) + size_t(e.y) * TILE_TRIS) * 9;
    return t;
}

// Sum over a workgroup of up to 16 wavefronts; the result in thread 0.
template <int N>
__device__ __forceinline__ void block_sum(double (&v)[N], double (*s)[N]) {
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[k] = v[k] + __shfl_xor(v[k], off, 64);
    if ((threadIdx.x & 63u) == 0)
#pragma unroll
        for (int k = 0; k < N; ++k) s[threadIdx.x >> 6][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
        for (uint32_t w = 1; w < blockDim.x / 64; ++w)
#pragma unroll
            for (int k = 0; k < N; ++k) v[k] = v[k] + s[w][k];
}

__global__ __launch_bounds__(256) void k_big_sums(BigArgs a, const uint4* lv) {
    __shared__ float s[TILE_LDS];
    __shared__ double s_sum[4][9];
    if (blockIdx.x >= lv[0].w) return;
    const BigTile t = big_tile(a, blockIdx.x);
    load_tile(t.src, t.nt, s);
    const float* P = a.lv.pos_in + size_t(t.b.beg) * 9;
    const float x0 = P[0], y0 = P[1], z0 = P[2];
    double v[9] = {};
    bool multi = false;
    for (uint32_t i = threadIdx.x; i < t.nt; i += blockDim.x) {
        float T[9];
        tri_of(s, i, T);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            multi |= !(T[3 * k] == x0 && T[3 * k + 1] == y0 && T[3 * k + 2] == z0);
            const double x = T[3 * k], y = T[3 * k + 1], z = T[3 * k + 2];
            v[0] += x;
            v[1] += y;
            v[2] += z;
            v[3] += x * x;
            v[4] += y * y;
            v[5] += z * z;
            v[6] += x * y;
            v[7] += x * z;
            v[8] += y * z;
        }
    }
    const int any = __syncthreads_or(multi);
    block_sum(v, s_sum);
    if (threadIdx.x == 0) {
        TileSums& o = a.sums[blockIdx.x];
#pragma unroll
        for (int k = 0; k < 9; ++k) o.s[k] = v[k];
        o.multi = any != 0;
    }
}

// What a chunk's additions do to a running double sum, as a function of the
// sum at its start.  While the sum stays inside one binade [2^e, 2^(e+1))
// (or its negative), every addition rounds to a multiple of the same ulp u,
// half-way cases to the even multiple, so a start moved by an even number of
// ulps moves every partial sum, and the end, by just as much.  A lane
// therefore runs the chunk's additions twice, from a guessed start g and from
// g + u (the other parity), and keeps the two changes (exact: start and end
// are multiples of u in one binade) with the range of starts whose partial
// sums all stay strictly inside the binade:
//   start in [lo, hi], start's last bit 0: end = start + d_even (exact), 1: + d_odd.
// A chunk whose simulation leaves the binade has an empty range; chunks of
// zeros keep any start.  The guess decides only how often the range holds.
struct ChunkFn {
    double d_even, d_odd, lo, hi;
};
__device__ __forceinline__ uint32_t hi32(double v) { return uint32_t(__double2hiint(v)); }
__device__ __forceinline__ uint32_t lo32(double v) { return uint32_t(__double2loint(v)); }
__device__ __forceinline__ uint32_t binade(double v) { return hi32(v) >> 20; }  // sign and exponent

struct ChunkSim {
    double g, g1, r0, r1, mn, mx;
    bool zero = true;
    __device__ explicit ChunkSim(double guess) {
        g = guess;
        g1 = __longlong_as_double(__double_as_longlong(g) + 1);
        r0 = g;
        r1 = g1;
        mn = fmin(g, g1);
        mx = fmax(g, g1);
    }
    __device__ __forceinline__ void add(double t) {
        zero &= t == 0.0;
        r0 = r0 + t;
        r1 = r1 + t;
        mn = fmin(mn, fmin(r0, r1));
        mx = fmax(mx, fmax(r0, r1));
    }
    __device__ ChunkFn result() const {
        ChunkFn f = {0.0, 0.0, -INFINITY, INFINITY};
        if (zero) return f;
        const uint32_t b = binade(g), e = b & 0x7FFu;
        if (e < 64u || e > 2000u || binade(mn) != b || binade(mx) != b) {
            f.lo = INFINITY;
            f.hi = -INFINITY;
            return f;
        }
        const double step = __hiloint2double(int((e - 52u) << 20), 0);  // u
        const double edge = __hiloint2double(int(e << 20), 0);          // 2^e
        const double b_lo = g > 0.0 ? edge : -2.0 * edge, b_hi = g > 0.0 ? 2.0 * edge : -edge;
        // a start of parity p is a_p + t with a_p within u of g: four ulps cover that and both ends' strictness
        f.lo = b_lo + (g - mn) + 4.0 * step;
        f.hi = b_hi - (mx - g) - 4.0 * step;
        const double d0 = r0 - g, d1 = r1 - g1;
        const bool odd = (lo32(g) & 1u) != 0u;
        f.d_even = odd ? d1 : d0;
        f.d_odd = odd ? d0 : d1;
        return f;
    }
};

// Coordinates of the terms of the covariance chains (OBB.cpp:56-73: xx, yy, zz, xy, xz, yz).
__device__ __forceinline__ uint32_t cov_a(uint32_t c) { return c < 3 ? c : (c == 5 ? 1u : 0u); }
__device__ __forceinline__ uint32_t cov_b(uint32_t c) { return c < 3 ? c : (c == 3 ? 1u : 2u); }

// K = 3: mean chains, K = 6: covariance chains; one wavefront per chain, one
// lane per chunk.
template <int K>
__global__ __launch_bounds__(64 * K) void k_big_sim(BigArgs a, const uint4* lv) {
    __shared__ float s[TILE_LDS];
    if (blockIdx.x >= lv[0].w) return;
    const BigTile t = big_tile(a, blockIdx.x);
    const uint32_t lane = threadIdx.x & 63u, c = threadIdx.x >> 6;
    const uint32_t ca = K == 3 ? c : cov_a(c), cb = cov_b(c);
    double ma = 0.0, mb = 0.0;
    if (K == 6) {
        ma = a.state[t.slot].mean[ca];
        mb = a.state[t.slot].mean[cb];
    }
    // the guess at the tile's start: the earlier tiles' sums
    double base = 0.0;
    for (uint32_t k = lane; k < t.tile; k += 64) {
        const TileSums& q = a.sums[t.b.tile0 + k];
        if (K == 3) base += q.s[c];
        else base += q.s[3 + c] - mb * q.s[ca] - ma * q.s[cb] + double(TILE_PTS) * ma * mb;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) base = base + __shfl_xor(base, off, 64);
    load_tile(t.src, t.nt, s);
    const float* p = s + lane * (CHUNK_FLOATS + 1);
    const uint32_t first = lane * CHUNK_PTS, np = 3 * t.nt;
    const uint32_t m = first < np ? min(CHUNK_PTS, np - first) : 0u;
    auto term = [&](uint32_t j) -> double {
        if (j >= m) return 0.0;  // adding +0 changes no sum (none is ever -0)
        if (K == 3) return double(p[3 * j + ca]);
        const double da = double(p[3 * j + ca]) - ma, db = double(p[3 * j + cb]) - mb;
        return da * db;
    };
    double own = 0.0;
#pragma unroll 8
    for (uint32_t j = 0; j < CHUNK_PTS; ++j) own = own + term(j);
    double incl = own;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double up = __shfl_up(incl, off, 64);
        if (lane >= uint32_t(off)) incl = incl + up;
    }
    ChunkSim sim(base + (incl - own));
#pragma unroll 8
    for (uint32_t j = 0; j < CHUNK_PTS; ++j) sim.add(term(j));
    const ChunkFn f = sim.result();
    double2* o = a.fn + (size_t(c) * a.tile_cap + blockIdx.x) * 128 + lane;
    o[0] = make_double2(f.d_even, f.d_odd);
    o[64] = make_double2(f.lo, f.hi);
}

__device__ __forceinline__ double lane_value(double v, uint32_t l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), int(l)),
                            __builtin_amdgcn_readlane(__double2loint(v), int(l)));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v, bool on) {
    const int h = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
    const int l = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
    return v + (on ? __hiloint2double(h, l) : 0.0);
}
// Inclusive sums over runs of lanes, a run starting at every set bit of
// `heads` (bit 0 counts as set): shifts by 1, 2, 4 and 8 within the rows of
// 16, then the row ends carried on (DPP: no LDS round trips), each only from
// lanes of the same run.
__device__ __forceinline__ double run_sums(double v, unsigned long long heads, uint32_t lane) {
    const unsigned long long upto = (heads | 1ull) & (~0ull >> (63 - lane));
    const uint32_t head = 63u - uint32_t(__builtin_clzll(upto));
    v = dpp_add<0x111, 0xf>(v, lane >= head + 1);
    v = dpp_add<0x112, 0xf>(v, lane >= head + 2);
    v = dpp_add<0x114, 0xf>(v, lane >= head + 4);
    v = dpp_add<0x118, 0xf>(v, lane >= head + 8);
    v = dpp_add<0x142, 0xa>(v, (lane & ~15u) > head);  // lane 15 of a row into the next row (rows 1 and 3)
    v = dpp_add<0x143, 0xc>(v, 31u >= head);           // lane 31 into rows 2 and 3
    return v;
}

// The true chains: one workgroup per big node and chain.  Its first wavefront
// takes a tile's 64 chunk functions at a time.  Runs of chunks in one binade
// whose change does not depend on the parity are summed over the lanes once
// per tile; from a run's true start every chunk's start follows, and all that
// lie in their ranges are done at once (the sums are exact up to the first
// that does not: each is a difference of two partial sums of the chain).  A
// chunk in no run, or outside its range, is applied by itself, by its parity
// or point by point.  The other wavefronts bring the next RESOLVE_TILES tiles'
// functions into LDS meanwhile, and the terms of the chunks whose range is
// empty: both come from memory that other XCDs wrote, and one wavefront
// fetching for itself waited 2.7 us per tile.
constexpr uint32_t RESOLVE_TILES = 4, STAGED = 64;
struct ResolveTile {
    double2 d[64], w[64];
    double term[STAGED][CHUNK_PTS];  // of the chunks with an empty range, in order
};
template <int K>
__global__ __launch_bounds__(64 * (1 + RESOLVE_TILES)) void k_big_resolve(BigArgs a, const uint4* lv) {
    __shared__ ResolveTile s_tile[2][RESOLVE_TILES];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
    const uint32_t slot = blockIdx.x / K, c = blockIdx.x % K;
    const uint32_t ca = K == 3 ? c : cov_a(c), cb = cov_b(c);
    if (slot >= lv[0].z) return;
    const BigNode b = a.big[slot];
    BigState& st = a.state[slot];
    const uint32_t ntile = big_tiles(b.n), npts = 3 * b.n;
    const uint32_t nstep = (ntile + RESOLVE_TILES - 1) / RESOLVE_TILES;
    const float* P = a.lv.pos_in + size_t(b.beg) * 9;
    double ma = 0.0, mb = 0.0;
    if (K == 6) {
        ma = st.mean[ca];
        mb = st.mean[cb];
    }
    // point l of chunk h of tile t; +0 past the node's points (adding it changes no sum: none is ever -0)
    auto load = [&](uint32_t t, uint32_t h, uint32_t l, float& xa, float& xb) -> bool {
        const size_t k = size_t(t) * TILE_PTS + h * CHUNK_PTS + l;
        const size_t q = 3 * min(k, size_t(npts - 1));
        xa = P[q + ca];
        xb = K == 6 ? P[q + cb] : 0.f;
        return l < CHUNK_PTS && k < npts;
    };
    auto term = [&](float xa, float xb) -> double {
        return K == 3 ? double(xa) : (double(xa) - ma) * (double(xb) - mb);
    };
    // A fetching wavefront keeps two loads in flight over every step: the
    // terms of its tile of the next step (IN_FLIGHT pairs of chunks), and its
    // functions of the step after that.
    constexpr int IN_FLIGHT = 8;
    const double2* fn = a.fn + (size_t(c) * a.tile_cap + b.tile0) * 128 + lane;
    double2 d = make_double2(0.0, 0.0), w = d, d2 = d, w2 = d;
    float xa[IN_FLIGHT], xb[IN_FLIGHT];
    bool in[IN_FLIGHT];
    unsigned long long open = 0;
    auto functions = [&](uint32_t step) {
        const size_t t = min(step * RESOLVE_TILES + (wave - 1), ntile - 1);
        d2 = fn[t * 128];
        w2 = fn[t * 128 + 64];
    };
    auto terms = [&](uint32_t t) {
#pragma unroll
        for (int i = 0; i < IN_FLIGHT; ++i) {  // two chunks per load
            const uint32_t h0 = open ? uint32_t(__builtin_ctzll(open)) : 0u;
            open &= open - 1;
            const uint32_t h1 = open ? uint32_t(__builtin_ctzll(open)) : 0u;
            open &= open - 1;
            in[i] = load(t, lane < 32 ? h0 : h1, lane & 31u, xa[i], xb[i]);
        }
    };
    auto next = [&](uint32_t step) {  // the functions of `step` have arrived
        d = d2;
        w = w2;
        open = __ballot(!(w.x <= w.y));
        terms(min(step * RESOLVE_TILES + (wave - 1), ntile - 1));
        functions(step + 1);
    };
    auto put = [&](uint32_t step) {
        const uint32_t t = step * RESOLVE_TILES + (wave - 1);
        if (t >= ntile) return;
        ResolveTile& o = s_tile[step & 1][wave - 1];
        o.d[lane] = d;
        o.w[lane] = w;
        for (uint32_t r0 = 0; r0 < STAGED; r0 += 2 * IN_FLIGHT) {
#pragma unroll
            for (int i = 0; i < IN_FLIGHT; ++i)
                if ((lane & 31u) < CHUNK_PTS)
                    o.term[r0 + 2 * i + (lane >> 5)][lane & 31u] = in[i] ? term(xa[i], xb[i]) : 0.0;
            if (!open) break;
            terms(t);
        }
    };
    // LDS is all that the wavefronts share: the barrier leaves loads in flight
    auto sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    if (wave) {
        functions(0);
        next(0);
        put(0);
        next(1);
    }
    sync();
    double acc = 0.0;
    for (uint32_t step = 0; step < nstep; ++step) {
        if (wave) {
            if (step + 1 < nstep) {
                put(step + 1);
                next(step + 2);
            }
        } else {
            const uint32_t nt = min(RESOLVE_TILES, ntile - step * RESOLVE_TILES);
            for (uint32_t u = 0; u < nt; ++u) {
                const ResolveTile& q = s_tile[step & 1][u];
                const double2 qd = q.d[lane], qw = q.w[lane];
                const bool open = qw.x <= qw.y;
                const bool simple = open && qd.x == qd.y;
                const unsigned long long closed = __ballot(!open);
                const unsigned long long alone = __ballot(!simple);
                // a run starts where the binade of the range changes, and after a chunk in no run
                const uint32_t bin = binade(qw.x);
                const uint32_t prev = uint32_t(__builtin_amdgcn_update_dpp(0, int(bin), 0x138, 0xf, 0xf, false));
                unsigned long long heads = __ballot(bin != prev) | alone | (alone << 1) | 1ull;
                double incl = run_sums(simple ? qd.x : 0.0, heads, lane);
                uint32_t at = 0;
                while (at < 64) {
                    uint32_t h = at;
                    if (!((alone >> at) & 1ull)) {
                        const unsigned long long later = at < 63 ? heads & (~0ull << (at + 1)) : 0ull;
                        const uint32_t end = later ? uint32_t(__builtin_ctzll(later)) : 64u;
                        const double start = acc + (incl - qd.x);
                        const unsigned long long bad =
                            __ballot(lane >= at && lane < end && !(qw.x <= start && start <= qw.y));
                        if (!bad) {
                            acc = acc + lane_value(incl, end - 1);
                            at = end;
                            continue;
                        }
                        h = uint32_t(__builtin_ctzll(bad));
                        acc = lane_value(start, h);
                        if (h < 63) {  // the lanes after it start a run of their own
                            heads |= 2ull << h;
                            incl = run_sums(simple ? qd.x : 0.0, heads, lane);
                        }
                    } else if (lane_value(qw.x, h) <= acc && acc <= lane_value(qw.y, h)) {
                        acc = acc + ((lo32(acc) & 1u) ? lane_value(qd.y, h) : lane_value(qd.x, h));
                        at = h + 1;
                        continue;
                    }
                    at = h + 1;
                    if ((closed >> h) & 1ull) {
                        // this chunk and those with empty ranges right after it
                        const double2* x = reinterpret_cast<const double2*>(
                            q.term[__popcll(closed & ((1ull << h) - 1ull))]);
                        const unsigned long long not_closed = ~(closed >> h);
                        const uint32_t run = not_closed ? uint32_t(__builtin_ctzll(not_closed)) : 64u;
                        for (uint32_t k = 0; k < run; ++k, x += CHUNK_PTS / 2) {
                            double2 v[CHUNK_PTS / 2];
#pragma unroll
                            for (uint32_t j = 0; j < CHUNK_PTS / 2; ++j) v[j] = x[j];
#pragma unroll
                            for (uint32_t j = 0; j < CHUNK_PTS / 2; ++j) {
                                acc = acc + v[j].x;
                                acc = acc + v[j].y;
                            }
                        }
                        at = h + run;
                    } else {
                        float ya, yb;
                        const bool ok = load(step * RESOLVE_TILES + u, h, min(lane, CHUNK_PTS), ya, yb);
                        const double x = ok ? term(ya, yb) : 0.0;
#pragma unroll
                        for (uint32_t j = 0; j < CHUNK_PTS; ++j) acc = acc + lane_value(x, j);
                    }
                }
            }
        }
        sync();
    }
    if (wave) return;
    const double N = double(npts);
    if (lane == 0) (K == 3 ? st.mean : st.cov)[c] = acc / N;
    if (K == 3 && c == 0) {
        bool multi = false;
        for (uint32_t k = lane; k < ntile; k += 64) multi |= a.sums[b.tile0 + k].multi != 0;
        const unsigned long long m = __ballot(multi);
        if (lane == 0) st.multi = m != 0;
    }
}

// The axes of a big node: the ROWS of eig3's V (OBB.cpp:80-87).
__device__ inline void big_axes(const BigState& st, double* ax) {
    const double xx = st.cov[0], yy = st.cov[1], zz = st.cov[2], xy = st.cov[3], xz = st.cov[4], yz = st.cov[5];
    double A[3][3] = {{xx, xy, xz}, {xy, yy, yz}, {xz, yz, zz}};
    double V[3][3], d[3];
    eig3(A, V, d);
    for (int r = 0; r < 3; ++r)
        for (int q = 0; q < 3; ++q) ax[r * 3 + q] = V[r][q];
}

// Merges two extents whose points come from anywhere in the node: equal
// values go to the larger index for the minimum, the smaller for the maximum
// (std::min / std::max visiting the points in order).
__device__ __forceinline__ void merge_extents(TileExtents& a, const TileExtents& b) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        if (b.lo[q] < a.lo[q] || (b.lo[q] == a.lo[q] && b.loi[q] > a.loi[q])) {
            a.lo[q] = b.lo[q];
            a.loi[q] = b.loi[q];
        }
        if (b.hi[q] > a.hi[q] || (b.hi[q] == a.hi[q] && b.hii[q] < a.hii[q])) {
            a.hi[q] = b.hi[q];
            a.hii[q] = b.hii[q];
        }
    }
}
__device__ __forceinline__ TileExtents no_extents() {
    TileExtents e;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        e.lo[q] = INFINITY;
        e.hi[q] = -INFINITY;
        e.loi[q] = -1;
        e.hii[q] = 0x7FFFFFFF;
    }
    return e;
}
// Over a workgroup of four wavefronts; the result in thread 0.
__device__ __forceinline__ void block_extents(TileExtents& e, TileExtents* s) {
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        wave_min_last(e.lo[q], e.loi[q]);
        wave_max_first(e.hi[q], e.hii[q]);
    }
    if ((threadIdx.x & 63u) == 0) s[threadIdx.x >> 6] = e;
    __syncthreads();
    if (threadIdx.x == 0)
        for (uint32_t w = 1; w < blockDim.x / 64; ++w) merge_extents(e, s[w]);
}

__global__ __launch_bounds__(256) void k_big_project(BigArgs a, const uint4* lv) {
    __shared__ float s[TILE_LDS];
    __shared__ TileExtents s_ext[4];
    __shared__ double s_ax[9];
    if (blockIdx.x >= lv[0].w) return;
    const BigTile t = big_tile(a, blockIdx.x);
    BigState& st = a.state[t.slot];
    if (!st.multi) return;
    if (threadIdx.x == 0) {  // every workgroup of the node for itself, while its tile loads
        big_axes(st, s_ax);
        if (t.tile == 0)
            for (int q = 0; q < 9; ++q) st.ax[q] = s_ax[q];
    }
    load_tile(t.src, t.nt, s);
    double ax[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) ax[q] = s_ax[q];
    TileExtents e = no_extents();
    for (uint32_t i = threadIdx.x; i < 3 * t.nt; i += blockDim.x) {
        const float* p = s + lds_at(3 * i);
        const int k = int(t.tile * TILE_PTS + i);
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const double pr = (ax[3 * q] * double(p[0]) + ax[3 * q + 1] * double(p[1])) + ax[3 * q + 2] * double(p[2]);
            if (!(e.lo[q] < pr)) { e.lo[q] = pr; e.loi[q] = k; }
            if (e.hi[q] < pr) { e.hi[q] = pr; e.hii[q] = k; }
        }
    }
    block_extents(e, s_ext);
    if (threadIdx.x == 0) a.ext[blockIdx.x] = e;
}

__global__ __launch_bounds__(256) void k_big_count(BigArgs a, const uint4* lv) {
    __shared__ float s[TILE_LDS];
    __shared__ TileExtents s_ext[4];
    __shared__ float s_box[12];
    __shared__ uint32_t s_cnt[4][3];
    __shared__ double s_ex[4][2];
    if (blockIdx.x >= lv[0].w) return;
    const BigTile t = big_tile(a, blockIdx.x);
    BNode* nd = &a.lv.nodes[t.b.node];
    load_tile(t.src, t.nt, s);
    if (a.state[t.slot].multi) {  // every workgroup of the node merges its tiles' extents for itself
        TileExtents e = no_extents();
        for (uint32_t k = threadIdx.x; k < big_tiles(t.b.n); k += blockDim.x) merge_extents(e, a.ext[t.b.tile0 + k]);
        block_extents(e, s_ext);
        if (threadIdx.x == 0) box_of_extents(a.state[t.slot].ax, e.lo, e.hi, s_box);
    } else if (threadIdx.x == 0) {
        const float* P = a.lv.pos_in + size_t(t.b.beg) * 9;
        box_to12(empty_box(mk(P[0], P[1], P[2])), s_box);
    }
    __syncthreads();
    const Box box = box_from12(s_box);
    if (t.tile == 0 && threadIdx.x == 0) {
        box_to12(box, nd->box);
        nd->surf = surface(box);
    }
    AxisCand cand[3];
    float cp[3];
    split_candidates(box, cand, cp);
    const Excess ex(box);
    double worst = 0.0, rad2 = 0.0;
    uint32_t cnt[3] = {0, 0, 0};
    for (uint32_t i = threadIdx.x; i < t.nt; i += blockDim.x) {
        float T[9];
        tri_of(s, i, T);
        ex.take(T, worst, rad2);
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) cnt[ch] += goes_left(T, cand[ch].dir, cp[ch]) ? 1u : 0u;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        worst = fmax(worst, __shfl_xor(worst, off, 64));
        rad2 = fmax(rad2, __shfl_xor(rad2, off, 64));
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) cnt[ch] += __shfl_xor(cnt[ch], off, 64);
    }
    const uint32_t wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 0) {
        for (int ch = 0; ch < 3; ++ch) s_cnt[wv][ch] = cnt[ch];
        s_ex[wv][0] = worst;
        s_ex[wv][1] = rad2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) {
            for (int ch = 0; ch < 3; ++ch) cnt[ch] += s_cnt[w][ch];
            worst = fmax(worst, s_ex[w][0]);
            rad2 = fmax(rad2, s_ex[w][1]);
        }
        a.counts[blockIdx.x] = make_uint4(cnt[0], cnt[1], cnt[2], 0u);
        post_excess(a.lv, *nd, blockIdx.x, worst, rad2);
    }
}

__global__ __launch_bounds__(256) void k_big_scatter(BigArgs a, uint4* lv) {
    __shared__ float s[TILE_LDS];
    __shared__ uint32_t s_cnt[4][6];
    __shared__ uint32_t s_left[TILE_TRIS / 64];  // left triangles of each 64
    __shared__ uint32_t s_kid[2][2];             // per big child: its slot, its first tile
    if (blockIdx.x >= lv[0].w) return;
    const BigTile t = big_tile(a, blockIdx.x);
    BNode* nd = &a.lv.nodes[t.b.node];
    const uint32_t n = t.b.n, beg = t.b.beg, lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    load_tile(t.src, t.nt, s);
    // the candidates' counts over the whole node and over the tiles before this one
    uint32_t v[6] = {0, 0, 0, 0, 0, 0};
    for (uint32_t k = threadIdx.x; k < big_tiles(n); k += blockDim.x) {
        const uint4 q = a.counts[t.b.tile0 + k];
        const uint32_t m = k < t.tile ? ~0u : 0u;
        v[0] += q.x;
        v[1] += q.y;
        v[2] += q.z;
        v[3] += q.x & m;
        v[4] += q.y & m;
        v[5] += q.z & m;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] += __shfl_xor(v[k], off, 64);
    if (lane == 0)
        for (int k = 0; k < 6; ++k) s_cnt[wv][k] = v[k];
    __syncthreads();
    uint32_t cnt[3], before[3];
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) {
        cnt[ch] = (s_cnt[0][ch] + s_cnt[1][ch]) + (s_cnt[2][ch] + s_cnt[3][ch]);
        before[ch] = (s_cnt[0][3 + ch] + s_cnt[1][3 + ch]) + (s_cnt[2][3 + ch] + s_cnt[3][3 + ch]);
    }
    AxisCand cand[3];
    float cp[3];
    split_candidates(box_from12(nd->box), cand, cp);
    const int pick = split_pick(cnt, n);
    f3 axis = cand[0].dir;
    float cproj = 0.f;
    const uint32_t first = t.tile * TILE_TRIS;
    uint32_t nl = n / 2, left_before = min(first, n / 2);
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
        if (ch == pick) {
            axis = cand[ch].dir;
            cproj = cp[ch];
            nl = cnt[ch];
            left_before = before[ch];
        }
    // 64 triangles per wavefront and step, in order
    constexpr int STEPS = int(TILE_TRIS / 256);
    unsigned long long mask[STEPS];
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const uint32_t i = j * 256 + threadIdx.x;
        bool left = false;
        if (i < t.nt) {
            float T[9];
            tri_of(s, i, T);
            left = pick >= 0 ? goes_left(T, axis, cproj) : first + i < n / 2;
        }
        mask[j] = __ballot(left);
        if (lane == 0) s_left[j * 4 + wv] = uint32_t(__popcll(mask[j]));
    }
    __syncthreads();
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
        const uint32_t i = j * 256 + threadIdx.x;
        if (i >= t.nt) continue;
        uint32_t l = left_before + uint32_t(__popcll(mask[j] & below));  // left triangles before this one
        for (uint32_t k = 0; k < j * 4 + wv; ++k) l += s_left[k];
        const uint32_t dst = ((mask[j] >> lane) & 1ull) ? beg + l : beg + nl + (first + i - l);
        float T[9];
        tri_of(s, i, T);
        float* o = a.lv.pos_out + size_t(dst) * 9;
#pragma unroll
        for (int q = 0; q < 9; ++q) o[q] = T[q];
        a.lv.id_out[dst] = a.lv.id_in[beg + first + i];
    }
    if (t.tile != 0) return;
    // the node's first workgroup makes the children and lists the big ones' tiles
    if (threadIdx.x == 0) {
        const uint32_t slot = append_kids(a.lv, nd, nl, lv[0].x + lv[0].y, &lv[1].y);
        for (uint32_t k = 0; k < 2; ++k) {
            const uint32_t m = k ? n - nl : nl;
            s_kid[k][0] = ~0u;
            if (m <= a.lv.big_min) continue;
            const uint32_t bi = atomicAdd(&lv[1].z, 1u), t0 = atomicAdd(&lv[1].w, big_tiles(m));
            a.big_out[bi] = BigNode{slot + k, k ? beg + nl : beg, m, t0};
            s_kid[k][0] = bi;
            s_kid[k][1] = t0;
        }
    }
    __syncthreads();
    for (uint32_t k = 0; k < 2; ++k) {
        if (s_kid[k][0] == ~0u) continue;
        const uint32_t m = k ? n - nl : nl;
        for (uint32_t q = threadIdx.x; q < big_tiles(m); q += blockDim.x)
            a.tiles_out[s_kid[k][1] + q] = make_uint2(s_kid[k][0], q);
    }
}

}  // namespace cdk
