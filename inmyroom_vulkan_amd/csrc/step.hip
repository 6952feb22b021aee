// Glue of the one-call scene step (cd_step): the counts that the separate
// calls read back between their stages stay on the device, in a count block
// (DC_* words), so that the whole step, from the entity matrices to the pair
// responses, is enqueued at once and can be replayed as one graph.  Every
// stage is shaped for a capacity and reads its count from the block; the
// host checks the counts once, after the step, and runs it again with larger
// capacities when one was exceeded.
//  k_step_pairs   pairs the sweep kept: the batched traversal's query count
//  k_step_contacts contacts the later stages take
//  k_seg_*        the contacts grouped by pair and ordered within each pair
//                 (below)
//  k_pair_begins  per side, the first ray of every pair (exclusive scan of
//                 the pairs' ray counts)
//  k_pack         the step's results gathered into one block for a single
//                 copy to the host
#include "kernels.hpp"

namespace cdk {

__global__ void k_step_pairs(const unsigned int* __restrict__ sweep, uint32_t cap, uint32_t* __restrict__ dc,
                             unsigned int* __restrict__ d_nq) {
    if (threadIdx.x != 0) return;
    const uint32_t found = *sweep;
    const uint32_t kept = min(found, cap);
    dc[DC_SWEEP] = found;
    dc[DC_NQ] = kept;
    *d_nq = kept;
}

// qcnt (np words, when given) cleared for k_seg_count
__global__ __launch_bounds__(1024) void k_step_contacts(const RunCounters* __restrict__ ctr, uint64_t cap,
                                                        uint32_t* __restrict__ dc, uint32_t* __restrict__ qcnt,
                                                        uint32_t np) {
    if (threadIdx.x == 0) dc[DC_NC] = uint32_t(min(ctr->contacts, cap));
    if (qcnt)
        for (uint32_t i = threadIdx.x; i < np; i += blockDim.x) qcnt[i] = 0u;
}

// ---- contact order ------------------------------------------------------------
// The rays need a run's contacts ordered by (pair, tri_a, tri_b), and a
// permutation of them by (pair, tri_b, tri_a).  A run tests a triangle pair
// of an entity pair once, so these keys are distinct and every sort gives
// the order the separate calls' multi-pass radix sorts give.  Here:
//  k_seg_count    contacts per pair
//  k_scan_one     each pair's first slot (and a copy the scatter advances)
//  k_seg_scatter  every contact into its pair's slots, in any order
//  k_seg_sort     one workgroup per pair: its contacts ranked by (tri_a,
//                 tri_b) and by (tri_b, tri_a) together, by merging runs in
//                 LDS.  Pairs of up to SEG_SMALL contacts take a small workgroup
//                 each, the larger ones (listed by k_scan_one) a large one; a
//                 pair of more than SEG_MAX sets a flag, and the caller runs
//                 the radix sorts instead.
// The count and the scatter add to a pair's counter once per wavefront and
// pair (a run's contacts of one pair lie together), not once per contact.
// Sorting the two orders one after the other by a bitonic network (66 stages
// of a barrier and two LDS round trips each for 2,048 contacts) took 38 us in
// the 512-entity scene, 112 us over 4,099 entities; the query batches and
// deformables, which used up to 24 radix passes, 0.27-1.2 ms.
constexpr uint32_t SEG_MAX = 4096, SEG_THREADS = 1024;
constexpr uint32_t SEG_SMALL = 256;
constexpr uint32_t SEG_GRID = 1024;   // workgroups of the larger pairs' launch at most
constexpr uint32_t SEG_SMALL_GRID = 1u << 20;  // of the small ones': a launch takes fewer than 2^32 threads
// A key: both triangles, and the contact's place.  Where a mesh has more than
// 2^25 triangles (WIDE) both take 32 bits each, and the places lie beside the
// keys: 96 KB of LDS a workgroup (one to a CU) instead of 80 (two), against the
// radix sorts such meshes would need (a frame of 63 pairs on a 34M-triangle
// terrain: 0.49 against 0.62 ms).
constexpr uint32_t SEG_TRI_BITS = 25, SEG_POS_BITS = 13;
static_assert(2 * SEG_TRI_BITS + SEG_POS_BITS < 64 && SEG_MAX < (1u << SEG_POS_BITS), "key fields");

// Slot of each lane's contact among its pair's (base + rank among the
// wavefront's lanes of that pair); valid lanes only.  One atomic add per
// pair the wavefront holds.
__device__ __forceinline__ uint32_t seg_slot(uint32_t* __restrict__ ctr, uint32_t q, bool valid) {
    const uint32_t lane = threadIdx.x & 63;
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    unsigned long long todo = __ballot(valid), mine = 0;
    while (todo) {  // the lanes of each pair the wavefront holds
        const int first = __ffsll(static_cast<long long>(todo)) - 1;
        const uint32_t lq = __shfl(q, first, 64);
        const unsigned long long peers = __ballot(valid && q == lq);
        if (valid && q == lq) mine = peers;
        todo &= ~peers;
    }
    // the pairs' adds together: one round trip, not one per pair
    const int leader = valid ? __ffsll(static_cast<long long>(mine)) - 1 : 0;
    uint32_t base = 0;
    if (valid && int(lane) == leader) base = atomicAdd(&ctr[q], uint32_t(__popcll(mine)));
    base = __shfl(base, leader, 64);
    const uint32_t slot = base + uint32_t(__popcll(mine & below));
    return slot;
}

__global__ __launch_bounds__(256) void k_seg_count(const cd_contact* __restrict__ c, uint32_t cap,
                                                   const uint32_t* __restrict__ nc_dev, uint32_t* __restrict__ qcnt) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < count_of(cap, nc_dev);
    (void)seg_slot(qcnt, valid ? c[i].query : 0u, valid);
}

// Exclusive scan of n_dev (min with cap) counts in one workgroup, into out
// and out2; the counts above SEG_SMALL are listed (large[0] of them, from
// large[1]), and one above SEG_MAX sets *flag.
__global__ __launch_bounds__(1024) void k_scan_one(const uint32_t* __restrict__ in, uint32_t cap,
                                                   const uint32_t* __restrict__ n_dev, uint32_t* __restrict__ out,
                                                   uint32_t* __restrict__ out2, uint32_t* __restrict__ large,
                                                   uint32_t* __restrict__ flag) {
    __shared__ uint32_t s_w[16];
    __shared__ uint32_t s_large;
    if (threadIdx.x == 0) s_large = 0;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t n = count_of(cap, n_dev);
    uint32_t carry = 0;
    for (uint32_t base = 0; base < n; base += 1024) {
        const uint32_t i = base + tid;
        const uint32_t v = i < n ? in[i] : 0u;
        uint32_t x = v;
#pragma unroll
        for (uint32_t off = 1; off < 64; off <<= 1) {
            const uint32_t y = __shfl_up(x, off, 64);
            if (lane >= off) x += y;
        }
        if (lane == 63) s_w[wave] = x;
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (uint32_t w = 0; w < 16; ++w) {
            before += w < wave ? s_w[w] : 0u;
            all += s_w[w];
        }
        if (i < n) {
            out[i] = carry + before + x - v;
            out2[i] = carry + before + x - v;
            if (v > SEG_SMALL) large[1 + atomicAdd(&s_large, 1u)] = i;
            if (v > SEG_MAX) *flag = 1u;
        }
        carry += all;
        __syncthreads();
    }
    if (tid == 0) large[0] = s_large;
}

__global__ __launch_bounds__(256) void k_seg_scatter(const cd_contact* __restrict__ c, uint32_t cap,
                                                     const uint32_t* __restrict__ nc_dev, uint32_t* __restrict__ qfill,
                                                     cd_contact* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < count_of(cap, nc_dev);
    cd_contact r = {};
    if (valid) r = c[i];
    const uint32_t slot = seg_slot(qfill, r.query, valid);
    if (valid) out[slot] = r;
}

// The contacts of one pair, n <= CAP, ranked by both orders.  Runs of L keys
// are merged into runs of 2 L, every key by a binary search of the run next
// to it (keys are distinct): each level's searches of all of a thread's keys
// in both orders are in flight together, and a level costs two barriers.
template <uint32_t CAP, bool WIDE>
struct SegShared {
    unsigned long long key[2][CAP];
    uint32_t place[CAP];
};
template <uint32_t CAP>
struct SegShared<CAP, true> {
    unsigned long long key[2][CAP];
    uint32_t place[CAP];
    uint16_t pos[2][CAP];
};
static_assert(sizeof(SegShared<SEG_MAX, false>) <= 80 * 1024, "two large workgroups share a CU's LDS");
template <uint32_t THREADS, uint32_t CAP, bool WIDE>
__device__ __forceinline__ void seg_rank(const cd_contact* __restrict__ seg, uint32_t base, uint32_t n,
                                         SegShared<CAP, WIDE>& S, cd_contact* __restrict__ sorted,
                                         uint32_t* __restrict__ order_b) {
    unsigned long long(*const key)[CAP] = S.key;
    uint32_t* const place = S.place;
    constexpr uint32_t E = CAP / THREADS;
    const uint32_t tid = threadIdx.x;
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) {
        const uint32_t i = e * THREADS + tid;
        if (i < n) {
            const unsigned long long a = seg[base + i].tri_a, b = seg[base + i].tri_b;
            if constexpr (WIDE) {
                key[0][i] = (a << 32) | b;
                key[1][i] = (b << 32) | a;
                S.pos[0][i] = S.pos[1][i] = uint16_t(i);
            } else {
                key[0][i] = (((a << SEG_TRI_BITS) | b) << SEG_POS_BITS) | i;
                key[1][i] = (((b << SEG_TRI_BITS) | a) << SEG_POS_BITS) | i;
            }
        }
    }
    __syncthreads();
    for (uint32_t lg = 0, L = 1; L < n; ++lg, L <<= 1) {
        unsigned long long v[2][E];
        uint32_t s0[E], len[E], lo[2][E];
        uint16_t p[2][E];
#pragma unroll
        for (uint32_t e = 0; e < E; ++e) {
            const uint32_t i = min(e * THREADS + tid, n - 1);
            v[0][e] = key[0][i];
            v[1][e] = key[1][i];
            if constexpr (WIDE) {
                p[0][e] = S.pos[0][i];
                p[1][e] = S.pos[1][i];
            }
            s0[e] = min(((i >> lg) ^ 1u) << lg, n);  // the run next to key i's
            len[e] = min(L, n - s0[e]);
            lo[0][e] = lo[1][e] = 0;
        }
        for (uint32_t step = L; step > 0; step >>= 1)
#pragma unroll
            for (uint32_t e = 0; e < E; ++e) {
                if (e * THREADS >= n) break;
                // read whether or not the step stays inside the run: the loads then need no branches
#pragma unroll
                for (int o = 0; o < 2; ++o) {
                    const uint32_t m = lo[o][e] + step;
                    const unsigned long long k = key[o][min(s0[e] + m, n) - 1];
                    lo[o][e] = ((m <= len[e]) & (k < v[o][e])) ? m : lo[o][e];
                }
            }
        __syncthreads();
#pragma unroll
        for (uint32_t e = 0; e < E; ++e) {
            const uint32_t i = e * THREADS + tid;
            if (i < n) {
                const uint32_t at = (((i >> lg) & ~1u) << lg) + (i & (L - 1));
                key[0][at + lo[0][e]] = v[0][e];
                key[1][at + lo[1][e]] = v[1][e];
                if constexpr (WIDE) {
                    S.pos[0][at + lo[0][e]] = p[0][e];
                    S.pos[1][at + lo[1][e]] = p[1][e];
                }
            }
        }
        __syncthreads();
    }
    // slot r of the sorted array holds the contact at key r's place; the second order lists those slots
    auto placed = [&](int o, uint32_t r) -> uint32_t {
        if constexpr (WIDE) return S.pos[o][r];
        else return uint32_t(key[o][r]) & ((1u << SEG_POS_BITS) - 1u);
    };
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) {
        const uint32_t r = e * THREADS + tid;
        if (r < n) {
            const uint32_t i = placed(0, r);
            place[i] = r;
            sorted[base + r] = seg[base + i];
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) {
        const uint32_t r = e * THREADS + tid;
        if (r < n) order_b[base + r] = base + place[placed(1, r)];
    }
}

template <bool WIDE>
__global__ __launch_bounds__(SEG_SMALL) void k_seg_sort_small(const cd_contact* __restrict__ seg,
                                                       const uint32_t* __restrict__ qoff,
                                                       const uint32_t* __restrict__ qcnt,
                                                       const uint32_t* __restrict__ nq_dev, uint32_t cap,
                                                       cd_contact* __restrict__ sorted, uint32_t* __restrict__ order_b) {
    __shared__ SegShared<SEG_SMALL, WIDE> S;
    const uint32_t nq = count_of(cap, nq_dev);
    for (uint32_t q = blockIdx.x; q < nq; q += gridDim.x) {
        const uint32_t n = qcnt[q];
        if (n == 0 || n > SEG_SMALL) continue;
        seg_rank<SEG_SMALL, SEG_SMALL, WIDE>(seg, qoff[q], n, S, sorted, order_b);
        __syncthreads();  // the next pair reuses the LDS
    }
}

template <bool WIDE>
__global__ __launch_bounds__(SEG_THREADS) void k_seg_sort(const cd_contact* __restrict__ seg,
                                                          const uint32_t* __restrict__ qoff,
                                                          const uint32_t* __restrict__ qcnt,
                                                          const uint32_t* __restrict__ large,
                                                          cd_contact* __restrict__ sorted,
                                                          uint32_t* __restrict__ order_b) {
    __shared__ SegShared<SEG_MAX, WIDE> S;
    for (uint32_t k = blockIdx.x; k < large[0]; k += gridDim.x) {
        const uint32_t q = large[1 + k], n = qcnt[q];
        if (n > SEG_MAX) {  // flagged: in any order, so that what follows reads contacts
            for (uint32_t r = threadIdx.x; r < n; r += SEG_THREADS) {
                sorted[qoff[q] + r] = seg[qoff[q] + r];
                order_b[qoff[q] + r] = qoff[q] + r;
            }
            continue;
        }
        seg_rank<SEG_THREADS, SEG_MAX, WIDE>(seg, qoff[q], n, S, sorted, order_b);
        __syncthreads();  // the next pair reuses the LDS
    }
}

// One workgroup: each side's counts (qw + 2 stride side) scanned 1024 at a
// time, the wavefronts' sums combined through LDS.
__global__ __launch_bounds__(1024) void k_pair_begins(const uint32_t* __restrict__ qw, uint32_t stride,
                                                      const uint32_t* __restrict__ dc, uint32_t* __restrict__ pbegin) {
    __shared__ uint32_t s_w[16];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t nq = min(dc[DC_NQ], stride);
    for (int side = 0; side < 2; ++side) {
        const uint32_t* cnt = qw + 2 * size_t(stride) * side;
        uint32_t* out = pbegin + size_t(stride) * side;
        uint32_t carry = 0;
        for (uint32_t base = 0; base < nq; base += 1024) {
            const uint32_t i = base + tid;
            const uint32_t v = i < nq ? cnt[i] : 0u;
            uint32_t x = v;
#pragma unroll
            for (uint32_t off = 1; off < 64; off <<= 1) {
                const uint32_t y = __shfl_up(x, off, 64);
                if (lane >= off) x += y;
            }
            if (lane == 63) s_w[wave] = x;
            __syncthreads();
            uint32_t before = 0, all = 0;
            for (uint32_t w = 0; w < 16; ++w) {
                before += w < wave ? s_w[w] : 0u;
                all += s_w[w];
            }
            if (i < nq) out[i] = carry + before + x - v;
            carry += all;
            __syncthreads();
        }
    }
}

__global__ void k_pack(PackSpans sp, uint32_t* __restrict__ dst) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t s = 0; s < sp.n; ++s) {
        const uint32_t* src = sp.src[s];
        uint32_t* d = dst + sp.dst[s];
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < sp.words[s]; i += stride) d[i] = src[i];
    }
}

hipError_t launch_step_pairs(const unsigned int* sweep, uint32_t cap, uint32_t* dc, unsigned int* d_nq, hipStream_t st) {
    hipLaunchKernelGGL(k_step_pairs, dim3(1), dim3(64), 0, st, sweep, cap, dc, d_nq);
    return hipGetLastError();
}
hipError_t launch_step_contacts(const RunCounters* ctr, uint64_t cap, uint32_t* dc, hipStream_t st, uint32_t* qcnt,
                                uint32_t np) {
    hipLaunchKernelGGL(k_step_contacts, dim3(1), dim3(1024), 0, st, ctr, cap, dc, qcnt, np);
    return hipGetLastError();
}
size_t seg_order_words(uint32_t np_cap) { return 4 * size_t(np_cap) + 1; }
hipError_t launch_seg_order(const cd_contact* c, uint32_t tri_bits, uint32_t nc_cap, const uint32_t* nc_dev,
                            uint32_t np_cap, const uint32_t* np_dev, uint32_t* flag, uint32_t* work, cd_contact* seg,
                            cd_contact* sorted, uint32_t* order_b, hipStream_t st) {
    uint32_t* qcnt = work;
    uint32_t* qoff = work + np_cap;
    uint32_t* qfill = work + 2 * size_t(np_cap);
    uint32_t* large = work + 3 * size_t(np_cap);
    const dim3 gc((std::max(nc_cap, 1u) + 255) / 256);
    hipLaunchKernelGGL(k_seg_count, gc, dim3(256), 0, st, c, nc_cap, nc_dev, qcnt);
    hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(1024), 0, st, qcnt, np_cap, np_dev, qoff, qfill, large, flag);
    hipLaunchKernelGGL(k_seg_scatter, gc, dim3(256), 0, st, c, nc_cap, nc_dev, qfill, seg);
    // no more pairs than contacts / SEG_SMALL are large
    const dim3 gs(std::min(std::max(np_cap, 1u), SEG_SMALL_GRID)),
        gl(std::min(std::min(np_cap, nc_cap / SEG_SMALL), SEG_GRID));
    if (tri_bits > SEG_TRI_BITS) {
        hipLaunchKernelGGL(k_seg_sort_small<true>, gs, dim3(SEG_SMALL), 0, st, seg, qoff, qcnt, np_dev, np_cap, sorted,
                           order_b);
        if (gl.x)
            hipLaunchKernelGGL(k_seg_sort<true>, gl, dim3(SEG_THREADS), 0, st, seg, qoff, qcnt, large, sorted, order_b);
    } else {
        hipLaunchKernelGGL(k_seg_sort_small<false>, gs, dim3(SEG_SMALL), 0, st, seg, qoff, qcnt, np_dev, np_cap, sorted,
                           order_b);
        if (gl.x)
            hipLaunchKernelGGL(k_seg_sort<false>, gl, dim3(SEG_THREADS), 0, st, seg, qoff, qcnt, large, sorted, order_b);
    }
    return hipGetLastError();
}
hipError_t launch_pair_begins(const uint32_t* qw, uint32_t stride, const uint32_t* dc, uint32_t* pbegin, hipStream_t st) {
    hipLaunchKernelGGL(k_pair_begins, dim3(1), dim3(1024), 0, st, qw, stride, dc, pbegin);
    return hipGetLastError();
}
hipError_t launch_pack(const PackSpans& sp, uint32_t* dst, hipStream_t st) {
    if (sp.n > PackSpans::MAX) return hipErrorInvalidValue;
    uint64_t most = 0;
    for (uint32_t s = 0; s < sp.n; ++s) most = std::max<uint64_t>(most, sp.words[s]);
    const uint32_t blocks = uint32_t(std::min<uint64_t>(256, std::max<uint64_t>(1, (most + 255) / 256)));
    hipLaunchKernelGGL(k_pack, dim3(blocks), dim3(256), 0, st, sp, dst);
    return hipGetLastError();
}

}  // namespace cdk
