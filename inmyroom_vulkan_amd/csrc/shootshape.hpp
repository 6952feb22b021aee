// Launch shape of the ray shooting (no HIP dependency).
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace cdk {

// Rays of one wavefront: 32 fill its lanes; a call of few rays spreads them
// over more wavefronts (at least 8 each), as long as these still fit
// SHOOT_SPREAD, four per SIMD: a wavefront takes as many steps as its longest
// walk and pays every step for the union of what its lanes need, so fewer
// walks in each end sooner when the chip has room for them (512-entity scene
// step spread over 2,048 wavefronts 1.04 ms, 4,096: 0.92, 16,384: 1.00).
constexpr uint32_t SHOOT_SPREAD = 4096;
constexpr uint32_t rays_per_wave(uint32_t nrays, uint32_t blocks) {
    const uint32_t most = blocks < SHOOT_SPREAD ? blocks : SHOOT_SPREAD;
    return (uint64_t(nrays) + 7) / 8 <= most ? 8u : (uint64_t(nrays) + 15) / 16 <= most ? 16u : 32u;
}

// Bytes of one wavefront's stacks in HBM, when its trees are too deep for the LDS ones.
constexpr size_t shoot_stack_bytes(uint32_t stack_entries) { return size_t(2) * stack_entries * 64 * sizeof(uint32_t); }

// Wavefronts of a launch over up to nrays rays.  Stacks in HBM (deep: a
// tree's depth sets their size) bound the spread: at most 256 MiB of them,
// unless 32 rays to a wavefront, the least there can be, need more.
constexpr size_t SHOOT_STACK_SPREAD = size_t(256) << 20;
constexpr uint32_t shoot_blocks(uint32_t nrays, uint32_t stack_entries, bool deep) {
    const uint32_t least = uint32_t((uint64_t(nrays) + 31) / 32);
    uint64_t most = (uint64_t(nrays) + 7) / 8;
    if (most > SHOOT_SPREAD) most = SHOOT_SPREAD;
    if (deep && most > SHOOT_STACK_SPREAD / shoot_stack_bytes(stack_entries))
        most = SHOOT_STACK_SPREAD / shoot_stack_bytes(stack_entries);
    return most > least ? uint32_t(most) : least;
}

}  // namespace cdk
