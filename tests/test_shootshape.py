"""Launch shape of the ray shooting (csrc/shootshape.hpp), on the CPU.

The grid is shaped for a capacity, the rays per wavefront for the rays there
are: every count up to the capacity must be covered, and the stacks in HBM,
whose size a tree's depth sets, must not grow with the spread of few rays over
many wavefronts past 256 MiB.
"""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "inmyroom_vulkan_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_ray_has_a_wavefront_and_stacks_are_bounded(tmp_path):
    src = tmp_path / "shape.cpp"
    src.write_text(r'''
#include "shootshape.hpp"
#include <cstdio>
using namespace cdk;
int main() {
    const uint32_t entries[] = {49, 62, 128, 129, 255, 2000, 70000};
    const uint32_t caps[] = {1, 7, 8, 9, 31, 32, 33, 64, 4096, 32767, 32768, 32769, 65536, 65537, 131071, 131072,
                             131073, 1u << 20, 0x7FFFFFFFu, 0xFFFFFFFFu};
    for (uint32_t cap : caps)
        for (int deep = 0; deep < 2; ++deep)
            for (uint32_t e : entries) {
                const uint32_t blocks = shoot_blocks(cap, e, deep != 0), least = uint32_t((uint64_t(cap) + 31) / 32);
                for (uint32_t n : caps) {
                    if (n > cap) continue;
                    const uint32_t w = rays_per_wave(n, blocks);
                    if (uint64_t(w) * blocks < n || (w != 8 && w != 16 && w != 32))
                        return std::printf("%u of %u rays, %u entries: %u wavefronts of %u\n", n, cap, e, blocks, w), 1;
                }
                if (deep && blocks > least && blocks * shoot_stack_bytes(e) > (size_t(256) << 20))
                    return std::printf("%u rays, %u entries: %zu bytes\n", cap, e, blocks * shoot_stack_bytes(e)), 1;
            }
    // 32 rays fill a wavefront, few rays spread over up to 4,096
    std::printf("%u %u %u %u\n", shoot_blocks(8000, 20, false), shoot_blocks(40000, 20, false),
                shoot_blocks(40000, 2000, true), shoot_blocks(1u << 20, 20, false));
    return 0;
}
''')
    exe = tmp_path / "shape"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-I", CSRC,
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split() == ["1000", "4096", "1250", "32768"]
