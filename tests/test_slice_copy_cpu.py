"""The addresses of the update GEMM's clamped one-element copies (csrc/slice_copy.hpp), compiled for the host: a wave's base
element plus a lane's 32-bit byte offset is the lane's element clamped into the buffer, at buffers on both sides of 2^32 bytes
and at slices that start before, inside, at the end of and past them."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / 'noise_amd' / 'csrc'
SOURCE = r'''
#include <cstdio>
#include "slice_copy.hpp"
int main() {
    // a [65280, 256] parameter at 16,385 directions and [4096, 512] tables at 233,017 pass 2^30 elements
    const int64_t lengths[] = {1, 63, 64, 700, (1ll << 30) - 1, 1ll << 30, (1ll << 30) + 65536, 233017ll * 4608, 1ll << 38};
    long checked = 0;
    for (int64_t numel : lengths) {
        const int64_t around[] = {0, numel / 2, numel - 64, numel, 1ll << 30, (1ll << 30) + 65280};
        for (int64_t at : around)
            for (int64_t first = at - 130; first <= at + 130; ++first) {
                const int64_t base = noise::slice_base(first, numel);
                for (int lane = 0; lane < 64; ++lane) {
                    const uint32_t off = noise::slice_lane(first, lane, base, numel);
                    int64_t want = first + lane;
                    if (want < 0) want = 0;
                    if (want > numel - 1) want = numel - 1;
                    if (base < 0 || base >= numel || off % 4 || off > 252 || base + off / 4 != want) {
                        std::printf("numel %lld first %lld lane %d: base %lld offset %u\n", (long long)numel, (long long)first,
                                    lane, (long long)base, off);
                        return 1;
                    }
                    ++checked;
                }
            }
    }
    std::printf("%ld\n", checked);
    return 0;
}
'''


def test_clamped_copies(tmp_path):
    gxx = shutil.which('g++')
    if gxx is None:
        pytest.skip('no host C++ compiler')
    src, exe = tmp_path / 'slice_copy.cpp', tmp_path / 'slice_copy'
    src.write_text(SOURCE)
    subprocess.run([gxx, '-std=c++17', '-Wall', '-Werror', '-I', str(CSRC), str(src), '-o', str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True)
    assert res.returncode == 0 and int(res.stdout) == 9 * 6 * 261 * 64, res.stdout
