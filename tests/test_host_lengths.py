"""The host's running sums of stream lengths (csrc/host_lengths.hpp) at every byte address, built by the
host compiler with its undefined-behaviour checks: a container's sections lie anywhere in a pickle blob."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include <vector>
#include "host_lengths.hpp"

template <typename T>
int run(int64_t C, int at)
{
    const int64_t nsub = 2, rows = 3, tiles = (C + 63) / 64, n = nsub * rows * C;
    std::vector<char> raw(n * sizeof(T) + 16);
    std::vector<uint32_t> starts(nsub * rows * tiles);
    int64_t sub_bytes[2];
    for (int64_t i = 0; i < n; ++i) {
        const T v = (T)(i * 37 % 300);
        memcpy(raw.data() + at + i * sizeof(T), &v, sizeof(v));
    }
    if (!host_tile_starts<T>(raw.data() + at, nsub, rows, C, 256, starts.data(), sub_bytes)) return 1;
    for (int64_t s = 0, i = 0; s < nsub; ++s) {
        uint32_t sum = 0;
        for (int64_t r = 0; r < rows; ++r)
            for (int64_t c = 0; c < C; ++c, ++i) {
                if (c % 64 == 0 && starts[(s * rows + r) * tiles + c / 64] != sum) return 2;
                sum += i * 37 % 300 < 256 ? i * 37 % 300 : 256;
            }
        if (sub_bytes[s] != sum) return 3;
    }
    if (sizeof(T) == 4) {
        const T v = (T)-1;
        memcpy(raw.data() + at + (n - 1) * sizeof(T), &v, sizeof(v));
        if (host_tile_starts<T>(raw.data() + at, nsub, rows, C, 256, starts.data(), sub_bytes)) return 4;
    }
    return 0;
}

int main()
{
    for (int64_t C : {1, 63, 64, 65, 192})
        for (int at = 0; at < 8; ++at) {
            const int wrong = 10 * run<int32_t>(C, at) + run<uint16_t>(C, at);
            if (wrong) {
                printf("%lld channels at byte %d: %d\n", (long long)C, at, wrong);
                return 1;
            }
        }
    return 0;
}
"""


@pytest.mark.parametrize("level", ["-O0", "-O3"])
def test_lengths_are_read_at_any_address(tmp_path, level):
    source, program = tmp_path / "driver.cpp", str(tmp_path / "driver")
    source.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", level, "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    "-I", os.path.join(ROOT, "cachegen_amd", "csrc"), str(source), "-o", program], check=True)
    done = subprocess.run([program], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert done.returncode == 0, done.stdout
