"""Segments of the CSR-Adaptive products (moquimc_amd/csrc/mqi_plan.h,
cut_segments), compiled with g++: the bisected cut equals the row-by-row one
for 32- and 64-bit row pointers."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <cstdio>
#include <vector>
#include "mqi_plan.h"
template<typename T> int run(long long rows) {
    std::vector<T> ip(rows + 1);
    for (auto& v : ip) {
        long long x;
        if (std::scanf("%lld", &x) != 1) return 1;
        v = (T) x;
    }
    std::vector<int64_t> sk; std::vector<uint32_t> si; std::vector<int32_t> sp;
    if (!cut_segments(ip.data(), rows, 16, 40, 8, sk, si, sp)) return 1;
    for (auto v : sk) std::printf("%lld ", (long long) v);
    for (auto v : si) std::printf("%u ", v);
    for (auto v : sp) std::printf("%d ", v);
    std::printf("\n");
    return 0;
}
int main() {
    long long bits, rows;
    while (std::scanf("%lld %lld", &bits, &rows) == 2)
        if (bits == 32 ? run<uint32_t>(rows) : run<int64_t>(rows)) return 1;
    return 0;
}
"""


def _rows_one_by_one(ip, shrt=16, lng=40, max_rows=8):
    rows, r = len(ip) - 1, 0
    sk, si, split = [], [], []
    while r < rows:
        n = ip[r + 1] - ip[r]
        if n > shrt:
            split.append(len(sk))
            for off in range(0, n, lng):
                sk.append(ip[r] + off)
                si.append(r | 0x80000000)
            split.append(len(sk))
            r += 1
        else:
            r0 = r
            while r < rows and r - r0 < max_rows and ip[r + 1] - ip[r0] <= shrt:
                r += 1
            sk.append(ip[r0])
            si.append(r0)
    return sk + [ip[rows]] + si + [rows] + split


@pytest.mark.parametrize("bits", [32, 64])
def test_segments_match_the_row_by_row_cut(tmp_path, bits):
    src, exe = tmp_path / "seg.cpp", str(tmp_path / "seg")
    src.write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "moquimc_amd", "csrc"),
                    str(src), "-o", exe], check=True)
    rng = np.random.default_rng(bits)
    lens = [[], [0], [16], [17], [40], [41], [0] * 30, [16] * 9, [1] * 16 + [2], [8, 8, 1], [17, 0, 16, 81, 15, 1, 1]]
    lens += [rng.integers(0, hi, 200) for hi in (2, 6, 18, 100)]
    ips = [np.r_[0, np.cumsum(x)].astype(int).tolist() for x in lens]
    out = subprocess.run([exe], input="".join("%d %d %s\n" % (bits, len(ip) - 1, " ".join(map(str, ip))) for ip in ips),
                         capture_output=True, text=True, check=True).stdout.split("\n")
    for ip, line in zip(ips, out):
        assert [int(x) for x in line.split()] == _rows_one_by_one(ip), ip
