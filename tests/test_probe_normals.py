"""The blocks of the seeded normals against the standard distribution's own serial sequence, bit for
bit: one block, an odd count, the ends of one and of several blocks, more than one round of blocks."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pdlsm-fem_mpi_amd", "csrc")

MAIN = r"""
#include <cstdio>
#include <cstring>
#include "normals.hpp"
int main() {
    for (size_t n : {1ul, 2ul, 7ul, 6433ul, 6434ul, 12868ul, 100003ul, 1700001ul})
        for (unsigned long long seed : {0ull, 5ull, 12345678901ull}) {
            std::vector<double> want(n), got(n, -9.0);
            std::mt19937_64 rng(seed);
            std::normal_distribution<double> nd(0.0, 1.0);
            for (auto &x : want) x = nd(rng);
            pdx::seeded_normals(seed, n, [&](size_t i, double v) { got[i] = v; });
            if (std::memcmp(want.data(), got.data(), n * 8)) return std::printf("n %zu seed %llu\n", n, seed), 1;
        }
    return 0;
}
"""


def test_seeded_normals_bits(tmp_path):
    src, exe = tmp_path / "normals.cpp", tmp_path / "normals"
    src.write_text(MAIN)
    subprocess.run(["g++", "-O2", "-std=c++17", "-fopenmp", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
