"""Host half of the element tiles (csrc/hex.hip) on the CPU: the file is compiled for the host with a runtime whose
allocations are host memory and fail on demand.

A context whose tile arrays do not fit walks K: each allocation failing in turn, the call succeeds without tiles,
nothing is left allocated, a second call does not try (or read) again, and a new context builds the same tiles as
one that never failed.
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "pdlsm-fem_mpi_amd", "csrc")

RUNTIME = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include "hex.hip"
#include "setup.hpp"

static int g_fail_at = -1, g_calls = 0;
static std::set<void *> g_live;
extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
    if (g_calls++ == g_fail_at) return hipErrorOutOfMemory;
    g_live.insert(*p = std::malloc(n));
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (p && !g_live.erase(p)) std::abort();
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "out of memory"; }
}

namespace pdx {
int setup_device() { return -1; }
int dev_cell_search(int, int, const double *, const double *, const std::vector<int> &, const std::vector<int> &,
                    const CellGrid &, long long, const int *, double, std::vector<long long> &, std::vector<int> *, int &,
                    int **, std::string &) { std::abort(); }
int dev_node_graph(int, const Model &, const std::vector<int> &, const std::vector<int> &, std::vector<int> &,
                   std::vector<int> &, std::string &) { std::abort(); }
}  // namespace pdx
using namespace pdx;

// box of nx x ny x nz nodes with spacing (hx, hy, hz); elements whose cell index is below pd in every direction are PD
static void box(Model &m, int nx, int ny, int nz, double hx, double hy, double hz, int pd) {
    m.dim = 3;
    m.E = 1e9;
    m.nu = 0.3;
    m.rho = 1000;
    m.nn = nx * ny * nz;
    for (int k = 0; k < nz; k++)
        for (int j = 0; j < ny; j++)
            for (int i = 0; i < nx; i++) m.x.insert(m.x.end(), {i * hx, j * hy, k * hz});
    auto id = [&](int i, int j, int k) { return i + nx * (j + ny * k); };
    for (int k = 0; k + 1 < nz; k++)
        for (int j = 0; j + 1 < ny; j++)
            for (int i = 0; i + 1 < nx; i++) {
                const int e[8] = {id(i, j, k), id(i + 1, j, k), id(i + 1, j + 1, k), id(i, j + 1, k),
                                  id(i, j, k + 1), id(i + 1, j, k + 1), id(i + 1, j + 1, k + 1), id(i, j + 1, k + 1)};
                m.econ.insert(m.econ.end(), e, e + 8);
                m.nen.push_back(8);
                m.algo.push_back(i < pd && j < pd && k < pd ? 1 : 2);
            }
    m.ne = (int)m.nen.size();
    std::string err;
    if (m.setup(err)) {
        std::puts(err.c_str());
        std::exit(2);
    }
}

// a context with the fields that the tiles read: dimension, sizes, the FE elements of every node
struct Host {
    Ctx c;
    std::vector<int> off, item;
    explicit Host(const Model &m) : off(m.nn + 1, 0) {
        for (int e : m.fe)
            for (int a = 0; a < m.nen[e]; a++) off[m.econ[e * 8 + a] + 1]++;
        for (int k = 0; k < m.nn; k++) off[k + 1] += off[k];
        item.resize(off[m.nn]);
        std::vector<int> fill(off.begin(), off.end() - 1);
        for (size_t t = 0; t < m.fe.size(); t++)
            for (int a = 0; a < m.nen[m.fe[t]]; a++) item[fill[m.econ[m.fe[t] * 8 + a]]++] = int(t) * 8 + a;
        c.dim = 3;
        c.nn = m.nn;
        c.nfam = m.nfam;
        c.host = &m;
        c.nfe_off = off.data();
        c.nfe_item = item.data();
    }
};
"""

FAILING = RUNTIME + r"""
int main() {
    Model m;
    box(m, 30, 30, 30, 1e-3, 1e-3, 1e-3, 6);
    std::string err;
    const HexTiles *t = nullptr;
    int work = 0, calls = 0;
    {
        Host h(m);
        if (hex_tiles(h.c, t, err) || !t || !t->n_fam) return 3;
        work = t->n_work;
        calls = g_calls;
        free_hex_tiles(h.c);
    }
    for (int at = 0; at < calls; at++) {
        Host h(m);
        g_calls = 0;
        g_fail_at = at;
        for (int rep = 0; rep < 2; rep++)
            if (hex_tiles(h.c, t, err) || t || h.c.hex || !g_live.empty()) return std::printf("allocation %d, call %d\n", at, rep), 4;
        g_fail_at = -1;
        Host n(m);
        if (hex_tiles(n.c, t, err) || !t || t->n_work != work) return 5;
        free_hex_tiles(n.c);
    }
    std::printf("%d allocations, %d blocks\n", calls, work);
    return g_live.empty() ? 0 : 6;
}
"""


def _run(tmp_path, code, *args):
    src, exe = tmp_path / "tiles.cpp", tmp_path / "tiles"
    src.write_text(code)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-O1", "-g", "-std=c++17", "-fopenmp", "-Wno-unused-result", "-Wno-unused-value", "--offload-arch=gfx950",
                    "--offload-host-only", "-I", CSRC, "-I", os.path.join(CSRC, "..", "..", "include"), "-x", "hip",
                    str(src), "-x", "c++", os.path.join(CSRC, "model.cpp"), "-o", str(exe), "-Wl,-rpath,/opt/rocm/llvm/lib",
                    *args], check=True)
    return subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)


def test_tiles_that_do_not_fit(tmp_path):
    r = _run(tmp_path, FAILING)
    assert r.returncode == 0, f"exit {r.returncode}: {r.stdout}{r.stderr}"
