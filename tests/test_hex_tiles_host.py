"""Host half of the element tiles (csrc/hex.hip) on the CPU: the file is compiled for the host with a runtime whose
allocations are host memory and fail on demand.

A context whose tile arrays do not fit (on the device or the host) walks K: each device allocation failing in turn, the call succeeds without tiles,
nothing is left allocated, a second call does not try (or read) again, and a new context builds the same tiles as
one that never failed.

Which models get tiles: those whose tiles take less time than the walk of K by the counts in hex.hpp.  Where there
are tiles, they, the families and the rows left to K hold every node once, and a tile lists every element of the
nodes it owns.
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
static std::atomic<long> g_new_calls{0}, g_new_fail_at{-1};
void *operator new(size_t n) {
    if (g_new_calls++ == g_new_fail_at) throw std::bad_alloc();
    return std::malloc(n ? n : 1);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
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

static void material(Model &m) {
    m.dim = 3;
    m.E = 1e9;
    m.nu = 0.3;
    m.rho = 1000;
}

static void finish(Model &m) {
    m.ne = (int)m.nen.size();
    std::string err;
    if (m.setup(err)) {
        std::puts(err.c_str());
        std::exit(2);
    }
}

// box of nx x ny x nz nodes with spacing (hx, hy, hz); elements whose cell index is below pd in every direction are
// PD, those of the lowest `tets` layers are split into five tetrahedra
static void box(Model &m, int nx, int ny, int nz, double hx, double hy, double hz, int pd, int tets = 0) {
    material(m);
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
                static const int part[5][4] = {{0, 1, 2, 5}, {0, 2, 3, 7}, {0, 5, 7, 4}, {2, 7, 5, 6}, {0, 2, 7, 5}};
                if (k < tets) {
                    for (auto &t : part) {
                        for (int a = 0; a < 8; a++) m.econ.push_back(a < 4 ? e[t[a]] : -1);
                        m.nen.push_back(4);
                        m.algo.push_back(2);
                    }
                    continue;
                }
                m.econ.insert(m.econ.end(), e, e + 8);
                m.nen.push_back(8);
                m.algo.push_back(i < pd && j < pd && k < pd ? 1 : 2);
            }
    finish(m);
}

// cylinder of `sectors` wedge-shaped hexahedra around an axis node, `rings` more rings and `layers` layers of nodes:
// a node of the axis belongs to 2 * sectors elements
static void fan(Model &m, int sectors, int rings, int layers, double h) {
    material(m);
    const int n = 2 * sectors, per = 1 + n * rings;
    auto id = [&](int r, int s, int k) { return k * per + (r ? 1 + (r - 1) * n + (s % n) : 0); };
    for (int k = 0; k < layers; k++) {
        m.x.insert(m.x.end(), {0.0, 0.0, k * h});
        for (int r = 1; r <= rings; r++)
            for (int s = 0; s < n; s++) {
                const double a = 2 * M_PI * s / n, d = (r + n / 6.3) * h;
                m.x.insert(m.x.end(), {d * std::cos(a), d * std::sin(a), k * h});
            }
    }
    m.nn = per * layers;
    auto add = [&](int a, int b, int c, int d) {
        for (int q : {a, b, c, d, a + per, b + per, c + per, d + per}) m.econ.push_back(q);
        m.nen.push_back(8);
        m.algo.push_back(2);
    };
    for (int k = 0; k + 1 < layers; k++) {
        for (int s = 0; s < sectors; s++) add(id(0, 0, k), id(1, 2 * s, k), id(1, 2 * s + 1, k), id(1, 2 * s + 2, k));
        for (int r = 1; r < rings; r++)
            for (int s = 0; s < n; s++) add(id(r, s, k), id(r + 1, s, k), id(r + 1, s + 1, k), id(r, s + 1, k));
    }
    finish(m);
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
        c.nfe_off_host = off;
        c.nfe_item_host = item;
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
        if (hex_tiles(h.c, 0, t, err) || !t || !t->n_fam) return 3;
        work = t->n_work;
        calls = g_calls;
        free_hex_tiles(h.c);
    }
    for (int at = 0; at < calls; at++) {
        Host h(m);
        g_calls = 0;
        g_fail_at = at;
        for (int rep = 0; rep < 2; rep++)
            if (hex_tiles(h.c, 0, t, err) || t || h.c.hex || !g_live.empty()) return std::printf("allocation %d, call %d\n", at, rep), 4;
        g_fail_at = -1;
        Host n(m);
        if (hex_tiles(n.c, 0, t, err) || !t || t->n_work != work) return 5;
        free_hex_tiles(n.c);
    }
    // host memory too, on whichever thread it runs out
    long news = 0, failed = 0;
    for (long at = 0;; at += 1 + at / 3) {
        Host h(m);
        g_new_calls = 0;
        g_new_fail_at = at;
        const int rc = hex_tiles(h.c, 0, t, err);
        g_new_fail_at = -1;
        if (rc || !t != !h.c.hex || (!t && !g_live.empty())) return std::printf("host allocation %ld\n", at), 7;
        news = g_new_calls;
        failed += !t;
        free_hex_tiles(h.c);
        if (at > 2 * news) break;
    }
    if (failed < 10) return 8;
    std::printf("%d allocations, %d blocks; %ld host allocations, %ld failed\n", calls, work, news, failed);
    return g_live.empty() ? 0 : 6;
}
"""

RULE = RUNTIME + r"""
// tiles of m: whether there are any, the rows left to K; checks that every node is held once
static bool tiles(const char *name, const Model &m, size_t *rows = nullptr) {
    Host h(m);
    HexTilesHost H;
    hex_tiles_host(m, h.off, h.item, H);
    std::printf("%s: %d nodes, %zu tiles, %lld elements of %zu, %zu rows, %zu families, use %d %d\n", name, m.nn, H.tile.size(),
                H.n_ele, m.fe.size(), H.rows.size(), H.fams.size(), H.use[0], H.use[1]);
    if (rows) *rows = H.rows.size();
    if (H.tile.empty()) return false;
    std::vector<int> held(m.nn, 0);
    for (int r : H.rows) held[r]++;
    for (int f : H.fams) held[m.fam_node[f]]++;
    for (const HexTile &t : H.tile) {
        std::vector<int> seen(t.n_own, 0);  // corners of the tile's elements at each owned node
        if (t.n_node > HT_NODES || t.n_own > HT_OWN || t.n_ele % HT_GROUP) std::exit(7);
        for (int e = 0; e < t.n_ele * 8; e++) {
            const int l = H.conn[(size_t)t.ele0 * 8 + e];
            if (l != 0xffff && l >= t.n_node) std::exit(8);
            if (l < t.n_own) seen[l]++;
        }
        for (int i = 0; i < t.n_own; i++) {
            const int k = H.nodes[t.node0 + i];
            held[k]++;
            if (seen[i] != h.off[k + 1] - h.off[k]) std::exit(9);
        }
    }
    for (int k = 0; k < m.nn; k++)
        if (held[k] != 1) std::exit(10);
    return true;
}
int main() {
    const double s = 1e-3;
    struct { const char *name; int nx, ny, nz; double hz; int pd, tets; bool want; } c[] = {
        {"cube", 30, 30, 30, s, 8, 0, true},          {"plate of 4 layers", 80, 80, 4, s, 0, 0, true},
        {"bar", 5, 5, 1000, s, 0, 0, true},           {"few nodes", 26, 26, 30, s, 0, 0, false},
        {"small with PD", 28, 28, 28, s, 10, 0, false}, {"plate of 2 layers", 120, 120, 2, s, 0, 0, false}, {"spacing 100 : 1", 31, 31, 31, s / 100, 0, 0, false},
        {"a fifth tetrahedra", 33, 33, 33, s, 0, 6, false},
        {"mostly tetrahedra", 30, 30, 90, s, 0, 60, false}};
    for (auto &q : c) {
        Model m;
        box(m, q.nx, q.ny, q.nz, s, s, q.hz, q.pd, q.tets);
        if (tiles(q.name, m) != q.want) return 3;
    }
    // the axis nodes of a fan have more elements than a tile holds: their rows go to K, all others have tiles
    Model m;
    fan(m, 36, 12, 30, s);
    size_t rows = 0;
    if (!tiles("fan", m, &rows) || rows != 28) return 4;
    return 0;
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


def test_which_models_get_tiles(tmp_path):
    r = _run(tmp_path, RULE)
    assert r.returncode == 0, f"exit {r.returncode}: {r.stdout}{r.stderr}"
    print(r.stdout)
