// Node tiles for the products with hex8 elements without their K blocks (hex.hpp): host set-up.
#include <hip/hip_runtime.h>
#include <omp.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <bitset>
#include <cmath>
#include <cstring>
#include <new>
#include <numeric>
#include <vector>

#include "hex.hpp"

namespace pdx {

namespace {

// one tile under construction on the host
struct HostTile {
    int n_own = 0;
    std::vector<int> node, ele, place;  // place: positions in ele in groups of HT_GROUP, -1 for an empty place
    std::vector<unsigned short> corner, conn;  // local numbers of the corners, by element and by place
};

// Out of memory inside a parallel loop: an exception must not leave the loop's body, so the first one is noted and
// thrown again behind the loop
class LoopMemory {
    std::atomic<bool> out{false};

public:
    template <typename F>
    void body(F &&f) {
        try {
            f();
        } catch (const std::bad_alloc &) {
            out = true;
        }
    }
    void check() const {
        if (out) throw std::bad_alloc();
    }
};

// v[b, e) by coordinate, then node
void sort_along(std::vector<int> &v, size_t b, size_t e, const double *x, int axis) {
    std::vector<std::pair<double, int>> k(e - b);
    for (size_t i = b; i < e; i++) k[i - b] = {x[(size_t)v[i] * 3 + axis], v[i]};
    std::sort(k.begin(), k.end());
    for (size_t i = b; i < e; i++) v[i] = k[i - b].second;
}

// the same for a long list: equal bins of the coordinate range, each sorted by itself
void sort_along_parallel(std::vector<int> &v, const double *x, int axis) {
    constexpr int NB = 1024;
    const size_t n = v.size();
    double lo = 1e300, hi = -1e300;
#pragma omp parallel for schedule(static) reduction(min : lo) reduction(max : hi)
    for (size_t i = 0; i < n; i++) {
        const double c = x[(size_t)v[i] * 3 + axis];
        lo = std::min(lo, c);
        hi = std::max(hi, c);
    }
    const double scale = hi > lo ? NB / (hi - lo) : 0.0;
    auto bin = [&](int k) { return std::min(NB - 1, std::max(0, int((x[(size_t)k * 3 + axis] - lo) * scale))); };
    std::vector<unsigned short> at(n);
#pragma omp parallel for schedule(static)
    for (size_t i = 0; i < n; i++) at[i] = (unsigned short)bin(v[i]);
    std::vector<size_t> off(NB + 1, 0);
    for (size_t i = 0; i < n; i++) off[at[i] + 1]++;
    for (int i = 0; i < NB; i++) off[i + 1] += off[i];
    std::vector<size_t> fill(off.begin(), off.end() - 1);
    std::vector<int> out(n);
    for (size_t i = 0; i < n; i++) out[fill[at[i]]++] = v[i];
    v.swap(out);
    LoopMemory mem;
#pragma omp parallel for schedule(dynamic, 8)
    for (int i = 0; i < NB; i++) mem.body([&] { sort_along(v, off[i], off[i + 1], x, axis); });
    mem.check();
}

// Nodes in slabs along x, the slabs in columns along y, each about `w` node spacings wide, the cuts
// (v[b, e) is sorted along the axis) moved to the widest gap between neighbouring coordinates near the even position (so that a mesh
// with layers is cut between layers); a column is then filled from below, node by node in z, until a
// tile is full.
void cut_even(const std::vector<int> &v, size_t b, size_t e, const double *x, int axis, double width,
              std::vector<size_t> &cuts) {
    cuts.assign(1, b);
    const size_t n = e - b;
    const double ext = n ? x[(size_t)v[e - 1] * 3 + axis] - x[(size_t)v[b] * 3 + axis] : 0.0;
    const size_t k = std::max<size_t>(1, (size_t)std::llround(ext / width));
    for (size_t i = 1; i < k; i++) {
        const size_t at = b + n * i / k, half = n / (4 * k) + 1;
        size_t lo = at > cuts.back() + half ? at - half : cuts.back() + 1, best = at;
        double gap = -1.0;
        for (size_t q = lo; q < std::min(e, at + half); q++) {
            const double d = x[(size_t)v[q] * 3 + axis] - x[(size_t)v[q - 1] * 3 + axis];
            if (d > gap) {
                gap = d;
                best = q;
            }
        }
        if (best > cuts.back()) cuts.push_back(best);
    }
    cuts.push_back(e);
}

// Elements into groups of HT_GROUP, in order, none beside another with the same node in the same
// corner (two elements of a consistently numbered mesh never are)
void place_elements(HostTile &t) {
    using Used = std::bitset<HT_NODES>;
    std::vector<std::array<Used, 8>> used;  // nodes in each corner of each group
    std::vector<int> count;                 // elements of each group
    size_t first = 0;                       // the first group with a place left
    t.place.clear();
    for (int e = 0; e < (int)t.ele.size(); e++) {
        const unsigned short *l = &t.corner[(size_t)e * 8];
        while (first < count.size() && count[first] == HT_GROUP) first++;
        size_t g = first;
        for (; g < count.size(); g++) {
            bool free = count[g] < HT_GROUP;
            for (int a = 0; a < 8 && free; a++) free = !used[g][a][l[a]];
            if (free) break;
        }
        if (g == count.size()) {
            count.push_back(0);
            used.emplace_back();
            t.place.resize(count.size() * HT_GROUP, -1);
        }
        for (int a = 0; a < 8; a++) used[g][a][l[a]] = true;
        t.place[g * HT_GROUP + count[g]++] = e;
    }
}

}  // namespace

// The tiles of a model on the host (nfe_off, nfe_item: per node its FE elements in element order, as
// FE position * 8 + corner); empty where no product would go through them
void hex_tiles_host(const Model &m, const std::vector<int> &nfe_off, const std::vector<int> &nfe_item, HexTilesHost &H) {
    // nodes whose row is a sum of hex8 elements only
    const std::vector<int> &off = nfe_off;
    auto inc = [&](int j) { return m.fe[nfe_item[j] >> 3]; };
    std::vector<char> hex((size_t)m.nn, 0);
#pragma omp parallel for schedule(static)
    for (int k = 0; k < m.nn; k++) {
        bool all = off[k + 1] > off[k] && m.famid[k] < 0;
        for (int j = off[k]; j < off[k + 1] && all; j++) all = m.nen[inc(j)] == 8;
        hex[k] = all;
    }
    std::vector<int> nodes;
    for (int k = 0; k < m.nn; k++)
        if (hex[k]) nodes.push_back(k);
    if ((long long)nodes.size() < HEX_MIN_NODES) return;
    // families of nodes without elements and without boundary terms; the other rows are left to K
    std::vector<char> edge((size_t)m.nn, 0);
    for (int p = 0; p < m.npdbe; p++)
        for (int a = 0; a < 4; a++) edge[m.pdbe[(size_t)p * 4 + a]] = 1;
    auto by_family = [&](int k) { return m.famid[k] >= 0 && !edge[k] && off[k + 1] == off[k]; };
    long long n_fam = 0, n_row = 0;
    for (int k = 0; k < m.nn; k++)
        if (!hex[k]) (by_family(k) ? n_fam : n_row)++;
    // no need to build them where even full tiles with the fewest elements would take too long
    const double limit = HEX_WALK * hex_walk_us(m.adj_off[m.nn]), nh = (double)nodes.size();
    const double limit32 = m.nn >= HEX_MIN_NODES_F32 ? hex_walk_f32_us(m.adj_off[m.nn]) : 0.0;
    if (hex_tiles_us(nh / 8, nh / HT_OWN, (double)n_row, (double)n_fam) > std::max(limit, limit32)) return;
    // mean node spacing, from the volume of the elements around the nodes
    double vol = 0.0;
    for (int k : nodes) vol += m.nv[k];
    const double sp = std::cbrt(vol / (double)nodes.size()), width = 5.0 * sp;
    std::vector<size_t> xs;
    sort_along_parallel(nodes, m.x.data(), 0);
    cut_even(nodes, 0, nodes.size(), m.x.data(), 0, width, xs);
    // columns: the slabs cut along y, each sorted along z
    std::vector<std::vector<size_t>> ys(xs.size() - 1);
    LoopMemory mem;
#pragma omp parallel for schedule(dynamic, 1)
    for (int s = 0; s < (int)xs.size() - 1; s++)
        mem.body([&] {
            sort_along(nodes, xs[s], xs[s + 1], m.x.data(), 1);
            cut_even(nodes, xs[s], xs[s + 1], m.x.data(), 1, width, ys[s]);
        });
    mem.check();
    std::vector<std::pair<size_t, size_t>> column;
    for (auto &y : ys)
        for (size_t q = 0; q + 1 < y.size(); q++) column.push_back({y[q], y[q + 1]});
    std::vector<std::vector<HostTile>> per_column(column.size());
    // a thread's marks are 10 bytes per node and element: as many threads as a gigabyte holds
    const double marks = 4.0 * m.ne + 6.0 * m.nn;
    const int threads = (int)std::max(1.0, std::min((double)omp_get_max_threads(), 1e9 / marks));
#pragma omp parallel num_threads(threads)
    {
        // number of the last tile that took the element / node
        std::vector<int> in_e, in_n;
        std::vector<unsigned short> loc;  // local number of a node of the current tile
        mem.body([&] {
            in_e.assign((size_t)m.ne, -1);
            in_n.assign((size_t)m.nn, -1);
            loc.resize((size_t)m.nn);
        });
        int serial = 0;
#pragma omp for schedule(dynamic, 1)
        for (int q = 0; q < (int)column.size(); q++) mem.body([&] {
            if (loc.size() != (size_t)m.nn) return;  // this thread's marks did not fit
            const size_t last = column[q].second;
            sort_along(nodes, column[q].first, last, m.x.data(), 2);
            size_t at = column[q].first;
            while (at < last) {
                HostTile t;
                serial++;
                size_t end = at, layer = at, ne = 0, nn = 0;
                for (size_t k = at; k < last; k++) {
                    const int nd = nodes[k];
                    if (k > at && m.x[(size_t)nd * 3 + 2] - m.x[(size_t)nodes[k - 1] * 3 + 2] > 0.3 * sp) layer = k;
                    size_t add = 0;
                    for (int j = off[nd]; j < off[nd + 1]; j++) add += in_e[inc(j)] != serial;
                    // eight new nodes per new element at most
                    if (ne + add > (size_t)HT_ELE || k - at + 1 > (size_t)HT_OWN || nn + 8 * add > (size_t)HT_NODES) break;
                    for (int j = off[nd]; j < off[nd + 1]; j++) {
                        const int e = inc(j);
                        if (in_e[e] == serial) continue;
                        in_e[e] = serial;
                        ne++;
                        for (int a = 0; a < 8; a++) {
                            int &v = in_n[m.econ[(size_t)e * 8 + a]];
                            nn += v != serial;
                            v = serial;
                        }
                    }
                    end = k + 1;
                }
                if (end == at) {  // a node of more elements than a tile holds: left to its row of K
                    at++;
                    continue;
                }
                // end on a layer of nodes where that keeps most of the tile
                if (end < last && layer > at && layer < end && layer - at >= (end - at) * 6 / 10) end = layer;
                // the owned nodes in node order, then the other nodes of their elements as these list them
                t.node.assign(nodes.begin() + at, nodes.begin() + end);
                std::sort(t.node.begin(), t.node.end());
                t.n_own = int(t.node.size());
                t.corner.reserve(HT_ELE * 8);
                serial++;
                for (int i = 0; i < t.n_own; i++) {
                    const int nd = t.node[i];
                    in_n[nd] = serial;
                    loc[nd] = (unsigned short)i;
                    for (int j = off[nd]; j < off[nd + 1]; j++) {
                        const int e = inc(j);
                        if (in_e[e] == serial) continue;
                        in_e[e] = serial;
                        t.ele.push_back(e);
                    }
                }
                std::sort(t.ele.begin(), t.ele.end());
                for (int e : t.ele)
                    for (int a = 0; a < 8; a++) {
                        const int v = m.econ[(size_t)e * 8 + a];
                        if (in_n[v] != serial) {
                            in_n[v] = serial;
                            loc[v] = (unsigned short)t.node.size();
                            t.node.push_back(v);
                        }
                        t.corner.push_back(loc[v]);
                    }
                place_elements(t);
                t.conn.assign(t.place.size() * 8, 0xffff);
                for (size_t i = 0; i < t.place.size(); i++)
                    if (t.place[i] >= 0) std::copy_n(&t.corner[(size_t)t.place[i] * 8], 8, &t.conn[i * 8]);
                t.corner = std::vector<unsigned short>();
                per_column[q].push_back(std::move(t));
                at = end;
            }
        });
    }
    mem.check();
    // flat arrays
    std::vector<const HostTile *> all;
    for (auto &col : per_column)
        for (auto &t : col) all.push_back(&t);
    H.tile.resize(all.size());
    size_t n_node = 0, n_ele = 0;
    for (size_t k = 0; k < all.size(); k++) {
        HexTile h{};
        h.node0 = (int)n_node;
        h.n_node = (int)all[k]->node.size();
        h.ele0 = (int)n_ele;
        h.n_ele = (int)all[k]->place.size();
        h.n_own = all[k]->n_own;
        for (int c = 0; c < 3; c++) h.x[c] = m.x[(size_t)all[k]->node[0] * 3 + c];
        n_node += all[k]->node.size();
        n_ele += all[k]->place.size();
        H.n_ele += (long long)all[k]->ele.size();
        H.tile[k] = h;
    }
    H.nodes.resize(n_node);
    H.conn.resize(n_ele * 8);
    std::vector<char> owned((size_t)m.nn, 0);
#pragma omp parallel for schedule(static)
    for (int k = 0; k < (int)all.size(); k++) {
        std::copy(all[k]->node.begin(), all[k]->node.end(), H.nodes.begin() + H.tile[k].node0);
        std::copy(all[k]->conn.begin(), all[k]->conn.end(), H.conn.begin() + (size_t)H.tile[k].ele0 * 8);
        for (int i = 0; i < all[k]->n_own; i++) owned[all[k]->node[i]] = 1;
    }
    for (int k = 0; k < m.nn; k++) {
        if (owned[k]) continue;
        if (by_family(k)) H.fams.push_back(m.famid[k]);
        else H.rows.push_back(k);
    }
    const double us = hex_tiles_us((double)H.n_ele, (double)all.size(), (double)H.rows.size(), (double)H.fams.size());
    H.use[0] = us <= limit;
    H.use[1] = us <= limit32;
    if (!H.use[0] && !H.use[1]) {
        H = HexTilesHost();
        return;
    }
    // each XCD's list: its eighth of the tiles, families and rows, evenly mixed
    const int n[3] = {(int)H.tile.size(), int(H.fams.size() + HEX_FAMS - 1) / HEX_FAMS,
                      int(H.rows.size() + HEX_ROWS - 1) / HEX_ROWS};
    std::vector<std::vector<HexTile>> list(8);
    size_t per = 0;
    for (int x = 0; x < 8; x++) {
        std::vector<std::pair<double, HexTile>> l;
        for (int kind = 0; kind < 3; kind++) {
            const int b = int((long long)n[kind] * x / 8), e = int((long long)n[kind] * (x + 1) / 8);
            for (int k = b; k < e; k++) {
                HexTile w{};
                if (kind == 0) {
                    w = H.tile[k];
                } else {
                    const int size = kind == 1 ? HEX_FAMS : HEX_ROWS, all = int(kind == 1 ? H.fams.size() : H.rows.size());
                    w.n_own = kind == 1 ? -1 : 0;
                    w.node0 = k * size;
                    w.n_node = std::min(size, all - w.node0);
                }
                l.push_back({(k - b + 0.5) / (e - b), w});
            }
        }
        std::stable_sort(l.begin(), l.end(), [](const auto &a, const auto &b) { return a.first < b.first; });
        for (auto &w : l) list[x].push_back(w.second);
        per = std::max(per, l.size());
    }
    H.work.assign(per * 8, HexTile{});
    for (int x = 0; x < 8; x++)
        for (size_t q = 0; q < list[x].size(); q++) H.work[q * 8 + x] = list[x][q];
}

// The device arrays of the tiles, and those of the family moments, which only products through the
// tiles read
static int build_hex_tiles(Ctx &c, HexTilesHost &H, std::string &err) {
    hex_tiles_host(*c.host, c.nfe_off_host, c.nfe_item_host, H);
    if (H.tile.empty()) return PDX_OK;
    auto *T = new HexTiles();
    c.hex = T;
    T->n_work = (int)H.work.size();
    T->n_fam = (int)H.fams.size();
    T->n_tile = (int)H.tile.size();
    T->n_row = (int)H.rows.size();
    T->n_ele = H.n_ele;
    T->use[0] = H.use[0];
    T->use[1] = H.use[1];
    auto alloc = [&](auto *&dst, size_t n) -> int {
        const hipError_t e = hipMalloc((void **)&dst, std::max<size_t>(n, 1) * sizeof(*dst));
        if (e == hipSuccess) return PDX_OK;
        dst = nullptr;
        (void)hipGetLastError();
        err = std::string("element tiles: ") + hipGetErrorString(e);
        return e == hipErrorOutOfMemory ? PDX_ERR_LIMIT : PDX_ERR_HIP;
    };
    auto up = [&](auto *&dst, const auto &src) -> int {
        if (int rc = alloc(dst, src.size())) return rc;
        if (!src.empty()) PDX_HIP(hipMemcpy(dst, src.data(), src.size() * sizeof(src[0]), hipMemcpyHostToDevice));
        return PDX_OK;
    };
    int rc;
    if ((rc = up(T->nodes, H.nodes)) || (rc = up(T->conn, H.conn)) || (rc = up(T->rows, H.rows)) ||
        (rc = up(T->work, H.work)) || (rc = up(T->fams, H.fams)))
        return rc;
    if (T->n_fam && ((rc = alloc(c.mom_w, c.host->fam_mem.size())) || (rc = alloc(c.mom_T, (size_t)c.nfam * 54)))) return rc;
    return PDX_OK;
}

int hex_tiles(Ctx &c, int pi, const HexTiles *&out, std::string &err) {
    out = nullptr;
    if (pi && c.nn < HEX_MIN_NODES_F32) return PDX_OK;
    if (!c.hex_tried && c.dim == 3 && c.host && c.host->dim == 3 && !c.nfe_off_host.empty()) {
        HexTilesHost H;
        int rc;
        try {
            rc = build_hex_tiles(c, H, err);
        } catch (const std::bad_alloc &) {
            rc = PDX_ERR_LIMIT;
        }
        if (rc) {
            free_hex_tiles(c);
            // out of memory: the walk of K needs none of these arrays, so this context keeps to it
            if (rc != PDX_ERR_LIMIT) return rc;
            err.clear();
        }
    }
    if (!c.hex_tried) {  // built, or never to be: the lists have served
        c.hex_tried = true;
        c.nfe_off_host = std::vector<int>();
        c.nfe_item_host = std::vector<int>();
    }
    const auto *T = (const HexTiles *)c.hex;
    if (T && T->use[pi]) out = T;
    return PDX_OK;
}

void free_hex_tiles(Ctx &c) {
    auto *T = (HexTiles *)c.hex;
    if (!T) return;
    for (void *p : {(void *)T->nodes, (void *)T->conn, (void *)T->rows, (void *)T->work, (void *)T->fams})
        if (p) hipFree(p);
    for (double **p : {&c.mom_w, &c.mom_T}) {
        if (*p) hipFree(*p);
        *p = nullptr;
    }
    c.mom_gen = -1;
    delete T;
    c.hex = nullptr;
    c.hex_tried = false;
}

}  // namespace pdx
