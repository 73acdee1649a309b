// Products with the stiffness of hex8 elements without their K blocks (hex.hip): the node tiles and
// the device code of one element, shared by the explicit step and the Krylov products.
#pragma once
#include <hip/hip_runtime.h>

#include "device.hpp"

namespace pdx {

constexpr int HT_THREADS = 256;           // a workgroup: four wavefronts, two threads per element
constexpr int HT_WAVES = 2;               // wavefronts per SIMD: an element's FP64 arithmetic holds about 180 registers
constexpr int HT_GROUP = 32;              // elements a wavefront takes at once
constexpr int HT_ELE = 256;               // element places of a tile, at most (a multiple of HT_GROUP)
constexpr int HT_OWN = 170;               // owned nodes of a tile, at most
constexpr int HT_NODES = 448;             // nodes staged per tile, at most
constexpr int HT_ACC = HT_OWN * 3;        // sums of one wavefront
constexpr int HT_LDS = HT_NODES * 6 + HT_THREADS / 64 * HT_ACC;  // doubles of LDS (37 KB)

// A tile owns up to HT_OWN nodes whose rows of K are sums of hex8 elements only and lists every
// element incident to them, so the workgroup of a tile forms the whole product of its nodes: no
// atomics and no second pass, at the price of computing the elements between two tiles in both.
struct HexTile {
    int node0, n_node;  // nodes[node0 ...]: the owned nodes, then the other nodes of the elements
    int ele0, n_ele;    // conn[(ele0 + e) * 8 ...]: local node numbers of element place e (0xffff: an empty place)
    // owned nodes; 0: not a tile but the n_node rows rows[node0 ...], -1: the n_node families fams[node0 ...]
    int n_own;
    int pad;
    double x[3];        // a point of the tile: coordinates are taken relative to it
};

struct HexTiles {
    // Work of every block.  The hardware deals blocks to the 8 XCDs round-robin; XCD x takes the
    // x-th contiguous eighth of the tiles and of the row blocks, the two spread evenly over its
    // list, so that the rows' K reads run beside the tiles' arithmetic.
    int n_work = 0;  // blocks: a multiple of 8, some without work
    HexTile *work = nullptr;
    int *nodes = nullptr;
    unsigned short *conn = nullptr;
    int *rows = nullptr;  // rows formed from K, a wavefront each
    int n_fam = 0;
    int *fams = nullptr;  // families whose rows hold nothing but their bonds, 16 lanes each
    int n_tile = 0, n_row = 0;
    long long n_ele = 0;  // elements of all tiles
    bool use[2] = {false, false};  // whether products of FP64 / FP32 vectors go through them
};
constexpr int HEX_ROWS = HT_THREADS / 64;  // rows of a block
constexpr int HEX_FAMS = HT_THREADS / 16;  // families of a block

struct HexTilesHost {
    std::vector<HexTile> tile, work;
    std::vector<int> nodes, rows, fams;
    std::vector<unsigned short> conn;
    long long n_ele = 0;
    bool use[2] = {false, false};  // as in HexTiles
};
void hex_tiles_host(const Model &m, const std::vector<int> &nfe_off, const std::vector<int> &nfe_item, HexTilesHost &H);

// Fewer nodes than this keep their rows in K: their tiles leave CUs idle through the several
// microseconds of one tile (explicit step at 24^3 nodes, 8^3 of them PD: 8.7 us against 6.8 for the walk of
// K; at 31^3, 10^3 PD: 12.2 against 12.7)
constexpr long long HEX_MIN_NODES = 20480;
// FP32 products walk the blocks up to this many nodes: 4-byte blocks stay in the 256 MB Infinity Cache
// so long.  Explicit step: 31^3 nodes 9.3 us against 12.2 through the tiles; 60^3: 44.6 against 44.5,
// for a longer first call; 66^3: 58.8 against 55.6; 80^3: 120 against 81.  Newmark iteration, penny
// box: 48^3 107 against 110, 60^3 156 against 169, 80^3 409 against 349.
constexpr int HEX_MIN_NODES_F32 = 262144;

// Microseconds of a product through the tiles and of one that walks K, as sums over what they consist
// of.  Least squares over explicit steps of 35 models of 24,000 to 720,000 nodes: cubes, plates of 2 to
// 6 node layers, bars, boxes with spacings up to 1 : 100, boxes partly of tetrahedra, PD blocks of 41^3
// and 49^3 nodes.  The tiles' sum is within 17% of each, the walk's within 20%.  A tile of a cube holds
// 143 nodes and an element is computed 1.6 times; at a spacing of 1 : 10 it is 50 and 3.8, at 1 : 100 19
// and 7.3.  A row left to K costs a wavefront that reads it unmirrored.  A family's chain of loads shows in
// a short launch: 28^3 nodes 9.0 us against 9.3 for the walk, with 9^3 PD nodes 11.5 against 9.7; 33^3 with
// 8^3 12.5 against 13.6, 48^3 with 10^3 24.9 against 32.9.
inline double hex_tiles_us(double elements, double tiles, double rows, double families) {
    return 6.0 + 5.7e-5 * elements + 5.9e-3 * tiles + 1.5e-3 * rows + 1.4e-3 * families + (families > 0.0 ? 1.8 : 0.0);
}
inline double hex_walk_us(double blocks) { return 3.3 + 1.11e-5 * blocks; }
// FP32 blocks in mirrored storage, from HEX_MIN_NODES_F32 nodes on: up to some 9M blocks stay in the
// Infinity Cache (15 models of 216,000 to 1,080,000 nodes, within 10%)
inline double hex_walk_f32_us(double blocks) {
    return blocks <= 9e6 ? 7.0e-6 * blocks : 63.0 + 1.45e-5 * (blocks - 9e6);
}
// FP64 products go through the tiles up to this multiple of the walk's sum, FP32 products up to the walk's
// own: on these models that is the faster way, or one within 3% of it (elsewhere the worst seen is 30^3 with
// 8^3 PD nodes, 11.4 us through the tiles and 10.8 by the walk).  FP64 steps through the tiles
// against the walk: 60^3 35 and 62 us, plate of 400 x 400 x 4 87 and 204, bar 5 x 5 x 8000 21 and 41; but
// 300 x 300 x 2 52 and 38, 60^3 with a spacing of 1 : 10 70 and 62, of 1 : 100 148 and 62, with a fifth of
// tetrahedra 95 and 59, a tenth of them spread out 216 and 62.  FP32: 80^3 72 and 113, 600 x 600 x 2 192
// and 116, 70^3 with a spacing of 1 : 3 55 and 63, of 1 : 5 70 and 62.
constexpr double HEX_WALK = 1.1;

// The context's tiles (built on first use) for products of vectors of precision index pi (0 FP64, 1 FP32),
// or null where these walk K: 2D models, models with few nodes whose rows are hex8 sums (HEX_MIN_NODES,
// HEX_MIN_NODES_F32), and those whose tiles would take longer (HEX_WALK)
int hex_tiles(Ctx &c, int pi, const HexTiles *&out, std::string &err);
void free_hex_tiles(Ctx &c);

// lane l ^ 1's value
__device__ inline double pair_swap(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

// Half of an element's product: the four Gauss points of the plane zeta = -g (h = 0) or +g (h = 1).
// n[0..3] / n[4..7]: x (comps 0-2) and u (3-5) of the lower / upper corners, u relative or not.
// f[i][c], i < 4: force on corner 4 h + i of both planes together (the two threads of an element
// are lanes 2 e and 2 e + 1 of one wavefront, and both run this together).
//
// With xp, xd the trilinear interpolation to the plane and its zeta derivative at the four edges,
// every parent derivative in the plane is (a corner difference) + (position) * (a difference of
// differences): 30 differences serve the four points.  All derivatives are taken for parent
// coordinates in [0, 1] (twice the ones of [-1, 1]): J and H = du/dxi scale alike, so grad u does not
// change, and the 1/8 left in w detJ J^-1 sits in lam and mu.  Per point, with the cofactor rows A_k
// (J^-1 = A / det): G = A^T H, sigma = lam tr(G) I + mu (G + G^T) over det, P_k = A_k . sigma (detJ
// cancels), then the transposes of the interpolations.  About 700 VALU instructions per thread.
// MASS adds rho N_a N_b detJ of the consistent mass to the product (rho8 = rho / 8).
// FP64 for FP32 vectors too: without packed instructions FP32 arithmetic has FP64's rate, and the
// FP32 form of this code took longer (115 us against 92 per product on the 80^3 box: its additions in
// LDS, ds_add_f32, waited ten times as long).
template <bool MASS>
__device__ inline void hex_plane(const double (&nb)[4][6], const double (&nt)[4][6], int h, double lam8, double mu8,
                                 double rho8, double (&f)[4][3]) {
    using T = double;
    const T g0 = T(0.21132486540518711775), g1 = T(0.78867513459481288225);  // (1 -+ 1/sqrt 3) / 2
    const T mz = h ? g1 : g0;
    T s0[6], e0[6], cc[6], z0[6], zs[6], ze[6], zc[6], v0[3];
#pragma unroll
    for (int c = 0; c < 6; c++) {
        T d[4], p[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            d[i] = nt[i][c] - nb[i][c];
            p[i] = nb[i][c] + mz * d[i];
        }
        s0[c] = p[1] - p[0];
        e0[c] = p[3] - p[0];
        cc[c] = (p[2] - p[3]) - s0[c];
        z0[c] = d[0];
        zs[c] = d[1] - d[0];
        ze[c] = d[3] - d[0];
        zc[c] = (d[2] - d[3]) - zs[c];
        if (MASS && c >= 3) v0[c - 3] = p[0];
    }
    // sums of the transposed products, one per coefficient above
    T S[3], E[3], C[3], D[3], ZS[3], ZE[3], ZC[3], V[3];
#pragma unroll
    for (int c = 0; c < 3; c++) S[c] = E[c] = C[c] = D[c] = ZS[c] = ZE[c] = ZC[c] = V[c] = T(0);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const T m = q & 2 ? g1 : g0, l = q & 1 ? g1 : g0, lm = m * l;
        T rx[6], re[6], rz[6];  // d/dxi, d/deta, d/dzeta of x and u
#pragma unroll
        for (int c = 0; c < 6; c++) {
            rx[c] = s0[c] + m * cc[c];
            re[c] = e0[c] + l * cc[c];
            rz[c] = z0[c] + l * zs[c] + m * ze[c] + lm * zc[c];
        }
        T A0[3], A1[3], A2[3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int j = (i + 1) % 3, k = (i + 2) % 3;
            A0[i] = re[j] * rz[k] - re[k] * rz[j];
            A1[i] = rz[j] * rx[k] - rz[k] * rx[j];
            A2[i] = rx[j] * re[k] - rx[k] * re[j];
        }
        const T det = rx[0] * A0[0] + rx[1] * A0[1] + rx[2] * A0[2];
        // 1 / det: the hardware estimate and two Newton steps, within a unit in the last place
        T inv = __builtin_amdgcn_rcp(det);
        inv = inv + inv * (T(1) - det * inv);
        inv = inv + inv * (T(1) - det * inv);
        T G[3][3];
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
            for (int c = 0; c < 3; c++) G[i][c] = A0[i] * rx[3 + c] + A1[i] * re[3 + c] + A2[i] * rz[3 + c];
        const T mu = mu8 * inv, lt = lam8 * inv * (G[0][0] + G[1][1] + G[2][2]), m2 = mu + mu;
        const T sxx = lt + m2 * G[0][0], syy = lt + m2 * G[1][1], szz = lt + m2 * G[2][2];
        const T sxy = mu * (G[0][1] + G[1][0]), syz = mu * (G[1][2] + G[2][1]), szx = mu * (G[2][0] + G[0][2]);
        const T sg[3][3] = {{sxx, sxy, szx}, {sxy, syy, syz}, {szx, syz, szz}};
#pragma unroll
        for (int c = 0; c < 3; c++) {
            T px = A0[0] * sg[0][c] + A0[1] * sg[1][c] + A0[2] * sg[2][c];
            T pe = A1[0] * sg[0][c] + A1[1] * sg[1][c] + A1[2] * sg[2][c];
            const T pz = A2[0] * sg[0][c] + A2[1] * sg[1][c] + A2[2] * sg[2][c];
            if (MASS) {
                // the value of u at the point, times rho detJ
                const T v = (v0[c] + m * e0[3 + c] + l * rx[3 + c]) * (rho8 * det);
                V[c] += v;
                S[c] += l * v;
                E[c] += m * v;
                C[c] += lm * v;
            }
            S[c] += px;
            E[c] += pe;
            C[c] += m * px + l * pe;
            D[c] += pz;
            ZS[c] += l * pz;
            ZE[c] += m * pz;
            ZC[c] += lm * pz;
        }
    }
    const T cm = h ? mz : T(1) - mz, sm = h ? T(1) : T(-1);
#pragma unroll
    for (int c = 0; c < 3; c++) {
        T fp[4], fd[4];
        fp[0] = C[c] - S[c] - E[c];
        if (MASS) fp[0] += V[c];
        fp[1] = S[c] - C[c];
        fp[2] = C[c];
        fp[3] = E[c] - C[c];
        fd[0] = D[c] - ZS[c] - ZE[c] + ZC[c];
        fd[1] = ZS[c] - ZC[c];
        fd[2] = ZC[c];
        fd[3] = ZE[c] - ZC[c];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // this plane's share of this thread's corner and of the other thread's
            const T mine = cm * fp[i] + sm * fd[i], other = fp[i] - mine;
            f[i][c] = mine + pair_swap(other);
        }
    }
}

// addition to a sum in LDS in one operation (ds_add), and a point that the additions of a wavefront
// are not moved across
__device__ inline void lds_add(double *p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Sums of the element forces of a tile: x and u of the tile's nodes are staged in LDS, and each
// wavefront takes every fourth group of 32 elements and adds their corner forces to sums of its own.
// The LDS operations of a wavefront run in order, and the host places the elements so that no two of
// one group have a node in the same corner: each addition has its place in a fixed order, so the sums
// are the same bits every time.  x is kept relative to a point of the tile, so that J does not lose
// digits far from the origin.  Every thread of the workgroup must call it; after a barrier
// hex_tile_sum(lds, n * 3 + c) is component c of owned node n and hex_tile_u(lds, n, c) its u.
template <bool MASS, typename X>
__device__ inline void hex_tile_product(const HexTile &t, const HexTiles &ht, const double *__restrict__ x,
                                        const X *__restrict__ u, double lam8, double mu8, double rho8, double *lds) {
    const int tid = threadIdx.x, wave = tid >> 6, h = tid & 1;
    // everything that depends on the tile alone is loaded before anything is waited for
    const uint4 *cn = reinterpret_cast<const uint4 *>(ht.conn) + t.ele0 + ((tid & 63) >> 1);
    uint4 w = make_uint4(~0u, ~0u, ~0u, ~0u);
    if (wave * HT_GROUP < t.n_ele) w = cn[wave * HT_GROUP];
    constexpr int NS = (HT_NODES + HT_THREADS - 1) / HT_THREADS;
    int id[NS];
#pragma unroll
    for (int k = 0; k < NS; k++) id[k] = tid + k * HT_THREADS < t.n_node ? ht.nodes[t.node0 + tid + k * HT_THREADS] : -1;
    double xv[NS][3];
    X uv[NS][3];
#pragma unroll
    for (int k = 0; k < NS; k++)
        if (id[k] >= 0) {
            const size_t o = (size_t)id[k] * 3;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                xv[k][c] = x[o + c];
                uv[k][c] = u[o + c];
            }
        }
    double *acc = lds + HT_NODES * 6 + wave * HT_ACC;
    for (int k = tid & 63; k < t.n_own * 3; k += 64) acc[k] = 0.0;
#pragma unroll
    for (int k = 0; k < NS; k++)
        if (id[k] >= 0) {
            double *d = lds + (tid + k * HT_THREADS) * 6;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                d[c] = xv[k][c] - t.x[c];
                d[3 + c] = double(uv[k][c]);
            }
        }
    __syncthreads();
    for (int g = wave; g * HT_GROUP < t.n_ele; g += HT_THREADS / 64) {
        // the pair of threads of an element: lanes 2 e and 2 e + 1; eight 16-bit node numbers in one load
        const unsigned l[4] = {w.x, w.y, w.z, w.w};
        if ((g + HT_THREADS / 64) * HT_GROUP < t.n_ele) w = cn[(g + HT_THREADS / 64) * HT_GROUP];
        auto local = [&](int i) { return (l[i >> 1] >> (16 * (i & 1))) & 0xffffu; };
        if (local(0) == 0xffffu) continue;  // both threads of the pair
        double nb[4][6], nt[4][6], f[4][3];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const double *b = lds + local(i) * 6, *a = lds + local(4 + i) * 6;
#pragma unroll
            for (int c = 0; c < 6; c++) {
                nb[i][c] = b[c];
                nt[i][c] = a[c];
            }
        }
        hex_plane<MASS>(nb, nt, h, lam8, mu8, rho8, f);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int n = h ? local(4 + i) : local(i);
            // one corner of the 32 elements per addition: no two of its lanes add to one sum
            if (n < t.n_own && h == 0)
#pragma unroll
                for (int c = 0; c < 3; c++) lds_add(&acc[n * 3 + c], f[i][c]);
            wave_order();
            if (n < t.n_own && h == 1)
#pragma unroll
                for (int c = 0; c < 3; c++) lds_add(&acc[n * 3 + c], f[i][c]);
            wave_order();
        }
    }
}

__device__ inline double hex_tile_u(const double *lds, int n, int c) { return lds[n * 6 + 3 + c]; }
__device__ inline double hex_tile_sum(const double *lds, int k) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < HT_THREADS / 64; w++) s += lds[HT_NODES * 6 + w * HT_ACC + k];
    return s;
}

// v of lane (l + N) % 16 of each 16 lanes
template <int N>
__device__ inline double row_rotate(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + N, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + N, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

struct MomentArgs {
    const int *fam_off, *fam_mem;
    const double *fam_v, *w, *T;
    double lam, mu;
};

// Row of K u of a family whose row holds nothing but its bonds, without the bonds' blocks.  The block
// of a bond is -v_k w_m M(A^-1 p(xi_m)) with M linear, so
//   sum_m K_km (u_m - u_k) = -v_k M(A^-1 sum_m w_m p(xi_m) (u_m - u_k)^T):
// 27 moments over the bonds, then 6 x 9 rows of the inverse shape tensor times three columns.  A bond
// is read as its weight and node (12 bytes) instead of a block and a column (76 bytes).  16 lanes per
// family; the result is in all of them.
template <typename X>
__device__ inline void family_row(const MomentArgs &A, int f, int lane, const double *__restrict__ x,
                                  const X *__restrict__ u, double (&v)[3]) {
    const int off = A.fam_off[f], n = A.fam_off[f + 1] - off;
    const size_t k = (size_t)A.fam_mem[off] * 3;
    const double xk[3] = {x[k], x[k + 1], x[k + 2]};
    const X uk[3] = {u[k], u[k + 1], u[k + 2]};
    double Q[9][3];
#pragma unroll
    for (int j = 0; j < 9; j++) Q[j][0] = Q[j][1] = Q[j][2] = 0.0;
#pragma unroll 2
    for (int m = 1 + lane; m < n; m += 16) {
        const size_t o = (size_t)A.fam_mem[off + m] * 3;
        const double w = A.w[off + m];
        const double a = x[o] - xk[0], b = x[o + 1] - xk[1], c = x[o + 2] - xk[2];
        const double p[9] = {a, b, c, a * a, b * b, c * c, a * b, b * c, c * a};
        const double d[3] = {w * double(u[o] - uk[0]), w * double(u[o + 1] - uk[1]), w * double(u[o + 2] - uk[2])};
#pragma unroll
        for (int j = 0; j < 9; j++)
#pragma unroll
            for (int i = 0; i < 3; i++) Q[j][i] += p[j] * d[i];
    }
    // lane r < 6: row r of the inverse shape tensor (xx, yy, zz, xy, yz, zx)
    double T[9];
#pragma unroll
    for (int j = 0; j < 9; j++) T[j] = lane < 6 ? A.T[(size_t)f * 54 + lane * 9 + j] : 0.0;
    double D[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 9; j++)
#pragma unroll
        for (int i = 0; i < 3; i++) {
            double q = Q[j][i];
            q += row_rotate<8>(q);
            q += row_rotate<4>(q);
            q += row_rotate<2>(q);
            q += row_rotate<1>(q);
            D[i] += T[j] * q;
        }
    // (lam + mu) grad div u + mu laplacian u, lane by lane
    const double l2 = A.lam + 2.0 * A.mu, lm = A.lam + A.mu, mu = A.mu;
    v[0] = lane < 3 ? (lane == 0 ? l2 : mu) * D[0] : lane == 3 ? lm * D[1] : lane == 5 ? lm * D[2] : 0.0;
    v[1] = lane < 3 ? (lane == 1 ? l2 : mu) * D[1] : lane == 3 ? lm * D[0] : lane == 4 ? lm * D[2] : 0.0;
    v[2] = lane < 3 ? (lane == 2 ? l2 : mu) * D[2] : lane == 4 ? lm * D[1] : lane == 5 ? lm * D[0] : 0.0;
    const double cdv = A.fam_v[f];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        v[i] += row_rotate<8>(v[i]);
        v[i] += row_rotate<4>(v[i]);
        v[i] += row_rotate<2>(v[i]);
        v[i] += row_rotate<1>(v[i]);
        v[i] = -(v[i] * cdv);
    }
}

inline MomentArgs moment_args(const Ctx &c) {
    return MomentArgs{c.fam_off, c.fam_mem, c.fam_v, c.mom_w, c.mom_T, c.lambda, c.mu};
}

}  // namespace pdx
