// Seeded normal values of the learned smoother's probes.
#pragma once

#include <algorithm>
#include <cstddef>
#include <random>
#include <vector>

namespace pdx {

// The generator's draws of one block, handed out in order; past the block's end it returns a value
// that every attempt accepts, so a block's last attempt ends without a read past its draws.
struct BlockDraws {
    typedef std::mt19937_64::result_type result_type;
    const result_type *p;
    int n, i;
    static constexpr result_type min() { return std::mt19937_64::min(); }
    static constexpr result_type max() { return std::mt19937_64::max(); }
    result_type operator()() { return i < n ? p[i++] : (i++, result_type(3) << 62); }
};

// v(i), i < n: the first n values of std::normal_distribution<double> on std::mt19937_64(seed), bit
// for bit, given to put(i, v) in blocks on several threads.  The distribution's polar method spends
// two draws an attempt and gives two values for an accepted one, so any even position of the
// generator's sequence starts an attempt: one thread draws, blocks of PROBE_PAIRS attempts become
// values on the others, and the values of a block follow those of the blocks before it.
// 1,008,016 values and their copy to the device in loss_grad: 21.3 ms serial, 4.2 ms on 16 threads.
constexpr int PROBE_PAIRS = 4096, PROBE_BLOCKS = 256;

template <class PUT>
void seeded_normals(unsigned long long seed, size_t n, const PUT &put) {
    std::mt19937_64 rng(seed);
    size_t done = 0;
    std::vector<std::mt19937_64::result_type> raw;
    std::vector<double> val;
    std::vector<size_t> first(PROBE_BLOCKS + 1);
    while (done < n) {
        // an attempt is accepted with probability pi/4, a value needs 2/pi attempts
        const size_t want = (size_t)((double)(n - done) * 0.6367) + 8;
        const int draws = 2 * (int)std::min<size_t>(want, PROBE_PAIRS);
        const int nb = (int)std::min<size_t>((want * 2 + draws - 1) / draws, PROBE_BLOCKS);
        if (raw.size() < (size_t)nb * draws) {
            raw.resize((size_t)nb * draws);
            val.resize((size_t)nb * draws);
        }
#pragma omp parallel if (nb > 1)
#pragma omp single
        for (int b = 0; b < nb; b++) {
            std::mt19937_64::result_type *r = raw.data() + (size_t)b * draws;
            for (int i = 0; i < draws; i++) r[i] = rng();
#pragma omp task firstprivate(b, r)
            {
                std::normal_distribution<double> nd(0.0, 1.0);
                BlockDraws u{r, draws, 0};
                double *v = val.data() + (size_t)b * draws;
                size_t k = 0;
                while (u.i < draws) {
                    const double a = nd(u), c = nd(u);
                    if (u.i > draws) break;
                    v[k] = a;
                    v[k + 1] = c;
                    k += 2;
                }
                first[b + 1] = k;
            }
        }
        first[0] = 0;
        for (int b = 0; b < nb; b++) first[b + 1] += first[b];
#pragma omp parallel for schedule(dynamic, 1) if (nb > 1)
        for (int b = 0; b < nb; b++) {
            const double *v = val.data() + (size_t)b * draws;
            for (size_t k = first[b]; k < first[b + 1] && done + k < n; k++) put(done + k, v[k - first[b]]);
        }
        done += first[nb];
    }
}

}  // namespace pdx
