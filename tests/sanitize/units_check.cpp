// Wave units of the batched queue (test infrastructure): for random problem sets and every wave
// tile size, the units that the workgroups of a launch read cover each 16 x 16 atom of every
// queue entry once, none is larger than the size allows, and no place of the array is left out.
#include "batched.hip"

#include <cstdio>
#include <random>

using namespace kami;

static int check(int prec, std::mt19937& rng, int count, int hi) {
    std::uniform_int_distribution<int> size(1, hi / 16);
    std::vector<kami_problem> probs(count);
    std::vector<int> bucket(count);
    int variants[125];
    std::uniform_int_distribution<int> any(0, variants_of(prec) - 1);
    for (int& v : variants) v = any(rng);
    for (int i = 0; i < count; ++i) {
        kami_problem& p = probs[i];
        p = kami_problem{16 * size(rng), 16 * size(rng), 16 * size(rng), 0, 0, 0, 0, nullptr, nullptr, nullptr};
        p.lda = p.ldb = p.k;
        p.ldc = p.n;
        bucket[i] = bucket_of(p);
    }
    std::vector<WorkItem> items;
    build_items(probs, bucket, variants, elt_in(prec), elt_out(prec), false, items);
    const int64_t n = (int64_t)items.size();
    int bad = 0;
    for (int cap = 0; cap < kCaps; ++cap) {
        const int64_t n_units = count_units(items.data(), n, cap);
        if (n_units % (kWavesPerGroup * kXcds)) ++bad;
        const WaveUnit none{UINT32_MAX, 0, 0, 0, 0};
        std::vector<WaveUnit> units(n_units, none);
        build_units(items.data(), n, cap, n_units, units.data());
        std::vector<std::vector<int>> covered(n);
        for (int64_t i = 0; i < n; ++i) covered[i].assign(64, 0);
        const int64_t groups = batched_groups(n_units);
        std::vector<char> read(n_units, 0);
        for (int64_t L = 0; L < groups; ++L)
            for (int w = 0; w < kWavesPerGroup; ++w) {
                const int64_t at = unit_at(L, groups, w);
                if (at < 0 || at >= n_units || read[at]++) { ++bad; continue; }
                const WaveUnit u = units[at];
                if (u.item == UINT32_MAX) { ++bad; continue; }
                if (u.im == 0) continue;
                if (u.item >= n || u.im > kCapM[cap] || u.jn > kCapN[cap] || u.jn == 0) { ++bad; continue; }
                for (int r = u.ra; r < u.ra + u.im; ++r)
                    for (int c = u.ca; c < u.ca + u.jn; ++c) {
                        if (r >= 8 || c >= 8) ++bad; else ++covered[u.item][r * 8 + c];
                    }
            }
        for (int64_t i = 0; i < n; ++i) {
            const WorkItem& w = items[i];
            const int am = std::min(w.mlim, kVariantTM[w.variant]) / 16, an = std::min(w.nlim, kVariantTN[w.variant]) / 16;
            for (int r = 0; r < 8; ++r)
                for (int c = 0; c < 8; ++c) bad += covered[i][r * 8 + c] != (r < am && c < an);
        }
    }
    return bad;
}

int main() {
    std::mt19937 rng(7);
    int bad = 0, sets = 0;
    for (int prec : {KAMI_PREC_F64, KAMI_PREC_F16_F32})
        for (int count : {1, 2, 7, 33, 100, 1000})
            for (int hi : {16, 64, 256, 400}) {
                bad += check(prec, rng, count, hi);
                ++sets;
            }
    std::printf("%d problem sets, %d faults\n", sets, bad);
    return bad != 0;
}
