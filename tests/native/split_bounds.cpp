// Random batches through the split choice of split_choice.hpp and the
// longest-first schedule's deal of groups to XCDs: the grid and the partial
// rows that split_bounds allows have to hold what the choice makes.  Prints
// how often each candidate was taken (4: none fits, 5: left whole) and how often a bound was
// met exactly; exits 1 at the first batch that breaks one.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <numeric>
#include <random>
#include <vector>

#include "split_choice.hpp"

int main(int argc, char **argv) {
    const int rounds = argc > 1 ? std::atoi(argv[1]) : 20000;
    std::mt19937 rng(7);
    auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    long taken[6] = {0, 0, 0, 0, 0, 0}, exact_wgs = 0, exact_rows = 0;
    for (int r = 0; r < rounds; ++r) {
        const int nx = pick(0, 3) ? 8 : pick(1, 6), Hkv = pick(1, 16), G = pick(1, 16), Hq = Hkv * G;
        const bool f32 = pick(0, 3) == 0;
        const int rows_wg = pick(0, 1) ? 128 : 256, slots = 256 * pick(1, 3), B = pick(1, 64);
        const int s_hi = 1 << pick(0, 14), p_hi = 1 << pick(0, 7), kind = pick(0, 3);
        std::vector<int> S(B), P(B), tiles(B), rb(B), ns(B), len(B);
        long total_q = 0, W = 0;
        for (int b = 0; b < B; ++b) {
            P[b] = kind == 1 ? p_hi : pick(pick(0, 9) ? 1 : 0, p_hi);
            S[b] = kind == 2 ? s_hi : kind == 3 && b ? pick(0, 64) : pick(0, s_hi);
            tiles[b] = P[b] ? (S[b] + P[b] + 63) / 64 : 0;
            rb[b] = P[b] ? (P[b] * G + rows_wg - 1) / rows_wg : 0;
            total_q += P[b];
            W += (long)tiles[b] * rb[b];
        }
        const long total = W * Hkv;
        if (!total) continue;
        const int share = std::max(1L, (total + slots - 1) / slots);
        const int start = cast::split_start(share, total, (int)(total / cast::split_few(f32, slots)), 2, f32, slots);
        auto items = [&](int c) {
            long n = 0;
            for (int b = 0; b < B; ++b) n += (long)rb[b] * ((tiles[b] + c - 1) / c);
            return n * Hkv;
        };
        bool fit[4];
        for (int w = 0; w < 4; ++w) fit[w] = items(cast::split_candidate(start, w)) <= slots;
        const int w = cast::split_pick(fit[0], fit[1], fit[2], fit[3]);
        const int t_max = *std::max_element(tiles.begin(), tiles.end());
        long rb_sum = 0, keys = 0;
        for (int b = 0; b < B; ++b) rb_sum += rb[b], keys += S[b] + P[b];
        const float limit =
            pick(0, 1) ? cast::split_even_limit(std::min((total_q + B - 1) / B, 128L) * G, (keys + B - 1) / B) : 0.f;
        const bool even = cast::split_even(t_max, (int)rb_sum, (int)W, limit);
        const int c = even ? t_max : cast::split_candidate(start, w);
        ++taken[even ? 5 : fit[w] ? w : 4];
        long part = 0;
        for (int b = 0; b < B; ++b) {
            ns[b] = (tiles[b] + c - 1) / c;
            len[b] = ns[b] ? (tiles[b] + ns[b] - 1) / ns[b] : 0;
            if (ns[b] > 1) part += (long)ns[b] * P[b];
        }
        // groups, longest first, dealt to the XCDs round-robin; a group takes
        // its request's row blocks in slots of one XCD
        std::vector<int> order(B);
        std::iota(order.begin(), order.end(), 0);
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return len[x] > len[y]; });
        std::vector<long> on(nx, 0);
        long g = 0;
        for (int b : order)
            for (long k = 0; k < (long)Hkv * ns[b]; ++k, ++g) on[g % nx] += rb[b];
        const long wgs = nx * *std::max_element(on.begin(), on.end());
        const int rbmax = (int)((std::min(total_q, 128L) * G + rows_wg - 1) / rows_wg);
        const cast::SplitBounds most = cast::split_bounds(B, total_q, Hq, Hkv, rows_wg, rbmax, slots, nx);
        if (wgs > most.wgs || part > most.part_rows) {
            std::printf("batch %d: %ld workgroups of %ld, %ld partial rows of %ld (nx %d Hkv %d G %d rows %d slots %d c %d)\n",
                        r, wgs, (long)most.wgs, part, (long)most.part_rows, nx, Hkv, G, rows_wg, slots, c);
            return 1;
        }
        exact_wgs += wgs == most.wgs;
        exact_rows += part == most.part_rows;
    }
    std::printf("taken %ld %ld %ld %ld %ld %ld exact %ld %ld ok\n", taken[0], taken[1], taken[2], taken[3], taken[4],
                taken[5], exact_wgs, exact_rows);
    return 0;
}
