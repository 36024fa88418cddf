// The locality order of host layouts (csrc/swe_order.h) on a row-numbered n x n lattice, large enough for its threads:
//   order_check N [REPEATS]
// prints "ok" and the longest and mean number of outside rows that runs of 256 consecutive rows border on, and the
// seconds per order; exits with 1 if an order is no permutation or differs from the first.  (Built with
// -fsanitize=thread by the test that runs it, it reports races.)
#include <chrono>
#include <cstdio>
#include <cstdlib>

#include "swe_order.h"

int main(int argc, char** argv) {
    const int n = argc > 1 ? std::atoi(argv[1]) : 300, repeats = argc > 2 ? std::atoi(argv[2]) : 1;
    const int np = n * n;
    std::vector<int> ia{1}, ja;
    for (int i = 0; i < np; ++i) {
        const int x = i % n, y = i / n;
        for (int dy = -1; dy <= 1; ++dy)
            for (int dx = -1; dx <= 1; ++dx)
                if (dx * dy >= 0 && x + dx >= 0 && x + dx < n && y + dy >= 0 && y + dy < n) ja.push_back(i + dx + n * dy + 1);
        ia.push_back((int)ja.size() + 1);
    }
    swe_mesh_desc d{};
    d.np = np;
    d.nnz = (int)ja.size();
    d.ia = ia.data();
    d.ja = ja.data();
    std::vector<int> first;
    double best = 1e30;
    for (int r = 0; r < repeats; ++r) {
        const auto t0 = std::chrono::steady_clock::now();
        const std::vector<int> order = swe::locality_order(d, 64, 256);
        best = std::min(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
        std::vector<char> seen((size_t)np, 0);
        for (int v : order)
            if (v < 0 || v >= np || seen[(size_t)v]++) return std::printf("not a permutation\n"), 1;
        if ((int)order.size() != np) return std::printf("%d of %d rows\n", (int)order.size(), np), 1;
        if (r == 0) first = order;
        else if (order != first) return std::printf("run %d differs\n", r), 1;
    }
    std::vector<int> pos((size_t)np), far;
    for (int q = 0; q < np; ++q) pos[(size_t)first[(size_t)q]] = q;
    size_t longest = 0, all = 0;
    for (int b = 0; b < np; b += 256) {
        far.clear();
        for (int q = b; q < std::min(np, b + 256); ++q)
            for (int p = ia[(size_t)first[(size_t)q]] - 1; p < ia[(size_t)first[(size_t)q] + 1] - 1; ++p) {
                const int w = pos[(size_t)ja[(size_t)p] - 1];
                if (w < b || w >= b + 256) far.push_back(w);
            }
        std::sort(far.begin(), far.end());
        const size_t h = (size_t)(std::unique(far.begin(), far.end()) - far.begin());
        longest = std::max(longest, h);
        all += h;
    }
    std::printf("ok %zu %.1f %.4f\n", longest, (double)all / ((np + 255) / 256), best);
    return 0;
}
