// swe_order.h -- the internal numbering's base order of a mesh handed over as a matrix graph (host code only).
#pragma once
#include <algorithm>
#include <atomic>
#include <thread>
#include <utility>
#include <vector>

#include "swe_amd.h"

namespace swe {

// Locality order of the CSR graph, for a mesh handed over without coordinates: the rows are bisected
// recursively, each part in the order of a breadth-first sweep from an end of it, so that every cut goes
// across the part's longer dimension and runs of consecutive rows are compact in every direction.  Cuts
// fall on multiples of the largest tile's rows while a part is larger than that, of a slice's below.  (A
// reverse Cuthill-McKee order makes runs thin strips: the 256 rows of a tile of a 50,000-node mesh then
// border on about 450 rows instead of 80.)
struct Bisector {
    const swe_mesh_desc& d;
    const int small, large;            // rows of a slice and of the largest tile
    std::vector<int> order;
    // Stamp of the part or sweep that holds the node.  Threads bisect different parts, but a sweep looks at the marks
    // of neighbours in other parts too.  Every stamp belongs to one thread, so whichever value of another's it finds
    // there compares unequal; atomic words make that a defined read, at the cost of a plain one.
    std::vector<std::atomic<int>> mark;
    std::atomic<int> stamp{1};         // (marks start at 0, which is no stamp)

    Bisector(const swe_mesh_desc& m, int slice_rows, int tile_rows)
        : d(m), small(slice_rows), large(tile_rows), order((size_t)m.np), mark((size_t)m.np) {
        for (int i = 0; i < m.np; ++i) order[(size_t)i] = i;
    }
    int get(int v) const { return mark[(size_t)v].load(std::memory_order_relaxed); }
    void set(int v, int to) { mark[(size_t)v].store(to, std::memory_order_relaxed); }
    // Breadth-first sweep from s over the nodes stamped `from`, restamped `to`, appended to seq.
    void sweep(int s, int from, int to, std::vector<int>& seq) {
        size_t h = seq.size();
        seq.push_back(s);
        set(s, to);
        for (; h < seq.size(); ++h)
            for (int p = d.ia[seq[h]] - 1; p < d.ia[seq[h] + 1] - 1; ++p) {
                const int v = d.ja[p] - 1;
                if (get(v) == from) {
                    set(v, to);
                    seq.push_back(v);
                }
            }
    }
    void run(int b, int e, int depth) {
        const int n = e - b;
        if (n <= small) return;
        const int part = stamp.fetch_add(3), seen = part + 1, done = part + 2;
        for (int q = b; q < e; ++q) set(order[(size_t)q], part);
        std::vector<int> seq, first;
        seq.reserve((size_t)n);
        for (int q = b; q < e; ++q) {                      // one connected piece after another
            if (get(order[(size_t)q]) != part) continue;
            first.clear();
            sweep(order[(size_t)q], part, seen, first);
            sweep(first.back(), seen, done, seq);
            for (int u : first)                            // (one-way references may leave some behind)
                if (get(u) == seen) sweep(u, seen, done, seq);
        }
        std::copy(seq.begin(), seq.end(), order.begin() + b);
        std::vector<int>().swap(seq);
        const int unit = (n > large) ? large : small;
        const int m = b + std::max(1, (n / 2 + unit / 2) / unit) * unit;
        if (m >= e) return;
        if (depth < 5 && n > (1 << 15)) {
            std::thread t([=] { run(b, m, depth + 1); });
            run(m, e, depth + 1);
            t.join();
        } else {
            run(b, m, depth + 1);
            run(m, e, depth + 1);
        }
    }
};

inline std::vector<int> locality_order(const swe_mesh_desc& d, int slice_rows, int tile_rows) {
    Bisector B(d, slice_rows, tile_rows);
    B.run(0, d.np, 0);
    return std::move(B.order);
}

}  // namespace swe
