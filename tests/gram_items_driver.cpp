// Prints the Gram's work items of a launch as the kernels compute them
// (rocket_amd/csrc/gram_items.hpp, compiled for the host), one line per id and
// working wave: item, first slab, wave, first A and B pattern, the slabs of
// the LDS quarters that hold them, the wave's slab, partial tile, offset in it.
// Arguments: count ks S remap.  First line: items per slab, slab_split,
// ids, items of the busiest XCD.
#include <algorithm>
#include <cstdio>
#include <cstdlib>

using std::min;  // as device code finds it

#include "../rocket_amd/csrc/gram_items.hpp"

int main(int argc, char **argv) {
    if (argc != 5) return 2;
    const int count = std::atoi(argv[1]), ks = std::atoi(argv[2]), S = std::atoi(argv[3]), remap = std::atoi(argv[4]);
    using namespace prnu;
    const int T = tri_items_per_slab(count);
    const ItemIndex index(T, ks, S);
    std::printf("%d %d %lld %lld\n", T, slab_split(count), (long long)index.ids(remap), (long long)index.xcd_items());
    for (int64_t id = 0; id < index.ids(remap); ++id) {
        int u, s;
        if (!index.at(id, remap, u, s)) continue;
        for (int wave = 0; wave < 8; ++wave) {
            const ItemWaves w = item_waves(u, count, wave, ks);
            if (w.out_tile < 0) continue;
            if ((w.a_off >> 7) >= w.nq || (w.b_off >> 7) >= w.nq) return 3;  // rows that are not loaded
            std::printf("%lld %d %d %d %d %d %d %d %d %d %d\n", (long long)id, u, s, wave, row_pattern(w, w.a_off),
                        row_pattern(w, w.b_off), w.kq[w.a_off >> 7], w.kq[w.b_off >> 7], w.kw, w.out_tile, w.out_off);
        }
    }
    return 0;
}
