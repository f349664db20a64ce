// Walks the prefill schedules' partial regions with the kernel's own index functions (kernels.hpp) and prints every
// region that two parts of different query tiles share, part runs that leave or repeat a key tile, and regions past
// the workspace. Arguments: the CU count; per line of the standard input one launch:
//   query heads, KV heads, pos, n, max_tokens, count, count values
// the values taking turns as the visible key tiles of the query tiles (0 or past the tile's own: all of its tiles, as
// without key bits). Prints "launches L split S mixed M worst W": launches read, those of the split schedule, those
// of them whose tiles differ in parts, the most parts; exit status 1 after any fault.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <utility>
#include <vector>

#include "kernels.hpp"

int main(int argc, char** argv) {
    const int n_cu = argc > 1 ? std::atoi(argv[1]) : 256;
    int nh, nkv, pos, n, max_tokens, count, faults = 0, launches = 0, split = 0, mixed = 0, worst = 0;
    while (std::scanf("%d %d %d %d %d %d", &nh, &nkv, &pos, &n, &max_tokens, &count) == 6) {
        std::vector<int> see(count);
        for (int& v : see)
            if (std::scanf("%d", &v) != 1) return 2;
        const int G = nh / nkv, tok = 128 / G, n_qt = qw::pf_query_tiles(n, G);
        const int split_all = qw::pf_parts(n_qt, nkv, n_cu, (pos + n + 63) / 64);
        const int slots = qw::pf_split_slots(n_qt, split_all), qt_max = qw::pf_query_tiles(max_tokens, G);
        const int regions = nkv * qw::pf_regions_per_head(qt_max, nkv, n_cu);
        auto tiles = [&](int qt) {
            const int all = (std::min(pos + n, pos + (qt + 1) * tok) + 63) / 64, v = count ? see[qt % count] : 0;
            return v > 0 && v < all ? v : all;
        };
        auto bad = [&](const char* what, int kvh, int qt, int part, int region) {
            std::printf("%d/%d heads pos %d n %d (%d parts): %s: KV head %d tile %d part %d region %d\n", nh, nkv, pos, n,
                        split_all, what, kvh, qt, part, region);
            faults++;
        };
        std::map<int, std::pair<int, int>> owner;  // region: (slot, part)
        auto take = [&](int kvh, int qt, int slot, int part) {
            const int r = qw::pf_region(slot, part, split_all);
            if (r < 0 || r >= regions) bad("outside the workspace", kvh, qt, part, r);
            if (!owner.emplace(r, std::make_pair(slot, part)).second) bad("shared", kvh, qt, part, r);
        };
        if (slots > qw::pf_slots_per_head(qt_max, nkv, n_cu)) bad("too many slots", 0, 0, 0, 0);
        int least = 1 << 30, most = 0;
        for (int kvh = 0; kvh < nkv; kvh++) {
            if (split_all == 0)
                for (int p = 0; p < n_qt / 2; p++)
                    for (int own = 0; own < 2; own++) take(kvh, n_qt - 1 - p, kvh * slots + p, own);
            for (int qt = 0; split_all && qt < n_qt; qt++) {
                const int nt = tiles(qt), parts = qw::pf_part(nt, split_all, 0).parts;
                least = std::min(least, parts), most = std::max(most, parts);
                int at = 0;
                for (int part = 0; part < parts; part++) {
                    const qw::PfPart p = qw::pf_part(nt, split_all, part);
                    if (p.parts != parts || p.lo != at || p.hi <= p.lo) bad("key tiles", kvh, qt, part, p.lo);
                    at = p.hi;
                    if (parts > 1) take(kvh, qt, kvh * slots + qt, part);
                }
                if (at != nt) bad("key tiles left", kvh, qt, parts, at);
            }
        }
        launches++, split += split_all > 0, mixed += least < most, worst = std::max(worst, most);
    }
    std::printf("launches %d split %d mixed %d worst %d\n", launches, split, mixed, worst);
    return faults ? 1 : 0;
}
