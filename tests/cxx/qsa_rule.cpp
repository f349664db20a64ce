// Reads "pos n cr budget heads dims" lines and prints, for each, 1 where a block selection of such a call takes the
// many-token launches (the rule of kernels.hpp), else 0.
#include <cstdio>

#include "kernels.hpp"

int main() {
    int pos, n, cr, budget, ih, id;
    while (std::scanf("%d %d %d %d %d %d", &pos, &n, &cr, &budget, &ih, &id) == 6)
        std::printf("%d\n", (int)qw::qsa_many(pos, n, cr, budget, ih, id));
}
