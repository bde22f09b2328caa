// The library's choices by size and density, for the test beside it: one line in, one line out.
#include <stdio.h>

#include "wc_choose.hpp"

int main() {
    int scenes;
    while (scanf("%d", &scenes) == 1) {
        std::vector<wc::SceneFill> fills;
        for (int s = 0; s < scenes; ++s) {
            unsigned n;
            int R;
            double bin, h, rest, mass;
            if (scanf("%u %d %lf %lf %lf %lf", &n, &R, &bin, &h, &rest, &mass) != 6) return 1;
            fills.push_back(wc::scene_fill(n, R, bin, h, rest, mass));
        }
        const wc::TileShape t = wc::choose_tile_shape(fills);
        printf("%d %d %d %d\n", wc::start_on_tiles(fills, t) ? 1 : 0, t.x, t.y, t.z);
    }
    return 0;
}
