// The library's choices by size and density, for the test beside it: one line in, one line out.
#include <stdio.h>

#include "wc_choose.hpp"

// variants, whether the tile passes can run, then the times per mode and pass
static int tune() {
    int nv, tiles;
    while (scanf("%d %d", &nv, &tiles) == 2) {
        std::vector<double> t[2][2];
        for (auto& m : t)
            for (auto& v : m) {
                v.resize(nv);
                for (double& x : v)
                    if (scanf("%lf", &x) != 1) return 1;
            }
        for (const wc::TuningPick& p : wc::tuning_candidates(t, tiles != 0))
            printf("%d %d %d\n", p.density, p.update, p.lists ? 1 : 0);
    }
    return 0;
}

int main(int argc, char**) {
    if (argc > 1) return tune();
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
