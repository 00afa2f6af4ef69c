// gam_set_tile reaches the launches of its stage: the grid of the stage's kernel is that of the
// tile's bricks.  Where a block's step does not take the separate launches by itself,
// the stage timers do.  Built with EMF_COL_MIN=0 the I and K edges walk columns.
//
// TEST INFRASTRUCTURE ONLY.  Built for the CPU emulation with the step library's sources.
#include "gam_api.hip"

#include <cstdio>

static std::vector<unsigned> blocks_of_step(gam_handle *h) {   // of every launch of a step, in order
    static std::vector<unsigned> seen;
    seen.clear();
    emu_on_launch = [](dim3 g) { seen.push_back(g.x); };
    gam_step(h, 1);
    emu_on_launch = nullptr;
    return seen;
}

int main() {
    int bad = 0;
    for (int precision = 0; precision < 2; precision++) {
        gam_dims d = {40, 12, 6, 4};
        gam_params p = {};
        p.gamma = 5.0 / 3.0; p.CFL = 0.3; p.pdmb = 4.0; p.Vd0 = 0.5; p.cHogH = 0.25; p.cHogM = 0.25; p.Ca = 1e12;
        p.dFloor = 1e-6; p.pFloor = 1e-6; p.tFin = 1e8; p.limDT0 = 1e-4; p.limCPR = 0.25;
        p.rmeth = 1; p.doLFMLim = 1; p.doMHD = 1; p.precision = precision;
        gam_handle *h = nullptr;
        if (gam_create(&d, &p, &h)) return 2;
        const int n[3] = {d.Nip + 9, d.Njp + 9, d.Nkp + 9};
        const size_t F = (size_t)n[0] * n[1] * n[2];
        std::vector<double> xyz(3 * F);
        for (size_t q = 0; q < F; q++) {
            const int ijk[3] = {(int)(q % n[0]), (int)(q / n[0]) % n[1], (int)(q / n[0] / n[1])};
            for (int x = 0; x < 3; x++) xyz[x * F + q] = (ijk[x] - 4.0) / 40.0;
        }
        if (gam_set_corners(h, xyz.data()) || gam_ic_orszag_tang(h, 2.7, 1.6, 1.0, 6.0) || gam_hatch(h)) return 2;
        gam_set_timing(h, 1);
        for (int st = 0; st < ST_N; st++) {
            if (!tiled_stage(st) || st == ST_BPOST) continue;   // periodic 3D: no bflux_post launch
            int keep[4];
            if (gam_get_tile(h, st, keep)) return 2;
            const std::vector<unsigned> before = blocks_of_step(h);
            if (gam_set_tile(h, st, 1, 1, 256, 0)) return 2;   // bricks that hold at most a few points of this block
            const std::vector<unsigned> after = blocks_of_step(h);
            if (gam_set_tile(h, st, keep[0], keep[1], keep[2], keep[3])) return 2;
            if (before == after || before != blocks_of_step(h)) {
                std::printf("precision %d: the tile of %s reaches no launch\n", precision, gam_stage_name(st));
                bad++;
            }
        }
        gam_destroy(h);
    }
    return bad ? 1 : 0;
}
