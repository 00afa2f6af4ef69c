// The handle's host copy of the clock against the device's after every call that can
// change either: gam_put_state and gam_set_clock write the host copy back whole, so
// a word that differs would return to the device later.
//
// TEST INFRASTRUCTURE ONLY.  Built for the CPU emulation with the step library's sources.
#include "gam_api.hip"

#include <cstdio>

static int bad = 0;
static void same(gam_handle *h, const char *after) {
    gam_sync(h);
    if (std::memcmp(h->clk, h->clk_host, sizeof(DClock)) == 0) return;
    std::printf("the clock's copies differ after %s (halt %d/%d, halted %d/%d)\n", after, h->clk->halt, h->clk_host->halt,
                h->clk->halted, h->clk_host->halted);
    bad++;
}

int main() {
    for (int precision = 0; precision < 2; precision++) {
        gam_dims d = {9, 8, 2, 4};
        gam_params p = {};
        p.gamma = 5.0 / 3.0; p.CFL = 0.3; p.pdmb = 4.0; p.Vd0 = 0.5; p.cHogH = 0.25; p.cHogM = 0.25; p.Ca = 1e12;
        p.dFloor = 1e-6; p.pFloor = 1e-6; p.tFin = 1e8; p.limDT0 = 1e-4; p.limCPR = 0.25;
        p.rmeth = 1; p.doLFMLim = 1; p.doMHD = 1; p.precision = precision;
        gam_handle *h = nullptr;
        if (gam_create(&d, &p, &h)) return 2;
        same(h, "gam_create");
        const int n[3] = {d.Nip + 9, d.Njp + 9, d.Nkp + 9};
        const size_t F = (size_t)n[0] * n[1] * n[2];
        std::vector<double> xyz(3 * F), gas(5 * gsz(h)), mag(3 * F);
        for (size_t q = 0; q < F; q++) {
            const int ijk[3] = {(int)(q % n[0]), (int)(q / n[0]) % n[1], (int)(q / n[0] / n[1])};
            for (int x = 0; x < 3; x++) xyz[x * F + q] = (ijk[x] - 4.0) / 9.0;
        }
        if (gam_set_corners(h, xyz.data()) || gam_ic_orszag_tang(h, 2.7, 1.6, 1.0, 6.0)) return 2;
        if (gam_hatch(h)) return 2;
        same(h, "gam_hatch");
        if (gam_step(h, 2)) return 2;
        same(h, "gam_step");
        double t, dt;
        int st;
        if (gam_get_state(h, 0, &t, gas.data(), mag.data(), nullptr)) return 2;
        if (gam_put_state(h, 0, t, gas.data(), mag.data(), nullptr)) return 2;
        same(h, "gam_put_state");
        if (gam_advance_mhd(h)) return 2;
        same(h, "gam_advance_mhd");
        if (gam_calc_dt(h, &dt, &st)) return 2;
        same(h, "gam_calc_dt");
        if (gam_enforce_bcs(h)) return 2;
        same(h, "gam_enforce_bcs");
        gam_clock c;
        if (gam_get_clock(h, &c)) return 2;
        c.dt0 = 1e6 * c.dt;   // CalcDT's limit against dt0 fails in the first of the steps
        if (gam_set_clock(h, &c)) return 2;
        same(h, "gam_set_clock");
        if (gam_step(h, 3) != 1) return 2;
        same(h, "a halt before the last step");
        if (gam_step(h, 1) != 1) return 2;
        same(h, "a step of a halted block");
        if (gam_put_state_device(h, 0, t, gas.data(), mag.data())) return 2;
        same(h, "gam_put_state_device on a halted block");
        gam_destroy(h);
    }
    return bad ? 1 : 0;
}
