// The tuner's report and the tiling it keeps agree, also where two candidates
// are closer than a nanosecond.
#include "hip_host.h"

#include "../../include/rast3dmhd_ensemble.h"
#include "../../rast-3dmhd_amd/csrc/mhd_host.h"

int main() {
    int calls = 0;
    hh::elapsed_ms = [&] { return 0.0512345f - 1e-8f * (float)((calls++ * 7) % 13); };
    mhd_desc d{};
    d.npx = 40;
    d.npy = 13;
    d.npz = 9;
    d.gamma = 1.0;
    d.precision = MHD_MIXED;
    mhd_ens_t *e = nullptr;
    HH_CHECK(mhd_ens_create(&d, 1, &e) == MHD_OK);
    const std::vector<double> a(42 * 15 * 11, 1.0);
    const double *m = a.data();
    HH_CHECK(mhd_ens_set_metrics(e, 0, m, m, m, m, m, m, m, m, m, m, m) == MHD_OK);
    HH_CHECK(mhd_ens_set_background(e, 0, m, m) == MHD_OK);
    HH_CHECK(mhd_ens_upload(e, 0, m, m, m, m, m, nullptr, nullptr, nullptr) == MHD_OK);
    char report[8192];
    HH_CHECK(mhd_ens_autotune(e, 1, report, sizeof report) == MHD_OK);
    HH_CHECK(report[strlen(report) - 1] == ']');
    int n = 0, best[4] = {0, 0, 0, 0}, t[4];
    double ms, least = 1e300;
    for (const char *p = report; (p = strchr(p, '{')); ++p, ++n) {
        HH_CHECK(sscanf(p, "{\"tile_x\": %d, \"tile_y\": %d, \"kdepth\": %d, \"grid\": %d, \"ms_step\": %lf}", &t[0], &t[1], &t[2],
                        &t[3], &ms) == 5);
        if (ms < least) {
            least = ms;
            memcpy(best, t, sizeof best);
        }
    }
    HH_CHECK(n == 84);
    HH_CHECK(mhd_ens_get_tile(e, &t[0], &t[1], &t[2], &t[3]) == MHD_OK);
    HH_CHECK(memcmp(best, t, sizeof best) == 0);
    mhd_ens_destroy(e);
    HH_CHECK(hh::ranges.empty());
    return 0;
}
