// A box where no memory can be pinned: the handle is created, single and
// repeated steps return the scalars of the step that ran last, and the state
// comes down.
#include "hip_host.h"

#include "../../rast-3dmhd_amd/csrc/mhd_host.h"

using namespace rmhd;

// The close of a step, as its third stage does it: dt of the step that ran.
static void stage(const char *name, void **args) {
    if (!strstr(name, "7k_stageI") || !strstr(name, "ELi3ELi")) return;
    const BoxArgs &b = *static_cast<BoxArgs *>(args[0]);
    DevScalars *const sc = *static_cast<DevScalars **>(args[5]);
    sc->nit += 1;
    sc->dt_used = 0.25 * sc->nit;
    sc->umach_used = 0.5;
    if (b.p.report) *b.p.report = *sc;
}

int main(int argc, char **argv) {
    hh::no_pinned = argc > 1 && !strcmp(argv[1], "none");
    hh::on_launch = stage;
    mhd_desc d{};
    d.npx = d.npy = 8;
    d.npz = 6;
    d.gamma = 1.0;
    d.izcon = 1;
    mhd_t *h = nullptr;
    HH_CHECK(mhd_create(&d, &h) == MHD_OK);
    const std::vector<double> a(10, 1.0);
    const double *m = a.data();
    HH_CHECK(mhd_set_metrics(h, m, m, m, m, m, m, m, m, m, m, m) == MHD_OK);
    std::vector<double> field(10 * 10 * 8, 1.0);
    double *f = field.data();
    HH_CHECK(mhd_upload(h, f, f, f, f, f, nullptr, nullptr, nullptr) == MHD_OK);
    double dt = 0.0, um = 0.0;
    HH_CHECK(mhd_step(h, &dt, &um) == MHD_OK && dt == 0.25 && um == 0.5);
    HH_CHECK(mhd_steps(h, 3, &dt, &um) == MHD_OK && dt == 1.0);
    HH_CHECK(mhd_steps(h, 0, &dt, &um) == MHD_OK && dt == 1.0);
    HH_CHECK(mhd_download(h, f, nullptr, nullptr, f, nullptr, nullptr, nullptr, nullptr) == MHD_OK);
    mhd_destroy(h);
    HH_CHECK(hh::ranges.empty());
    return 0;
}
