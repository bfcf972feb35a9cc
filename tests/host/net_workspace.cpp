// A network's workspace that could not grow: every later use of the network,
// by itself, in training and in a box's closure step, either reports the error
// or runs on buffers that exist and hold its volume.
#include "hip_host.h"

#include "../../include/rast3dmhd_closure.h"
#include "../../rast-3dmhd_amd/csrc/mhd_host.h"

static long long need;  // voxels of the volume in hand
static int launches, bad;

static void check(const char *name, void **args) {
    auto ptr = [&](int i, size_t bytes) {
        if (!hh::on_device(*static_cast<void **>(args[i]), bytes)) {
            printf("%s: argument %d\n", name, i);
            ++bad;
        }
    };
    const size_t v = (size_t)need;
    int cin, nt, epi;
    const char *const conv = strstr(name, "k_convILi");
    if (conv && sscanf(conv, "k_convILi%dELi%dELi%d", &cin, &nt, &epi) == 3) {
        ++launches;
        ptr(0, v * cin * 2);
        if (epi == 2) ptr(4, v * 32 * 4);
        if (epi == 1 || epi == 2 || epi == 4) ptr(5, v * 32 * 2);
        if (epi == 0 || epi == 3 || epi == 5) ptr(6, v * 8 * 4);
        if (epi == 1) ptr(7, v * 32 * 4);
    } else if (strstr(name, "k_dwI")) {
        ptr(0, v * 8 * 2), ptr(2, v * 8 * 2);
    } else if (strstr(name, "k_loss")) {
        ptr(0, v * 8 * 4);
    } else if (strstr(name, "k_f32_to_bf16")) {
        ptr(0, v * 7 * 4), ptr(1, v * 8 * 2);
    }
}

int main() {
    hh::on_launch = check;
    mhd_net_t *net = nullptr;
    HH_CHECK(mhd_net_create(8, 32, 7, &net) == MHD_OK);
    const std::vector<float> par((size_t)mhd_net_num_params(net), 0.1f);
    HH_CHECK(mhd_net_set_params(net, par.data()) == MHD_OK);

    mhd_desc d{};
    d.npx = d.npy = 8;
    d.npz = 6;
    d.lmag = 1;
    d.gamma = 1.0;
    d.izcon = 1;
    d.precision = MHD_MIXED;
    mhd_t *h = nullptr;
    HH_CHECK(mhd_create(&d, &h) == MHD_OK);
    const std::vector<double> a(10 * 10 * 8, 1.0);
    const double *m = a.data();
    HH_CHECK(mhd_set_metrics(h, m, m, m, m, m, m, m, m, m, m, m) == MHD_OK);
    HH_CHECK(mhd_set_background(h, m, m) == MHD_OK);
    HH_CHECK(mhd_upload(h, m, m, m, m, m, m, m, m) == MHD_OK);
    HH_CHECK(mhd_set_closure(h, net, m, m, m, m, 0.0, 1.0) == MHD_OK && mhd_closure_active(h));

    const long long small = 8 * 8 * 6, large = 16 * 16 * 16;
    const std::vector<float> x((size_t)large * 8, 1.0f), t((size_t)large * 7, 1.0f);
    std::vector<float> y((size_t)large * 7);
    need = small;
    HH_CHECK(mhd_net_add_sample(net, 8, 8, 6, x.data(), t.data()) == MHD_OK);
    HH_CHECK(mhd_step(h, nullptr, nullptr) == MHD_OK && launches == 3);
    for (int ok = 0; ok < 11; ++ok) {  // the allocations of the workspace that succeed
        const size_t before = hh::ranges.size();
        need = large;
        hh::malloc_until = ok;
        HH_CHECK(mhd_net_forward(net, 16, 16, 16, x.data(), y.data()) == MHD_ERR_HIP);
        need = small;
        hh::malloc_until = 0;  // and nothing after: errors, no launch
        launches = 0;
        HH_CHECK(mhd_step(h, nullptr, nullptr) == MHD_ERR_HIP && launches == 0);
        HH_CHECK(mhd_net_forward(net, 8, 8, 6, x.data(), y.data()) == MHD_ERR_HIP && launches == 0);
        double loss;
        HH_CHECK(mhd_net_loss(net, 0, &loss) == MHD_ERR_HIP && launches == 0);
        hh::malloc_until = -1;  // memory again: they run
        if (ok % 3 == 0) HH_CHECK(mhd_step(h, nullptr, nullptr) == MHD_OK && launches == 3);
        if (ok % 3 == 1) HH_CHECK(mhd_net_train(net, 1, 1e-3f, &loss, nullptr) == MHD_OK && launches == 5);
        if (ok % 3 == 2) HH_CHECK(mhd_net_forward(net, 8, 8, 6, x.data(), y.data()) == MHD_OK && launches == 3);
        HH_CHECK(hh::ranges.size() == before && bad == 0);
    }
    mhd_destroy(h);
    mhd_net_destroy(net);
    HH_CHECK(hh::ranges.empty() && bad == 0);
    return 0;
}
