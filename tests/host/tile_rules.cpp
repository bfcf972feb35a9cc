// The tile and the z chunks that the rules of mhd_host.h give boxes, as
// "width height chunks" per line of "npx npy npz lmag mixed id" on the standard
// input (0 0: tiles of 64x4).  Every box's chunks are checked: planes
// 1..npz without gap or overlap, three at least in the first and the last, no
// chunk deeper than said; its tile: at most 256 points and threads for the halo,
// the LDS plane within its bound.
#include "hip_host.h"

#include "../../rast-3dmhd_amd/csrc/mhd_host.h"

using namespace rmhd;

static int check_chunks(int npz, int nc) {
    HH_CHECK(nc >= 1 && nc <= max_chunks(npz));
    HH_CHECK(chunk_begin(npz, nc, 0) == 1 && chunk_begin(npz, nc, nc) == npz + 1);
    for (int c = 0; c < nc; ++c) {
        const int n = chunk_begin(npz, nc, c + 1) - chunk_begin(npz, nc, c);
        HH_CHECK(n >= 1 && n <= (nc == 1 ? npz : chunk_depth(npz, nc)));
        if (c == 0 || c == nc - 1) HH_CHECK(n >= 3);
    }
    return 0;
}

int main() {
    for (int npz = 4; npz < 300; ++npz)
        for (int nc = 1; nc <= max_chunks(npz); ++nc)
            if (check_chunks(npz, nc)) return 1;
    mhd_desc d{};
    d.gamma = 1.0;
    int lmag, mixed, id;
    while (scanf("%d %d %d %d %d %d", &d.npx, &d.npy, &d.npz, &lmag, &mixed, &id) == 6) {
        d.lmag = lmag;
        d.precision = mixed ? MHD_MIXED : MHD_FP64;
        d.id = id;
        const Params p = params_from_desc(&d);
        const int w = p.tile_w ? p.tile_w : 64, h = p.tile_w ? p.tile_h : p.tile_y;
        HH_CHECK(w >= 1 && h >= 1 && w * h <= 256 && 2 * (w + 2 + h) <= 256);
        HH_CHECK((w + 2) * (h + 2) <= (mixed ? FIT_POINTS_MIXED : FIT_POINTS_FP64));
        if (p.tile_w) HH_CHECK(w <= d.npx && h <= d.npy);
        if (check_chunks(p.npz, p.nchunks)) return 1;
        printf("%d %d %d\n", p.tile_w, p.tile_h, p.nchunks);
    }
    return 0;
}
