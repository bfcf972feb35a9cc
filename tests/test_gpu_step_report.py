"""What a step call reports (DT, UMACH, written to the host by the step's
close) against the same scalars copied from the device (a call of zero steps),
and mhd_step_noalloc's one-launch upload with the CFL reduction against a
handle's at planes around its 512-point blocks: bit for bit."""

import pytest

import helpers as H
from test_gpu_stage_split import _box
from test_zz_no_alloc import handle_steps, noalloc_step, same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmag", [True, False], ids=["mhd", "hydro"])
@pytest.mark.parametrize("size", [(9, 6, 4), (16, 32, 6), (27, 19, 5), (33, 31, 5), (257, 4, 7)],
                         ids=lambda s: "x".join(map(str, s)))
def test_noalloc_upload_matches_the_handle(size, lmag):
    meta, st = _box(*size, lmag)
    got, dt, um, clk = noalloc_step(meta, st, (2, 0.5, 1.0))
    ref, dtr, umr, clkr = handle_steps(meta, st, (2, 0.5, 1.0))
    assert (dt, um, clk) == (dtr, umr, clkr)
    same(got, ref, lmag)


@pytest.mark.parametrize("precision,every", [("fp64", 0), ("mixed", 0), ("mixed", 2)])
def test_reported_scalars_are_the_devices(precision, every):
    meta, st = _box(20, 12, 10, True)
    with H.pkg().Box(meta, precision=precision) as box:
        box.upload(st)
        if every:
            box.set_rebase_interval(every)
        for call in (box.step, lambda: box.steps(3), lambda: box.steps(2), box.step):
            assert call() == box.steps(0)
        assert box.clock()[0] == 7
