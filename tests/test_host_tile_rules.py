"""The rules that choose a box's stage tile and z chunks, on the CPU: the tile of
the boxes that the GPU tests step with fitted tiles, and the bounds that the
kernels rely on over many boxes."""

import random

import hostbuild

# (npx, npy, npz, magnetic, precision, density diffusion), its tile
FITTED = [
    ((96, 96, 48, True, "fp64", True), (48, 5)),     # half rows
    ((40, 72, 54, True, "fp64", True), (40, 6)),     # whole rows, threads left over
    ((33, 47, 40, False, "fp64", True), (33, 7)),    # the same, a short last tile
    ((130, 90, 41, False, "fp64", False), (44, 5)),  # a third of the rows, its last column tile short
    ((20, 33, 40, False, "fp64", False), (20, 11)),  # three tiles high
    ((72, 200, 64, True, "fp64", False), (72, 3)),   # wider than a wavefront
    ((83, 128, 36, True, "fp64", False), (83, 2)),
    ((72, 200, 64, True, "mixed", False), (72, 3)),
    ((40, 72, 54, True, "mixed", False), (40, 6)),
    ((36, 77, 64, True, "mixed", False), (36, 7)),
    ((20, 33, 40, False, "mixed", False), (20, 11)),
    ((83, 128, 36, False, "mixed", False), (83, 2)),
    ((160, 160, 64, True, "mixed", False), (0, 0)),  # 64x4
]


def _tiles(boxes):
    line = "{} {} {} {:d} {:d} {:d}".format
    out = hostbuild.run("tile_rules", stdin="\n".join(line(*b[:4], b[4] == "mixed", b[5]) for b in boxes))
    return [tuple(int(v) for v in row.split()) for row in out.splitlines()]


def test_tiles_of_the_stepped_boxes():
    assert [t[:2] for t in _tiles([b for b, _ in FITTED])] == [t for _, t in FITTED]


def test_tiles_and_chunks_hold_their_bounds():
    rng = random.Random(1)
    size = lambda lo, hi: int(lo * (hi / lo) ** rng.random())  # noqa: E731
    boxes = [(size(3, 700), size(3, 700), size(4, 500), rng.random() < 0.5, rng.choice(["fp64", "mixed"]), False)
             for _ in range(3000)]
    assert len(_tiles(boxes)) == len(boxes)  # (the program checks each)
