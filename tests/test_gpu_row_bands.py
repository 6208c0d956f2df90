"""Single-step launches on both sides of the rule that gives each XCD a band of rows: rows added to
fill the bands or not, short and long rows, lattices that stay in the L2s or not, against launches
whose waves span rows.  The same per-cell arithmetic, so the same bits.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALL = {"kind": "wall"}
MOVING = {"kind": "moving_wall", "u": (0.02, 0.0, 0.0)}
BOX = {f: WALL for f in ("west", "east", "south", "bottom", "top")}
SHAPES = [
    (100, 23, 5), (65, 47, 4), (33, 60, 5),  # a few rows added
    (65, 40, 4),                             # none added
    (65, 9, 6), (300, 17, 4),                # too many to add: no bands
    (700, 17, 1), (60, 3, 1),                # D2Q9 in the L2s: bands whatever they add
    (1200, 403, 1), (1100, 409, 1),          # beyond them, rows of up to 10 KB and longer (F64)
    (2600, 203, 1),                          # (FP32)
]


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s", "f16s"])
def test_bands_equal_patch_launches(kmi, backend, storage):
    for k, shape in enumerate(SHAPES):
        print(f"[bands] {storage} {shape}", flush=True)
        stencil = "d2q9" if shape[2] == 1 else "d3q19"
        faces = dict(BOX, north=MOVING)
        if stencil == "d2q9":
            faces = {f: faces[f] for f in ("west", "east", "south", "north")}
        d = kmi.make_desc(stencil, *shape, 0.05, storage=storage, collision="trt", faces=faces)
        field = shape if stencil == "d3q19" else shape[:2]
        r = np.random.default_rng(k)
        u = 0.02 * r.uniform(-1, 1, (4,) + field)
        out = []
        for bx, by in ((16, 4), (64, 1), (64, 3), (256, 1)):
            with kmi.Lattice(d, backend) as lat:
                lat.set_launch(bx, by)
                lat.set_temporal(0)
                lat.init_equilibrium(*((1 + u[0], u[1], u[2], u[3])[:len(field) + 1]))
                lat.step(5)
                out.append(lat.download_raw())
        for o in out[1:]:
            assert np.array_equal(out[0], o), (storage, shape)
