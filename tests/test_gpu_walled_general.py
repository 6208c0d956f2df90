"""Two D3Q19 steps per launch under walls of every kind: moving walls and Zou–He faces across x and y,
solid masks with bounce-back, one tile along an axis, odd numbers of planes.

Each step evaluates the same per-cell arithmetic in the same order as a single-step launch, so the
populations must be equal bit for bit: the tolerance is zero.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALLS = {f: {"kind": "wall"} for f in ("west", "east", "south", "north", "bottom", "top")}


def _moving(*u):
    return {"kind": "moving_wall", "u": u, "rho": 1.02}


FACES = {
    "one moving x wall": dict(WALLS, west=_moving(0.0, 0.03, -0.02)),
    "all moving": dict(west=_moving(0.0, 0.03, 0.01), east=_moving(0.0, -0.02, 0.02), south=_moving(0.03, 0.0, 0.01),
                       north=_moving(-0.01, 0.0, 0.02), bottom=_moving(0.02, 0.01, 0.0), top=_moving(0.01, -0.03, 0.0)),
    "Zou–He x": dict(WALLS, west={"kind": "zouhe_velocity", "u": (0.03, 0.0, 0.0)},
                     east={"kind": "zouhe_pressure", "rho": 1.0}),
    "walls": WALLS,
}


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s"])
@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("mask", [False, True])
@pytest.mark.parametrize("tile", [12, 14])
def test_two_steps_under_general_walls(kmi, backend, storage, faces, mask, tile):
    for shape, coll in (((64, 32, 24), "trt"), ((64, 8, 7), "bgk"), ((128, 16, 31), "trt")):
        print(f"[general walls] {faces} {storage} tile {tile} {shape} mask {mask}", flush=True)
        r = np.random.default_rng(shape[1])
        fields = [1 + 0.02 * r.uniform(-1, 1, shape)] + [0.02 * r.uniform(-1, 1, shape) for _ in range(3)]
        solid = (r.uniform(size=shape) < 0.1).astype(np.uint8)
        d = kmi.make_desc("d3q19", *shape, 0.02, storage=storage, collision=coll, faces=FACES[faces])
        got = []
        for span in ((0, 1), (tile, 1), (tile, 3)):
            with kmi.Lattice(d, backend) as lat:
                lat.set_temporal(*span)
                lat.init_equilibrium(*fields)
                if mask:
                    lat.set_mask(solid)
                lat.step(9)
                got.append(lat.download_raw())
        assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2]), (shape, coll)
