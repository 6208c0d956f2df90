"""Tile 2 of large D2Q9 lattices on both sides of the rule that sends it to the register march.

The march, the LDS tile and single steps run the same per-cell arithmetic in the same order and
round every intermediate value to the storage, so the populations must be equal bit for bit: the
tolerance is zero.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALL, PERIODIC = {"kind": "wall"}, {"kind": "periodic"}
FACES = {
    "periodic": dict(west=PERIODIC, east=PERIODIC, south=PERIODIC, north=PERIODIC),
    "box": dict(west=WALL, east=WALL, south=WALL, north=WALL),
    "cavity": dict(west=WALL, east=WALL, south=WALL, north={"kind": "zouhe_velocity", "u": (0.08, 0.0, 0.0)}),
    "shaft": dict(west=WALL, east={"kind": "moving_wall", "u": (0.0, 0.03, 0.0)}, south=PERIODIC, north=PERIODIC),
    "couette": dict(west=PERIODIC, east=PERIODIC, south={"kind": "zouhe_velocity", "u": (0.03, 0.0, 0.0)}, north=WALL),
    "channel": dict(west={"kind": "zouhe_velocity", "u": (0.03, 0.0, 0.0)}, east={"kind": "zouhe_pressure", "rho": 1.0},
                    south=WALL, north=WALL),
}
# the march in every storage: strips just full and just over, half empty, few rows; x faces with a
# closure or a Ladd term need more cells
MARCH = [(f, n) for f in ("periodic", "cavity", "couette") for n in
         ((58, 7500), (64, 7600), (65, 10800), (116, 4600), (117, 4600), (1300, 420), (4001, 130), (731, 733))] + \
        [(f, n) for f in ("shaft", "channel") for n in ((122, 9200), (1300, 1000), (1137, 1139), (6003, 220))]
# both sides of the lines: 512, 840, 1800 and 2200 tiles of 24×24, and the shapes that decide below
EDGE = [("cavity", (384, 768)), ("cavity", (385, 768)), ("periodic", (384, 768)), ("periodic", (385, 768)),
        ("cavity", (720, 672)), ("cavity", (720, 673)), ("channel", (720, 672)), ("channel", (721, 672)),
        ("shaft", (1080, 960)), ("shaft", (1081, 960)), ("channel", (1200, 1056)), ("channel", (1201, 1056)),
        ("couette", (400, 400)), ("periodic", (70, 3000)), ("couette", (5000, 33)), ("cavity", (56, 2900)),
        ("cavity", (48, 8400)), ("box", (118, 1400)), ("box", (5000, 33)), ("box", (401, 403))]


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s", "f16s"])
@pytest.mark.parametrize("sizes", ["march", "edge"])
def test_tile_2_equals_single_steps(kmi, backend, storage, sizes):
    for k, (faces, shape) in enumerate(MARCH if sizes == "march" else EDGE):
        collision = ("bgk", "trt", "mrt")[(k + len(storage)) % 3]
        print(f"[march routes] {storage} {collision} {faces} {shape}", flush=True)
        d = kmi.make_desc("d2q9", *shape, 1, 0.05, storage=storage, collision=collision, faces=FACES[faces])
        r = np.random.default_rng(k)
        fields = (1 + 0.02 * r.uniform(-1, 1, shape), 0.02 * r.uniform(-1, 1, shape), 0.02 * r.uniform(-1, 1, shape))
        got = []
        for tile in (0, 2):
            with kmi.Lattice(d, backend) as lat:
                lat.set_temporal(tile)
                lat.init_equilibrium(*fields)
                lat.step(9 + k % 4)
                got.append(lat.download_raw())
        assert np.array_equal(got[0], got[1]), (faces, collision, shape)
