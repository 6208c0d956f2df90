"""D2Q9 LDS tiles on both sides of the number of work-groups at which a launch takes the form that
lets groups share a CU: 256 for regions of 576 cells (16×16 with four steps, 8×8 with eight), 1024
for the 8×8 tile with four; and the tiles that always take it.

Both forms run the single step's per-cell arithmetic in the same order and round every
intermediate value to the storage, so the populations must equal single steps bit for bit: the
tolerance is zero.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALL, PERIODIC = {"kind": "wall"}, {"kind": "periodic"}
FACES = {
    "periodic": dict(west=PERIODIC, east=PERIODIC, south=PERIODIC, north=PERIODIC),
    "cavity": dict(west=WALL, east=WALL, south=WALL, north={"kind": "zouhe_velocity", "u": (0.08, 0.0, 0.0)}),
    "channel": dict(west={"kind": "zouhe_velocity", "u": (0.03, 0.0, 0.0)}, east={"kind": "zouhe_pressure", "rho": 1.0},
                    south=WALL, north={"kind": "moving_wall", "u": (0.05, 0.0, 0.0)}),
}
# 256 groups and one row or column of groups more, the last tiles cut; many groups
SIZES = {7: [(256, 256), (257, 250), (250, 257), (519, 301)], 8: [(128, 128), (129, 121), (121, 130), (333, 207)],
         6: [(256, 256), (257, 250), (250, 257), (401, 333)], 1: [(64, 61), (133, 57)], 5: [(64, 64), (128, 127)],
         3: [(64, 64), (129, 40)]}


def _fields(shape, seed):
    r = np.random.default_rng(seed)
    return 1 + 0.02 * r.uniform(-1, 1, shape), 0.02 * r.uniform(-1, 1, shape), 0.02 * r.uniform(-1, 1, shape)


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s", "f16s"])
@pytest.mark.parametrize("tile", sorted(SIZES))
def test_tiles_equal_single_steps(kmi, backend, tile, storage):
    for k, shape in enumerate(SIZES[tile]):
        for m, (faces, collision) in enumerate([("periodic", "bgk"), ("cavity", "mrt"), ("channel", "trt")]):
            print(f"[tile {tile}] {storage} {faces} {collision} {shape}", flush=True)
            d = kmi.make_desc("d2q9", *shape, 1, 0.05, storage=storage, collision=collision, faces=FACES[faces])
            got = []
            for t in (0, tile):
                with kmi.Lattice(d, backend) as lat:
                    lat.set_temporal(t)
                    lat.init_equilibrium(*_fields(shape, 3 * k + m))
                    lat.step(21)
                    got.append(lat.download_raw())
            assert np.array_equal(got[0], got[1]), (faces, collision, shape)


@pytest.mark.parametrize("storage", ["f32", "f32s", "f16s"])
@pytest.mark.parametrize("tile", sorted(SIZES))
def test_thermal_tiles_equal_single_steps(kmi, backend, tile, storage):
    for shape in SIZES[tile]:
        print(f"[tile {tile}] Rayleigh-Benard {storage} {shape}", flush=True)
        d, _ = kmi.rayleigh_benard_desc(*shape, 1e5, 0.71, storage=storage)
        got = []
        for t in (0, tile):
            with kmi.Lattice(d, backend) as lat:
                lat.set_temporal(t)
                lat.init_equilibrium(*_fields(shape, 7))
                lat.init_temperature(kmi.rb_initial_temperature(*shape, 1.0, 0.0))
                lat.step(21)
                got.append((lat.download_raw(), lat.download_raw("g")))
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1]), shape
