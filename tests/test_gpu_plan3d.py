"""The launch a D3Q19 lattice takes when none is set: several steps per launch where that is the
faster one, whatever the x–y extent, against single-step launches (set_temporal(0)).

Both run the same per-cell arithmetic in the same order and round every intermediate value to
the storage, so the populations must be equal bit for bit: the tolerance is zero.  Where no tile
divides an extent the last tile overlaps its neighbour; the extents leave remainders from one
cell to a tile less one.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALL, PERIODIC = {"kind": "wall"}, {"kind": "periodic"}
LID = {"kind": "moving_wall", "u": (0.05, 0.02, 0.0), "rho": 1.0}
BOX = {f: WALL for f in ("west", "east", "south", "north", "bottom")}
FACES = {
    "periodic": {},
    "cavity": dict(BOX, top={"kind": "zouhe_velocity", "u": (0.08, 0.0, 0.0)}),
    "ladd": dict(BOX, top=LID),
    "x_walls": dict(west=WALL, east=WALL, south=PERIODIC, north=PERIODIC, bottom=LID, top=WALL),
    "duct": dict(west=PERIODIC, east=PERIODIC, south=WALL, north=WALL, bottom=PERIODIC, top=PERIODIC),
    "couette": dict(west=PERIODIC, east=PERIODIC, south=PERIODIC, north=PERIODIC, bottom=WALL, top=LID),
}
SHAPES = [(128, 96, 101), (97, 105, 113), (129, 73, 131), (191, 95, 67), (66, 161, 127), (64, 200, 96),
          (96, 39, 131), (187, 99, 96), (229, 81, 96), (159, 147, 40)]


def _lattice(kmi, backend, faces, shape, storage, collision="trt"):
    return kmi.Lattice(kmi.make_desc("d3q19", *shape, 0.02, storage=storage, collision=collision,
                                     faces=FACES[faces]), backend)


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s"])
@pytest.mark.parametrize("forcing", ["guo", "guo_plain"])
def test_forced_default_launch_equals_single_steps(kmi, backend, storage, forcing):
    """A constant body force in a duct, a moving-lid box and a fully periodic lattice."""
    for k, (faces, shape) in enumerate([("duct", (96, 39, 131)), ("duct", (187, 135, 40)), ("duct", (124, 63, 96)),
                                        ("ladd", (161, 129, 129)), ("periodic", (225, 119, 67)),
                                        ("cavity", (96, 39, 131))]):
        print(f"[plan] forced {faces} {storage} {shape}", flush=True)
        d = kmi.make_desc("d3q19", *shape, 0.02, storage=storage, faces=FACES[faces], forcing=forcing,
                          force=(2e-4, -1e-4, 3e-5))
        got = []
        for single in (False, True):
            with kmi.Lattice(d, backend) as lat:
                if single:
                    lat.set_temporal(0)
                else:
                    with pytest.raises(kmi.KrakenError):
                        lat.set_temporal(14, 1)
                lat.init_equilibrium(*_fields(shape, k))
                for n in (7, 33, 1):
                    lat.step(n)
                got.append(lat.download_raw())
        assert np.array_equal(got[0], got[1]), (faces, storage, shape)


def _fields(shape, seed):
    r = np.random.default_rng(seed)
    return [1 + 0.02 * r.uniform(-1, 1, shape)] + [0.02 * r.uniform(-1, 1, shape) for _ in range(3)]


CASES = [(f, s) for f in FACES for s in ("f64", "f32", "f32s")] + [("periodic", "f16s")]


@pytest.mark.parametrize("faces,storage", CASES)
def test_default_launch_equals_single_steps(kmi, backend, faces, storage):
    for k, shape in enumerate(SHAPES):
        print(f"[plan] {faces} {storage} {shape}", flush=True)
        fields = _fields(shape, k)
        got = []
        for single in (False, True):
            with _lattice(kmi, backend, faces, shape, storage, "trt" if k % 2 else "bgk") as lat:
                if single:
                    lat.set_temporal(0)
                lat.init_equilibrium(*fields)
                for n in (7, 33, 2, 1):
                    lat.step(n)
                assert lat.temporal == {"tile": 0, "zchunks": 1} and lat.steps == 43
                got.append(lat.download_raw())
        assert np.array_equal(got[0], got[1]), (faces, storage, shape)


def test_setters_masks_and_tuning(kmi, backend):
    """An explicit launch replaces the lattice's own, refusals stay, a mask set between two runs
    takes effect, and tuning leaves the results as they are."""
    shape = (97, 105, 113)
    fields = _fields(shape, 9)
    mask = np.zeros(shape, dtype=np.uint8)
    mask[40:50, 40:52, 30:50] = 1
    got = []
    for how in ("own", "single", "shape"):
        with _lattice(kmi, backend, "ladd", shape, "f64") as lat:
            with pytest.raises(kmi.KrakenError):
                lat.set_temporal(14, 1)  # no tile divides the extents
            if how == "single":
                lat.set_temporal(0)
            if how == "shape":
                lat.set_launch(64, 2)
                assert lat.temporal == {"tile": 0, "zchunks": 1}
            lat.init_equilibrium(*fields)
            lat.step(9)
            lat.set_mask(mask)
            lat.step(9)
            got.append(lat.download())
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    got = []
    for tune in (False, True):
        with _lattice(kmi, backend, "periodic", shape, "f32") as lat:
            lat.init_equilibrium(*fields)
            if tune:
                assert lat.autotune(32) > 0
            lat.step(35)
            got.append(lat.download())
    assert np.array_equal(got[0], got[1])
