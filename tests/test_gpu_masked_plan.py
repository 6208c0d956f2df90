"""D3Q19 lattices with a solid mask and no launch set, with and without a constant body force.

The multi-step launches the lattice would choose by itself are the ones without a mask: with one
(and no cut links) it takes single steps.  Both sides run the same per-cell arithmetic in the same
order, so the populations must be equal bit for bit: the tolerance is zero.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALL, PERIODIC = {"kind": "wall"}, {"kind": "periodic"}
FACES = {
    "periodic": {f: PERIODIC for f in ("west", "east", "south", "north", "bottom", "top")},
    "duct": dict(west=PERIODIC, east=PERIODIC, south=WALL, north=WALL, bottom=WALL, top=WALL),
    "ladd": dict({f: WALL for f in ("west", "east", "south", "north", "bottom")},
                 top={"kind": "moving_wall", "u": (0.05, 0.02, 0.0), "rho": 1.0}),
}
FORCE = dict(forcing="guo", force=(2e-4, -1e-4, 3e-5))


def _block(shape):
    m = np.zeros(shape, dtype=np.uint8)
    m[tuple(slice(n // 3, n // 3 + n // 4) for n in shape)] = 1
    return m


def _fields(shape, seed):
    r = np.random.default_rng(seed)
    return [1 + 0.02 * r.uniform(-1, 1, shape)] + [0.02 * r.uniform(-1, 1, shape) for _ in range(3)]


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s"])
@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("force", [False, True])
def test_masked_lattice_steps_and_equals_single_steps(kmi, backend, storage, faces, force):
    for shape, solid in (((128, 128, 128), "bounce_back"), ((128, 97, 130), "inert"), ((300, 128, 150), "bounce_back")):
        if shape[0] == 300 and not (force and faces == "duct"):
            continue
        print(f"[masked] {faces} {storage} {shape} {solid} force {force}", flush=True)
        d = kmi.make_desc("d3q19", *shape, 0.02, storage=storage, collision="bgk", faces=FACES[faces],
                          solid_mode=solid, **(FORCE if force else {}))
        fields = _fields(shape, shape[1])
        got = []
        for single in (False, True):
            with kmi.Lattice(d, backend) as lat:
                if single:
                    lat.set_temporal(0)
                lat.init_equilibrium(*fields)
                lat.step(5)  # several steps per launch where the lattice chooses so
                lat.set_mask(_block(shape))
                for n in (7, 33, 2, 1):
                    lat.step(n)
                lat.set_mask(None)
                lat.step(6)
                got.append(lat.download_raw())
        assert np.array_equal(got[0], got[1]), (faces, storage, shape)


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("force", [False, True])
def test_masked_lattice_tunes(kmi, backend, storage, force):
    """Tuning finds a launch where no tile divides the extents, and results stay as they are."""
    shape = (130, 129, 131)
    d = kmi.make_desc("d3q19", *shape, 0.02, storage=storage, collision="bgk", faces=FACES["duct"],
                      **(FORCE if force else {}))
    got = []
    for tune in (False, True):
        with kmi.Lattice(d, backend) as lat:
            lat.set_mask(_block(shape))
            if tune:
                assert lat.autotune(8) > 0
            else:
                lat.set_temporal(0)
            lat.init_equilibrium(*_fields(shape, 4))
            lat.step(35)
            got.append(lat.download_raw())
    assert np.array_equal(got[0], got[1])


def test_masked_lattice_is_not_slower_than_single_steps(kmi, backend):
    """With a mask the multi-step kernel takes its full walled form for every tile, 2.5 times as
    long as single steps on this lattice; both sides here run the same kernel, so half as much
    again covers any noise."""
    shape = (128, 128, 128)
    d = kmi.make_desc("d3q19", *shape, 0.02, storage="f64", collision="trt", faces=FACES["ladd"])
    ms = []
    for single in (False, True):
        with kmi.Lattice(d, backend) as lat:
            if single:
                lat.set_temporal(0)
            lat.set_mask(_block(shape))
            lat.step(60)
            ms.append(min(lat.step_timed(60) for _ in range(5)))
    assert ms[0] <= 1.5 * ms[1], ms
