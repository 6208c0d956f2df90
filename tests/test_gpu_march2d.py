"""The register march of D2Q9 lattices (kmi_march2d.h) against single-step launches.

Both run the same per-cell arithmetic in the same order and round every intermediate value to
the storage, so the populations must be equal bit for bit: the tolerance is zero.  Sizes sit at
the edges of the strips (64 − 2 (K − 1) columns, wider by K − 1 at a wall) and of the rows of a
piece; step counts leave remainders of one to three steps.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALL, PERIODIC = {"kind": "wall"}, {"kind": "periodic"}
FACES = {
    "periodic": dict(west=PERIODIC, east=PERIODIC, south=PERIODIC, north=PERIODIC),
    "cavity": dict(west=WALL, east=WALL, south=WALL, north={"kind": "zouhe_velocity", "u": (0.08, 0.0, 0.0)}),
    "moving": dict(west=WALL, east={"kind": "moving_wall", "u": (0.0, 0.03, 0.0)},
                   south={"kind": "moving_wall", "u": (-0.02, 0.0, 0.0)},
                   north={"kind": "moving_wall", "u": (0.05, 0.0, 0.0)}),
    "couette": dict(west=PERIODIC, east=PERIODIC, south={"kind": "zouhe_velocity", "u": (0.03, 0.0, 0.0)}, north=WALL),
    "shaft": dict(west=WALL, east={"kind": "moving_wall", "u": (0.0, 0.03, 0.0)}, south=PERIODIC, north=PERIODIC),
    "channel": dict(west={"kind": "zouhe_velocity", "u": (0.03, 0.0, 0.0)}, east={"kind": "zouhe_pressure", "rho": 1.0},
                    south=WALL, north=WALL),
    "pressure": dict(west={"kind": "zouhe_pressure", "rho": 1.01}, east={"kind": "zouhe_pressure", "rho": 1.0},
                     south=WALL, north=WALL),
}
# the march needs 160,000 cells: one strip, strips just full and just over, more rows than
# one wave per SIMD, fewer
SIZES = [(64, 2500), (58, 2760), (116, 1380), (117, 1400), (122, 1312), (1300, 130), (4001, 41), (401, 403)]


def _fields(shape, seed):
    r = np.random.default_rng(seed)
    return 1 + 0.02 * r.uniform(-1, 1, shape), 0.02 * r.uniform(-1, 1, shape), 0.02 * r.uniform(-1, 1, shape)


@pytest.mark.parametrize("faces", list(FACES))
@pytest.mark.parametrize("storage", ["f64", "f32", "f32s", "f16s"])
def test_march_equals_single_steps(kmi, backend, storage, faces):
    for k, (nx, ny) in enumerate(SIZES):
        collision = ("bgk", "trt", "mrt")[(k + len(storage) + len(faces)) % 3]
        steps = 9 + k % 4
        print(f"[march] {storage} {collision} {faces} {nx}x{ny}, {steps} steps", flush=True)
        d = kmi.make_desc("d2q9", nx, ny, 1, 0.05, storage=storage, collision=collision, faces=FACES[faces])
        out = []
        for tile in (0, 2):
            with kmi.Lattice(d, backend) as lat:
                lat.init_equilibrium(*_fields((nx, ny), k))
                lat.set_temporal(tile, 1)
                lat.step(steps)
                assert lat.steps == steps
                out.append(lat.download_raw())
        assert np.array_equal(out[0], out[1]), (storage, collision, faces, nx, ny)


def test_march_follows_mask_and_size(kmi, backend):
    """A mask, a force or a smaller lattice takes tile 2 back to the LDS tile kernel; setting
    and clearing the mask between runs changes nothing but the mask's own effect."""
    nx, ny = 500, 400
    mask = np.zeros((nx, ny), dtype=np.uint8)
    mask[200:230, 100:160] = 1
    d = kmi.make_desc("d2q9", nx, ny, 1, 0.05, storage="f32s", faces=FACES["cavity"])
    out = []
    for tile in (0, 2):
        with kmi.Lattice(d, backend) as lat:
            lat.init_equilibrium(*_fields((nx, ny), 5))
            lat.set_temporal(tile, 1)
            lat.step(41)
            lat.set_mask(mask)
            lat.step(41)
            lat.set_mask(None)
            lat.step(41)
            out.append(lat.download_raw())
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("storage", ["f64", "f32s", "f16s"])
@pytest.mark.parametrize("collision,lid", [("mrt", "zouhe"), ("bgk", "ladd"), ("trt", "zouhe")])
def test_batch_march_equals_single_steps(kmi, backend, storage, collision, lid):
    """Cavities from two cells a side to several strips, three and four steps per launch."""
    sizes = [2, 3, 5, 30, 58, 61, 64, 65, 70, 117, 122, 123, 128, 200, 319]
    nus = [0.1 * n / 100 + 0.02 for n in sizes]
    print(f"[batch march] {storage} {collision} {lid}", flush=True)
    ref = None
    for span in (1, 3, 4):
        with kmi.Batch(sizes, nus, storage=storage, collision=collision, lid=lid, backend=backend) as b:
            b.set_temporal(span)
            for c, n in enumerate(sizes):
                b.init_equilibrium(c, *_fields((n, n), c))
            b.step(39)
            got = [b.download(c) for c in range(len(sizes))]
        ref = ref or got
        for c in range(len(sizes)):
            assert np.array_equal(got[c], ref[c], equal_nan=True), (span, sizes[c])
