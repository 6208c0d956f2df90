"""Multi-step D3Q19 launches against lattices that provably run single steps.

A D3Q19 lattice on which no launch was set chooses its own, several steps per launch where that
is the faster one; set_temporal(0) asks for single steps.  Here every reference asks for them.
Both sides run the same per-cell arithmetic in the same order and round every intermediate value
to the storage, so the populations must be equal bit for bit: the tolerance is zero.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PERIODIC = {f: {"kind": "periodic"} for f in ("west", "east", "south", "north", "bottom", "top")}


def _run(kmi, backend, desc, launch, steps, fields=None):
    with kmi.Lattice(desc, backend) as lat:
        if fields is not None:
            lat.init_equilibrium(*fields)
        if launch == "tuned":
            lat.autotune(32)
        elif launch != "own":
            lat.set_temporal(*launch)
        for n in steps:
            lat.step(n)
        return lat.download_raw()


def test_tgv_256_fp64_single_steps_equal_the_oracle(kmi, po, backend):
    d = kmi.taylor_green_3d_desc(256, 0.01, "f64")
    f0 = po.equilibrium(*kmi.taylor_green_3d_fields(256, 0.05))
    with kmi.Lattice(d, backend) as lat:
        lat.set_temporal(0)
        lat.upload(f0)
        lat.step(2)
        fg = lat.download()
    po.run(d, f0, None, 2)
    assert np.array_equal(fg, f0)


@pytest.mark.parametrize("storage,tile", [("f32s", 11), ("f16s", 12)])
def test_tgv_256_launches_equal_single_steps(kmi, backend, storage, tile):
    d = kmi.taylor_green_3d_desc(256, 0.01, storage)
    fields = kmi.taylor_green_3d_fields(256, 0.05)
    ref = _run(kmi, backend, d, (0,), (6,), fields)
    for launch in ((tile, 2), "own"):
        assert np.array_equal(_run(kmi, backend, d, launch, (6,), fields), ref), launch


def test_walled_cube_256_launches_equal_single_steps(kmi, backend):
    d = kmi.cavity_3d_desc(256, 256, 256, 0.05, 0.05, storage="f32s")
    ref = _run(kmi, backend, d, (0,), (30,))
    for launch in ((12, 6), (14, 3), (9, 2), "own"):
        assert np.array_equal(_run(kmi, backend, d, launch, (30,)), ref), launch


def test_walled_cavity_128_tuned_equals_single_steps(kmi, backend):
    d = kmi.cavity_3d_desc(128, 128, 128, 0.05, 0.1, storage="f32s")
    ref = _run(kmi, backend, d, (0,), (30,))
    for launch in ("tuned", "own"):
        assert np.array_equal(_run(kmi, backend, d, launch, (30,)), ref), launch


# extents that leave remainders from one cell to a tile less one
SHAPES = [(128, 96, 101), (97, 105, 113), (129, 73, 131), (191, 95, 67), (66, 161, 127), (64, 200, 96),
          (96, 39, 131), (187, 99, 96), (229, 81, 96), (159, 147, 40)]


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s", "f16s"])
@pytest.mark.parametrize("forcing", [None, "guo"])
def test_periodic_lattices_of_any_extent_equal_single_steps(kmi, backend, storage, forcing):
    """Every face periodic: the halo of an overlapping last tile wraps round."""
    force = {} if forcing is None else dict(forcing=forcing, force=(2e-4, -1e-4, 3e-5))
    for k, shape in enumerate(SHAPES):
        if forcing and k % 3:
            continue
        print(f"[periodic] {storage} {forcing} {shape}", flush=True)
        r = np.random.default_rng(k)
        fields = [1 + 0.02 * r.uniform(-1, 1, shape)] + [0.02 * r.uniform(-1, 1, shape) for _ in range(3)]
        d = kmi.make_desc("d3q19", *shape, 0.02, storage=storage, collision="trt" if k % 2 and not forcing else "bgk",
                          faces=PERIODIC, **force)
        steps = (7, 33, 2, 1)
        ref = _run(kmi, backend, d, (0,), steps, fields)
        assert np.array_equal(_run(kmi, backend, d, "own", steps, fields), ref), shape
