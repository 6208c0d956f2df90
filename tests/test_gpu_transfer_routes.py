"""Host transfers on both sides of the sizes at which they go over from the context's ring to the
runtime's own copy and back, single arrays and several, whole and with a last piece of a few bytes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# cells of D2Q9 FP64 lattices (72 bytes a cell): around 128 KB, 1 MB, two and four pieces, and 48 MB
CELLS = [1820, 1821, 14563, 14564, 14565, 58254, 58255, 29127, 29128, 699050, 699051, 700001]


@pytest.mark.parametrize("cells", CELLS)
def test_arrays_round_trip(kmi, backend, cells):
    r = np.random.default_rng(cells)
    for storage, collision in (("f64", "mrt"), ("f32s", "mrt"), ("f16s", "bgk")):
        print(f"[transfer routes] {cells} cells {storage}", flush=True)
        with kmi.Lattice(kmi.make_desc("d2q9", cells, 1, 1, 0.05, storage=storage, collision=collision), backend) as lat:
            dt = lat.storage_dtype()
            for k in range(3):
                a = r.integers(0, 2 ** 15 - 2 ** 10, size=(cells, 1, 9)).astype(dt)
                lat.upload_raw(np.asfortranarray(a))
                assert np.array_equal(lat.download_raw(), a)
            if storage == "f64":
                lat.upload(a)
                assert np.array_equal(lat.download(), a)


@pytest.mark.parametrize("cells", [5461, 5462, 43690, 43691, 2097152, 2097153])
def test_several_arrays(kmi, backend, cells):
    """Three fields up and three down (24 bytes a cell: 128 KB, 1 MB, 48 MB), then two of them."""
    r = np.random.default_rng(cells)
    f = [1 + 0.01 * r.uniform(-1, 1, (cells, 1)), 0.02 * r.uniform(-1, 1, (cells, 1)), 0.02 * r.uniform(-1, 1, (cells, 1))]
    with kmi.Lattice(kmi.make_desc("d2q9", cells, 1, 1, 0.05), backend) as lat:
        for rho in (f[0], None):
            lat.init_equilibrium(rho, f[1], f[2])
            m = lat.moments()
            # moments of an equilibrium: rounding of 9 terms in FP64
            assert np.max(np.abs(m["rho"] - (1.0 if rho is None else rho))) < 1e-15 * 8
            assert np.max(np.abs(m["ux"] - f[1])) < 1e-15 and np.max(np.abs(m["uy"] - f[2])) < 1e-15


def test_a_copy_waits_for_the_steps_before_it(kmi, backend):
    """One piece and many: what comes back is the state after the steps, and an upload's array may be
    overwritten as soon as the call returns."""
    for n in (40, 300, 1100):
        d = kmi.make_desc("d2q9", n, n, 1, 0.05, storage="f64")
        r = np.random.default_rng(n)
        a = np.asfortranarray(r.uniform(0.01, 0.1, (n, n, 9)))
        want = None
        for _ in range(3):
            with kmi.Lattice(d, backend) as lat:
                b = a.copy(order="F")
                lat.upload(b)
                b[:] = 0.0
                lat.step(7)
                got = lat.download()
            want = got if want is None else want
            assert np.array_equal(got, want) and np.all(np.isfinite(got)) and np.max(got) > 0.01
