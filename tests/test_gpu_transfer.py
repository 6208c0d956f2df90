"""Host transfers through the context's pinned ring: contents at the sizes where the path
changes (one piece, the calling thread alone, fewer and more pieces than ring slots, a last
piece of one element), several arrays in one call, and two threads at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# D2Q9 F64 lattices: 72 bytes a cell — 72 B, just below and above 512 KiB, a few MB, one piece
# more than the 24 MB ring, and 130 MB
CELLS = [(1, 1), (7281, 1), (7282, 1), (701, 67), (1999, 175), (2000, 181), (1357, 1329)]


@pytest.mark.parametrize("shape", CELLS)
@pytest.mark.parametrize("storage", ["f64", "f16s"])
def test_round_trip(kmi, backend, shape, storage):
    r = np.random.default_rng(shape[0])
    print(f"[transfer] {storage} {shape}", flush=True)
    with kmi.Lattice(kmi.make_desc("d2q9", *shape, 1, 0.05, storage=storage), backend) as lat:
        dt = lat.storage_dtype()
        if storage == "f64":
            a = np.asfortranarray(r.standard_normal(shape + (9,)))
        else:
            a = np.asfortranarray(r.integers(0, 2 ** 15 - 2 ** 10, size=shape + (9,)).astype(dt))
        for _ in range(3):  # the ring is reused, uploads and downloads in turn
            lat.upload_raw(a)
            b = lat.download_raw()
            assert np.array_equal(a, b)
            a = np.asfortranarray(b[::-1].copy() if storage == "f64" else b)
        if storage == "f64":
            lat.upload(a)
            assert np.array_equal(lat.download(), a)


def test_moment_planes_and_threads(kmi, backend):
    """Each plane lands in its own array, also when two threads read two lattices at once."""
    shape = (96, 80, 64)
    r = np.random.default_rng(3)
    fields = [1 + 0.01 * r.uniform(-1, 1, shape)] + [0.02 * r.uniform(-1, 1, shape) for _ in range(3)]
    with kmi.Lattice(kmi.make_desc("d3q19", *shape, 0.05), backend) as one, \
            kmi.Lattice(kmi.make_desc("d3q19", *shape, 0.05), backend) as two:
        one.init_equilibrium(*fields)
        two.init_equilibrium(fields[0], fields[3], fields[2], fields[1])
        alone = [one.moments(), two.moments()]
        for m, order in zip(alone, ((1, 2, 3), (3, 2, 1))):
            # moments of an equilibrium: rounding of 19 terms in FP64
            for name, k in zip(("ux", "uy", "uz"), order):
                assert np.max(np.abs(m[name] - fields[k])) < 1e-15
        got = {}

        def read(key, lat):
            got[key] = [lat.moments() for _ in range(10)]

        threads = [threading.Thread(target=read, args=(k, lat)) for k, lat in enumerate((one, two))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for k in range(2):
            for m in got[k]:
                assert all(np.array_equal(m[n], alone[k][n]) for n in m)


def test_reductions_repeat(kmi, backend):
    """The last group to finish folds the partial sums in a fixed order: the same bits every
    time, for one group, a few and the most there are."""
    for shape in ((5, 3), (200, 130), (1100, 900)):
        r = np.random.default_rng(shape[0])
        with kmi.Lattice(kmi.make_desc("d2q9", *shape, 1, 0.05), backend) as lat:
            rho = 1 + 0.1 * r.uniform(-1, 1, shape)
            lat.init_equilibrium(rho, 0.02 * r.uniform(-1, 1, shape), 0.0)
            first = [lat.reduce(k) for k in ("mass", "momentum", "kinetic_energy", "max_speed")]
            for _ in range(5):
                assert first == [lat.reduce(k) for k in ("mass", "momentum", "kinetic_energy", "max_speed")]
            m = lat.moments()
            import math
            # compensated sum of FP64 values: a few ulps of the exact one
            assert abs(first[0] - math.fsum(m["rho"].ravel())) <= 4e-16 * first[0]
            assert first[3] == pytest.approx(float(np.max(np.hypot(m["ux"], m["uy"]))), rel=1e-15)


@pytest.mark.parametrize("cells", [256, 257, 513, 2304, 3841, 4096, 4097])
def test_reductions_of_few_groups(kmi, backend, cells):
    """One group, two to sixteen (summed by the last of them) and seventeen."""
    import math

    r = np.random.default_rng(cells)
    shape = (cells, 1) if cells % 2 else (cells // 2, 2)
    with kmi.Lattice(kmi.make_desc("d2q9", *shape, 1, 0.05), backend) as lat:
        lat.init_equilibrium(1 + 0.1 * r.uniform(-1, 1, shape), 0.02 * r.uniform(-1, 1, shape),
                             0.02 * r.uniform(-1, 1, shape))
        mass, mom, speed = lat.reduce("mass"), lat.reduce("momentum"), lat.reduce("max_speed")
        m = lat.moments()
        # compensated sums of FP64 values: a few ulps of the exact ones (of Σ|x| for the momentum)
        assert abs(mass - math.fsum(m["rho"].ravel())) <= 4e-16 * mass
        for k, u in enumerate(("ux", "uy")):
            x = (m["rho"] * m[u]).ravel()
            assert abs(mom[k] - math.fsum(x)) <= 4e-16 * np.abs(x).sum() + 1e-300
        assert speed == pytest.approx(float(np.max(np.hypot(m["ux"], m["uy"]))), rel=1e-15)
