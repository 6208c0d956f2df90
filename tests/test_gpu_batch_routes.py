"""Three and four steps per launch of a batch on both sides of the number of tiles at which it goes
over from LDS tiles to the register march, and across it as cavities retire.

All forms run the single step's per-cell arithmetic in the same order and round every
intermediate value to the storage, so the populations must equal single steps bit for bit: the
tolerance is zero.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# tile width, steps per launch, cavities of 64² (16 tiles of any width) at the last number on the LDS tiles
EDGES = {
    "f64": [(16, 3, 64), (32, 3, 48), (64, 3, 32), (16, 4, 48), (32, 4, 48), (64, 4, 32)],
    "f32": [(16, 3, 256), (32, 3, 64), (64, 3, 64), (16, 4, 80), (32, 4, 64), (64, 4, 40)],
    "f32s": [(16, 3, 256), (32, 3, 112), (64, 3, 72), (16, 4, 144), (32, 4, 112), (64, 4, 60)],
    "f16s": [(16, 3, 256), (64, 4, 60)],
}


def _u(n, seed):
    r = np.random.default_rng(seed)
    return 1 + 0.02 * r.uniform(-1, 1, (n, n)), 0.02 * r.uniform(-1, 1, (n, n)), 0.02 * r.uniform(-1, 1, (n, n))


def _run(kmi, backend, sizes, storage, collision, lid, launch, steps):
    with kmi.Batch(sizes, [0.03 + 0.001 * (c % 7) for c in range(len(sizes))], storage=storage, collision=collision,
                   lid=lid, backend=backend) as b:
        tw, span = launch
        b.set_launch(tw, 256 // tw)
        b.set_temporal(span)
        for c, n in enumerate(sizes):
            b.init_equilibrium(c, *_u(n, c % 11))
        b.step(steps)
        return [b.download(c) for c in range(len(sizes))]


@pytest.mark.parametrize("storage", list(EDGES))
def test_both_routes_equal_single_steps(kmi, backend, storage):
    for k, (tw, span, edge) in enumerate(EDGES[storage]):
        collision, lid = ("mrt", "bgk", "trt")[k % 3], ("zouhe", "ladd")[k % 2]
        for count in (edge, edge + 1):
            print(f"[batch routes] {storage} {collision} {lid} width {tw} span {span}, {count} cavities", flush=True)
            sizes = [64] * count
            ref = _run(kmi, backend, sizes, storage, collision, lid, (64, 1), 4 * span + 1)
            got = _run(kmi, backend, sizes, storage, collision, lid, (tw, span), 4 * span + 1)
            assert all(np.array_equal(a, b) for a, b in zip(ref, got)), (tw, span, count)


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s", "f16s"])
@pytest.mark.parametrize("collision,lid", [("mrt", "zouhe"), ("bgk", "ladd"), ("trt", "zouhe")])
def test_uneven_batches_equal_single_steps(kmi, backend, storage, collision, lid):
    """Cavities from two cells a side: few tiles, and enough of them for the march."""
    few = [2, 3, 5, 7, 13, 30, 58, 61, 64, 65, 70]
    many = few + [117, 122, 123, 128, 200, 319, 401, 255]
    for sizes in (few, many):
        ref = _run(kmi, backend, sizes, storage, collision, lid, (64, 1), 39)
        for launch in ((64, 3), (64, 4), (32, 4), (16, 3)):
            print(f"[batch routes] {storage} {collision} {lid} {len(sizes)} cavities {launch}", flush=True)
            got = _run(kmi, backend, sizes, storage, collision, lid, launch, 39)
            assert all(np.array_equal(a, b, equal_nan=True) for a, b in zip(ref, got)), (len(sizes), launch)


@pytest.mark.parametrize("storage", ["f64", "f32s"])
def test_route_changes_while_cavities_retire(kmi, backend, storage):
    """Small cavities converge first; the rest go over to the LDS tiles in mid-run."""
    sizes = [16] * 40 + [96] * 12 + [128] * 12
    out = []
    for span in (1, 4):
        with kmi.Batch(sizes, [0.1 * n / 16 for n in sizes], storage=storage, collision="mrt", backend=backend) as b:
            b.set_temporal(span)
            b.run(tol=1e-4, check_every=40, max_steps=4000)
            out.append(([b.download(c) for c in range(len(sizes))], b.status()["steps"]))
    assert np.array_equal(out[0][1], out[1][1]) and len(set(out[0][1])) > 1
    assert all(np.array_equal(a, b) for a, b in zip(out[0][0], out[1][0]))
