"""Single-step launches whose waves lie in one row of cells (work-group width a multiple of 64)
against the ones whose waves span rows: the same per-cell arithmetic, so the same bits.

Row lengths around a wave, odd rows, one or several groups across a row (each deals the rows to
the XCDs differently) and every kind of face and cell class that the pull selects on.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WALL, PER = {"kind": "wall"}, {"kind": "periodic"}


def _cases(kmi, nx, ny, nz):
    moving = {"kind": "moving_wall", "u": (0.02, 0.01, 0.03)}
    r = np.random.default_rng(nx + ny)
    blob = (r.uniform(size=(nx, ny, nz)) < 0.03).astype(np.uint8)
    lid = {"kind": "zouhe_velocity", "u": (0.05, 0.0, 0.0)}
    yield "lid", "trt", dict(west=WALL, east=WALL, south=WALL, north=WALL, bottom=WALL, top=lid), None, {}
    yield "moving", "bgk", dict(west=moving, east=WALL, south=moving, north=WALL, bottom=WALL, top=moving), blob, {}
    yield "duct", "bgk", dict(west=PER, east=PER), blob, dict(forcing="guo", force=(1e-5, 0.0, 2e-5))
    yield "slab", "trt", dict(west=PER, east=PER, south=PER, north=PER, bottom=moving, top=WALL), None, {}
    yield "rebuilt", "trt", dict(west={"kind": "zouhe_velocity_rebuild"},
                                 east={"kind": "zouhe_pressure_rebuild", "rho": 1.0}), None, {}
    yield "thermal", "bgk", dict(west=dict(WALL, thermal="dirichlet", T=1.0), east=dict(WALL, thermal="dirichlet", T=0.0)), \
        blob, dict(thermal=True, omega_T=1.4, beta_g=1e-4, T_ref=0.5)


@pytest.mark.parametrize("storage", ["f64", "f32", "f32s", "f16s"])
@pytest.mark.parametrize("shape", [(63, 9, 7), (64, 8, 5), (65, 17, 4), (130, 5, 6), (300, 3, 4)])
def test_row_launch_equals_patch_launch(kmi, backend, storage, shape):
    for name, collision, faces, mask, more in _cases(kmi, *shape):
        print(f"[rows] {storage} {shape} {name}", flush=True)
        d = kmi.make_desc("d3q19", *shape, 0.05, storage=storage, collision=collision, faces=faces, **more)
        r = np.random.default_rng(5)
        u = 0.02 * r.uniform(-1, 1, (4,) + shape)
        out = []
        for bx, by in ((16, 4), (64, 1), (64, 2), (128, 1), (256, 1)):
            with kmi.Lattice(d, backend) as lat:
                if mask is not None:
                    lat.set_mask(mask)
                lat.init_equilibrium(1 + u[0], u[1], u[2], u[3])
                if more.get("thermal"):
                    lat.init_temperature(0.5 + u[0])
                if name == "rebuilt":
                    lat.set_face_profile("west", 0.03 + u[1][0])
                lat.set_launch(bx, by)
                lat.set_temporal(0, 1)
                lat.step(5)
                out.append([lat.download_raw()] + ([lat.download_raw("g")] if more.get("thermal") else []))
        for o in out[1:]:
            assert all(np.array_equal(a, b) for a, b in zip(out[0], o)), (storage, shape, name)
