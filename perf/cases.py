"""Performance cases of the stream–collide framework: the runs its users make of it.

Each case is one kind of simulation (`problem`) at one size, storage type and collision.  A pass
advances the state by `steps` time steps (or serves / trains the warm-start decoder) through the
public entry points and hands back everything that a program reads afterwards: the moment planes,
sampled forces, Nusselt numbers, residuals, the network's outputs or weights.  `exact` computes the
same values in 64 bits with plain torch.

What a program has in hand before a pass — the lattice with its geometry, initial state and chosen
launch, the batch, the network with its weights and dataset — is made by `prepare`.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "krakenn.jl_amd"))

import kraken_mi355x as kmi  # noqa: E402
from kraken_mi355x import warmstart as ws  # noqa: E402
from kraken_mi355x.nn import WarmStartNet  # noqa: E402

BYTES = {"f64": 8, "f32": 4, "f32s": 4, "f16s": 2}


def listed():
    return [
        # run_cylinder_libb_2d at its default size: every step of the averaging window is one
        # step and one drag sample on 24,000 cells, the smallest calls there are.
        dict(name="cylinder drag 300x80 f64", problem="cylinder", nx=300, ny=80, storage="f64", steps=100),
        # run_cavity_2d, the plain small run: BGK, Zou–He lid, 128², double precision.
        dict(name="cavity 128x128 f64", problem="cavity2d", nx=128, ny=128, storage="f64", collision="bgk",
             steps=2000, check=0),
        # run_rayleigh_benard_2d at 512×256, Ra = 1e5: f and g, shifted FP32 storage.
        dict(name="rayleigh-benard 512x256 f32s", problem="rayleigh_benard", nx=512, ny=256, storage="f32s",
             steps=2000),
        # run_taylor_green_2d at the reference's certification size: a large periodic 2D lattice.
        dict(name="taylor-green 2048x2048 f64", problem="taylor_green_2d", nx=2048, ny=2048, storage="f64",
             collision="bgk", steps=400),
        # The benchmark: D3Q19 TRT Taylor–Green, 256³, shifted FP32, launch chosen beforehand.
        dict(name="taylor-green 256^3 f32s", problem="taylor_green_3d", nx=256, ny=256, nz=256, storage="f32s",
             steps=600, tile=11, zchunks=2),
        # run_cavity_3d as the driver runs it: the reference's default precision and launch.
        dict(name="cavity 128^3 f64", problem="cavity3d", nx=128, ny=128, nz=128, storage="f64",
             collision="bgk", steps=400),
        # A body-force-driven duct at sizes that no tile divides.
        dict(name="duct 150x75x61 f32", problem="duct3d", nx=150, ny=75, nz=61, storage="f32", steps=400),
        # run_sphere_libb_3d at its default size, run-up and a short drag window.
        dict(name="sphere 120x60x60 f64", problem="sphere", nx=120, ny=60, nz=60, storage="f64", steps=200,
             samples=50),
        # run_natural_convection_3d: f and g on D3Q19 in double precision.
        dict(name="natural convection 64^3 f64", problem="natural_convection_3d", nx=64, ny=64, nz=64,
             storage="f64", steps=400),
        # The batched ensemble: 256 cavities of uneven side and Reynolds number with residual checks.
        dict(name="256 uneven cavities f32s", problem="ensemble", cavities=256, low=64, high=512, storage="f32s",
             collision="mrt", steps=1000),
        # Warm start, serving: initial fields for 256 held-out cavities.
        dict(name="decoder 256 fields 128x128", problem="decoder", samples=256, side=128, batch=32),
        # Warm start, training: epochs of forward, both gradients and Adam.
        dict(name="decoder training 128x128", problem="training", samples=256, side=128, batch=32, epochs=4),
    ]


def draw(rng):
    """One more case of the same ranges."""
    between = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    problem = rng.choice(["cylinder", "cavity2d", "rayleigh_benard", "taylor_green_2d", "taylor_green_3d", "cavity3d",
                          "duct3d", "sphere", "natural_convection_3d", "ensemble", "decoder", "training"])
    c = {"problem": problem}
    if problem == "cylinder":
        ny = between(40, 160)
        c.update(nx=int(ny * rng.uniform(3, 5)), ny=ny, storage=rng.choice(["f64", "f32"]), steps=rng.randint(40, 120))
    elif problem == "cavity2d":
        n = between(64, 1024)
        c.update(nx=n, ny=n, storage=rng.choice(["f64", "f32", "f32s"]), collision=rng.choice(["bgk", "trt", "mrt"]),
                 steps=100 * rng.randint(4, 12), check=rng.choice([0, 100]))
    elif problem == "rayleigh_benard":
        ny = between(64, 320)
        c.update(nx=int(ny * rng.uniform(1.5, 4)), ny=ny, storage=rng.choice(["f64", "f32", "f32s", "f16s"]),
                 steps=rng.randint(300, 1000))
    elif problem == "taylor_green_2d":
        n = between(256, 2500)
        c.update(nx=n, ny=n, storage=rng.choice(["f64", "f32"]), collision="bgk", steps=rng.randint(200, 400))
    elif problem == "taylor_green_3d":
        n = between(48, 256)
        c.update(nx=n, ny=n, nz=n, storage=rng.choice(["f64", "f32", "f32s", "f16s"]), steps=rng.randint(100, 250),
                 tile=0, zchunks=1)
    elif problem == "cavity3d":
        n = between(48, 200)
        c.update(nx=n, ny=n, nz=n, storage=rng.choice(["f64", "f64", "f32", "f32s"]),
                 collision=rng.choice(["bgk", "trt"]), steps=rng.randint(100, 250))
    elif problem == "duct3d":
        ny = between(32, 128)
        c.update(nx=int(ny * rng.uniform(1, 3)), ny=ny, nz=int(ny * rng.uniform(0.7, 1.2)),
                 storage=rng.choice(["f64", "f32", "f32s"]), steps=rng.randint(100, 300))
    elif problem == "sphere":
        ny = between(40, 96)
        c.update(nx=int(ny * rng.uniform(1.6, 2.4)), ny=ny, nz=ny, storage=rng.choice(["f64", "f32"]),
                 steps=rng.randint(60, 200), samples=rng.randint(10, 50))
    elif problem == "natural_convection_3d":
        n = between(32, 112)
        c.update(nx=n, ny=n, nz=n, storage=rng.choice(["f64", "f32", "f32s"]), steps=rng.randint(100, 300))
    elif problem == "ensemble":
        low = between(32, 160)
        c.update(cavities=between(16, 256), low=low, high=low + between(32, 300),
                 storage=rng.choice(["f64", "f32", "f32s"]), collision=rng.choice(["mrt", "mrt", "trt", "bgk"]),
                 steps=100 * rng.randint(2, 5))
    elif problem == "decoder":
        c.update(samples=between(16, 512), side=rng.choice([64, 128]), batch=rng.choice([16, 32]))
    else:
        batch = rng.choice([16, 32])
        c.update(samples=batch * rng.randint(2, 8), side=rng.choice([64, 128]), batch=batch, epochs=rng.randint(1, 3))
    return c


# ---- what the seed decides ---------------------------------------------------------------------
def _flow(case, seed):
    """Physical parameters and initial fields of a single-lattice case."""
    r = np.random.default_rng([int(seed), 7])
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    jig = lambda v, rel=0.2: float(v * (1 + rel * r.uniform(-1, 1)))  # noqa: E731
    p = case["problem"]
    if p in ("cavity2d", "cavity3d"):
        u = jig(0.08)
        re = math.exp(r.uniform(math.log(100.0), math.log(400.0)))
        return {"u": u, "nu": max(u * nx / re, 0.012)}
    if p == "taylor_green_2d":
        return {"u": jig(0.02), "nu": jig(0.02), "phase": r.uniform(0, 2 * math.pi, 2).tolist()}
    if p == "taylor_green_3d":
        return {"u": jig(0.05), "nu": jig(0.01), "phase": r.uniform(0, 2 * math.pi, 3).tolist()}
    if p == "duct3d":
        return {"nu": jig(0.05), "force": (jig(2e-6), 0.0, 0.0), "u": jig(0.03), "phase": float(r.uniform())}
    if p in ("cylinder", "sphere"):
        return {"u": jig(0.04), "nu": jig(0.04), "radius": ny / 8.0}
    if p == "rayleigh_benard":
        return {"ra": 1e5, "pr": 0.71, "t0": kmi.rb_initial_temperature(nx, ny, 1.0, 0.0, seed="noise",
                                                                        rng_seed=int(seed))}
    t0 = kmi.natural_convection_3d_initial_temperature(nx) + 1e-2 * r.uniform(-1, 1, (nx, ny, nz))
    return {"ra": math.exp(r.uniform(math.log(1e3), math.log(1e5))), "pr": 0.71, "t0": np.asfortranarray(t0)}


def _vortex(case, w):
    """Taylor–Green fields with shifted origins (ρ, u, v(, w)), arrays [i, j(, k)]."""
    if case["problem"] == "taylor_green_2d":
        k = 2 * math.pi / case["nx"]
        x = k * np.arange(case["nx"])[:, None] + w["phase"][0]
        y = k * np.arange(case["ny"])[None, :] + w["phase"][1]
        u0 = w["u"]
        rho = 1.0 - 0.75 * u0 ** 2 * (np.cos(2 * x) + np.cos(2 * y))
        return rho, -u0 * np.cos(x) * np.sin(y), u0 * np.sin(x) * np.cos(y)
    x, y, z = (2 * math.pi / n * np.arange(n) + ph for n, ph in zip((case["nx"], case["ny"], case["nz"]), w["phase"]))
    col = lambda a, b, c: np.multiply(a[:, None, None] * b[None, :, None], c[None, None, :], order="F")  # noqa: E731
    u = col(w["u"] * np.sin(x), np.cos(y), np.cos(z))
    v = col(-w["u"] * np.cos(x), np.sin(y), np.cos(z))
    return np.ones_like(u), u, v, np.zeros_like(u)


def _swirl(case, w):
    """Stream along the duct with swirling disturbances (ρ, u, v, w), arrays [i, j, k]."""
    x, y, z = (np.arange(n) / n for n in (case["nx"], case["ny"], case["nz"]))
    x = 2 * math.pi * (x + w["phase"])
    col = lambda a, b, c: np.multiply(a[:, None, None] * b[None, :, None], c[None, None, :], order="F")  # noqa: E731
    wall = lambda t: np.sin(math.pi * t)  # noqa: E731
    u = col(1 + 0.2 * np.cos(x), wall(y), wall(z))
    v = col(0.3 * np.sin(x), wall(y), np.cos(math.pi * z))
    s = col(0.3 * np.cos(x), np.cos(math.pi * y), wall(z))
    return np.ones_like(u), w["u"] * u, w["u"] * v, w["u"] * s


def _ensemble(case, seed):
    r = np.random.default_rng([int(seed), 11])
    sides = np.arange(case["low"], case["high"] + 1, 32)
    n = np.random.default_rng(2024).choice(sides, size=case["cavities"]).astype(np.int32)
    # Reynolds numbers log-uniform from 100 up to where the relaxation time stays above 0.53
    top = np.minimum(3200.0, 0.1 * n / 0.012)
    re = np.exp(r.uniform(np.log(min(100.0, top.min() * 0.9)), np.log(top)))
    return n, 0.1 * n / re


def _net_inputs(case, seed):
    re, a = ws.draw_cases(case["samples"], seed=int(seed))
    x = ws.encode(re, a)
    side = case["side"]
    if case["problem"] == "decoder":
        return x, None
    yy, xx = np.meshgrid(np.linspace(0, 1, side), np.linspace(0, 1, side), indexing="ij")
    x0, x1 = x[:, 0, None, None], x[:, 1, None, None]
    y = np.stack([np.sin(np.pi * (1 + c) * xx + x0) * np.cos(np.pi * yy * (1 + x1)) for c in range(3)], axis=-1)
    return x, y.astype(np.float32)


def _net(case, seed):
    return WarmStartNet(latent_hw=case["side"] // 8, max_batch=case["batch"], seed=1 + int(seed) % 1000)


# ---- state -------------------------------------------------------------------------------------
def _channel(case, w):
    """Descriptor, cut links, solid mask and inlet profile of the cylinder / sphere drivers."""
    nx, ny, nz, rad = case["nx"], case["ny"], case.get("nz", 1), w["radius"]
    faces = {"west": {"kind": "zouhe_velocity_rebuild"}, "east": {"kind": "zouhe_pressure_rebuild", "rho": 1.0}}
    if case["problem"] == "cylinder":
        qw, solid = kmi.precompute_q_wall_cylinder(nx, ny, nx // 4, ny // 2, rad)
        j = np.arange(ny, dtype=np.float64)
        prof = 4.0 * w["u"] * j * (ny - 1 - j) / float(ny - 1) ** 2
        d = kmi.make_desc("d2q9", nx, ny, 1, w["nu"], storage=case["storage"], collision="trt", faces=faces,
                          solid_mode="inert")
        return d, qw, solid, prof
    qw, solid = kmi.precompute_q_wall_sphere_3d(nx, ny, nz, nx // 4, ny // 2, nz // 2, rad)
    d = kmi.make_desc("d3q19", nx, ny, nz, w["nu"], storage=case["storage"], collision="trt", faces=faces,
                      solid_mode="inert")
    return d, qw, solid, np.full((ny, nz), w["u"])


def prepare(case, seed):
    p = case["problem"]
    state = {"case": case}
    if p in ("decoder", "training"):
        state["net"] = _net(case, seed)
        state["x"], y = _net_inputs(case, seed)
        if y is not None:
            state["net"].set_dataset(state["x"], y)
        return state
    if p == "ensemble":
        n, nu = _ensemble(case, seed)
        b = kmi.Batch(n, nu, storage=case["storage"], collision=case["collision"], u_lid=0.1)
        b.autotune(4)
        cells = n.astype(np.int64) ** 2
        at = np.concatenate([[0], np.cumsum(cells)])
        state.update(batch=b, cap=0, at=at, fields={k: np.zeros(at[-1]) for k in ("rho", "ux", "uy")})
        return state
    w = _flow(case, seed)
    shape = (case["nx"], case["ny"]) if "nz" not in case else (case["nx"], case["ny"], case["nz"])
    st = case["storage"]
    if p == "cavity2d":
        lat = kmi.Lattice(kmi.cavity_desc(case["nx"], w["nu"], w["u"], storage=st, collision=case["collision"]))
    elif p == "cavity3d":
        lat = kmi.Lattice(kmi.cavity_3d_desc(*shape, w["nu"], w["u"], storage=st, collision=case["collision"]))
    elif p == "rayleigh_benard":
        lat = kmi.Lattice(kmi.rayleigh_benard_desc(*shape, w["ra"], w["pr"], storage=st)[0])
        lat.init_temperature(w["t0"])
    elif p == "natural_convection_3d":
        lat = kmi.Lattice(kmi.natural_convection_3d_desc(case["nx"], w["ra"], w["pr"], storage=st)[0])
        lat.init_temperature(w["t0"])
    elif p == "taylor_green_2d":
        per = {f: {"kind": "periodic"} for f in ("west", "east", "south", "north")}
        lat = kmi.Lattice(kmi.make_desc("d2q9", *shape, 1, w["nu"], storage=st, faces=per))
        lat.init_equilibrium(*_vortex(case, w))
    elif p == "taylor_green_3d":
        lat = kmi.Lattice(kmi.taylor_green_3d_desc(case["nx"], w["nu"], st))
        lat.init_equilibrium(*_vortex(case, w))
        if case["tile"]:
            lat.set_temporal(case["tile"], case["zchunks"])
    elif p == "duct3d":
        per = {"west": {"kind": "periodic"}, "east": {"kind": "periodic"}}
        lat = kmi.Lattice(kmi.make_desc("d3q19", *shape, w["nu"], storage=st, faces=per, forcing="guo",
                                        force=w["force"]))
        lat.init_equilibrium(*_swirl(case, w))
    else:
        d, qw, solid, prof = _channel(case, w)
        lat = kmi.Lattice(d)
        lat.set_mask(solid)
        lat.set_cut_links(*kmi.cut_links_from_dense(qw))
        lat.set_face_profile("west", prof)
        lat.init_equilibrium(1.0, np.broadcast_to(prof[None], shape))
    if p in ("cavity2d", "rayleigh_benard", "taylor_green_2d"):
        lat.autotune(64)  # as the 2D drivers do for runs of this length
    state["lat"] = lat
    return state


# ---- one pass ----------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    p = case["problem"]
    if p == "decoder":
        return {"fields": state["net"].predict(state["x"])}
    if p == "training":
        loss = state["net"].train_epochs(case["epochs"], case["batch"], 1e-3, seed=5)
        return {"loss": loss, "params": state["net"].get_params()}
    if p == "ensemble":
        b = state["batch"]
        state["cap"] += case["steps"]
        b.resume()
        b.run(1e-9, 100, state["cap"], window=100)
        st = b.status()
        for c in range(len(b)):
            m = b.moments(c)
            for k, a in state["fields"].items():
                a[state["at"][c]:state["at"][c + 1]] = m[k].ravel(order="F")
        return {"steps": st["steps"], "residual": st["residual"], **state["fields"]}
    lat = state["lat"]
    if p in ("cylinder", "sphere"):
        kind = "drag_mea" if p == "cylinder" else "drag_halfway"
        samples = case.get("samples", case["steps"])
        if case["steps"] > samples:
            lat.step(case["steps"] - samples)
        drag = np.empty((samples, 3))
        for k in range(samples):
            lat.step(1)
            drag[k] = lat.reduce(kind)
        return {"drag": drag[:, 0].copy(), **lat.moments()}
    if case.get("check"):
        res = [lat.step_residual(case["check"], case["check"]) for _ in range(case["steps"] // case["check"])]
        return {"residual": np.array(res), **lat.moments()}
    lat.step(case["steps"])
    if p == "rayleigh_benard":
        return {**lat.moments(temperature=True), "nu": lat.reduce("nusselt", "south")}
    if p == "natural_convection_3d":
        return {**lat.moments(temperature=True), "nu": lat.reduce("nusselt", "west")}
    return lat.moments()


# ---- work --------------------------------------------------------------------------------------
def work(case):
    """State and inputs read once, state and outputs written once; the updates' arithmetic."""
    p = case["problem"]
    if p in ("decoder", "training"):
        hw = case["side"] // 8
        lat = hw * hw * 64
        fwd = 2 * (2 * 256 + 256 * lat)
        for hi, ci, co in ((hw, 64, 64), (2 * hw, 64, 32), (4 * hw, 32, 3)):
            fwd += 2 * (2 * hi) ** 2 * 9 * ci * co
        weights = 2 * 256 + 256 + 256 * lat + lat + 9 * 64 * 64 + 64 + 9 * 64 * 32 + 32 + 9 * 32 * 3 + 3
        image = case["side"] ** 2 * 3 * 4
        if p == "decoder":
            return {"bytes": 4 * weights + case["samples"] * image, "flops": fwd * case["samples"]}
        n = case["samples"] // case["batch"] * case["batch"] * case["epochs"]
        return {"bytes": 6 * 4 * weights + case["samples"] * image, "flops": 3 * fwd * n}
    flow = {"bgk": (130, 290), "trt": (150, 330), "mrt": (190, 0)}
    if p == "ensemble":
        sides = np.arange(case["low"], case["high"] + 1, 32, dtype=np.float64)
        cells = case["cavities"] * float(np.mean(sides ** 2))
        return {"bytes": cells * (18 * BYTES[case["storage"]] + 24), "flops": cells * case["steps"] * flow[case["collision"]][0]}
    q, dim = (9, 0) if "nz" not in case else (19, 1)
    cells = case["nx"] * case["ny"] * case.get("nz", 1)
    thermal = p in ("rayleigh_benard", "natural_convection_3d")
    coll = "trt" if p in ("cylinder", "sphere", "taylor_green_3d") else case.get("collision", "bgk")
    flops = flow[coll][dim] + (80, 170)[dim] * (thermal + (p == "duct3d"))
    b = BYTES[case["storage"]]
    pops = 2 * q * (b + (max(b, 4) if thermal else 0))
    return {"bytes": cells * (pops + 8 * (3 + dim + thermal)), "flops": cells * case["steps"] * flops}


# ---- the same values in 64 bits, plain torch ---------------------------------------------------
C9 = [(0, 0, 0), (1, 0, 0), (0, 1, 0), (-1, 0, 0), (0, -1, 0), (1, 1, 0), (-1, 1, 0), (-1, -1, 0), (1, -1, 0)]
W9 = [4 / 9] + [1 / 9] * 4 + [1 / 36] * 4
C19 = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1), (1, 1, 0), (-1, 1, 0), (1, -1, 0),
       (-1, -1, 0), (1, 0, 1), (-1, 0, 1), (1, 0, -1), (-1, 0, -1), (0, 1, 1), (0, -1, 1), (0, 1, -1), (0, -1, -1)]
W19 = [1 / 3] + [1 / 18] * 6 + [1 / 36] * 12


class Plain:
    """Populations [q, (batch,) z, y, x] in float64; one method per stage of a step."""

    def __init__(self, q, periodic, device):
        self.c, self.w = (C9, W9) if q == 9 else (C19, W19)
        self.q, self.periodic = q, periodic
        self.opp = [self.c.index(tuple(-v for v in c)) for c in self.c]
        self.dev = device
        self.cm = torch.tensor(self.c, dtype=torch.float64, device=device).T.contiguous()
        self.wv = torch.tensor(self.w, dtype=torch.float64, device=device)

    def per_q(self, v, like):
        return v.reshape((self.q,) + (1,) * (like.dim() - 1))

    def sides(self, a, face):
        """The planes of a tensor [..., z, y, x] on a face: west, east, south, north, bottom, top."""
        ax = -1 - face // 2
        return a.select(ax, 0 if face % 2 == 0 else a.shape[ax] - 1)

    def stream(self, f):
        out = torch.empty_like(f)
        for k, c in enumerate(self.c):
            out[k] = torch.roll(f[k], shifts=(c[2], c[1], c[0]), dims=(-3, -2, -1)) if any(c) else f[k]
            for ax in range(3):
                if c[ax] and not self.periodic[ax]:  # halfway bounce-back: the cell's own opposite
                    face = 2 * ax + (0 if c[ax] > 0 else 1)
                    self.sides(out[k], face).copy_(self.sides(f[self.opp[k]], face))
        return out

    def moments(self, f):
        rho = f.sum(0)
        j = (self.cm @ f.reshape(self.q, -1)).reshape((3,) + f.shape[1:])
        return rho, j

    def feq(self, rho, u):
        cu = (self.cm.T @ u.reshape(3, -1)).reshape((self.q,) + u.shape[1:])
        usq = (u * u).sum(0)
        e = cu.mul(4.5).add_(3.0).mul_(cu).add_(1.0).sub_(1.5 * usq)
        return e.mul_(rho).mul_(self.per_q(self.wv, e))

    def bgk(self, f, om):
        rho, j = self.moments(f)
        return f + om * (self.feq(rho, j / rho) - f)

    def trt(self, f, sp, sm):
        rho, j = self.moments(f)
        n = f - self.feq(rho, j / rho)
        return f - (0.5 * (sp + sm)) * n - (0.5 * (sp - sm)) * n[self.opp]

    def guo(self, f, om, force, rho=None, j=None):
        """BGK with the Guo source; force: a list of three numbers or planes."""
        if rho is None:
            rho, j = self.moments(f)
        F = torch.stack([torch.as_tensor(v, dtype=torch.float64, device=self.dev).expand_as(rho) for v in force])
        u = (j + 0.5 * F) / rho
        cu = (self.cm.T @ u.reshape(3, -1)).reshape((self.q,) + rho.shape)
        cf = (self.cm.T @ F.reshape(3, -1)).reshape((self.q,) + rho.shape)
        s = self.per_q(self.wv, f) * (3.0 * (cf - (u * F).sum(0)) + 9.0 * cu * cf)
        return f + om * (self.feq(rho, u) - f) + (1.0 - 0.5 * om) * s

    def mrt(self, f, s_nu, s_e=1.4, s_eps=1.4, s_q=1.2):
        cx, cy = self.cm[0], self.cm[1]
        r2 = cx * cx + cy * cy
        m = torch.stack([torch.ones_like(cx), -4 + 3 * r2, 4 - 10.5 * r2 + 4.5 * r2 * r2, cx, (3 * r2 - 5) * cx, cy,
                         (3 * r2 - 5) * cy, cx * cx - cy * cy, cx * cy])
        mom = (m @ f.reshape(9, -1)).reshape(f.shape)
        rho, jx, jy = mom[0], mom[3], mom[5]
        sq = 3.0 * (jx * jx + jy * jy) / rho
        eq = torch.stack([rho, -2 * rho + sq, rho - sq, jx, -jx, jy, -jy, (jx * jx - jy * jy) / rho, jx * jy / rho])
        zero = torch.zeros_like(rho)
        one = lambda v: torch.as_tensor(v, dtype=torch.float64, device=self.dev) + zero  # noqa: E731
        rate = torch.stack([zero, one(s_e), one(s_eps), zero, one(s_q), zero, one(s_q), one(s_nu), one(s_nu)])
        return f - (torch.linalg.inv(m) @ (rate * (mom - eq)).reshape(9, -1)).reshape(f.shape)

    def lid2(self, f, u):
        """Zou–He velocity (u, 0) on the north row."""
        n = [self.sides(f[k], 3) for k in range(9)]
        rw = n[0] + n[1] + n[3] + 2 * (n[2] + n[5] + n[6])
        d = 0.5 * (n[1] - n[3])
        n[4].copy_(n[2])
        n[8].copy_(n[6] - d + 0.5 * rw * u)
        n[7].copy_(n[5] + d - 0.5 * rw * u)

    def lid3(self, f, u):
        """Zou–He velocity (u, 0, 0) on the top plane."""
        n = [self.sides(f[k], 5) for k in range(19)]
        rw = sum(n[k] for k in (0, 1, 2, 3, 4, 7, 8, 9, 10)) + 2 * sum(n[k] for k in (5, 11, 12, 15, 16))
        t1 = 0.5 * ((n[1] - n[2]) + (n[7] - n[8] + n[9] - n[10]))
        t2 = 0.5 * ((n[3] - n[4]) + (n[7] + n[8] - n[9] - n[10]))
        n[6].copy_(n[5])
        n[13].copy_(n[12] - t1 + 0.5 * rw * u)
        n[14].copy_(n[11] + t1 - 0.5 * rw * u)
        n[17].copy_(n[16] - t2)
        n[18].copy_(n[15] + t2)

    def hot_cold(self, g, face_t):
        """Anti-bounce-back g = −g + 2 w T of the links that enter through a Dirichlet face."""
        for face, t in face_t.items():
            ax, sign = face // 2, 1 if face % 2 == 0 else -1
            for k, c in enumerate(self.c):
                if c[ax] == sign:
                    s = self.sides(g[k], face)
                    s.copy_(2 * self.w[k] * t - s)

    def thermal(self, f, g, om, om_t, buoyancy, t_ref, face_t):
        f, g = self.stream(f), self.stream(g)
        self.hot_cold(g, face_t)
        t = g.sum(0)
        rho, j = self.moments(f)
        u = j / rho
        cu = (self.cm.T @ u.reshape(3, -1)).reshape((self.q,) + rho.shape)
        geq = self.per_q(self.wv, g) * t * (1 + 3 * cu)
        return self.guo(f, om, [0.0, buoyancy * (t - t_ref), 0.0], rho, j), g + om_t * (geq - g)


def _planes(P, f, shape, shift=None):
    """Moment planes as the framework lays them out: [i, j(, k)] in float64."""
    rho, j = P.moments(f)
    if shift is not None:
        j = j + 0.5 * torch.tensor(shift, dtype=torch.float64, device=f.device).reshape(3, 1, 1, 1)
    u = j / rho
    host = lambda a: a.permute(2, 1, 0).reshape(shape).cpu().numpy()  # noqa: E731
    out = {"rho": host(rho), "ux": host(u[0]), "uy": host(u[1])}
    if P.q == 19:
        out["uz"] = host(u[2])
    return out


def _to(a, shape3, device):
    """Host field [i, j(, k)] → device [z, y, x]."""
    return torch.from_numpy(np.ascontiguousarray(np.asarray(a, dtype=np.float64).reshape(shape3).transpose(2, 1, 0))).to(device)


def _rebuilt(P, node, west, value, sp, sm):
    """A rebuilt inlet (west: normal velocity) or outlet (density) node: Zou–He closure, then the local
    collision of the face: regularised TRT on D2Q9, TRT on D3Q19."""
    n = [v.clone() for v in node]
    pair = [(k, P.opp[k]) for k in range(P.q) if P.c[k][0] == (1 if west else -1)]
    par = sum(n[k] for k in range(P.q) if P.c[k][0] == 0)
    out = sum(n[o] for _, o in pair)
    if west:
        rho = (par + 2 * out) / (1 - value)
        ru = rho * value
    else:
        rho = torch.zeros_like(par) + value
        ru = -rho * (1 - (par + 2 * out) / rho)
    sign = 1.0 if west else -1.0
    axis = {0: 0, 1: 2.0 / 3.0 if P.q == 9 else 1.0 / 3.0}
    ty = n[P.c.index((0, 1, 0))] - n[P.c.index((0, -1, 0))]
    tz = n[P.c.index((0, 0, 1))] - n[P.c.index((0, 0, -1))] if P.q == 19 else None
    for k, o in pair:
        c = P.c[k]
        if c[1] == 0 and c[2] == 0:
            n[k] = n[o] + sign * axis[1] * ru
        else:
            t = c[1] * ty if c[1] else c[2] * tz
            n[k] = n[o] - 0.5 * t + sign * ru / 6.0
    f = torch.stack(n)
    rho, j = P.moments(f)
    e = P.feq(rho, j / rho)
    if P.q == 19:
        d = f - e
        return f - (0.5 * (sp + sm)) * d - (0.5 * (sp - sm)) * d[P.opp]
    d = f - e
    pxx = d[1] + d[3] + d[5] + d[6] + d[7] + d[8]
    pyy = d[2] + d[4] + d[5] + d[6] + d[7] + d[8]
    pxy = d[5] - d[6] + d[7] - d[8]
    m0 = -(pxx + pyy) / 9
    m1, m2 = (2 * pxx - pyy) / 18, (2 * pyy - pxx) / 18
    m5, m6 = (pxx + pyy) / 72 + pxy / 4, (pxx + pyy) / 72 - pxy / 4
    m = torch.stack([m0, m1, m2, m1, m2, m5, m6, m5, m6])
    rate = torch.tensor([sp] + [0.5 * (sp + sm) + 0.5 * (sp - sm)] * 8, dtype=torch.float64, device=f.device)
    return e + (1 - P.per_q(rate, m)) * m


def _exact_channel(case, seed, dev):
    w = _flow(case, seed)
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    two = case["problem"] == "cylinder"
    _, qw, solid, prof = _channel(case, w)
    P = Plain(9 if two else 19, (False, False, True) if two else (False,) * 3, dev)
    qw = torch.stack([_to(qw[..., k], (nx, ny, nz), dev) for k in range(P.q)])
    solid = _to(solid, (nx, ny, nz), dev) > 0
    prof = torch.from_numpy(np.ascontiguousarray(prof.reshape(ny, nz).T)).to(dev)  # [z, y]
    u = torch.zeros((3, nz, ny, nx), dtype=torch.float64, device=dev)
    u[0] = prof[..., None]
    f = P.feq(torch.ones_like(u[0]), u)
    sp, sm = 1 / (3 * w["nu"] + 0.5), 1 / (3.0 / 16.0 / (3 * w["nu"]) + 0.5)
    inner = (slice(None) if two else slice(1, nz - 1), slice(1, ny - 1))
    cut = [k for k in range(1, P.q) if bool((qw[k] > 0).any())]
    near = {k: qw[k] > 0 for k in cut}
    mirrored = lambda fw, back, bar, q: torch.where(q <= 0.5, 2 * q * fw + (1 - 2 * q) * back,  # noqa: E731
                                                    fw / (2 * q) + (1 - 1 / (2 * q)) * bar)
    rest = P.per_q(P.wv, f)
    cut_q = {k: torch.where(near[k], qw[k], torch.ones_like(qw[k])) for k in cut}
    drag = []
    samples = case.get("samples", case["steps"])
    for n in range(case["steps"]):
        s = P.stream(f)
        pulled = s.clone()
        for k in cut:
            o = P.opp[k]
            s[o] = torch.where(near[k], mirrored(f[k], pulled[k], f[o], cut_q[k]), s[o])
        out = P.trt(s, sp, sm)
        out = torch.where(solid, rest, out)
        for west in (True, False):
            x = 0 if west else nx - 1
            node = [pulled[k][inner[0], inner[1], x] for k in range(P.q)]
            value = prof[inner] if west else 1.0
            out[:, inner[0], inner[1], x] = _rebuilt(P, node, west, value, sp, sm)
        f = out
        if n >= case["steps"] - samples:
            total = 0.0
            for k in cut:
                if P.c[k][0] == 0:
                    continue
                if two:
                    b = torch.roll(f[k], shifts=(P.c[k][2], P.c[k][1], P.c[k][0]), dims=(-3, -2, -1))
                    force = f[k] + mirrored(f[k], b, f[P.opp[k]], cut_q[k])
                else:
                    force = 2 * f[k]
                total = total + P.c[k][0] * torch.where(near[k], force, torch.zeros_like(force)).sum()
            drag.append(float(total))
    return {"drag": np.array(drag), **_planes(P, f, (nx, ny) if two else (nx, ny, nz))}


def _residual(u, before, window):
    return float(torch.sqrt(((u - before) ** 2).sum() / (u ** 2).sum()) / window)


def _exact_flow(case, seed, dev):
    w = _flow(case, seed)
    p = case["problem"]
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    shape = (nx, ny) if "nz" not in case else (nx, ny, nz)
    q = 9 if "nz" not in case else 19
    if p in ("rayleigh_benard", "natural_convection_3d"):
        side = ny if q == 9 else nx
        nu, alpha = 0.05, 0.05 / w["pr"]
        P = Plain(q, (True, False, True) if q == 9 else (False,) * 3, dev)
        t0 = _to(w["t0"], (nx, ny, nz), dev)
        f = P.per_q(P.wv, t0[None]).expand((q, nz, ny, nx)).clone()
        g = P.per_q(P.wv, t0[None]) * t0
        faces = {2: 1.0, 3: 0.0} if q == 9 else {0: 1.0, 1: 0.0}
        for _ in range(case["steps"]):
            f, g = P.thermal(f, g, 1 / (3 * nu + 0.5), 1 / (3 * alpha + 0.5), w["ra"] * nu * alpha / float(side) ** 3,
                             0.5, faces)
        t = g.sum(0)
        t1, t2 = (t[0, 0], t[0, 1]) if q == 9 else (t[1:-1, 1:-1, 0], t[1:-1, 1:-1, 1])
        number = float((-side * (-8 * 1.0 + 9 * t1 - t2) / 3.0).mean())
        return {**_planes(P, f, shape), "Temp": t.permute(2, 1, 0).reshape(shape).cpu().numpy(), "nu": number}
    om = 1 / (3 * w["nu"] + 0.5)
    sm = 1 / (3.0 / 16.0 / (3 * w["nu"]) + 0.5)
    if p in ("taylor_green_2d", "taylor_green_3d"):
        P = Plain(q, (True,) * 3, dev)
        fields = _vortex(case, w)
    elif p == "duct3d":
        P = Plain(q, (True, False, False), dev)
        fields = _swirl(case, w)
    else:
        P = Plain(q, (False, False, q == 9), dev)
        fields = (np.ones(shape),)
    fields = [_to(a, (nx, ny, nz), dev) for a in fields]
    u = torch.zeros((3, nz, ny, nx), dtype=torch.float64, device=dev)
    for k, a in enumerate(fields[1:]):
        u[k] = a
    f = P.feq(fields[0], u)
    del u, fields
    coll = "trt" if p == "taylor_green_3d" else case.get("collision", "bgk")
    res, before, check = [], None, case.get("check", 0)
    velocity = lambda f: (lambda rho, j: j / rho)(*P.moments(f))  # noqa: E731
    for n in range(case["steps"]):
        if check and n % check == 0:
            before = velocity(f)
        f = P.stream(f)
        if p == "cavity2d":
            P.lid2(f, w["u"])
        if p == "cavity3d":
            P.lid3(f, w["u"])
        if p == "duct3d":
            f = P.guo(f, om, w["force"])
        elif coll == "trt":
            f = P.trt(f, om, sm)
        else:
            f = P.mrt(f, om) if coll == "mrt" else P.bgk(f, om)
        if check and n % check == check - 1:
            res.append(_residual(velocity(f), before, check))
    out = _planes(P, f, shape, w["force"] if p == "duct3d" else None)
    return {"residual": np.array(res), **out} if check else out


def _exact_ensemble(case, seed, dev):
    n, nu = _ensemble(case, seed)
    P = Plain(9, (False, False, True), dev)
    at = np.concatenate([[0], np.cumsum(n.astype(np.int64) ** 2)])
    out = {k: np.zeros(at[-1]) for k in ("rho", "ux", "uy")}
    res = np.zeros(len(n))
    for side in np.unique(n):
        who = np.where(n == side)[0]
        om = torch.tensor(1 / (3 * nu[who] + 0.5), dtype=torch.float64, device=dev).reshape(-1, 1, 1, 1)
        sm = torch.tensor(1 / (3.0 / 16.0 / (3 * nu[who]) + 0.5), dtype=torch.float64, device=dev).reshape(-1, 1, 1, 1)
        f = P.wv.reshape(9, 1, 1, 1, 1).expand(9, len(who), 1, side, side).clone()
        for k in range(case["steps"]):
            if k == case["steps"] - 100:
                rho, j = P.moments(f)
                before = j / rho
            f = P.stream(f)
            P.lid2(f, 0.1)
            f = P.mrt(f, om) if case["collision"] == "mrt" else P.trt(f, om, sm) if case["collision"] == "trt" else P.bgk(f, om)
        rho, j = P.moments(f)
        u = j / rho
        for i, c in enumerate(who):
            res[c] = _residual(u[:, i], before[:, i], 100)
            for name, a in (("rho", rho[i]), ("ux", u[0, i]), ("uy", u[1, i])):
                out[name][at[c]:at[c + 1]] = a.reshape(-1).cpu().numpy()
    return {"steps": None, "residual": res, **out}


def _net_split(case, flat):
    hw = case["side"] // 8
    lat = hw * hw * 64
    shapes = [(2, 256), (256,), (256, lat), (lat,), (9 * 64, 64), (64,), (9 * 64, 32), (32,), (9 * 32, 3), (3,)]
    out, at = [], 0
    for s in shapes:
        k = int(np.prod(s))
        out.append(flat[at:at + k].reshape(s))
        at += k
    return out


def _net_forward(case, flat, x):
    p = _net_split(case, flat)
    silu = lambda z: z * torch.sigmoid(z)  # noqa: E731
    h = silu(silu(x @ p[0] + p[1]) @ p[2] + p[3])
    hw = case["side"] // 8
    h = h.reshape(-1, hw, hw, 64)
    for k in range(3):
        w, b = p[4 + 2 * k], p[5 + 2 * k]
        up = h.repeat_interleave(2, 1).repeat_interleave(2, 2)
        n = up.shape[1]
        pad = torch.nn.functional.pad(up, (0, 0, 1, 1, 1, 1))
        cols = torch.cat([pad[:, ky:ky + n, kx:kx + n] for ky in range(3) for kx in range(3)], dim=-1)
        h = (cols.reshape(-1, cols.shape[-1]) @ w + b).reshape(*cols.shape[:3], -1)
        h = silu(h) if k < 2 else h
    return h


def _shuffles(n, epochs, seed):
    """The epochs' permutations: Fisher–Yates on splitmix64 (Steele, Lea and Flood 2014)."""
    mask, s = (1 << 64) - 1, seed
    for _ in range(epochs):
        perm = list(range(n))
        for i in range(n - 1, 0, -1):
            s = (s + 0x9E3779B97F4A7C15) & mask
            z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            z ^= z >> 31
            k = z % (i + 1)
            perm[i], perm[k] = perm[k], perm[i]
        yield perm


def _exact_net(case, seed, dev):
    x, y = _net_inputs(case, seed)
    net = _net(case, seed)
    flat = torch.from_numpy(net.get_params().astype(np.float64)).to(dev)  # the weights it starts from
    net.close()
    xt = torch.from_numpy(x.astype(np.float64)).to(dev)
    if case["problem"] == "decoder":
        with torch.no_grad():
            return {"fields": np.concatenate([_net_forward(case, flat, xt[i:i + 32]).cpu().numpy()
                                              for i in range(0, len(x), 32)])}
    yt = torch.from_numpy(y).to(dev)
    m, v, t, loss = torch.zeros_like(flat), torch.zeros_like(flat), 0, []
    batch = case["batch"]
    for perm in _shuffles(len(x), case["epochs"], 5):
        loss = []
        for b in range(len(x) // batch):
            idx = torch.tensor(perm[b * batch:(b + 1) * batch], device=dev)
            w = flat.detach().clone().requires_grad_(True)
            e = ((_net_forward(case, w, xt[idx]) - yt[idx].double()) ** 2).mean()
            e.backward()
            g, t = w.grad, t + 1
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            flat = flat - 1e-3 * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
            loss.append(float(e))
    return {"loss": float(np.mean(loss)), "params": flat.cpu().numpy()}


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    p = case["problem"]
    if p in ("decoder", "training"):
        return _exact_net(case, seed, dev)
    if p == "ensemble":
        return _exact_ensemble(case, seed, dev)
    if p in ("cylinder", "sphere"):
        return _exact_channel(case, seed, dev)
    return _exact_flow(case, seed, dev)
