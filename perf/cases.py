"""The timed workloads of the framework: what a program asks of it through its
public entry points, with sizes from one small scene to the 64-scene batch.

Kinds of case (`kind`):
  rollout    Engine: upload a state, advance `steps` substeps, download it.
  batch      The same for many independent scenes in one engine.
  solve      solve_mls_mpm_3d, the drop-in substep, called `steps` times.
  phases3d   three_d.p2g / grid_op / g2p on caller grids, `steps` substeps.
  phases2d   two_d.p2g / grid_op / g2p on caller grids, `steps` substeps.
  bin        bin_particles: cell keys and their stable ordering.
  gradient   adjoint.rollout forward and backward: gradients of a loss on the
             final positions with respect to the initial velocities and E.
  train      One training step of the corrector network (forward, loss,
             backward, Adam).
  corrected  Engine with the learned corrector on, `steps` big steps.

Scenes are boxes of particles in the middle of a motion: a box has a mean
velocity, a velocity gradient (its affine matrices C agree with it) and a
smooth strain.  Particles come in arbitrary order, as a caller has them.
`exact` restates the step in FP64 with torch operations only.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

import femflow_amd
from femflow_amd import adjoint
from femflow_amd.corrector import CorrectorMLP
from femflow_amd.engine import Engine, MaterialSpec, SceneSpec, bin_particles
from femflow_amd.solvers.mpm import solve_mls_mpm_3d, three_d, two_d
from femflow_amd.solvers.mpm.particle import ParticleSet

ELASTIC, SNOW, WATER = 0, 1, 2
#        kind     E    nu   h     theta_c theta_s (water: bulk modulus)
TABLE = ((ELASTIC, 5e3, 0.2, 1.0, 2.5e-2, 7.5e-3), (SNOW, 5e3, 0.2, 10.0, 2.5e-2, 7.5e-3),
         (WATER, 1e4, 0.0, 1.0, 2.5e-2, 7.5e-3))
CORNERS = ((0.15, 0.45, 0.40), (0.42, 0.20, 0.40), (0.65, 0.45, 0.40))
GRAVITY = -9.8
M_REF_OF = 1.0  # rho: mass of a full cell is rho dx^3
DTYPES = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # one small body on a coarse grid: an interactive scene, launch-bound
        dict(name="rollout_4k_64", kind="rollout", n=4096, res=64, mats="elastic", steps=64, sticky=False, textbook=False),
        # a mid-size snow scene, odd count and grid, sticky walls, textbook stress
        dict(name="rollout_snow_100k_90", kind="rollout", n=100_003, res=90, mats="snow", steps=48, sticky=True,
             textbook=True),
        # the headline configuration: three materials at 128^3
        dict(name="rollout_1m_128", kind="rollout", n=1 << 20, res=128, mats="three", steps=64, sticky=False,
             textbook=False),
        # the batched configuration: 64 scenes of 4k-256k particles, 64^3..128^3
        dict(name="batch_64_scenes", kind="batch", scenes=64, n_lo=4096, n_hi=262144, steps=24, spec_seed=0),
        # a program that keeps the reference's one-call-per-substep loop, FP32
        dict(name="solve_f32_131k_64", kind="solve", n=1 << 17, res=64, steps=8, dtype="f32"),
        # the same loop in the reference's own precision
        dict(name="solve_f64_131k_64", kind="solve", n=1 << 17, res=64, steps=4, dtype="f64"),
        # a program that calls the three phases itself, snow, FP32, odd sizes
        dict(name="phases3d_snow_200k_96", kind="phases3d", n=200_001, res=96, steps=4, dtype="f32", model="snow"),
        # the 2D configuration (8,192 particles, 128^2, FP64), 20 of its substeps
        dict(name="phases2d_8k_128", kind="phases2d", n=8192, res=128, steps=20, dtype="f64", model="neo_hookean"),
        # standalone binning of the headline positions
        dict(name="bin_1m_128", kind="bin", n=1 << 20, res=128, dim=3, layout="blocked"),
        # the differentiable rollout: 2^17 particles, 64^3
        dict(name="gradient_131k_64", kind="gradient", n=1 << 17, res=64, steps=60),
        # one mini-batch of the corrector's training
        dict(name="train_32k_rows", kind="train", rows=32768),
        # one judged window of the corrector: a big step (8 dt) of the three cubes
        # from a given state (at finer grids a big step lies so far beyond the
        # stability limit that its light nodes amplify every rounding)
        dict(name="corrected_262k_80", kind="corrected", n=1 << 18, res=80, steps=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("rollout", "rollout", "rollout", "batch", "solve", "phases3d", "phases2d", "bin", "gradient",
                       "train", "corrected"))
    if kind == "rollout":
        n = _log_int(rng, 4096, 1 << 21)
        # grids from a few to about a hundred particles per occupied cell
        res = min(256, max(32, int(round((n / _log_int(rng, 2, 60)) ** (1 / 3) / 0.25))))
        return dict(kind=kind, n=n, res=res, mats=rng.choice(("elastic", "snow", "water", "three")),
                    steps=rng.randint(8, 48), sticky=rng.random() < 0.3, textbook=rng.random() < 0.3)
    if kind == "batch":
        lo = _log_int(rng, 1024, 16384)
        return dict(kind=kind, scenes=rng.randint(2, 48), n_lo=lo, n_hi=lo * rng.randint(2, 12),
                    steps=rng.randint(8, 24), spec_seed=rng.randint(1, 10 ** 6))
    if kind == "solve":
        dtype = rng.choice(("f32", "f64"))
        return dict(kind=kind, n=_log_int(rng, 2048, 1 << 19), res=rng.randint(32, 128), steps=rng.randint(2, 6),
                    dtype=dtype)
    if kind == "phases3d":
        return dict(kind=kind, n=_log_int(rng, 1024, 1 << 19), res=rng.randint(32, 128), steps=rng.randint(1, 4),
                    dtype=rng.choice(("f32", "f64")), model=rng.choice(("neo_hookean", "snow")))
    if kind == "phases2d":
        return dict(kind=kind, n=_log_int(rng, 1024, 1 << 19), res=rng.randint(48, 512), steps=rng.randint(4, 20),
                    dtype=rng.choice(("f32", "f64")), model=rng.choice(("neo_hookean", "snow")))
    if kind == "bin":
        return dict(kind=kind, n=_log_int(rng, 4096, 1 << 22), res=rng.randint(48, 256), dim=rng.choice((2, 3, 3)),
                    layout=rng.choice(("blocked", "rowmajor")))
    if kind == "gradient":
        return dict(kind=kind, n=_log_int(rng, 4096, 1 << 18), res=rng.randint(32, 96), steps=rng.randint(10, 60))
    if kind == "train":
        return dict(kind=kind, rows=_log_int(rng, 1024, 131072))
    return dict(kind=kind, n=_log_int(rng, 1 << 15, 1 << 19), res=rng.randint(48, 80), steps=1)


# --------------------------------------------------------------- inputs ----
def _batch_specs(case):
    """(n, res, material, side, corner) of each scene; fixed by the case."""
    rng = np.random.default_rng(case["spec_seed"])
    out = []
    for _ in range(case["scenes"]):
        n = int(round(math.exp(rng.uniform(math.log(case["n_lo"]), math.log(case["n_hi"])))))
        res, mat, side = int(rng.integers(64, 129)), int(rng.integers(0, 3)), float(rng.uniform(0.1, 0.3))
        out.append((n, res, mat, side, tuple(float(c) for c in rng.uniform(0.1, 0.9 - side, size=3))))
    return out


def _boxes(case):
    """[(n, scene, material, side, corner)] of a 3D case."""
    if case["kind"] == "batch":
        return [(n, i, mat, side, corner) for i, (n, _, mat, side, corner) in enumerate(_batch_specs(case))]
    n, mats = case["n"], case.get("mats", "elastic")
    if case["kind"] == "corrected":
        mats = "three"
    if mats == "three":
        per = n // 3
        return [(n - 2 * per if k == 0 else per, 0, k, 0.2, CORNERS[k]) for k in range(3)]
    return [(n, 0, {"elastic": ELASTIC, "snow": SNOW, "water": WATER}[mats], 0.2, (0.4, 0.4, 0.4))]


def _scene_res(case):
    return [s[1] for s in _batch_specs(case)] if case["kind"] == "batch" else [case["res"]]


def _volumes(case):
    """Particle volume of each scene (its boxes filled at unit density)."""
    vol = [0.0] * len(_scene_res(case))
    for n, scene, _, side, _ in _boxes(case):
        vol[scene] = side ** 3 / n
    return vol


def _dt(case):
    return {"solve": 1e-4, "phases3d": 1e-4, "gradient": 1e-4, "phases2d": 1e-4, "corrected": 4e-4}.get(case["kind"], 5e-5)


def _gradient_of_motion(host, d, size):
    """A velocity gradient that turns and shears a body without compressing it
    (an impact at metres per second over some centimetres)."""
    M = host.normal(0.0, size, (d, d))
    sym = 0.5 * (M + M.T)
    return 0.8 * 0.5 * (M - M.T) + 0.4 * (sym - np.trace(sym) / d * np.eye(d))


def _state3d(case, seed, dtype=torch.float32):
    """The particles of a 3D case in arbitrary order."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed * 7919 + 17)
    host = np.random.default_rng(seed)
    rand = lambda *s: torch.rand(*s, generator=g, device=dev, dtype=torch.float64)  # noqa: E731
    parts, vols = [], _volumes(case)
    for n, scene, mat, side, corner in _boxes(case):
        kind, E, nu, h, tc, ts = TABLE[mat]
        u = rand(n, 3)
        x = torch.tensor(corner, dtype=torch.float64, device=dev) + side * u
        B = torch.tensor(_gradient_of_motion(host, 3, 40.0), device=dev)
        v0 = torch.tensor(host.normal(0.0, 0.5, 3), device=dev)
        v = v0 + side * (u - 0.5) @ B.T
        wave = torch.sin(2 * math.pi * u.roll(1, 1) + torch.tensor(host.uniform(0, 6.28, 3), device=dev))
        I3 = torch.eye(3, dtype=torch.float64, device=dev)
        Jp = torch.ones(n, dtype=torch.float64, device=dev)
        if kind == WATER:
            F = (1 + 0.002 * wave[:, 0])[:, None, None] * I3
            mu, lam = 0.0, E
        else:
            G = torch.tensor(host.normal(0.0, 0.001, (3, 3)), device=dev)
            F = I3 + G + 0.001 * wave[:, :, None] * torch.tensor(host.normal(0.0, 1.0, 3), device=dev)
            mu, lam = E / (2 * (1 + nu)), E * nu / ((1 + nu) * (1 - 2 * nu))
            if kind == SNOW:
                Jp = 1 - 0.03 * u[:, 0]
        full = lambda a: torch.full((n,), a, dtype=torch.float64, device=dev)  # noqa: E731
        if case["kind"] == "gradient":  # a field of stiffnesses
            mu, lam = 1.0, 1.0
        parts.append(dict(x=x, v=v, F=F, C=B.expand(n, 3, 3), Jp=Jp, mass=full(vols[scene]), mu0=full(mu),
                          lam0=full(lam), material=full(mat).int(), scene=full(scene).int()))
    perm = torch.randperm(sum(len(p["x"]) for p in parts), generator=g, device=dev)
    out = {k: torch.cat([p[k] for p in parts])[perm] for k in parts[0]}
    return {k: (a.contiguous() if a.dtype == torch.int32 else a.to(dtype).contiguous()) for k, a in out.items()}


def _state2d(case, seed, dtype):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed * 7919 + 17)
    host = np.random.default_rng(seed)
    n = case["n"]
    u = torch.rand(n, 2, generator=g, device=dev, dtype=torch.float64)
    x = torch.tensor((0.4, 0.6), dtype=torch.float64, device=dev) + 0.2 * u
    B = torch.tensor(_gradient_of_motion(host, 2, 40.0), device=dev)
    v = torch.tensor(host.normal(0.0, 0.5, 2), device=dev) + 0.2 * (u - 0.5) @ B.T
    wave = torch.sin(2 * math.pi * u.roll(1, 1))
    F = torch.eye(2, dtype=torch.float64, device=dev) + 0.004 * wave[:, :, None] * torch.tensor(
        host.normal(0.0, 1.0, 2), device=dev)
    s = dict(x=x, v=v, F=F, C=B.expand(n, 2, 2), Jp=1 - 0.03 * u[:, :1])
    return {k: a.to(dtype).contiguous() for k, a in s.items()}


def _train_inputs(case, seed):
    """Features with the layout of the network (27 neighbours x 13 values:
    mass, momentum, F - I), targets and row weights."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed * 7919 + 17)
    rows = case["rows"]
    f = torch.randn(rows, 27, 13, generator=g, device=dev)
    f[:, :, 0] = f[:, :, 0].abs()
    f[:, :, 1:4] *= 0.5
    f[:, :, 4:] *= 0.02
    X = torch.zeros(rows, 352, dtype=torch.bfloat16, device=dev)
    X[:, :351] = f.reshape(rows, 351).to(torch.bfloat16)
    T = 0.1 * torch.randn(rows, 3, generator=g, device=dev)
    w = 0.1 + torch.rand(rows, generator=g, device=dev)
    host = np.random.default_rng(seed)
    params = []
    for o, i in ((128, 351), (128, 128), (3, 128)):
        params += [host.uniform(-1, 1, o * i) / math.sqrt(i), host.uniform(-1, 1, o) / math.sqrt(i)]
    return X, T, w, torch.from_numpy(np.concatenate(params).astype(np.float32))


def _network_file():
    return os.path.join(os.path.dirname(femflow_amd.__file__), "data", "corrector_c5.npz")


def _positions(case, seed):
    """Headline-like positions (three boxes) in 2D or 3D, FP32, arbitrary order."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed * 7919 + 17)
    n, d = case["n"], case["dim"]
    c = torch.tensor(CORNERS, device=dev)[torch.randint(0, 3, (n,), generator=g, device=dev), :d]
    return (c + 0.2 * torch.rand(n, d, generator=g, device=dev)).contiguous()


# -------------------------------------------------------------- prepare ----
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("rollout", "batch", "corrected"):
        s = _state3d(case, seed)
        dt, vols = _dt(case), _volumes(case)
        scenes = [SceneSpec(res=r, dt=dt, gravity=GRAVITY, volume=vol,
                            boundary="sticky" if case.get("sticky") else "reference",
                            quirks="textbook" if case.get("textbook") else "reference")
                  for r, vol in zip(_scene_res(case), vols)]
        eng = Engine(scenes, [MaterialSpec(("elastic", "snow", "water")[k], h, tc, ts) for k, _, _, h, tc, ts in TABLE],
                     n_max=len(s["x"]))
        if kind == "corrected":
            net = CorrectorMLP.load(_network_file())
            eng.set_corrector(net.params, M_REF_OF / case["res"] ** 3, 1.0)
        out = {k: torch.empty_like(s[k]) for k in ("x", "v", "F", "C", "Jp")}
        return dict(kind=kind, s=s, eng=eng, out=out, steps=case["steps"], scene=s["scene"] if kind == "batch" else None)
    if kind in ("solve", "phases3d"):
        s = _state3d(case, seed, DTYPES[case["dtype"]])
        s["Jp"] = s["Jp"].reshape(-1, 1)
        cur = {k: s[k].clone() for k in ("x", "v", "F", "C", "Jp")}
        return dict(kind=kind, s=s, cur=cur, case=case, particles=ParticleSet(cur["x"], s["mass"], s["mu0"], s["lam0"]),
                    volume=_volumes(case)[0])
    if kind == "phases2d":
        s = _state2d(case, seed, DTYPES[case["dtype"]])
        return dict(kind=kind, s=s, cur={k: a.clone() for k, a in s.items()}, case=case)
    if kind == "bin":
        return dict(kind=kind, x=_positions(case, seed), case=case)
    if kind == "gradient":
        s = _state3d(case, seed)
        E, target = _gradient_extras(case, seed, s)
        cfg = adjoint.RolloutConfig(res=case["res"], dt=_dt(case), volume=_volumes(case)[0], nsteps=case["steps"])
        return dict(kind=kind, s=s, v0=s["v"].clone().requires_grad_(True), E=E.requires_grad_(True), target=target,
                    cfg=cfg)
    X, T, w, params = _train_inputs(case, seed)
    return dict(kind=kind, X=X, T=T, w=w, net=CorrectorMLP(params=params))


def _gradient_extras(case, seed, s):
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 18)
    E = 1e3 + 9e3 * torch.rand(case["n"], generator=g, device="cuda")
    target = s["x"] + 0.02 * torch.randn(case["n"], 3, generator=g, device="cuda")
    return E, target


# ------------------------------------------------------------------ run ----
def run(st):
    kind = st["kind"]
    if kind in ("rollout", "batch", "corrected"):
        s, eng, out = st["s"], st["eng"], st["out"]
        eng.upload(s["x"], s["v"], s["F"], s["C"], s["Jp"], s["mass"], s["mu0"], s["lam0"], s["material"], st["scene"])
        eng.run(st["steps"])
        eng.download(out["x"], out["v"], out["F"], out["C"], out["Jp"])
        return out
    if kind == "bin":
        c = st["case"]
        return bin_particles(st["x"], c["res"], float(c["res"]), c["layout"])
    if kind == "gradient":
        mu0, lam0 = adjoint.lame_from_E(st["E"], 0.2)
        xT, vT = adjoint.rollout(st["s"]["x"], st["v0"], mu0, lam0, st["s"]["mass"], st["cfg"])
        loss = ((xT - st["target"]) ** 2).sum(1).mean()
        gv, gE = torch.autograd.grad(loss, (st["v0"], st["E"]))
        return dict(loss=loss.detach(), x=xT.detach(), v=vT.detach(), v0_grad=gv, E_grad=gE)
    if kind == "train":
        net = st["net"]
        loss = net.train_step(st["X"], st["T"], st["w"], lr=1e-3)
        return dict(loss=loss, grads=net.grads, params=net.params)
    # the remaining kinds mutate the caller's arrays: start from the initial state
    s, cur, c = st["s"], st["cur"], st["case"]
    for k, a in cur.items():
        a.copy_(s[k])
    res, dt = c["res"], _dt(c)
    dx, inv_dx, r1, dtype = 1.0 / res, float(res), res + 1, DTYPES[c["dtype"]]
    for _ in range(c["steps"]):
        if kind == "solve":
            solve_mls_mpm_3d(res, inv_dx, 1.0, dx, dt, st["volume"], GRAVITY, st["particles"], cur["v"], cur["F"],
                             cur["C"], cur["Jp"])
        elif kind == "phases3d":
            gv = torch.zeros((r1, r1, r1, 3), dtype=dtype, device="cuda")
            gm = torch.zeros((r1, r1, r1, 1), dtype=dtype, device="cuda")
            args = (st["particles"], cur["v"], cur["F"], cur["C"], cur["Jp"])
            three_d.p2g(inv_dx, _hardening(c), dx, dt, st["volume"], gv, gm, *args, model=c["model"])
            three_d.grid_op(res, dx, dt, GRAVITY, gv, gm)
            three_d.g2p(inv_dx, dt, gv, *args, model=c["model"])
        else:
            mu0, lam0, vol = 1e3 / 2.4, 1e3 * 0.2 / (1.2 * 0.6), (0.5 * dx) ** 2
            gv = torch.zeros((r1, r1, 2), dtype=dtype, device="cuda")
            gm = torch.zeros((r1, r1), dtype=dtype, device="cuda")
            args = (cur["x"], cur["v"], cur["F"], cur["C"], cur["Jp"])
            two_d.p2g(inv_dx, _hardening(c), mu0, lam0, vol, dx, dt, vol, gv, gm, *args, model=c["model"])
            two_d.grid_op(res, dt, GRAVITY, gv, gm)
            two_d.g2p(inv_dx, dt, gv, *args, model=c["model"])
    return dict(cur)


def _hardening(case):
    return 10.0 if case.get("model") == "snow" else 1.0


# ----------------------------------------------------------------- work ----
def _occupied_nodes(case):
    """Grid nodes that a substep has to touch: those of the occupied boxes
    with a one-cell margin on each side."""
    res = _scene_res(case)
    return sum((side * res[scene] + 3) ** 3 for _, scene, _, side, _ in _boxes(case))


def work(case):
    """Each input once, each output once, and the arithmetic of the step:
    about 2,600 operations per particle-substep in 3D (stress, 27-node
    scatter and gather), 700 in 2D."""
    kind = case["kind"]
    if kind == "bin":
        return dict(bytes=case["n"] * (4.0 * case["dim"] + 8), flops=0.0)
    if kind == "train":
        macs = 351 * 128 + 128 * 128 + 128 * 3
        # features, targets, weights; parameters, moments and gradients
        return dict(bytes=case["rows"] * (704.0 + 12 + 4) + 4.0 * macs * 7, flops=case["rows"] * 2.0 * (3 * macs - 351 * 128))
    n = sum(b[0] for b in _boxes(case)) if kind != "phases2d" else case["n"]
    steps = case["steps"]
    if kind == "phases2d":
        size = 8 if case["dtype"] == "f64" else 4
        nodes = (0.2 * case["res"] + 3) ** 2
        return dict(bytes=steps * size * (n * 26.0 + nodes * 11), flops=steps * n * 700.0)
    nodes = _occupied_nodes(case)
    if kind in ("solve", "phases3d"):
        size = 8 if case["dtype"] == "f64" else 4
        return dict(bytes=steps * size * (n * 53.0 + nodes * 14), flops=steps * n * 2600.0)
    if kind == "gradient":  # forward substep, then its reverse: state and adjoints in and out
        return dict(bytes=steps * (n * (212.0 + 96 + 2 * 100 + 16) + nodes * 100.0), flops=steps * n * 9000.0)
    extra_b = extra_f = 0.0
    if kind == "corrected":  # node features (13 values) and the network at every node with mass
        extra_b, extra_f = nodes * 13 * 8.0 + n * 48, nodes * 2.0 * (351 * 128 + 128 * 128 + 128 * 3)
    return dict(bytes=steps * (n * 212.0 + nodes * 56 + extra_b) + n * 212.0, flops=steps * (n * 2600.0 + extra_f))


# ---------------------------------------------------------------- exact ----
def _polar(F):
    """Rotation factor of F (d = 3) by Newton's iteration."""
    X = F
    for _ in range(9):
        X = 0.5 * (X + _cof(X) / _det(X)[..., None, None])
    return X


def _cof(X):
    a, b, c = X[..., 0, :], X[..., 1, :], X[..., 2, :]
    return torch.stack((torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)), -2)


def _det(X):
    if X.shape[-1] == 2:
        return X[..., 0, 0] * X[..., 1, 1] - X[..., 0, 1] * X[..., 1, 0]
    return (X[..., 0, :] * torch.linalg.cross(X[..., 1, :], X[..., 2, :])).sum(-1)


def _eig_sym(A):
    """Eigenvalues (…, d) and eigenvectors of symmetric A by Jacobi sweeps."""
    d = A.shape[-1]
    V = torch.eye(d, dtype=A.dtype, device=A.device).expand(A.shape).clone()
    for _ in range(6 if d == 3 else 1):
        for p, q in ((0, 1), (0, 2), (1, 2)) if d == 3 else ((0, 1),):
            apq, diff = A[..., p, q], A[..., q, q] - A[..., p, p]
            ang = 0.5 * torch.atan2(2 * apq, diff)
            R = torch.eye(d, dtype=A.dtype, device=A.device).expand(A.shape).clone()
            R[..., p, p] = R[..., q, q] = torch.cos(ang)
            R[..., p, q], R[..., q, p] = torch.sin(ang), -torch.sin(ang)
            A = R.transpose(-1, -2) @ A @ R
            V = V @ R
    return torch.diagonal(A, dim1=-2, dim2=-1), V


def _clamp_stretch(F, tc, ts):
    """F with its singular values clamped to [1 - tc, 1 + ts]."""
    e, V = _eig_sym(F.transpose(-1, -2) @ F)
    s = e.sqrt()
    r = s.clamp(1 - tc, 1 + ts) / s
    return F @ ((V * r[..., None, :]) @ V.transpose(-1, -2))


class _Exact:
    """FP64 substeps of the reference step on dense grids, 2D or 3D."""

    def __init__(self, d, res, dt, volume, sticky=False, textbook=False, scene=None, differentiable=False):
        dev = torch.device("cuda")
        f = lambda a: torch.tensor(a, dtype=torch.float64, device=dev)  # noqa: E731
        self.d, self.dt, self.textbook, self.sticky = d, dt, textbook, sticky
        sizes = [(r + 1) ** d for r in res]
        off = np.concatenate(([0], np.cumsum(sizes)[:-1]))
        self.nodes = int(sum(sizes))
        many = scene is not None
        pick = lambda a: a[scene.long()] if many else a[0]  # noqa: E731
        self.res_p, self.off_p = pick(f(np.array(res, float))), pick(torch.tensor(off, device=dev))
        self.vol_p = pick(f(np.array(volume, float)))
        self.inv_dx = self.res_p
        self.coords, self.res_n = [], []
        for r in res:
            ax = torch.arange(r + 1, device=dev, dtype=torch.int16)
            self.coords.append(torch.stack(torch.meshgrid(*([ax] * d), indexing="ij"), -1).reshape(-1, d))
            self.res_n.append(torch.full(((r + 1) ** d,), r, dtype=torch.int16, device=dev))
        self.coords, self.res_n = torch.cat(self.coords), torch.cat(self.res_n)
        self.offsets = [tuple(int(c) for c in o) for o in np.ndindex(*([3] * d))]
        self.differentiable = differentiable
        self.correct = None

    def weights(self, x):
        s = x * (self.inv_dx[:, None] if self.inv_dx.dim() else self.inv_dx)
        base = (s.detach() - 0.5).trunc()
        fx = s - base
        return base.long(), fx, (0.5 * (1.5 - fx) ** 2, 0.75 - (fx - 1) ** 2, 0.5 * (fx - 0.5) ** 2)

    def stress(self, F, mu, lam, water):
        J = _det(F)
        eye = torch.eye(self.d, dtype=torch.float64, device=F.device)
        if self.d == 3:
            PF = 2 * mu[:, None, None] * ((F - _polar(F)) @ F.transpose(-1, -2))
        else:
            a, b = F[:, 0, 0] + F[:, 1, 1], F[:, 1, 0] - F[:, 0, 1]
            sc = 1 / ((a * a + b * b).sqrt() + (0.0 if self.textbook else 1e-10))
            R = torch.stack((a * sc, -b * sc, b * sc, a * sc), -1).reshape(-1, 2, 2)
            PF = 2 * mu[:, None, None] * ((F - R) @ F.transpose(-1, -2))
        spread = torch.ones_like(eye)
        if self.textbook:
            spread = eye
        elif water is not None:
            spread = torch.where(water[:, None, None], eye, spread)
        return PF + (lam * (J - 1) * J)[:, None, None] * spread

    def node(self, base, o):
        r1 = (self.res_p + 1).long()
        idx = base[:, 0] + o[0]
        for a in range(1, self.d):
            idx = idx * r1 + base[:, a] + o[a]
        return idx + self.off_p

    def p2g(self, x, v, F, C, mass, mu, lam, water):
        base, fx, w = self.weights(x)
        dx = 1 / self.inv_dx
        k = -(self.dt * self.vol_p) * 4 * self.inv_dx ** 2
        A = (k[:, None, None] if k.dim() else k) * self.stress(F, mu, lam, water) + mass[:, None, None] * C
        mom = torch.zeros(self.nodes, self.d + 1, dtype=torch.float64, device=x.device)
        for o in self.offsets:
            wt = self.weight(w, o)
            dp = (torch.tensor(o, dtype=torch.float64, device=x.device) - fx) * (dx[:, None] if dx.dim() else dx)
            val = mass[:, None] * v + (A @ dp[:, :, None])[:, :, 0]
            val = wt[:, None] * torch.cat((val, mass[:, None]), 1)
            mom = mom.index_add(0, self.node(base, o), val) if self.differentiable else mom.index_add_(
                0, self.node(base, o), val)
        return mom

    def weight(self, w, o):
        wt = w[o[0]][:, 0]
        for a in range(1, self.d):
            wt = wt * w[o[a]][:, a]
        return wt

    def walls(self, v):
        I, R = self.coords, self.res_n
        if self.sticky:
            stop = ((I < 3) | (I > (R - 3)[:, None])).any(1)
            return torch.where(stop[:, None], 0.0, v)
        if self.d == 3:
            return torch.where((I < 1) | (I >= (R - 1)[:, None]), 0.0, v)
        p = I.double() / R.double()[:, None]
        stop = (p[:, 0] < 0.05) | (p[:, 0] > 0.95) | (p[:, 1] > 0.95)
        v = torch.where(stop[:, None], 0.0, v)
        return torch.stack((v[:, 0], torch.where(p[:, 1] < 0.05, v[:, 1].clamp(min=0.0), v[:, 1])), 1)

    def grid(self, mom):
        m = mom[:, self.d]
        has = m > 0
        v = mom[:, :self.d] / torch.where(has, m, 1.0)[:, None]
        g = torch.zeros(self.d, dtype=torch.float64, device=v.device)
        g[1] = self.dt * GRAVITY
        v = torch.where(has[:, None], v + g, 0.0)
        if self.d == 3:
            self.lim = (0.9 / self.dt / self.res_n.double())[:, None]
            v = torch.minimum(torch.maximum(v, -self.lim), self.lim)
        return self.walls(v)

    def g2p(self, x, v_grid):
        base, fx, w = self.weights(x)
        v = torch.zeros_like(x)
        C = torch.zeros(*x.shape, self.d, dtype=torch.float64, device=x.device)
        for o in self.offsets:
            g = self.weight(w, o)[:, None] * v_grid[self.node(base, o)]
            v = v + g
            dp = torch.tensor(o, dtype=torch.float64, device=x.device) - fx
            C = C + g[:, :, None] * dp[:, None, :]
        c4 = 4 * self.inv_dx
        C = (c4[:, None, None] if c4.dim() else c4) * C
        return x + self.dt * v, v, C

    def step(self, s, mats):
        """One substep of state s (x, v, F, C, Jp); mats: mass, mu0, lam0,
        material masks (snow, water; None = no particle) and the snow law."""
        snow, water, h, h_snow, tc, ts = (mats[k] for k in ("snow", "water", "h", "h_snow", "tc", "ts"))
        e = torch.full_like(s["Jp"], h)
        if snow is not None:
            e = torch.where(snow, torch.exp(h_snow * (1 - s["Jp"])), e)
        mu, lam = mats["mu0"] * e, mats["lam0"] * e
        if water is not None:
            mu, lam = torch.where(water, 0.0, mu), torch.where(water, mats["lam0"], lam)
        mom = self.p2g(s["x"], s["v"], s["F"], s["C"], mats["mass"], mu, lam, water)
        vg = self.grid(mom)
        if self.correct is not None:
            vg = self.correct(self, s, mats, mom, vg)
        x, v, C = self.g2p(s["x"], vg)
        eye = torch.eye(self.d, dtype=torch.float64, device=x.device)
        F = (eye + self.dt * C) @ s["F"]
        Jp = s["Jp"]
        if mats["project"] is not None:  # the snow particles
            i = mats["project"]
            old = _det(F[i])
            Fs = _clamp_stretch(F[i], tc, ts)
            Jp = Jp.clone()
            Jp[i] = (Jp[i] * old / (_det(Fs) + 1e-10)).clamp(0.6, 20)
            F = F.index_copy(0, i, Fs)
        elif self.d == 2:
            J = _det(F)
            Jp = (Jp * J / (J + 1e-10)).clamp(0.6, 20)
        if water is not None:
            J = _det(F)
            F = torch.where(water[:, None, None], (J.sign() * J.abs() ** (1 / 3))[:, None, None] * eye, F)
        return dict(x=x, v=v, F=F, C=C, Jp=Jp)


def _correction(case):
    """The learned corrector's node velocities in FP64."""
    with np.load(_network_file(), allow_pickle=False) as f:
        p = torch.from_numpy(f["params"].astype(np.float64)).cuda()
    (W1, b1, W2, b2, W3, b3) = _unpack(p)
    m_ref, r1 = M_REF_OF / case["res"] ** 3, case["res"] + 1

    def apply(ex, s, mats, mom, vg):
        base, _, _ = ex.weights(s["x"])
        cell = torch.zeros(ex.nodes, 10, dtype=torch.float64, device="cuda")
        vals = mats["mass"][:, None] * torch.cat((torch.ones_like(s["Jp"])[:, None], s["F"].reshape(-1, 9)), 1)
        cell.index_add_(0, ex.node(base, (0, 0, 0)), vals)
        feat = torch.zeros(ex.nodes, 13, dtype=torch.float64, device="cuda")
        has, full = mom[:, 3] > 0, cell[:, 0] > 0
        feat[has, 0] = mom[has, 3] / m_ref
        feat[has, 1:4] = mom[has, :3] / m_ref
        feat[full, 4:] = cell[full, 1:] / cell[full, :1] - torch.eye(3, dtype=torch.float64, device="cuda").reshape(9)
        pad = torch.nn.functional.pad(feat.reshape(r1, r1, r1, 13), (0, 0, 1, 1, 1, 1, 1, 1))
        ids = has.nonzero()[:, 0]
        I = ex.coords[ids].long()
        rows = torch.cat([pad[I[:, 0] + a, I[:, 1] + b, I[:, 2] + c] for a in range(3) for b in range(3)
                          for c in range(3)], 1)
        y = ((rows @ W1.T + b1).relu() @ W2.T + b2).relu() @ W3.T + b3
        gate = (mom[ids, 3] / (0.25 * m_ref)).clamp(max=1.0)
        out = vg.clone()
        out[ids] = torch.minimum(torch.maximum(out[ids] + gate[:, None] * y, -ex.lim[ids]), ex.lim[ids])
        return ex.walls(out)

    return apply


def _unpack(p):
    out, at = [], 0
    for o, i in ((128, 351), (128, 128), (3, 128)):
        out += [p[at:at + o * i].reshape(o, i), p[at + o * i:at + o * i + o]]
        at += o * i + o
    return out


def _exact_train(case, seed):
    X, T, w, params = _train_inputs(case, seed)
    p = params.double().cuda().requires_grad_(True)
    W1, b1, W2, b2, W3, b3 = _unpack(p)
    y = ((X[:, :351].double() @ W1.T + b1).relu() @ W2.T + b2).relu() @ W3.T + b3
    w = w.double()
    loss = (w[:, None] * (y - T.double()) ** 2).sum() / w.sum()
    g, = torch.autograd.grad(loss, p)
    step = 1e-3 * g / (g.abs() + 1e-8)
    return dict(loss=loss.detach().reshape(1), grads=g, params=(p - step).detach())


def _exact_gradient(case, seed):
    s32 = _state3d(case, seed)
    E, target = _gradient_extras(case, seed, s32)
    n, nu = case["n"], 0.2
    ex = _Exact(3, [case["res"]], _dt(case), _volumes(case), differentiable=True)
    mass = s32["mass"].double()
    mu, lam = E.double() / (2 * (1 + nu)), E.double() * nu / ((1 + nu) * (1 - 2 * nu))

    def step(x, v, F, C, mu, lam):
        vg = ex.grid(ex.p2g(x, v, F, C, mass, mu, lam, None))
        x, v, C = ex.g2p(x, vg)
        return x, v, (torch.eye(3, dtype=torch.float64, device="cuda") + ex.dt * C) @ F, C

    eye = torch.eye(3, dtype=torch.float64, device="cuda").expand(n, 3, 3)
    cur = (s32["x"].double(), s32["v"].double(), eye, torch.zeros_like(eye))
    states = []
    with torch.no_grad():
        for _ in range(case["steps"]):
            states.append(cur)
            cur = step(*cur, mu, lam)
    diff = cur[0] - target.double()
    bar = [2 * diff / n] + [torch.zeros_like(a) for a in cur[1:]]
    gmu, glam = torch.zeros_like(mu), torch.zeros_like(lam)
    for st in reversed(states):
        ins = [a.detach().clone().requires_grad_(True) for a in (*st, mu, lam)]
        got = torch.autograd.grad(step(*ins), ins, grad_outputs=bar)
        bar, gmu, glam = list(got[:4]), gmu + got[4], glam + got[5]
    gE = gmu / (2 * (1 + nu)) + glam * nu / ((1 + nu) * (1 - 2 * nu))
    return dict(loss=(diff ** 2).sum(1).mean(), x=cur[0], v=cur[1], v0_grad=bar[1], E_grad=gE)


def exact(case, seed):
    kind = case["kind"]
    if kind == "bin":
        return None  # whole numbers
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "gradient":
        return _exact_gradient(case, seed)
    if kind == "phases2d":
        dtype = DTYPES[case["dtype"]]
        s = _state2d(case, seed, dtype)
        n, vol, ids = case["n"], (0.5 / case["res"]) ** 2, torch.arange(case["n"], device="cuda")
        full = lambda a: torch.full((n,), a, dtype=torch.float64, device="cuda")  # noqa: E731
        mats = dict(mass=full(vol), mu0=full(1e3 / 2.4), lam0=full(1e3 * 0.2 / (1.2 * 0.6)))
        ex = _Exact(2, [case["res"]], _dt(case), [vol])
    else:
        s = _state3d(case, seed, DTYPES[case.get("dtype", "f32")])
        mats = {k: s[k].double() for k in ("mass", "mu0", "lam0")}
        ex = _Exact(3, _scene_res(case), _dt(case), _volumes(case), sticky=case.get("sticky", False),
                    textbook=case.get("textbook", False), scene=s["scene"] if kind == "batch" else None)
        ids = torch.arange(len(s["x"]), device="cuda")
        if kind == "corrected":
            ex.correct = _correction(case)
    if kind in ("rollout", "batch", "corrected"):
        snow, water = s["material"] == SNOW, s["material"] == WATER
        project = snow.nonzero()[:, 0]
        mats.update(snow=snow, water=water, h=1.0, h_snow=TABLE[SNOW][3], project=project if len(project) else None)
    else:
        law = case.get("model") == "snow"
        mats.update(snow=torch.ones_like(ids, dtype=torch.bool) if law else None, water=None, h=1.0,
                    h_snow=_hardening(case), project=ids if law else None)
    mats.update(tc=2.5e-2, ts=7.5e-3)
    cur = {k: s[k].double() for k in ("x", "v", "F", "C", "Jp")}
    cur["Jp"] = cur["Jp"].reshape(-1)
    for _ in range(case["steps"]):
        cur = ex.step(cur, mats)
    cur["Jp"] = cur["Jp"].reshape(s["Jp"].shape)
    return cur
