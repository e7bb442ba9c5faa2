"""Performance cases: the lattice updates, gradients and diagnostics that a
program built on this framework runs, through its public entry points.

Families (`kind` of a case):
- ``box``: periodic A-A steps, map-free: Taylor-Green and turbulence boxes, in
  every storage form and with every collision operator;
- ``channel``: steps with a geometry map: a duct with inlet, outlet and walls,
  or a channel driven by a body force between two walls, with macro output on
  the second step;
- ``coupled``: the flow with a passive scalar (D3Q7) and its source;
- ``inlet_gradient`` / ``source_gradient``: forward and backward passes of a
  differentiable run, for the duct's inlet profile and for the scalar source;
- ``diagnostics``: an output step followed by the FP64 reductions;
- ``slab``: one GPU's x-slab with ghost planes, stepped with its halo exchange.

``exact`` restates each path in FP64 torch operations.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "tnl-lbm_amd"))
from pytnl_lbm import (ADE_GEO, GEO, CheckpointedRun, CoupledScalarRun, D3Q7Lattice, D3Q27Lattice, _abi,  # noqa: E402
                       channel_geometry, lattice_run, populations, scalar_run, top_layer_variance)

DEVICE = "cuda:0"
# D3Q27 velocities in the storage order of the populations, and the weights
CX = (0, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1)
CY = (0, 0, 0, 1, -1, 0, 0, 1, -1, -1, 1, 0, 0, 0, 0, 1, -1, 1, -1, 1, -1, 1, -1, -1, 1, -1, 1)
CZ = (0, 0, 0, 0, 0, 1, -1, 0, 0, 0, 0, 1, -1, -1, 1, 1, -1, -1, 1, 1, -1, -1, 1, 1, -1, -1, 1)
VEL = tuple(zip(CX, CY, CZ))
W = tuple(math.prod((1 / 6, 2 / 3)[c == 0] for c in v) for v in VEL)
W7 = (0.25,) + (0.125,) * 6
INDEX = {v: q for q, v in enumerate(VEL)}
OPP = tuple(INDEX[(-x, -y, -z)] for x, y, z in VEL)
DTYPE = {"f64": torch.float64, "f32": torch.float32, "f32dev": torch.float32, "f16dev": torch.float16,
         "bf16dev": torch.bfloat16, "i16dev": torch.int16}
BYTES = {"f64": 8, "f32": 4, "f32dev": 4, "f16dev": 2, "bf16dev": 2, "i16dev": 2}
# bounds of the fixed-point form per direction class, for |u| up to 0.12
I16_RANGE = (0.08, 0.62, 0.9, 1.2)
SCALAR_SCALE = 1000.0  # store_scale of the D3Q7 deviation forms
ALTERNATIVE = ("CUM_2017", "CUM_2017_ANTIALIAS", "MRT_LES", "KBC_N1", "KBC_N2", "KBC_N3", "KBC_N4", "KBC_C1", "KBC_C2",
               "KBC_C3", "KBC_C4")


def listed():
    return [
        # a small Taylor-Green box as in convergence studies and unit runs: launches and latency
        dict(name="box-32", kind="box", X=32, Y=32, Z=32, storage="f64", collision="CUM", tau=0.52),
        # the production box: FP64 turbulence, the largest that a program holds next to others
        dict(name="box-512", kind="box", X=512, Y=512, Z=512, storage="f64", collision="CUM", tau=0.505),
        # the same flow in a 2-byte storage form
        dict(name="box-512-f16", kind="box", X=512, Y=512, Z=512, storage="f16dev", collision="CUM", tau=0.505),
        # a box whose sizes follow a domain, not the hardware
        dict(name="box-ragged-f32", kind="box", X=243, Y=205, Z=157, storage="f32dev", collision="CUM", tau=0.51),
        # an entropic operator, the choice for under-resolved turbulence
        dict(name="box-kbc", kind="box", X=192, Y=192, Z=192, storage="f64", collision="KBC_N4", tau=0.505),
        # duct flow with inlet, outlet and walls, A-B
        dict(name="duct", kind="channel", flow="duct", X=384, Y=128, Z=128, storage="f64", pattern="AB", tau=0.51),
        # ragged wall-bounded channel driven by a body force, 2-byte storage, A-A
        dict(name="channel-f16", kind="channel", flow="driven", X=301, Y=187, Z=129, storage="f16dev", pattern="AA",
             tau=0.51),
        # flow and scalar transport in one step
        dict(name="coupled-f16", kind="coupled", X=256, Y=256, Z=256, storage="f16dev", pattern="AB", operator="CLBM",
             tau=0.505),
        # gradient of an objective with respect to the inlet profile: forward and backward
        dict(name="inlet-gradient", kind="inlet_gradient", X=256, Y=96, Z=96, T=24, mode="mixed", storage="f64", tau=0.51),
        # gradient with respect to the scalar source: forward and backward
        dict(name="source-gradient", kind="source_gradient", X=192, Y=192, Z=192, T=12, storage="f16dev", operator="CLBM",
             tau=0.505),
        # an output step: macros and the energy, enstrophy and mass sums of a time series
        dict(name="diagnostics", kind="diagnostics", X=192, Y=192, Z=192, storage="f64", tau=0.52),
        # one GPU's share of a box split in x, with its halo exchange
        dict(name="slab", kind="slab", X=48, Y=320, Z=320, storage="f64", tau=0.505),
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(("box", "box", "channel", "coupled", "inlet_gradient", "source_gradient", "diagnostics", "slab"))
    tau = round(rng.uniform(0.505, 0.55), 4)
    if kind == "box":
        if rng.random() < 0.3:
            return dict(kind=kind, X=size(24, 256), Y=size(24, 256), Z=size(24, 256), storage=rng.choice(("f64", "f32")),
                        collision=rng.choice(ALTERNATIVE), tau=tau)
        return dict(kind=kind, X=size(24, 512), Y=size(24, 512), Z=size(24, 512), storage=rng.choice(tuple(DTYPE)),
                    collision="CUM", tau=tau)
    if kind == "channel":
        return dict(kind=kind, flow=rng.choice(("duct", "driven")), X=size(48, 384), Y=size(24, 256), Z=size(24, 256),
                    storage=rng.choice(("f64", "f32", "f32dev", "f16dev")), pattern=rng.choice(("AA", "AB")), tau=tau)
    if kind == "coupled":
        return dict(kind=kind, X=size(48, 320), Y=size(48, 320), Z=size(48, 320), storage=rng.choice(("f64", "f32", "f16dev")),
                    pattern=rng.choice(("AA", "AB")), operator=rng.choice(("SRT", "MRT", "CLBM")), tau=tau)
    if kind == "inlet_gradient":
        storage = rng.choice(("f64", "f64", "f32"))
        mode = rng.choice(("mixed", "segment", "recompute") if storage == "f64" else ("segment", "recompute", "tape"))
        return dict(kind=kind, X=size(32, 256), Y=size(16, 96), Z=size(16, 96), T=rng.randint(4, 24), mode=mode,
                    storage=storage, tau=tau)
    if kind == "source_gradient":
        return dict(kind=kind, X=size(32, 192), Y=size(32, 192), Z=size(32, 192), T=rng.randint(4, 12),
                    storage=rng.choice(("f64", "f32", "f16dev")), operator=rng.choice(("SRT", "MRT", "CLBM")), tau=tau)
    if kind == "diagnostics":
        return dict(kind=kind, X=size(32, 320), Y=size(32, 320), Z=size(32, 320), storage=rng.choice(("f64", "f32")), tau=tau)
    return dict(kind=kind, X=size(8, 128), Y=size(64, 512), Z=size(64, 512), storage=rng.choice(("f64", "f32", "f16dev")),
                tau=tau)


# ---- inputs, from the seed alone ----------------------------------------------------

def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _axes(case):
    """Site coordinates broadcast over the storage order (x, z, y)."""
    ax = [torch.arange(case[n], dtype=torch.float64, device=DEVICE) for n in "XYZ"]
    return ax[0].view(-1, 1, 1), ax[1].view(1, 1, -1), ax[2].view(1, -1, 1)


def _flow(case, seed):
    """rho and u of a seeded solenoidal flow, |u| up to about 0.1, shaped to
    the walls of the case, as (X, Z, Y) FP64 fields."""
    g = torch.Generator().manual_seed(seed)
    x, y, z = _axes(case)
    n = (case["X"], case["Y"], case["Z"])
    u = [torch.zeros(n[0], n[2], n[1], dtype=torch.float64, device=DEVICE) for _ in range(3)]
    for _ in range(5):
        m = torch.randint(-3, 4, (3,), generator=g).tolist()
        if not any(m):
            m[0] = 1
        k = [2 * math.pi * m[i] / n[i] for i in range(3)]
        a = torch.randn(3, generator=g, dtype=torch.float64)
        kt = torch.tensor(k, dtype=torch.float64)
        a = a - kt * (a @ kt) / (kt @ kt)
        a = (0.025 * a / a.norm().clamp_min(1e-3)).tolist()
        wave = torch.cos(k[0] * x + k[1] * y + k[2] * z + float(torch.rand(1, generator=g)) * 6.28)
        for i in range(3):
            u[i] += a[i] * wave
    walls = case["kind"] in ("coupled", "source_gradient") or case.get("flow") == "driven"
    if walls:
        for c in u:
            c *= torch.sin(math.pi * z / (case["Z"] - 1))
    if case["kind"] == "inlet_gradient" or case.get("flow") == "duct":
        shape = _duct_shape(case)
        for c in u:
            c *= 0.1 * shape
        u[0] += 0.04 * shape
    return 1.0 + 0.002 * torch.cos(2 * math.pi * (x / n[0] + y / n[1] + z / n[2])), u


def _duct_shape(case):
    _, y, z = _axes(case)
    y, z = y / (case["Y"] - 1), z / (case["Z"] - 1)
    return 16 * y * (1 - y) * z * (1 - z)


def _eq1(c, v):
    return 2 / 3 - v * v if c == 0 else 1 / 6 + 0.5 * (v * v + c * v)


def _equilibrium(q, rho, u):
    return rho * (_eq1(CX[q], u[0]) * _eq1(CY[q], u[1]) * _eq1(CZ[q], u[2]))


def _populations(case, seed):
    """(q, stored populations) in turn: the flow's equilibrium and a
    non-equilibrium part of about one per cent of its deviation."""
    rho, u = _flow(case, seed)
    g = _generator(seed)
    for q in range(27):
        f = _equilibrium(q, rho, u)
        f += (W[q] * 1e-3) * (torch.rand(f.shape, generator=g, dtype=torch.float64, device=DEVICE) - 0.5)
        yield q, _encode(f, q, case["storage"])


def _encode(f, q, storage):
    if storage == "i16dev":
        r = W[q] * I16_RANGE[sum(c != 0 for c in VEL[q])]
        return ((f - W[q]) / r).clamp_(-1, 1).mul_(32767).round_().to(torch.int16)
    return (f - W[q] if storage.endswith("dev") else f).to(DTYPE[storage])


def _decode(s, q, storage):
    return s.double() + W[q] if storage.endswith("dev") else s.double()


def _fill(lat, case, seed):
    """Sets the populations of a lattice without overlaps (array 0)."""
    dst = lat.df[0].view(27, case["X"], case["Z"], case["Y"])
    for q, s in _populations(case, seed):
        dst[q] = s
    for other in lat.df[1:]:
        other.zero_()


def _blobs(case, seed, count=8, amplitude=1e-3):
    """Scalar source: Gaussian blobs away from the walls, (X, Z, Y), values of
    the macro element type."""
    g = torch.Generator().manual_seed(seed + 77)
    out = torch.zeros(case["X"], case["Z"], case["Y"], dtype=torch.float64, device=DEVICE)
    sigma = max(2.0, min(case["X"], case["Y"], case["Z"]) / 24)
    for _ in range(count):
        f = []
        for p, n in zip(_axes(case), (case["X"], case["Y"], case["Z"])):
            c = (0.2 + 0.6 * float(torch.rand(1, generator=g))) * n
            f.append(torch.exp(-((p - c) ** 2) / (2 * sigma * sigma)))
        out += amplitude * f[0] * f[1] * f[2]
    return out if case["storage"] == "f64" else out.float()


def _profile(case, seed):
    """Inlet velocity profile (3, Z, Y): the duct profile with a smooth
    perturbation that vanishes on the walls."""
    g = torch.Generator().manual_seed(seed + 31)
    shape = _duct_shape(case)[0]
    _, y, z = _axes(case)
    out = torch.zeros(3, case["Z"], case["Y"], dtype=torch.float64, device=DEVICE)
    for k in range(3):
        m = torch.randn(2, generator=g).tolist()
        out[k] = 0.004 * shape * (m[0] * torch.sin(2 * math.pi * y[0] / case["Y"]) + m[1] * torch.cos(math.pi * z[0] / case["Z"]))
    out[0] += 0.04 * shape
    return out


def _walls(case, wall, other):
    geo = torch.full((case["X"], case["Y"], case["Z"]), other, dtype=torch.int16)
    geo[:, :, 0] = geo[:, :, -1] = wall
    return geo


def _lattice(case, **kw):
    return D3Q27Lattice(case["X"], case["Y"], case["Z"], storage=case["storage"], nu=(case["tau"] - 0.5) / 3,
                        device=DEVICE, **kw)


def _outlet(case):
    # the zero-gradient outlet is defined for the pull scheme only
    return GEO.OUTFLOW_RIGHT if case.get("pattern", "AB") == "AB" else GEO.OUTFLOW_EQ


def _force(case):
    """Body force that drives the channel towards a centre velocity of 0.05."""
    return 8 * (case["tau"] - 0.5) / 3 * 0.05 / case["Z"] ** 2


def _plane(case):
    """The measured plane: one that the inlet reaches within the run."""
    return min(case["X"] // 4, max(2, case["T"] // 2))


# A control kept in the precision of what is differentiated: float32 wherever
# the schedule's adjoint fields or the lattice are float32 or narrower.
def _control_dtype(case):
    return torch.float64 if case["storage"] == "f64" and case.get("mode") != "mixed" else torch.float32


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "box":
        lat = _lattice(case, collision=case["collision"], store_range_class=I16_RANGE)
        _fill(lat, case, seed)
    elif kind == "channel":
        duct = case["flow"] == "duct"
        geo = (channel_geometry(case["X"], case["Y"], case["Z"], _outlet(case)) if duct
               else _walls(case, GEO.WALL, GEO.PERIODIC))
        lat = _lattice(case, pattern=case["pattern"], geo=geo, force=(0.0 if duct else _force(case), 0.0, 0.0))
        if duct:
            p = _profile(case, seed)
            lat.set_inflow(profile=[p[0], p[1], p[2]])
        _fill(lat, case, seed)
    elif kind in ("coupled", "source_gradient"):
        lat = _lattice(case, pattern=case.get("pattern", "AB"), geo=_walls(case, GEO.WALL, GEO.PERIODIC))
        ade = D3Q7Lattice(lat, collision=case["operator"], diffusivity=0.0125,
                          geo=_walls(case, ADE_GEO.WALL, ADE_GEO.PERIODIC), phi_ref=0.0, store_scale=SCALAR_SCALE)
        _fill(lat, case, seed)
        for d in ade.df:
            d.zero_()
        source = _blobs(case, seed)
        s["ade"] = ade
        if kind == "coupled":
            ade.set_source(source.permute(0, 2, 1))
        else:
            s["run"] = CoupledScalarRun(lat, ade, case["T"])
            s["source"] = source.reshape(-1)
            s["f0"], s["g0"] = lat.df[0].clone(), ade.df[0].clone()
            s["layers"] = max(1, case["Z"] // 6)
    elif kind == "inlet_gradient":
        lat = _lattice(case, pattern="AB", geo=channel_geometry(case["X"], case["Y"], case["Z"], GEO.OUTFLOW_RIGHT))
        _fill(lat, case, seed)
        s["f0"] = lat.df[0].to(_control_dtype(case), copy=True)
        s["run"] = CheckpointedRun(lat, case["T"], mode=case["mode"])
        s["control"] = _profile(case, seed).to(_control_dtype(case))
        s["target"] = _profile(case, seed + 1).unsqueeze(1) * 0.9
        s["plane"] = _plane(case)
    elif kind == "diagnostics":
        lat = _lattice(case)
        _fill(lat, case, seed)
    else:
        lat = _lattice(case, overlap=(1, 0, 0))
        stored = lat.stored()
        for q, f in _populations(case, seed):
            stored[q, 0] = stored[q, -1] = 0
            stored[q, 1:-1] = f
    s["lat"] = lat
    return s


def run(s):
    lat, kind = s["lat"], s["kind"]
    if kind == "box":
        # the even and the odd step of the A-A pattern
        lat.step()
        lat.step()
        return lat.df[0]
    if kind == "channel":
        lat.step()
        lat.step(output_macro=True)
        return [lat.df[0], lat.macro]
    if kind == "coupled":
        lat.step_coupled(s["ade"])
        lat.step_coupled(s["ade"], output_macro=True)
        return [lat.df[0], lat.macro, s["ade"].df[0], s["ade"].phi]
    if kind == "inlet_gradient":
        p, f0 = s["control"].clone().requires_grad_(), s["f0"].detach().requires_grad_()
        fT = lattice_run(s["run"], p, f0)
        # misfit of the momentum on a plane
        f = populations(fT, lat)[:, s["plane"]].double()
        c = torch.tensor([CX, CY, CZ], dtype=torch.float64, device=DEVICE)
        j = torch.tensordot(c, f, dims=([1], [0]))
        loss = 0.5 * ((j - s["target"][:, 0]) ** 2).sum()
        loss.backward()
        return [fT.detach(), p.grad, f0.grad]
    if kind == "source_gradient":
        q = s["source"].clone().requires_grad_()
        gT = scalar_run(s["run"], q, s["g0"], s["f0"])
        loss = top_layer_variance(gT, lat, s["layers"])
        loss.backward()
        return [loss.detach().to(q.dtype), q.grad]
    if kind == "diagnostics":
        lat.step(output_macro=True)
        sums = lat.reduce_macro()
        return [lat.df[0], lat.macro, sums, lat.reduce_gradients()]
    for _ in range(2):
        lat.step(flags=_abi.FLAG_DISTRIBUTED_X)
        lat.halo_x(lat, _abi.HALO_PULL if lat.iterations % 2 == 1 else _abi.HALO_PUSH)
    return lat.df[0]


def work(case):
    """Bytes that a pass cannot do without (each population read and written
    once per step, the macro fields written, the map read) and about as many
    operations as the operator's formulas have."""
    n = case["X"] * case["Y"] * case["Z"]
    e = BYTES[case["storage"]]
    m = 8 if case["storage"] == "f64" else 4
    kind = case["kind"]
    step, flops = 54 * e, 600
    if kind == "box":
        return {"bytes": 2 * n * step, "flops": 2 * n * (flops if case["collision"] == "CUM" else 900)}
    if kind == "channel":
        return {"bytes": n * (2 * step + 4 + 4 * m), "flops": 2 * n * flops}
    if kind == "coupled":
        return {"bytes": n * (2 * (step + 14 * e + 4 + m) + 5 * m), "flops": 2 * n * (flops + 80)}
    if kind == "inlet_gradient":
        # forward, and the backward sweep's two adjoint fields and ten moments
        # per step, with the recomputation that the schedule asks for
        f = 4 if case["mode"] == "mixed" else e
        back = 54 * f + (27 * f if case["mode"] == "recompute" else 10 * f)
        again = {"mixed": 54 * 4 + 10 * 4, "segment": step + 10 * e, "recompute": step, "tape": 0}[case["mode"]]
        return {"bytes": case["T"] * n * (step + again + back), "flops": case["T"] * n * 3 * flops}
    if kind == "source_gradient":
        a = 8 if case["storage"] == "f64" else 4
        back = step + 3 * m + 14 * a + 3 * m
        return {"bytes": case["T"] * n * (step + 14 * e + 4 + m + back) + n * 8, "flops": case["T"] * n * (2 * flops + 160)}
    if kind == "diagnostics":
        return {"bytes": n * (step + 4 * m + 8 * m), "flops": n * (flops + 70)}
    return {"bytes": 2 * n * step + 4 * 18 * case["Y"] * case["Z"] * e, "flops": 2 * n * flops}


# ---- the same in FP64 torch operations ---------------------------------------------------

def _macro(f, force):
    rho = sum(f)
    j = [sum(c[q] * f[q] for q in range(27) if c[q]) for c in (CX, CY, CZ)]
    return rho, [(j[i] + 0.5 * force[i]) / rho for i in range(3)]


def _cumulant(f, rho, u, force, omega, mass=None):
    """Default cumulant: second order relaxed (trace at rate 1), every higher
    cumulant zero.  `mass`: the density that the products are divided by,
    where it is not the populations' own."""
    d = rho if mass is None else mass
    P = {}
    for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)):
        P[a, b] = sum(v[a] * v[b] * f[q] for q, v in enumerate(VEL) if v[a] * v[b])
    j = [rho * u[i] - 0.5 * force[i] for i in range(3)]
    k = {ab: P[ab] - u[ab[0]] * j[ab[1]] - u[ab[1]] * j[ab[0]] + rho * u[ab[0]] * u[ab[1]] for ab in P}
    r = 1 - omega
    e1, e2 = r * (k[0, 0] - k[1, 1]), r * (k[0, 0] - k[2, 2])
    a, b, c = (e1 + e2 + rho) / 3, (rho + e2 - 2 * e1) / 3, (rho + e1 - 2 * e2) / 3
    s, p, t = r * k[0, 1], r * k[0, 2], r * k[1, 2]
    K = {(0, 0, 0): rho, (2, 0, 0): a, (0, 2, 0): b, (0, 0, 2): c, (1, 1, 0): s, (1, 0, 1): p, (0, 1, 1): t}
    K[2, 1, 1], K[1, 2, 1], K[1, 1, 2] = (a * t + 2 * p * s) / d, (b * p + 2 * s * t) / d, (c * s + 2 * t * p) / d
    K[2, 2, 0], K[0, 2, 2], K[2, 0, 2] = (a * b + 2 * s * s) / d, (b * c + 2 * t * t) / d, (a * c + 2 * p * p) / d
    K[2, 2, 2] = ((a * K[0, 2, 2] + b * K[2, 0, 2] + c * K[2, 2, 0] + 4 * (t * K[2, 1, 1] + p * K[1, 2, 1] + s * K[1, 1, 2])) / d
                  - (16 * s * p * t + 4 * (p * p * b + t * t * a + s * s * c) + 2 * a * b * c) / (d * d))
    for i, n in enumerate(((1, 0, 0), (0, 1, 0), (0, 0, 1))):
        if force[i]:
            K[n] = torch.full_like(rho, 0.5 * force[i])
    for axis in range(3):  # central moments of one axis -> populations along it
        out = {}
        for n in {n[:axis] + (0,) + n[axis + 1:] for n in K}:
            def at(i):
                return K.get(n[:axis] + (i,) + n[axis + 1:], 0.0)
            v = u[axis]
            m0 = at(0)
            m1 = at(1) + v * m0
            m2 = at(2) + 2 * v * at(1) + v * v * m0
            for i, val in ((0, 0.5 * (m2 - m1)), (1, m0 - m2), (2, 0.5 * (m2 + m1))):
                out[n[:axis] + (i,) + n[axis + 1:]] = val
        K = out
    return [K[x + 1, y + 1, z + 1] for x, y, z in VEL]


def _mrt_les(f, rho, u, nu):
    P = [[sum(v[a] * v[b] * f[q] for q, v in enumerate(VEL) if v[a] * v[b]) for b in range(3)] for a in range(3)]
    N = [[P[a][b] - rho * ((a == b) / 3 + u[a] * u[b]) for b in range(3)] for a in range(3)]
    Q = 2 * sum(N[a][b] * N[a][b] for a in range(3) for b in range(3))
    tau = 3 * nu + 0.5
    omega = 2 / (torch.sqrt(tau * tau + 18 * 0.0342 * torch.sqrt(Q) / rho) + tau)
    P = [[P[a][b] - omega * N[a][b] for b in range(3)] for a in range(3)]
    trace = P[0][0] + P[1][1] + P[2][2]
    out = []
    for q, v in enumerate(VEL):
        cPc = sum(v[a] * v[b] * P[a][b] for a in range(3) for b in range(3) if v[a] * v[b]) + 0 * rho
        lin = 2.5 - 1.5 * sum(map(abs, v)) + 3 * sum(v[i] * u[i] for i in range(3))
        out.append(W[q] * (rho * lin + 4.5 * cPc - 1.5 * trace))
    return out


def _kbc_raw(f, rho, u, nu, variant):
    """KBC N1-N4 (raw moments): shear part D, D + T, D + Q or D + T + Q."""
    def mom(g, n):
        return sum(v[0] ** n[0] * v[1] ** n[1] * v[2] ** n[2] * g[q] for q, v in enumerate(VEL)
                   if all(v[i] or not n[i] for i in range(3)))

    feq = [_equilibrium(q, rho, u) for q in range(27)]
    delta = [a - b for a, b in zip(f, feq)]  # every part is linear in the populations
    T2 = [mom(delta, tuple(2 * (i == a) for i in range(3))) for a in range(3)]
    pair = {(a, b): mom(delta, tuple(int(i in (a, b)) for i in range(3))) for a in range(3) for b in range(a + 1, 3)}
    tr = sum(T2)
    cubic = {(a, b): mom(delta, tuple(2 * (i == a) + (i == b) for i in range(3))) for a in range(3) for b in range(3) if a != b}
    xyz = mom(delta, (1, 1, 1))
    ds = []
    for q, v in enumerate(VEL):
        on = [i for i in range(3) if v[i]]
        s = 0 * rho
        if len(on) == 1:
            s = s + (3 * T2[on[0]] - tr) / 6
        elif len(on) == 2:
            s = s + v[on[0]] * v[on[1]] * pair[on[0], on[1]] / 4
        if variant in (2, 4):
            s = s + (-tr if not on else tr / 6 if len(on) == 1 else 0)
        if variant in (3, 4):
            if len(on) == 1:
                s = s - v[on[0]] * sum(cubic[b, on[0]] for b in range(3) if b != on[0]) / 2
            elif len(on) == 2:
                s = s + (v[on[0]] * cubic[on[1], on[0]] + v[on[1]] * cubic[on[0], on[1]]) / 4
            elif len(on) == 3:
                s = s + v[0] * v[1] * v[2] * xyz / 8
        ds.append(s)
    dh = [a - b for a, b in zip(delta, ds)]
    beta = 1 / (6 * nu + 1)
    num = sum(a * b / e for a, b, e in zip(ds, dh, feq))
    den = sum(a * a / e for a, e in zip(dh, feq))
    gamma = 1 / beta - (2 - 1 / beta) * num / den
    return [f[q] - beta * (2 * ds[q] + gamma * dh[q]) for q in range(27)]


def _collide(case, f, force):
    rho, u = _macro(f, force)
    nu = (case["tau"] - 0.5) / 3
    op = case.get("collision", "CUM")
    if op == "CUM":
        return _cumulant(f, rho, u, force, 1 / case["tau"]), rho, u
    if op == "MRT_LES":
        return _mrt_les(f, rho, u, nu), rho, u
    return _kbc_raw(f, rho, u, nu, int(op[-1])), rho, u


def _wrap(a, v):
    """a(r - v) on the periodic box, a shaped (X, Z, Y)."""
    return torch.roll(a, (v[0], v[2], v[1]), (0, 1, 2)) if any(v) else a


def _clamp(a, v):
    """a(r - v) with indices clamped at the box's faces."""
    for c, d in ((v[0], 0), (v[2], 1), (v[1], 2)):
        if c:
            n = a.shape[d]
            edge = a.narrow(d, 0 if c > 0 else n - 1, 1)
            rest = a.narrow(d, 0 if c > 0 else 1, n - 1)
            a = torch.cat((edge, rest) if c > 0 else (rest, edge), d)
    return a


def _periodic_pair(case, seed, chunk=1 << 24):
    """An A-A even step and the odd step after it, on the slots of a periodic
    box: absolute FP64 populations, (27, X, Z, Y)."""
    X = case["X"]
    S = torch.empty(27, X, case["Z"], case["Y"], dtype=torch.float64, device=DEVICE)
    for q, s in _populations(case, seed):
        S[q] = _decode(s, q, case["storage"])
    width = max(1, chunk // (case["Y"] * case["Z"]))
    for x in range(0, X, width):
        f, _, _ = _collide(case, [S[q, x:x + width].clone() for q in range(27)], (0, 0, 0))
        for q in range(27):
            S[OPP[q], x:x + width] = f[q]
    out = torch.empty_like(S)
    for x in range(0, X, width):
        xs = torch.arange(x, min(X, x + width), device=DEVICE)
        f, _, _ = _collide(case, [_wrap(S[OPP[q]][(xs - CX[q]) % X], (0, CY[q], CZ[q])) for q in range(27)], (0, 0, 0))
        for q in range(27):
            out[q][(xs + CX[q]) % X] = _wrap(f[q], (0, CY[q], CZ[q]))
    return out


class _Walled:
    """Steps of a box with walls (and, for the duct, inlet and outlet)."""

    def __init__(self, case, seed):
        self.case = case
        X, Y, Z = case["X"], case["Y"], case["Z"]
        duct = case["kind"] == "inlet_gradient" or case.get("flow") == "duct"
        if duct:
            geo = torch.as_tensor(channel_geometry(X, Y, Z, _outlet(case))).to(torch.int16)
        else:
            geo = _walls(case, GEO.WALL, GEO.PERIODIC)
        geo = geo.permute(0, 2, 1).contiguous().to(DEVICE)
        self.wall, self.inlet = geo == GEO.WALL, geo == GEO.INFLOW
        self.right, self.eq = geo == GEO.OUTFLOW_RIGHT, geo == GEO.OUTFLOW_EQ
        self.periodic = geo == GEO.PERIODIC
        self.duct = duct
        self.force = (_force(case) if case.get("flow") == "driven" else 0.0, 0.0, 0.0)
        self.omega = 1 / case["tau"]

    def pull(self, f, v):
        """a(r - v): periodic sites wrap, the others clamp; the zero-gradient
        outlet pulls as if it lay one site upstream."""
        g = _clamp(f, v) if self.duct else torch.where(self.periodic, _wrap(f, v), _clamp(f, v))
        if self.duct and bool(self.right.any()):
            g = torch.where(self.right, _clamp(f, (1, v[1], v[2])), g)
        return g

    def site(self, f, profile=None):
        """Boundary conditions and collision of pulled populations: the
        post-collision populations and the site's rho and u."""
        rho, u = _macro(f, self.force)
        one, zero = torch.ones_like(rho), torch.zeros_like(rho)
        mass = torch.where(self.right, one, rho) if self.duct else rho
        post = _cumulant(f, rho, u, self.force, self.omega, mass)
        post = [torch.where(self.wall, f[OPP[q]], post[q]) for q in range(27)]
        u = [torch.where(self.wall, zero, c) for c in u]
        out_rho = torch.where(self.wall | self.right | self.eq | self.inlet, one, rho)
        if self.duct:
            ui = [torch.where(self.inlet, profile[k].unsqueeze(0).expand_as(u[k]), u[k]) for k in range(3)]
            given = self.inlet | self.eq
            post = [torch.where(given, _equilibrium(q, one, ui), post[q]) for q in range(27)]
            u = ui
        return post, out_rho, u

    def step_ab(self, f, profile=None):
        return self.site([self.pull(f[q], VEL[q]) for q in range(27)], profile)

    def pair_aa(self, S, profile=None):
        """Even and odd A-A step (non-periodic indices wrap at the array's end)."""
        f, _, _ = self.site(S, profile)
        S = [f[OPP[q]] for q in range(27)]
        f, rho, u = self.site([_wrap(S[OPP[q]], VEL[q]) for q in range(27)], profile)
        return [_wrap(f[q], VEL[q]) for q in range(27)], rho, u


def _initial(case, seed):
    return [_decode(s, q, case["storage"]) for q, s in _populations(case, seed)]


def _stored(f, case):
    """Absolute populations in the storage form's values, flat."""
    dev = case["storage"].endswith("dev")
    return torch.stack([f[q] - W[q] if dev else f[q] for q in range(27)]).reshape(-1)


def _scalar_collide(op, f, u, D, source):
    """D3Q7 collision: first moments relaxed (SRT: every population), second
    ones set to their equilibrium (MRT raw, CLBM central)."""
    omega = 1 / (0.5 + 4 * D)
    phi = sum(f)
    pairs = ((1, 2), (3, 4), (5, 6))
    if op == "SRT":
        uu = sum(c * c for c in u)
        out = []
        for q in range(7):
            cu = sum(VEL[q][i] * u[i] for i in range(3))
            out.append(f[q] + omega * (W7[q] * phi * (1 - 2 * uu + 4 * cu + 8 * cu * cu) - f[q]))
    else:
        out = [f[0]] + [None] * 6
        for a, (p, m) in enumerate(pairs):
            v = u[a]
            k1 = omega * (phi * v + f[m] - f[p])
            if op == "MRT":
                k2 = phi * (v * v + 0.25) - f[m] - f[p]
                out[0] = out[0] - k2
                out[p], out[m] = f[p] + 0.5 * (k2 + k1), f[m] + 0.5 * (k2 - k1)
            else:
                k2 = phi * (0.25 - v * v) + 2 * v * (f[p] - f[m]) - f[m] - f[p]
                out[0] = out[0] - 2 * k1 * v - k2
                out[p], out[m] = f[p] + k1 * v + 0.5 * (k2 + k1), f[m] + k1 * v + 0.5 * (k2 - k1)
    return [out[q] + W7[q] * source for q in range(7)], phi


class _Scalar:
    """The scalar's site update between the walls."""

    def __init__(self, case, box):
        self.case, self.box = case, box

    def site(self, g, u, source):
        post, phi = _scalar_collide(self.case["operator"], g, u, 0.0125, source)
        return [torch.where(self.box.wall, g[OPP[q]], post[q]) for q in range(7)], phi

    def step_ab(self, g, u, source):
        return self.site([self.box.pull(g[q], VEL[q]) for q in range(7)], u, source)


def _exact_coupled(case, seed):
    box = _Walled(case, seed)
    sc = _Scalar(case, box)
    f = _initial(case, seed)
    source = _blobs(case, seed).double()
    g = [torch.zeros_like(source) for _ in range(7)]
    if case["pattern"] == "AB":
        for _ in range(2):
            f, rho, u = box.step_ab(f)
            g, phi = sc.step_ab(g, u, source)
    else:
        f, rho, u = box.site(f)
        g, phi = sc.site(g, u, source)
        f, g = [f[OPP[q]] for q in range(27)], [g[OPP[q]] for q in range(7)]
        f, rho, u = box.site([_wrap(f[OPP[q]], VEL[q]) for q in range(27)])
        g, phi = sc.site([_wrap(g[OPP[q]], VEL[q]) for q in range(7)], u, source)
        f, g = [_wrap(f[q], VEL[q]) for q in range(27)], [_wrap(g[q], VEL[q]) for q in range(7)]
    scale = SCALAR_SCALE if case["storage"].endswith("dev") else 1.0
    return [_stored(f, case), torch.stack([rho] + u).reshape(-1), scale * torch.stack(g).reshape(-1), phi.reshape(-1)]


def _exact_inlet_gradient(case, seed):
    box = _Walled(case, seed)
    p = _profile(case, seed).to(_control_dtype(case)).double()
    states = [torch.stack(_initial(case, seed)).to(_control_dtype(case)).double()]
    with torch.no_grad():
        for _ in range(case["T"]):
            states.append(torch.stack(box.step_ab(states[-1], p)[0]))
    fT = states.pop()
    last = fT.clone().requires_grad_()
    c = torch.tensor([CX, CY, CZ], dtype=torch.float64, device=DEVICE)
    j = torch.tensordot(c, last[:, _plane(case)], dims=([1], [0]))
    target = _profile(case, seed + 1) * 0.9
    (lam,) = torch.autograd.grad(0.5 * ((j - target) ** 2).sum(), last)
    grad = torch.zeros_like(p)
    while states:
        s, pr = states.pop().requires_grad_(), p.clone().requires_grad_()
        out = torch.stack(box.step_ab(s, pr)[0])
        lam, gp = torch.autograd.grad(out, (s, pr), lam)
        grad += gp
        del s, out
    return [fT.reshape(-1), grad, lam.reshape(-1)]


def _exact_source_gradient(case, seed):
    box = _Walled(case, seed)
    sc = _Scalar(case, box)
    f = _initial(case, seed)
    source = _blobs(case, seed).double()
    g = torch.zeros(7, *source.shape, dtype=torch.float64, device=DEVICE)
    us = []
    with torch.no_grad():
        for _ in range(case["T"]):
            f, _, u = box.step_ab(f)
            us.append(u)
            g = torch.stack(sc.step_ab(g, u, source)[0])
    last = g.requires_grad_()
    layers = max(1, case["Z"] // 6)
    phi = last.sum(0)[:, case["Z"] - layers:, :]
    loss = ((phi - phi.mean()) ** 2).mean()
    (lam,) = torch.autograd.grad(loss, last)
    grad = torch.zeros_like(source)
    zero = torch.zeros_like(last)  # the step is linear in the scalar: its transpose at any state
    while us:
        z, sr = zero.clone().requires_grad_(), source.clone().requires_grad_()
        out = torch.stack(sc.step_ab(z, us.pop(), sr)[0])
        lam, gs = torch.autograd.grad(out, (z, sr), lam)
        grad += gs
    return [loss.detach(), grad.reshape(-1)]


def _exact_diagnostics(case, seed):
    f = _initial(case, seed)
    rho, u = _macro(f, (0, 0, 0))
    u2 = u[0] ** 2 + u[1] ** 2 + u[2] ** 2
    n = float(rho.numel())
    sums = [rho.sum(), (rho * u2).sum(), rho.new_zeros(()), ((rho - 1) ** 2).sum(), u2.sum(), rho.new_tensor(n)]
    axis = (0, 2, 1)  # of x, y, z in the storage order
    G = [[0.5 * (torch.roll(u[a], -1, axis[b]) - torch.roll(u[a], 1, axis[b])) for b in range(3)] for a in range(3)]
    g2 = sum(G[a][b] ** 2 for a in range(3) for b in range(3))
    curl = (G[2][1] - G[1][2]) ** 2 + (G[0][2] - G[2][0]) ** 2 + (G[1][0] - G[0][1]) ** 2
    post = _cumulant(f, rho, u, (0, 0, 0), 1 / case["tau"])
    state = _stored([post[OPP[q]] for q in range(27)], case)  # an even A-A step
    return [state, torch.stack([rho] + u).reshape(-1), sums, [(rho * g2).sum(), (rho * curl).sum()]]


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "box":
            if case["storage"] == "i16dev" or case["collision"].startswith(("CUM_2017", "KBC_C")):
                return None
            out = _periodic_pair(case, seed)
            if case["storage"].endswith("dev"):
                for q in range(27):
                    out[q] -= W[q]
            return out.reshape(-1)
        if kind == "channel":
            box = _Walled(case, seed)
            p = _profile(case, seed) if box.duct else None
            f = _initial(case, seed)
            if case["pattern"] == "AB":
                f, _, _ = box.step_ab(f, p)
                f, rho, u = box.step_ab(f, p)
            else:
                f, rho, u = box.pair_aa(f, p)
            return [_stored(f, case), torch.stack([rho] + u).reshape(-1)]
        if kind == "coupled":
            return _exact_coupled(case, seed)
        if kind == "diagnostics":
            return _exact_diagnostics(case, seed)
        if kind == "slab":
            out = _periodic_pair(case, seed)
            full = torch.zeros(27, case["X"] + 2, case["Z"], case["Y"], dtype=torch.float64, device=DEVICE)
            for q in range(27):
                full[q, 1:-1] = out[q] - W[q] if case["storage"].endswith("dev") else out[q]
                if CX[q]:  # the slots that the odd step pushed across a face
                    full[q, -1 if CX[q] > 0 else 0] = full[q, 1 if CX[q] > 0 else -2]
            return full.reshape(-1)
    return _exact_inlet_gradient(case, seed) if kind == "inlet_gradient" else _exact_source_gradient(case, seed)
