"""The work that a user of this framework has it do on the GPU, as cases to be timed.

One time step of the ocean model it serves runs, on 13 tiles of 90 x 90 with a halo of 4 and up to 50 levels: halo
exchanges, the operator and right-hand side of the free-surface equation, its solve (one member in the reference's
summation order; ensembles of members; the mixed-precision solve), the tracer advection with DST3 fluxes and the
implicit vertical solve; and, for gradients, the reverse modes of all of them. Each case is one of these calls:

  exchange   `Exchanger.exch_xy` of a scalar field, or `exch_uv_xy` of a pair
  solve      `cg2d.cg2d_fortran`: one member or a batch of right-hand sides on one operator
  mixed      `mixed.cg2d_mixed` for an ensemble whose members share operators by level count
  step       `ensemble.EnsembleStep.step`: the mixed solve and the tracer advection of an ensemble, prepared once
  advect     `gad.advect_tiles`: X/Y fluxes, or X/Y/R with the vertical velocity
  implicit   `tracer_implicit.gad_implicit_r`
  advect_grad, implicit_grad   forward and backward of the two through torch.autograd
  producers  `solve_for_pressure.update_cg2d` and `cg2d_rhs`
  rollout    a short coupled rollout with checkpoints, forward and backward

Grids, flows and operators are the package's seeded synthetic ones; `prepare` perturbs them from the seed.
`exact` restates every result in plain torch, FP64.
"""

from functools import lru_cache
from pathlib import Path
from types import SimpleNamespace

import numpy as np
import torch

from mit_jax_amd import cg2d, ensemble, gad, mixed, rollout, solve_for_pressure, synthetic, tracer_implicit
from mit_jax_amd.exchange import default_exchanger

T, N, OL, NI = 13, 98, 4, 90          # tiles, padded and interior points a side, halo
PLANE = N * N
LEVEL_CLASSES = (15, 30, 50)          # level counts of an ensemble's members
DT, GRAVITY = synthetic.DT, synthetic.G
IN = slice(OL, OL + NI)               # interior rows / columns
IN1 = slice(OL, OL + NI + 1)          # and one more (faces)


# ------------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call of a time step: the halo of one 2-D field (eta after each solve)
        dict(name="exchange-2d", kind="exchange", levels=0, vector=False),
        # what cg2d_solve runs by default in a model run: one member, the reference's summation order, tolerance 1e-7
        dict(name="solve-one", kind="solve", members=1, levels=50, order="fortran", tolerance=1e-7, precond="5point"),
        # many right-hand sides on one operator (sensitivities, a batch of forcings), FP64 to 1e-12
        dict(name="solve-batch", kind="solve", members=64, levels=50, order="tile", tolerance=1e-12,
             precond="diagonal"),
        # the ensemble's solve: 128 members of three level classes, FP32 inner iterations to the FP64 target
        dict(name="mixed-ensemble", kind="mixed", members=128),
        # a small ensemble's whole prepared step (solve and X/Y advection)
        dict(name="ensemble-step", kind="step", members=32),
        # tracer advection of one model run: X/Y, 50 levels
        dict(name="advect-one", kind="advect", members=1, levels=50, vertical=False, ragged=False),
        # tracer advection of an ensemble with level counts of its own per member, with the explicit vertical flux
        dict(name="advect-ensemble", kind="advect", members=24, levels=50, vertical=True, ragged=True),
        # the gradient of one tracer step in the tracer and the flow
        dict(name="advect-gradient", kind="advect_grad", members=1, levels=50, vertical=True, ragged=False),
        # implicit vertical advection and diffusion of an ensemble's tracer
        dict(name="implicit-ensemble", kind="implicit", members=24, levels=50, advection=True),
        # its gradient in the tracer, the diffusivity and the vertical velocity
        dict(name="implicit-gradient", kind="implicit_grad", members=2, levels=50, advection=True),
        # the operator and right-hand side before each solve of one model run
        dict(name="producers-one", kind="producers", members=1, levels=50),
        # a segment of an adjoint run: coupled steps with checkpoints, gradients of T0, u0, v0 and b
        dict(name="rollout-gradient", kind="rollout", steps=2, checkpoint=1),
    ]


def draw(rng):
    """One more case of the same ranges, without a name."""
    def log(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))
    kind = rng.choice(("exchange", "solve", "solve", "mixed", "mixed", "step", "advect", "advect", "advect_grad",
                       "implicit", "implicit", "implicit_grad", "producers"))
    levels = rng.choice((50, *(rng.randint(5, 49) for _ in range(3)), *LEVEL_CLASSES))
    if kind == "exchange":
        return dict(kind=kind, levels=log(1, 50) if rng.random() < 0.75 else 0, vector=rng.random() < 0.5)
    if kind == "solve":
        order = rng.choice(("fortran", "tile", "tile"))
        return dict(kind=kind, members=log(1, 6) if order == "fortran" else log(1, 64), levels=levels, order=order,
                    tolerance=rng.choice((1e-7, 1e-10, 1e-12)), precond=rng.choice(("5point", "diagonal")))
    if kind == "mixed":
        return dict(kind=kind, members=log(1, 127))
    if kind == "step":
        return dict(kind=kind, members=log(2, 31))
    if kind in ("advect", "advect_grad"):
        members = log(1, 23) if kind == "advect" else log(1, 4)
        ragged = members > 1 and rng.random() < 0.5
        return dict(kind=kind, members=members, levels=50 if ragged else levels, vertical=rng.random() < 0.5,
                    ragged=ragged)
    if kind in ("implicit", "implicit_grad"):
        return dict(kind=kind, members=log(1, 23) if kind == "implicit" else log(1, 4), levels=levels,
                    advection=rng.random() < 0.75)
    return dict(kind=kind, members=log(1, 16), levels=levels)


# ----------------------------------------------------------------------------------------------------- their inputs
@lru_cache(maxsize=8)
def _base(levels, precond="5point"):
    """Host arrays of the grid truncated to `levels` levels, its operator and its flow."""
    g, ops, norm = synthetic.cg2d_case(0, precond, nlev=levels)
    f = {k: np.ascontiguousarray(a[:, :levels]) if a.ndim == 4 else a for k, a in g.f.items()}
    v = {k: np.ascontiguousarray(a[:levels]) for k, a in g.v.items() if k not in ("rF",)}
    flow = [np.ascontiguousarray(a[:, :levels]) for a in synthetic.flow(g, 2)] if precond == "5point" else None
    return SimpleNamespace(L=g.L, ops=ops, norm=norm, flow=flow, f=f, v=v)


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _inputs(case, seed):
    """The device tensors of a case, from its seed."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind, B = case["kind"], case.get("members", 1)

    def normal(*shape):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64)

    def uniform(*shape):
        return torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64)

    ex = default_exchanger()
    if kind == "exchange":
        shape = (T, case["levels"], N, N) if case["levels"] else (T, N, N)
        return dict(a=normal(*shape), b=normal(*shape) if case["vector"] else None)

    ragged = kind in ("mixed", "step") or case.get("ragged")
    if ragged:  # every member has the level count of its class; a class shares its operator and masks
        rng = np.random.default_rng(seed)
        index = np.concatenate([np.arange(3)[:B], rng.integers(0, 3, max(B - 3, 0))]).astype(np.int32)
        index = index[rng.permutation(B)]
        levels, classes = 50, LEVEL_CLASSES
    else:
        levels = case.get("levels", 50)
        index, classes = np.zeros(B, np.int32), (levels,)
    bases = [_base(n, case.get("precond", "5point")) for n in classes]
    pick = torch.as_tensor(index, device="cuda", dtype=torch.int64)
    d = dict(index=pick.to(torch.int32), nlev=torch.as_tensor(np.asarray(classes, np.int32)[index], device="cuda"),
             levels=levels, shared=not ragged)

    def padded(a):  # a class's [T, k, N, N] field with the levels below it dry
        a = _dev(a)
        return torch.nn.functional.pad(a, (0, 0, 0, 0, 0, levels - a.shape[1]))

    def members(get):
        return torch.stack([get(b) for b in bases]).index_select(0, pick).contiguous()

    def fill(a):  # halos of [B, T, ...] fields
        for m in range(a.shape[0]):
            ex.fill_(a[m], "T")
        return a

    if kind in ("solve", "mixed", "step", "rollout"):
        d["ops"] = [_dev(bases[0].ops[k]) if not ragged else torch.stack([_dev(b.ops[k]) for b in bases])
                    for k in range(6)]
        d["norm"] = torch.as_tensor(np.asarray([b.norm for b in bases])[index], device="cuda")
        wet = torch.zeros(B, T, N, N, device="cuda", dtype=torch.float64)
        wet[:, :, IN, IN] = members(lambda b: _dev(b.f["maskInC"]))[:, :, IN, IN]
        b = normal(B, T, N, N) * wet
        d["b"] = b - wet * (b.sum((1, 2, 3)) / wet.sum((1, 2, 3)))[:, None, None, None]
        # a first guess with filled halos (the solve leaves it, normalised, on the halos of x)
        d["x0"] = fill(1e-5 * normal(B, T, N, N) * wet) if kind == "solve" else torch.zeros_like(d["b"])
        if kind in ("solve", "mixed"):
            return d
    f0, v0 = bases[-1].f, bases[-1].v
    d["g2"] = {k: _dev(f0[k]) for k in ("dyG", "dxG", "recip_dxC", "recip_dyC", "recip_rA", "rA", "maskInC")}
    d["vg"] = {k: _dev(v0[k]) for k in ("drF", "recip_drF", "rhoFacC", "recip_drC")}
    masks = {k: torch.stack([padded(b.f[k]) for b in bases]) for k in ("maskC", "maskW", "maskS")}
    d["masks"] = masks if ragged else {k: m[0] for k, m in masks.items()}
    maskC = masks["maskC"].index_select(0, pick)
    d["hW"], d["hS"] = members(lambda b: padded(b.f["hFacW"])), members(lambda b: padded(b.f["hFacS"]))
    d["rhC"] = members(lambda b: padded(b.f["recip_hFacC"]))
    shape = (B, T, levels, N, N)
    z = torch.as_tensor(-np.asarray(bases[-1].v["rC"]), device="cuda")[:, None, None]
    if kind == "producers":
        d.update(gU=normal(*shape) * 0.1, gV=normal(*shape) * 0.1, em=normal(B, T, N, N) * 1e-5,
                 etaN=normal(B, T, N, N) * 0.1, etaH=normal(B, T, N, N) * 0.1,
                 p0=[normal(B, T, N, N) for _ in range(3)], grid=bases[0])
        return d
    d["tr"] = fill(((2.0 + 25.0 * torch.exp(-z / 800.0)) + 0.1 * normal(*shape)) * maskC)
    u, v, w = (members(lambda b, k=k: padded(b.flow[k])) * (1.0 + 0.05 * normal(*shape)) for k in range(3))
    for m in range(B):
        uu, vv = ex.vector(u[m], v[m], "UVs")
        u[m].copy_(uu)
        v[m].copy_(vv)
    d.update(u=u, v=v, w=w, bar=normal(*shape) if kind in ("advect_grad", "implicit_grad") else None)
    if kind in ("implicit", "implicit_grad"):
        d["kappa"] = (1e-5 + 1e-2 * uniform(*shape)) * maskC
    if kind == "rollout":
        d["weight"] = _dev(f0["rA"][:, None] * f0["hFacC"]) * d["vg"]["drF"][:, None, None]
        d["weight"] = d["weight"] * torch.nn.functional.pad(torch.ones(NI, NI, device="cuda"), (OL,) * 4).double()
    return d


def _one(a, case):
    """A single member without its leading axis, as a model run holds it."""
    return a[0] if case.get("members", 1) == 1 else a


def prepare(case, seed):
    d = _inputs(case, seed)
    s = SimpleNamespace(case=case, kind=case["kind"], ex=default_exchanger())
    one = lambda a: _one(a, case)  # noqa: E731
    K = d.get("levels", 0)
    if s.kind == "exchange":
        s.a, s.b = d["a"], d["b"]
        return s
    if s.kind in ("solve", "mixed"):
        s.b, s.x0, s.ops = one(d["b"]), one(d["x0"]), d["ops"]
        s.norm = float(d["norm"][0]) if s.kind == "solve" else d["norm"]
        s.index = d["index"]
        return s
    if s.kind == "producers":
        s.g = SimpleNamespace(layout=d["grid"].L, **d["g2"], drF=d["vg"]["drF"])
        s.fs = solve_for_pressure.FreeSurfParams(deltaTMom=DT, deltaTFreeSurf=DT)
        s.cp = cg2d.Cg2dParams(cg2dMaxIters=1000, cg2dTolerance=1e-7, cg2dNorm=d["grid"].norm)
        s.rBo = torch.full((T, N, N), 1.0 / GRAVITY, device="cuda", dtype=torch.float64)
        s.Bo = torch.full((T, N, N), GRAVITY, device="cuda", dtype=torch.float64)
        s.h = one(d["hW"]), one(d["hS"])
        s.p0 = [one(a) for a in d["p0"]]
        s.rhs = [one(d[k]) for k in ("gU", "gV", "hW", "hS", "em", "etaN", "etaH")]
        return s
    if s.kind in ("implicit", "implicit_grad"):
        s.g = SimpleNamespace(layout=s.ex.L, maskC=d["masks"]["maskC"], rA=d["g2"]["rA"], recip_rA=d["g2"]["recip_rA"],
                              recip_drF=d["vg"]["recip_drF"].cpu().numpy(),
                              recip_drC=d["vg"]["recip_drC"].cpu().numpy())
        s.p = SimpleNamespace(dTtracerLev=np.full(K, DT), implicitDiffusion=True, rkSign=-1.0)
        s.args = [one(d[k]) for k in ("kappa", "rhC", "w", "tr")]
        if s.kind == "implicit_grad":
            s.bar = one(d["bar"])
            s.args = [a.requires_grad_() if n != 1 else a for n, a in enumerate(s.args)]
        return s
    s.g2 = dict(d["g2"], **d["masks"])
    if not d["shared"]:
        s.g2["mask_index"] = d["index"]
    s.vg, s.nlev = d["vg"], None if d["shared"] else d["nlev"]
    s.params = gad.GADParams.llc90(dt=DT, Nr=K, implicitAdvection=not case.get("vertical", False))
    s.fields = [one(d[k]) for k in ("u", "v", "tr", "hW", "hS", "rhC")]
    s.w = one(d["w"]) if case.get("vertical") else None
    if s.kind == "advect_grad":
        s.bar = one(d["bar"])
        s.leaves = [s.fields[2], s.fields[0], s.fields[1]] + ([s.w] if s.w is not None else [])
        for a in s.leaves:
            a.requires_grad_()
    if s.kind == "step":
        s.step = ensemble.EnsembleStep(s.ex, d["ops"], d["index"], d["norm"], d["b"], d["x0"], s.params, s.g2, s.vg,
                                       *s.fields, nlev=s.nlev)
    if s.kind == "rollout":
        u, v, tr, hW, hS, rhC = s.fields
        m = d["masks"]
        s.rc = rollout.RolloutCase(
            ops=d["ops"], p=cg2d.Cg2dParams(cg2dMaxIters=2000, cg2dTolerance=1e-12, cg2dNorm=float(d["norm"][0]),
                                            sum_order="tile"),
            params=s.params, g2d=s.g2, vg=s.vg, hFacW=hW, hFacS=hS, recip_hFacC=rhC, maskC=m["maskC"],
            maskW=m["maskW"], maskS=m["maskS"], recip_dxC=d["g2"]["recip_dxC"], recip_dyC=d["g2"]["recip_dyC"],
            weight=d["weight"], dt=DT)
        s.leaves = [a.requires_grad_() for a in (tr, u, v, _rollout_rhs(d)[0])]
    return s


def _rollout_rhs(d):
    # a surface of some centimetres to decimetres: its pressure gradient changes the flow and leaves it stable
    return d["b"] * 10.0


# -------------------------------------------------------------------------------------------------------- one pass
def run(s):
    c = s.case
    if s.kind == "exchange":
        return s.ex.exch_xy(s.a) if s.b is None else list(s.ex.exch_uv_xy(s.a, s.b))
    if s.kind == "solve":
        x, d = cg2d.cg2d_fortran(s.ex, s.ops, s.b, s.x0, cg2dNorm=s.norm, tolerance=c["tolerance"], max_iters=1000,
                                 sum_order=c["order"])
        return dict(x=x, iterations=d["numIters"], converged=d["converged"], residual=d["lastResidual"])
    if s.kind == "mixed":
        b, x0 = (a if a.dim() == 4 else a[None] for a in (s.b, s.x0))
        x, d = mixed.cg2d_mixed(s.ex, s.ops, b, x0, cg2dNorm=s.norm, tolerance=1e-12, max_iters=4000,
                                op_index=s.index)
        return dict(x=x, converged=d["converged"])
    if s.kind == "step":
        s.step.step()
        return dict(x=s.step.x, converged=s.step.diag()["converged"], gT=s.step.gT)
    if s.kind == "advect":
        u, v, tr, hW, hS, rhC = s.fields
        return gad.advect_tiles(s.params, None, s.g2, s.vg, u, v, tr, hW, hS, rhC, wFld=s.w, nlev=s.nlev)
    if s.kind == "advect_grad":
        u, v, tr, hW, hS, rhC = s.fields
        gT = gad.advect_tiles_ad(s.params, None, s.g2, s.vg, u, v, tr, hW, hS, rhC, nlev=s.nlev, wFld=s.w)
        return [gT.detach(), *torch.autograd.grad(gT, s.leaves, s.bar)]
    if s.kind == "implicit":
        return tracer_implicit.gad_implicit_r(s.p, s.g, c["advection"], 3, *s.args)
    if s.kind == "implicit_grad":
        out = tracer_implicit.gad_implicit_r_ad(s.p, s.g, c["advection"], 3, *s.args)
        leaves = [s.args[3], s.args[0]] + ([s.args[2]] if c["advection"] else [])
        return [out.detach(), *torch.autograd.grad(out, leaves, s.bar)]
    if s.kind == "producers":
        ops = solve_for_pressure.update_cg2d(s.fs, s.cp, s.g, s.ex, *s.h, s.rBo, *s.p0)
        return [*ops, *solve_for_pressure.cg2d_rhs(s.fs, s.g, *s.rhs, s.Bo)]
    Tn, un, vn = rollout.rollout(s.rc, *s.leaves, nsteps=c["steps"], checkpoint_every=c["checkpoint"], ex=s.ex)
    grads = torch.autograd.grad(rollout.loss(s.rc, Tn), s.leaves)
    return [Tn.detach(), un.detach(), vn.detach(), *grads]


# ------------------------------------------------------------------------------------------- what it cannot do without
def work(case):
    """Each input read once, each output written once; the operations of the recurrences on the interior points."""
    kind, B, K = case["kind"], case.get("members", 1), case.get("levels", 50)
    d2, n2 = 8 * T * PLANE, T * NI * NI            # bytes of a padded 2-D field, interior points of one level
    iterations = {15: 40, 30: 100, 50: 170}.get(K, 3.4 * K)
    if kind == "exchange":
        return dict(bytes=(4 if case["vector"] else 2) * d2 * max(K, 1), flops=0)
    cg = 31 * n2                                     # two stencils, three sums, three updates
    if kind == "solve":
        it = iterations * (1.0 if case["precond"] == "5point" else 1.9) * -np.log10(case["tolerance"]) / 12
        return dict(bytes=d2 * (3 * B + 6), flops=float(B * it * cg))
    if kind == "mixed":
        return dict(bytes=d2 * (3 * B + 18), flops=float(B * 100 * cg))
    d3 = d2 * K
    xy, r = 2.4 * 60, 45                             # sweeps of a tile on average x operations of a point; the R flux
    mean = 32 / 50 if case.get("ragged") or kind == "step" else 1.0  # levels of a member that are active
    if kind in ("advect", "step"):
        w = bool(case.get("vertical"))
        slots = 3 if mean < 1 else 1
        nbytes = (7 + w) * d3 * B * mean + (2 + w) * d3 * slots * (2 / 3 if mean < 1 else 1) + 7 * d2
        flops = (xy + r * w) * B * mean * K * T * PLANE
        if kind == "step":
            nbytes, flops = nbytes + d2 * (3 * B + 18), flops + B * 100 * cg
        return dict(bytes=float(nbytes), flops=float(flops))
    if kind == "advect_grad":  # forward, and per input a gradient; the reverse pass costs about three forwards
        w = bool(case.get("vertical"))
        return dict(bytes=float((8 + 3 + 2 * w) * d3 * B * mean + (2 + w) * d3 + 7 * d2),
                    flops=float(4 * (xy + r * w) * B * mean * K * T * PLANE))
    if kind in ("implicit", "implicit_grad"):
        a = bool(case["advection"])
        reads = (3 + a + (kind == "implicit_grad")) * d3 * B + d3
        writes = (1 if kind == "implicit" else 3 + a) * d3 * B
        return dict(bytes=float(reads + writes), flops=float((60 if kind == "implicit" else 180) * B * K * n2))
    if kind == "producers":
        return dict(bytes=float(B * (4 * d3 + 14 * d2) + 8 * d2), flops=float(B * 22 * K * n2))
    # rollout: per step the forward twice (checkpoints) and the reverse mode of a solve and an advection
    steps = case["steps"]
    return dict(bytes=float(9 * d3 + 4 * d3 + 20 * d2), flops=float(steps * (3 * 170 * cg + 5 * xy * K * T * PLANE)))


# ------------------------------------------------------------------------------------------ the results in plain torch
@lru_cache(maxsize=1)
def _maps():
    """The T map and the signed vector map as full gathers: (source, from the other component, sign) per point."""
    z = np.load(Path(__file__).resolve().parent.parent / "mit_jax_amd" / "data" / "exch2_halo_13x90x90.npz",
                allow_pickle=False)
    out = {}
    for name in ("T", "UVs_u", "UVs_v"):
        src, comp, sign = np.arange(T * PLANE), np.full(T * PLANE, 2 if name == "UVs_v" else 1), np.ones(T * PLANE)
        at = z[name + ".dst"]
        src[at], comp[at], sign[at] = z[name + ".src"], z[name + ".comp"], z[name + ".sign"]
        other = comp == (1 if name == "UVs_v" else 2)
        out[name] = tuple(torch.as_tensor(a, device="cuda") for a in (src, other, sign.astype(np.float64)))
    return out


def _gather(a, name, b=None):
    """The exchange of [..., T, (K,) N, N] fields given tile-first: [T, ..., N, N]."""
    src, other, sign = _maps()[name]
    lead = a.shape[1:-2]
    flat = lambda f: f.reshape(T, -1, PLANE).transpose(0, 1).reshape(-1, T * PLANE)  # noqa: E731
    out = flat(a)[:, src]
    if b is not None:
        out = torch.where(other, flat(b)[:, src], out)
    return (out * sign).reshape(-1, T, PLANE).transpose(0, 1).reshape((T,) + lead + (N, N))


def _halo_T(a):  # [B, T, (K,) N, N]
    return _gather(a.transpose(0, 1), "T").transpose(0, 1)


def _halo_uv(u, v):
    ut, vt = u.transpose(0, 1), v.transpose(0, 1)
    return _gather(ut, "UVs_u", vt).transpose(0, 1), _gather(vt, "UVs_v", ut).transpose(0, 1)


def _operator(ops, x):
    """A x on the interior of [B, T, N, N], 0 elsewhere."""
    aW, aS, aC = ops[:3]
    xe = _halo_T(x)
    i, e, w = IN, slice(OL + 1, OL + NI + 1), slice(OL - 1, OL + NI - 1)
    out = torch.zeros_like(x)
    out[..., i, i] = (aW[..., i, i] * xe[..., i, w] + aW[..., i, e] * xe[..., i, e] + aS[..., i, i] * xe[..., w, i]
                      + aS[..., e, i] * xe[..., e, i] + aC[..., i, i] * xe[..., i, i])
    return out


def _linear_solve(ops, b):
    """A x = b for [B, T, N, N]: conjugate gradients with the diagonal preconditioner, restarted from the true
    residual, to the last bits."""
    x = torch.zeros_like(b)
    diag = torch.ones_like(b)
    diag[..., IN, IN] = ops[2][..., IN, IN].expand_as(b[..., IN, IN])
    diag = torch.where(diag == 0.0, 1.0, diag)
    dot = lambda p, q: (p * q).sum((1, 2, 3), keepdim=True)  # noqa: E731
    for _ in range(4):
        r = b - _operator(ops, x)
        z = r / diag
        s, eta = z.clone(), dot(z, r)
        first = dot(r, r).amax()
        for n in range(500):
            q = _operator(ops, s)
            sq = dot(s, q)
            alpha = torch.where(sq == 0.0, 0.0, eta / torch.where(sq == 0.0, 1.0, sq))
            x, r = x + alpha * s, r - alpha * q
            z = r / diag
            new = dot(z, r)
            s = z + torch.where(eta == 0.0, 0.0, new / torch.where(eta == 0.0, 1.0, eta)) * s
            eta = new
            if n % 20 == 19 and bool(dot(r, r).amax() <= 1e-14 * first):
                break
    return x


def _solution(d):
    """x as the solve leaves it: A x = b cg2dNorm on the interior, halos from the normalised first guess."""
    n4 = lambda a: a[:, None, None, None]  # noqa: E731
    idx = d["index"].long()
    ops = [o if o.dim() == 3 else o[idx] for o in d["ops"][:3]]
    b = d["b"] * n4(d["norm"])
    scale = 1.0 / b.abs().amax((1, 2, 3))
    inner = torch.zeros(N, N, device="cuda", dtype=torch.bool)
    inner[IN, IN] = True
    x = _linear_solve(ops, torch.where(inner, b, 0.0))
    return torch.where(inner, x, _halo_T(torch.where(inner, d["x0"] * n4(scale), d["x0"])))


@lru_cache(maxsize=1)
def _advection_tables():
    """Per pass and direction (region [T, N, N], gather before, gather after) of the tiles' sweeps, and the gathers of
    the west and south masks (into both planes) at the facet corners."""
    tiles = []  # facet, and whether the tile's N, S, E, W edge is a facet edge
    for facet, (nx, ny) in enumerate(((1, 3), (1, 3), (1, 1), (3, 1), (3, 1)), 1):
        tiles += [(facet, ty == ny - 1, ty == 0, tx == nx - 1, tx == 0) for ty in range(ny) for tx in range(nx)]
    at = lambda i, j: (j - 1 + OL) * N + i - 1 + OL  # noqa: E731  (Fortran indices)
    R = range(1, OL + 1)
    M = NI

    def corner(t, direction):
        g = np.arange(PLANE)
        _, n, s, e, w = tiles[t]
        for i in R:
            for j in R:
                if direction == 1:
                    pairs = ((w and s, 1 - i, 1 - j, 1 - j, i), (e and s, M + i, 1 - j, M + j, i),
                             (w and n, 1 - i, M + j, 1 - j, M + 1 - i), (e and n, M + i, M + j, M + j, M + 1 - i))
                else:
                    pairs = ((w and s, 1 - i, 1 - j, j, 1 - i), (e and s, M + i, 1 - j, M + 1 - j, 1 - i),
                             (w and n, 1 - i, M + j, j, M + i), (e and n, M + i, M + j, M + 1 - j, M + i))
                for on, di, dj, si, sj in pairs:
                    if on:
                        g[at(di, dj)] = at(si, sj)
        return g

    sweeps = []
    for p in (1, 2, 3):
        for x in (True, False):
            region, before, after = np.zeros((T, N, N), bool), [], []
            for t, (f, n, s, e, w) in enumerate(tiles):
                overlap = f % 3 == 0 if p == 1 else f % 3 == 2 if p == 2 else False
                inside = f % 3 != 0 if p == 1 else f % 3 == 1 if p == 2 else True
                on = f in (((6, 1, 2), (2, 3, 4), (5, 6)) if x else ((3, 4, 5), (5, 6, 1), (2, 3)))[p - 1]
                lo, hi, left, right = (s, n, w, e) if x else (w, e, s, n)  # edges across and along the sweep
                r = region[t] if x else region[t].T
                fills = on and overlap and (lo or hi)
                if on and overlap:
                    cols = slice(OL if left else 1, OL + M if right else N - 1)
                    if lo:
                        r[:OL, cols] = True
                    if hi:
                        r[OL + M:, cols] = True
                elif on:
                    r[OL if inside and lo else 0:OL + M if inside and hi else N, 1:N - 1] = True
                same = np.arange(PLANE)
                before.append(corner(t, 1 if x else 2) if fills else same)
                after.append(corner(t, 2 if x else 1) if fills and p == 1 else same)
            sweeps.append(tuple(torch.as_tensor(np.asarray(a), device="cuda") for a in (region, before, after)))
    mu, mv = np.tile(np.arange(PLANE), (T, 1)), np.tile(np.arange(PLANE) + PLANE, (T, 1))
    for t, (_, n, s, e, w) in enumerate(tiles):
        for i in R:
            for j in R:
                if w and s:
                    mu[t, at(1 - i, 1 - j)] = PLANE + at(1 - j, 1 + i)
                    mv[t, at(1 - i, 1 - j)] = at(1 + j, 1 - i)
                if e and s:
                    if i >= 2:
                        mu[t, at(M + i, 1 - j)] = PLANE + at(M + j, i)
                    mv[t, at(M + i, 1 - j)] = at(M + 1 - j, 1 - i)
                if w and n:
                    mu[t, at(1 - i, M + j)] = PLANE + at(1 - j, M + 1 - i)
                    if j >= 2:
                        mv[t, at(1 - i, M + j)] = at(j, M + i)
                if e and n:
                    if i >= 2:
                        mu[t, at(M + i, M + j)] = PLANE + at(M + j, M + 2 - i)
                    if j >= 2:
                        mv[t, at(M + i, M + j)] = at(M + 2 - j, M + i)
    return sweeps, torch.as_tensor(mu, device="cuda"), torch.as_tensor(mv, device="cuda")


def _interface(trans, cfl, upup, up, down, downdown, m_up, m_0, m_down):
    """The DST3 interface value: `up` is the cell that positive transport comes from."""
    rj, rjm, rjp = (down - up) * m_0, (up - upup) * m_up, (downdown - down) * m_down
    d0, d1 = (2.0 - cfl) * (1.0 - cfl) / 6.0, (1.0 - cfl * cfl) / 6.0
    return (trans + trans.abs()) / 2 * (up + d0 * rj + d1 * rjm) + \
        (trans - trans.abs()) / 2 * (down - d0 * rj - d1 * rjp)


def _advect(d, u, v, tr, w=None):
    """The tracer tendency of [B, T, K, N, N] fields."""
    sweeps, mu, mv = _advection_tables()
    g, vg, idx = d["g2"], d["vg"], d["index"].long()
    level = lambda a: a[:, None, None]  # noqa: E731
    plane = lambda a: a[:, None]  # noqa: E731
    mask = {k: m if m.dim() == 4 else m[idx] for k, m in d["masks"].items()}
    both = torch.cat([mask[k].flatten(-2) for k in ("maskW", "maskS")], -1)
    loc_mask = [torch.gather(both, -1, i[:, None].expand(*both.shape[:-1], PLANE)).unflatten(-1, (N, N))
                for i in (mu, mv)]
    drF = level(vg["drF"])

    def refill(a, where):
        if bool((where == torch.arange(PLANE, device="cuda")).all()):
            return a
        return torch.gather(a.flatten(-2), -1, where[:, None].expand(*a.shape[:-2], PLANE)).unflatten(-1, (N, N))

    loc = tr
    for n, (region, before, after) in enumerate(sweeps):
        x = n % 2 == 0
        if not bool(region.any()):
            continue
        turn = (lambda a: a) if x else (lambda a: a.transpose(-1, -2))
        vel, h = (u, d["hW"]) if x else (v, d["hS"])
        length, rd = (g["dyG"], g["recip_dxC"]) if x else (g["dxG"], g["recip_dyC"])
        loc = refill(loc, before)
        trans = turn(vel * plane(length) * drF * h)
        c, m, q = turn((vel * DT * plane(rd)).abs()), turn(loc_mask[n % 2]), turn(loc)
        f = slice(2, N - 1)
        flux = _interface(trans[..., f], c[..., f], q[..., 0:N - 3], q[..., 1:N - 2], q[..., 2:N - 1], q[..., 3:N],
                          m[..., 1:N - 2], m[..., 2:N - 1], m[..., 3:N])
        flux = torch.nn.functional.pad(flux, (2, 1))
        nxt = lambda a: torch.nn.functional.pad(a[..., 1:] - a[..., :-1], (0, 1))  # noqa: E731
        change = turn(nxt(flux)) - tr * turn(nxt(trans))
        inc = DT * d["rhC"] * level(vg["recip_drF"]) * plane(g["recip_rA"]) * change * plane(g["maskInC"])
        loc = refill(loc, after)
        loc = torch.where(region[:, None], loc - inc, loc)
    if w is not None:
        mC = mask["maskC"]
        deep = (torch.arange(loc.shape[2], device="cuda") < d["nlev"][:, None])[:, None, :, None, None]
        mC = mC * deep
        below = lambda a: torch.nn.functional.pad(a[:, :, 1:], (0, 0, 0, 0, 0, 1))  # noqa: E731
        above = lambda a: torch.nn.functional.pad(a[:, :, :-1], (0, 0, 0, 0, 1, 0))  # noqa: E731
        q = loc * deep
        face = mC * above(mC)  # between level k - 1 and k
        trans = w * plane(g["rA"]) * face
        cfl = (w * DT * level(vg["recip_drC"])).abs()
        flux = _interface(trans, cfl, below(q), q, above(q), above(above(q)), below(face), face, above(face))
        change = (flux - below(flux)) - tr * (trans - below(trans))
        loc = loc - DT * d["rhC"] * level(vg["recip_drF"]) * plane(g["recip_rA"]) * change * mC
    gT = (loc - tr) / DT
    if not d["shared"]:
        gT = gT * (torch.arange(loc.shape[2], device="cuda") < d["nlev"][:, None])[:, None, :, None, None]
    return gT


def _implicit(d, kappa, w, tr, advection):
    """The tracer after the implicit vertical solve: pentadiagonal elimination of the interior columns."""
    K = tr.shape[2]
    col = lambda a: a[..., IN, IN].unbind(-3)  # noqa: E731
    mC, rh, kap, y = col(d["masks"]["maskC"]), col(d["rhC"]), col(kappa), list(col(tr))
    rdF, rdC = d["vg"]["recip_drF"], d["vg"]["recip_drC"]
    zero = torch.zeros_like(y[0])
    rows = []
    for k in range(K):
        s = DT * rh[k] * rdF[k]
        b = -s * mC[k - 1] * kap[k] * rdC[k] if k else zero
        dd = -s * mC[k + 1] * kap[k + 1] * rdC[k + 1] if k + 1 < K else zero
        rows.append([zero, b, 1.0 - (b + dd), dd, zero, s])
    if advection:
        wc = col(w)
        for k in range(1, K):  # the interface above level k; rkSign = -1
            rc = -0.5 * wc[k] * mC[k - 1]  # w rA / rA
            up = rc.abs() / 3.0
            km = (rc + rc.abs()) / 6.0 * mC[k - 2] if k >= 2 else zero
            kp = (rc - rc.abs()) / 6.0 * mC[k + 1] if k < K - 1 else zero
            terms = (-km, rc + up + km, rc - up + kp, -kp)
            for row, sign, first in ((rows[k - 1], 1.0, 1), (rows[k], -1.0, 0)):
                for n, term in enumerate(terms):
                    row[first + n] = row[first + n] + sign * term * row[5]
    e1 = e2 = d1 = d2 = y1 = y2 = zero
    done = []
    for k, (a, b, c, dd, e, _) in enumerate(rows):
        bb = b - a * d2
        pivot = c - a * e2 - bb * d1
        dn, en, yn = (dd - bb * e1) / pivot, e / pivot, (y[k] - a * y2 - bb * y1) / pivot
        d2, e2, y2, d1, e1, y1 = d1, e1, y1, dn, en, yn
        done.append((dn, en, yn))
    u1 = u2 = zero
    cols = []
    for dn, en, yn in reversed(done):
        u = yn - dn * u1 - en * u2
        u2, u1 = u1, u
        cols.append(u)
    inner = torch.nn.functional.pad(torch.stack(cols[::-1], -3), (OL,) * 4)
    edge = torch.ones(N, N, device="cuda", dtype=torch.float64)
    edge[IN, IN] = 0.0
    return inner + tr * edge


class _Surface(torch.autograd.Function):
    """The solution of A x = b cg2dNorm with 0 halos, and its (symmetric) reverse mode."""

    @staticmethod
    def forward(ctx, b, d):
        ctx.d = d
        return _Surface.solve(b, d)

    @staticmethod
    def solve(b, d):
        inner = torch.zeros_like(b)
        inner[..., IN, IN] = b[..., IN, IN]
        return _linear_solve(d["ops"][:3], inner) * d["norm"][0]

    @staticmethod
    def backward(ctx, g):
        return _Surface.solve(g, ctx.d), None


def _rollout(case, d):
    b = _rollout_rhs(d).requires_grad_()
    tr0, u0, v0 = (d[k].requires_grad_() for k in ("tr", "u", "v"))
    g, m = d["g2"], d["masks"]
    tr, u, v = tr0, u0, v0
    w = slice(OL - 1, OL + NI - 1)
    for _ in range(case["steps"]):
        eta = _halo_T(_Surface.apply(b, d))
        gx = (eta[..., IN, IN] - eta[..., IN, w]) * g["recip_dxC"][:, IN, IN]
        gy = (eta[..., IN, IN] - eta[..., w, IN]) * g["recip_dyC"][:, IN, IN]
        gx, gy = (torch.nn.functional.pad(a, (OL,) * 4)[:, :, None] for a in (gx, gy))
        u, v = _halo_uv(u - DT * GRAVITY * gx * m["maskW"], v - DT * GRAVITY * gy * m["maskS"])
        tr = _halo_T(tr + DT * _advect(d, u, v, tr) * m["maskC"])
    grads = torch.autograd.grad((d["weight"] * tr).sum(), (tr0, u0, v0, b))
    return [a.detach()[0] for a in (tr, u, v, *grads)]


def _producers(d):
    g, drF, norm = d["g2"], d["vg"]["drF"], d["grid"].norm
    e, e1 = slice(OL + 1, OL + NI + 1), IN1
    pad = lambda a, s: torch.nn.functional.pad(a, (OL, OL - 1) * 2 if s else (OL,) * 4)  # noqa: E731
    column = lambda h: (h * drF[:, None, None]).sum(2)  # noqa: E731
    aW = pad((column(d["hW"]) * g["dyG"] * g["recip_dxC"] * norm)[..., e1, e1], 1)
    aS = pad((column(d["hS"]) * g["dxG"] * g["recip_dyC"] * norm)[..., e1, e1], 1)
    aC = -(aW[..., IN, IN] + aW[..., IN, e] + aS[..., IN, IN] + aS[..., e, IN]
           + norm / GRAVITY * g["rA"][:, IN, IN] / DT / DT)
    aC = _halo_T(pad(aC, 0))
    c, cw, cs = aC[..., e1, e1], aC[..., e1, OL - 1:OL + NI], aC[..., OL - 1:OL + NI, e1]
    safe = lambda n, q: torch.where(q == 0.0, 0.0, n / torch.where(q == 0.0, 1.0, q))  # noqa: E731
    p = [a.clone() for a in d["p0"]]
    p[0][..., e1, e1] = safe(-aW[..., e1, e1], (0.51 * (c + cw)) ** 2)
    p[1][..., e1, e1] = safe(-aS[..., e1, e1], (0.51 * (c + cs)) ** 2)
    p[2][..., e1, e1] = torch.where(c == 0.0, 1.0, safe(torch.ones_like(c), c))
    fx = column(d["hW"] * d["gU"]) * g["dyG"] / DT
    fy = column(d["hS"] * d["gV"]) * g["dxG"] / DT
    b = fx[..., IN, e] - fx[..., IN, IN] + fy[..., e, IN] - fy[..., IN, IN]
    area = g["rA"][:, IN, IN]
    # fresh water (mass2rUnit = 1 / 1029) and the surface of the last step (Bo = g)
    b = b + d["em"][..., IN, IN] * area * g["maskInC"][:, IN, IN] / 1029.0 / DT - d["etaH"][..., IN, IN] * area / DT / DT
    return [aW, aS, aC, *p, pad(b, 0), d["etaN"] * GRAVITY]


def exact(case, seed):
    kind, B = case["kind"], case.get("members", 1)
    d = _inputs(case, seed)
    one = lambda a: _one(a, case)  # noqa: E731
    if kind == "exchange":
        return _gather(d["a"], "T") if d["b"] is None else \
            [_gather(d["a"], "UVs_u", d["b"]), _gather(d["b"], "UVs_v", d["a"])]
    if kind == "solve":
        return dict(x=one(_solution(d)), iterations=None, converged=None, residual=None)
    if kind == "mixed":
        return dict(x=_solution(d), converged=None)
    if kind == "step":
        return dict(x=_solution(d), converged=None, gT=_advect(d, d["u"], d["v"], d["tr"]))
    if kind == "advect":
        return one(_advect(d, d["u"], d["v"], d["tr"], d["w"] if case["vertical"] else None))
    if kind == "advect_grad":
        leaves = [d[k].requires_grad_() for k in ("tr", "u", "v", "w")[:4 if case["vertical"] else 3]]
        gT = _advect(d, d["u"], d["v"], d["tr"], d["w"] if case["vertical"] else None)
        return [one(a.detach()) for a in (gT, *torch.autograd.grad(gT, leaves, d["bar"]))]
    if kind == "implicit":
        return one(_implicit(d, d["kappa"], d["w"], d["tr"], case["advection"]))
    if kind == "implicit_grad":
        leaves = [d[k].requires_grad_() for k in (("tr", "kappa", "w") if case["advection"] else ("tr", "kappa"))]
        out = _implicit(d, d["kappa"], d["w"], d["tr"], case["advection"])
        return [one(a.detach()) for a in (out, *torch.autograd.grad(out, leaves, d["bar"]))]
    if kind == "producers":
        return [one(a) for a in _producers(d)]
    return _rollout(case, d)
