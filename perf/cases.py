"""The calls this framework is timed on: what a user of it has it do, through
``hawk.build`` / ``hawk.load`` / ``hawk.run`` and a loaded kernel's
``prepare``, over the sizes, scalar types and layouts those calls take.

A case is a dict of plain values whose ``"kind"`` names the work:

* ``calls``   small interactive calls: each a whole ``hawk.run``;
* ``energy``  the streaming kernels (a vector kernel, its VJP and its JVP);
* ``rows``    planes a program holds sample-major, ``(N, w)``, through
  ``hawk.run(..., layout="samples_first")``;
* ``orbit``   a leapfrog integrator and its reverse-mode derivative;
* ``solve``   a 6x6 SPD solve per sample and its reverse-mode derivative;
* ``matmul``  a 16x16 product per sample and its two transposed products;
* ``chain``   an elementwise chain, its ordered total and its ordered scatter
  into bins at Zipf keys;
* ``bins``    an ordered scatter alone: particles onto a mesh (uniform keys)
  or a histogram (Zipf keys), then its derivative (a gather);
* ``nets``    many small models in one launch: each one's loss and the
  gradient of its own weights;
* ``keyed``   one sum per key over its run of samples, under the ordered and
  the default policy;
* ``stats``   sum, mean of squares, extremes and ordered sum over every sample.
"""

from __future__ import annotations

import functools
import math
import tempfile

import numpy as np
import torch

import hawk_amd as hawk
from hawk_amd import Grid, Index, Kernel, Mutable, Scalar, diff
from hawk_amd import examples as E

DEVICE = "cuda:0"
MODES = ("float64", "float32")


# -- the kernels, as a user writes them (most are hawk_amd.examples') ----------

@hawk.kernel
def stats(x: Scalar, total: Mutable[Scalar], mean_sq: Mutable[Scalar], low: Mutable[Scalar],
          high: Mutable[Scalar], ordered: Mutable[Scalar]):
    total = hawk.sum(x)
    mean_sq = hawk.mean(x * x)
    low = hawk.min(x)
    high = hawk.max(x)
    ordered = hawk.sum(x, policy="ordered")


def per_key(samples: int, policy: str) -> Kernel:
    """One sum per key over its ``samples`` consecutive samples."""
    @hawk.kernel
    def key_total(lane: Grid["key", "sample":samples], x: Scalar) -> Scalar:
        return hawk.sum(x, over="sample", policy=policy)
    return Kernel(f"key_total_{samples}_{policy}", key_total.program)


@functools.lru_cache(maxsize=None)
def _unit(what: str, mode: str, samples: int = 0) -> dict:
    """The loaded kernels of one unit: a program builds and loads them once."""
    if what == "energy":
        kernels = [E.energy, E.energy_vjp, E.energy_jvp]
    elif what == "orbit":
        kernels = [E.twobody, E.twobody_vjp]
    elif what == "solve":
        kernels = [E.spd_solve, E.spd_solve_vjp]
    elif what == "matmul":
        kernels = [E.mm16, E.mm16_vjp]
    elif what == "chain":
        kernels = [E.chain]
    elif what == "bins":
        kernels = [E.add_sq, E.add_sq_grad]
    elif what == "nets":
        net = E.net_loss_for(samples)
        kernels = [net, Kernel(f"net_grad_{samples}", diff.vjp(net, wrt=("W",)))]
    elif what == "keyed":
        kernels = [per_key(samples, "ordered"), per_key(samples, "auto")]
    else:
        kernels = [stats]
    directory = tempfile.mkdtemp(prefix="hawk_perf_")
    hawk.build(kernels, directory, mode=mode)
    return [hawk.load(directory, k.name) for k in kernels]


# -- the cases ------------------------------------------------------------------

def listed() -> list:
    return [
        # An interactive call on a small batch: launches and host work are all of it.
        {"name": "calls_4096", "kind": "calls", "mode": "float64", "n": 4096},
        # The headline streams: a resident batch, every plane read or written once.
        {"name": "energy_f64_32m", "kind": "energy", "mode": "float64", "n": 1 << 25},
        # The same streams in the float32 mode, at a size that is no round number.
        {"name": "energy_f32_10m", "kind": "energy", "mode": "float32", "n": 10_000_019},
        # A program that keeps its arrays (N, 3), as numpy and torch code does.
        {"name": "rows_energy_4m", "kind": "rows", "mode": "float64", "what": "energy", "n": 4_000_037},
        # A batch of orbits stepped and differentiated.
        {"name": "orbit_1m", "kind": "orbit", "mode": "float64", "n": 1_000_003},
        # A batch of small SPD systems and the gradients of matrix and right side.
        {"name": "solve_1m", "kind": "solve", "mode": "float64", "n": 1 << 20},
        # Batched 16x16 products, forward and backward, a ragged batch.
        {"name": "matmul_f32_300k", "kind": "matmul", "mode": "float32", "n": 300_001},
        # The fused chain with both of its cross-sample sinks, at the benchmark's size.
        {"name": "chain_64m", "kind": "chain", "mode": "float64", "n": 1 << 26, "cells": 1 << 16},
        # Particles deposited onto a 64^3 mesh, and the force read back.
        {"name": "mesh_4m_262k", "kind": "bins", "mode": "float64", "n": 1 << 22, "cells": 1 << 18, "keys": "uniform"},
        # 16384 small models of 64 samples: losses and gradients.
        {"name": "nets_16k_64", "kind": "nets", "mode": "float64", "nets": 1 << 14, "samples": 64},
        # 20000 groups of 500 samples, each summed.
        {"name": "keyed_20k_500", "kind": "keyed", "mode": "float64", "keys": 20_000, "samples": 500},
        # Summary statistics of one large plane.
        {"name": "stats_10m", "kind": "stats", "mode": "float64", "n": 10_000_019},
    ]


def _log_int(rng, low: int, high: int) -> int:
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng) -> dict:
    kind = rng.choice(["calls", "energy", "energy", "rows", "orbit", "solve", "matmul", "chain", "bins", "bins",
                       "nets", "keyed", "stats"])
    if kind == "calls":
        return {"kind": kind, "mode": rng.choice(MODES), "n": _log_int(rng, 64, 20_000)}
    if kind == "energy":
        return {"kind": kind, "mode": rng.choice(MODES), "n": _log_int(rng, 1 << 16, 1 << 25)}
    if kind == "rows":
        what = rng.choice(["energy", "solve"])
        return {"kind": kind, "mode": rng.choice(MODES), "what": what,
                "n": _log_int(rng, 1 << 12, 1 << 23 if what == "energy" else 1 << 19)}
    if kind in ("orbit", "solve"):
        return {"kind": kind, "mode": "float64", "n": _log_int(rng, 1 << 12, 1 << 20)}
    if kind == "matmul":
        return {"kind": kind, "mode": rng.choice(MODES), "n": _log_int(rng, 1 << 10, 1 << 18)}
    if kind == "chain":
        return {"kind": kind, "mode": "float64", "n": _log_int(rng, 1 << 16, 1 << 25),
                "cells": _log_int(rng, 1 << 6, 1 << 16)}
    if kind == "bins":
        # from a few bins to a mesh of 64^3 cells, at least four lanes a cell
        cells = _log_int(rng, 1 << 6, 1 << 18)
        return {"kind": kind, "mode": rng.choice(MODES), "n": _log_int(rng, max(1 << 14, 4 * cells), 1 << 23),
                "cells": cells, "keys": rng.choice(["uniform", "zipf"])}
    if kind == "nets":
        samples = rng.choice([16, 40, 48, 64, 96])
        return {"kind": kind, "mode": "float64", "nets": _log_int(rng, 64, 1 << 15), "samples": samples}
    if kind == "keyed":
        samples = _log_int(rng, 4, 1 << 17)
        lanes = _log_int(rng, max(1 << 16, samples), 1 << 24)
        return {"kind": kind, "mode": rng.choice(MODES), "keys": max(1, lanes // samples), "samples": samples}
    return {"kind": "stats", "mode": rng.choice(MODES), "n": _log_int(rng, 1 << 10, 1 << 25)}


# -- inputs ----------------------------------------------------------------------

def _real(case) -> torch.dtype:
    return torch.float32 if case["mode"] == "float32" else torch.float64


def _zipf_keys(n: int, cells: int, g) -> torch.Tensor:
    """Zipf(1.1) keys folded into the cells: cell c has the weight of every
    rank that is c modulo the cell count (a Hurwitz zeta value)."""
    rank = torch.arange(1, cells + 1, dtype=torch.float64, device=DEVICE) / cells
    edges = torch.special.zeta(torch.full_like(rank, 1.1), rank).cumsum(0)
    u = torch.rand(n, dtype=torch.float64, device=DEVICE, generator=g) * edges[-1]
    return torch.searchsorted(edges, u, right=True).clamp_(max=cells - 1).to(torch.int32)


def _inputs(case, seed) -> dict:
    """The values of one case, on the GPU, from the seed alone."""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    real, kind = _real(case), case["kind"]

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, dtype=real, device=DEVICE, generator=g) * scale

    if kind == "rows":
        kind = case["what"]
    elif kind == "calls":
        kind = "energy"
    if kind == "energy":
        n = case["n"]
        return {"v": normal(3, n), "dot_v": normal(3, n), "bar_out": normal(n)}
    if kind == "orbit":
        n = case["n"]
        d = normal(3, n)
        r0 = d / d.norm(dim=0) * (0.5 + 1.5 * torch.rand(n, dtype=real, device=DEVICE, generator=g))
        return {"r0": r0, "v0": normal(3, n, scale=0.3), "bar_r": normal(3, n), "bar_v": normal(3, n)}
    if kind == "solve":
        n = case["n"]
        b = normal(n, 6, 6)
        a = torch.einsum("nik,njk->ijn", b, b) + 6.0 * torch.eye(6, dtype=real, device=DEVICE)[:, :, None]
        return {"A": a.contiguous(), "b": normal(6, n), "bar_x": normal(6, n)}
    if kind == "matmul":
        n = case["n"]
        return {p: normal(16, 16, n, scale=0.25) for p in ("A", "B", "bar_C")}
    if kind == "chain":
        n = case["n"]
        return {"x": normal(n), "key": _zipf_keys(n, case["cells"], g)}
    if kind == "bins":
        n, cells = case["n"], case["cells"]
        key = (_zipf_keys(n, cells, g) if case["keys"] == "zipf" else
               torch.randint(0, cells, (n,), dtype=torch.int32, device=DEVICE, generator=g))
        return {"key": key, "x": normal(n), "bar_acc": normal(cells)}
    if kind == "nets":
        k, s, units = case["nets"], case["samples"], E.NET_UNITS
        used = torch.tensor([8, 3, 5, 1, 6], device=DEVICE).repeat(-(-k // 5))[:k]
        mask = (torch.arange(units, device=DEVICE)[None, :] < used[:, None]).to(real)
        return {"W": normal(k, E.NET_WEIGHTS, scale=0.7).reshape(-1), "mask": mask.reshape(-1).contiguous(),
                "x": normal(k * s), "y": normal(k * s), "bar_out": normal(k)}
    if kind == "keyed":
        return {"x": normal(case["keys"] * case["samples"])}
    return {"x": normal(case["n"])}


def _empty(case, *shape) -> torch.Tensor:
    return torch.empty(*shape, dtype=_real(case), device=DEVICE)


# -- one pass --------------------------------------------------------------------

class _Prepared:
    """Planes bound once and launched per pass: a program's step over resident planes."""

    def __init__(self, launchers, outputs, zeroed=()):
        self.launchers, self.outputs, self.zeroed = launchers, outputs, zeroed

    def __call__(self):
        for x in self.zeroed:                     # accumulators a step starts from zero
            x.zero_()
        for launch in self.launchers:
            launch()
        return self.outputs


def prepare(case, seed):
    kind, mode = case["kind"], case["mode"]
    p = _inputs(case, seed)
    if kind in ("calls", "rows"):
        return _prepare_runs(case, p)
    if kind == "energy":
        n = case["n"]
        fwd, vjp, jvp = _unit("energy", mode)
        out, bar_v, dot_out = _empty(case, n), _empty(case, 3, n), _empty(case, n)
        return _Prepared([fwd.prepare(v=p["v"], out=out), vjp.prepare(v=p["v"], bar_out=p["bar_out"], bar_v=bar_v),
                          jvp.prepare(v=p["v"], dot_v=p["dot_v"], dot_out=dot_out)],
                         {"out": out, "bar_v": bar_v, "dot_out": dot_out})
    if kind == "orbit":
        n = case["n"]
        fwd, vjp = _unit("orbit", mode)
        o = {name: _empty(case, 3, n) for name in ("r", "v", "bar_r0", "bar_v0")}
        start = {"r0": p["r0"], "v0": p["v0"], "mu": 1.0}
        return _Prepared([fwd.prepare(**start, r=o["r"], v=o["v"]),
                          vjp.prepare(**start, bar_r=p["bar_r"], bar_v=p["bar_v"], bar_r0=o["bar_r0"],
                                      bar_v0=o["bar_v0"])], o)
    if kind == "solve":
        n = case["n"]
        fwd, vjp = _unit("solve", mode)
        o = {"x": _empty(case, 6, n), "bar_A": _empty(case, 6, 6, n), "bar_b": _empty(case, 6, n)}
        return _Prepared([fwd.prepare(A=p["A"], b=p["b"], x=o["x"]),
                          vjp.prepare(A=p["A"], b=p["b"], bar_x=p["bar_x"], bar_A=o["bar_A"], bar_b=o["bar_b"])], o)
    if kind == "matmul":
        n = case["n"]
        fwd, vjp = _unit("matmul", mode)
        o = {name: _empty(case, 16, 16, n) for name in ("C", "bar_A", "bar_B")}
        return _Prepared([fwd.prepare(A=p["A"], B=p["B"], C=o["C"]),
                          vjp.prepare(A=p["A"], B=p["B"], bar_C=p["bar_C"], bar_A=o["bar_A"], bar_B=o["bar_B"])], o)
    if kind == "chain":
        (k,) = _unit("chain", mode)
        o = {"y": _empty(case, case["n"]), "total": _empty(case, 1), "bins": _empty(case, case["cells"])}
        return _Prepared([k.prepare(x=p["x"], key=p["key"], **o)], o, (o["bins"],))
    if kind == "bins":
        fwd, vjp = _unit("bins", mode)
        o = {"acc": _empty(case, case["cells"]), "bar_x": _empty(case, case["n"])}
        return _Prepared([fwd.prepare(key=p["key"], x=p["x"], acc=o["acc"]),
                          vjp.prepare(key=p["key"], x=p["x"], bar_acc=p["bar_acc"], bar_x=o["bar_x"])], o,
                         (o["acc"],))
    if kind == "nets":
        fwd, vjp = _unit("nets", mode, case["samples"])
        o = {"out": _empty(case, case["nets"]), "bar_W": _empty(case, case["nets"] * E.NET_WEIGHTS)}
        read = {name: p[name] for name in ("W", "mask", "x", "y")}
        return _Prepared([fwd.prepare(**read, out=o["out"]),
                          vjp.prepare(**read, bar_out=p["bar_out"], bar_W=o["bar_W"])], o)
    if kind == "keyed":
        ordered, default = _unit("keyed", mode, case["samples"])
        o = {"ordered": _empty(case, case["keys"]), "default": _empty(case, case["keys"])}
        return _Prepared([ordered.prepare(x=p["x"], out=o["ordered"]), default.prepare(x=p["x"], out=o["default"])], o)
    (k,) = _unit("stats", mode)
    o = {name: _empty(case, 1) for name in ("total", "mean_sq", "low", "high", "ordered")}
    return _Prepared([k.prepare(x=p["x"], **o)], o)


def _prepare_runs(case, p):
    """Whole ``hawk.run`` calls: planes checked, bound and launched per call."""
    n = case["n"]
    first = case["kind"] == "rows"
    layout = {"layout": "samples_first"} if first else {}
    if first:                                     # (w, N) -> the program's own (N, w)
        p = {name: x.movedim(-1, 0).contiguous() for name, x in p.items()}

    def plane(*lead):
        return _empty(case, n, *lead) if first else _empty(case, *lead, n)

    if first and case["what"] == "solve":
        fwd, vjp = _unit("solve", case["mode"])
        o = {"x": plane(6), "bar_A": plane(6, 6), "bar_b": plane(6)}

        def step():
            hawk.run(fwd, A=p["A"], b=p["b"], x=o["x"], **layout)
            hawk.run(vjp, A=p["A"], b=p["b"], bar_x=p["bar_x"], bar_A=o["bar_A"], bar_b=o["bar_b"], **layout)
            return o
        return step
    fwd, vjp, jvp = _unit("energy", case["mode"])
    o = {"out": plane(), "bar_v": plane(3), "dot_out": plane()}

    def step():
        hawk.run(fwd, v=p["v"], out=o["out"], **layout)
        hawk.run(vjp, v=p["v"], bar_out=p["bar_out"], bar_v=o["bar_v"], **layout)
        hawk.run(jvp, v=p["v"], dot_v=p["dot_v"], dot_out=o["dot_out"], **layout)
        return o
    return step


def run(state):
    return state()


# -- what a pass cannot do without, and what its outputs are -----------------------

def work(case) -> dict:
    size = 4 if case["mode"] == "float32" else 8
    kind = case.get("what", case["kind"])
    if kind in ("calls", "energy"):               # v | v, bar_out | v, dot_v in; out | bar_v | dot_out out
        return {"bytes": case["n"] * 18 * size, "flops": case["n"] * 28}
    if kind == "orbit":                           # per substep: two accelerations and two kicks, and their reverse
        return {"bytes": case["n"] * 30 * size, "flops": case["n"] * (1280 + 4113)}
    if kind == "solve":
        return {"bytes": case["n"] * 138 * size, "flops": case["n"] * 632}
    if kind == "matmul":
        return {"bytes": case["n"] * 2048 * size, "flops": case["n"] * 3 * 8192}
    if kind == "chain":                           # x, key in, y out, every bin written
        return {"bytes": case["n"] * (2 * size + 4) + case["cells"] * size, "flops": case["n"] * 16}
    if kind == "bins":                            # key, x in, every cell out | key, x, cells in, bar_x out
        return {"bytes": case["n"] * (2 * 4 + 3 * size) + case["cells"] * 2 * size, "flops": case["n"] * 4}
    if kind == "nets":
        k, s = case["nets"], case["samples"]
        tables = E.NET_WEIGHTS + E.NET_UNITS
        return {"bytes": size * (2 * (2 * k * s + k * tables) + k * (2 + E.NET_WEIGHTS)), "flops": k * s * (287 + 603)}
    if kind == "keyed":                           # each policy's call reads every sample
        n = case["keys"] * case["samples"]
        return {"bytes": 2 * size * (n + case["keys"]), "flops": 2 * n}
    return {"bytes": case["n"] * size, "flops": case["n"] * 6}


#: About four times the largest relative error measured against ``exact`` over
#: 70 drawn cases (float32, float64).  A sum over every sample may cancel, and
#: a bin adds up to a 256th of the samples one after another.
TOLERANCE = {"stats": (5e-6, 1e-14), "bins": (1e-6, 1e-13), "chain": (1e-6, 1e-13), "keyed": (6e-7, 2e-15)}


def tolerance(case) -> dict:
    single, double = TOLERANCE.get(case["kind"], (3e-7, 2e-15))
    return {"rel": single if case["mode"] == "float32" else double}


# -- the same results in 64 bits, without this repository's code ---------------------

def _leapfrog(r, v, steps: int, dt: float):
    """``steps`` kick-drift-kick steps about a unit mass at the origin."""
    def pull(r):
        r2 = (r * r).sum(0)
        return -r / (r2 * r2.sqrt())
    for _ in range(steps):
        half = v + 0.5 * dt * pull(r)
        r = r + dt * half
        v = half + 0.5 * dt * pull(r)
    return r, v


def _blocks(n: int, block: int):
    return [slice(i, min(n, i + block)) for i in range(0, n, block)]


def _binned(key, value, cells: int):
    return torch.from_numpy(np.bincount(key.cpu().numpy(), value.cpu().numpy(), cells))


def exact(case, seed):
    kind = case["kind"]
    p = {name: x.double() if x.is_floating_point() else x for name, x in _inputs(case, seed).items()}
    what = case.get("what", kind)
    o = {}
    if what in ("calls", "energy"):
        o = {"out": 0.5 * (p["v"] * p["v"]).sum(0), "bar_v": p["bar_out"] * p["v"],
             "dot_out": (p["v"] * p["dot_v"]).sum(0)}
    elif what == "orbit":
        parts = []
        for s in _blocks(case["n"], 1 << 18):
            r0, v0 = (p[k][:, s].clone().requires_grad_() for k in ("r0", "v0"))
            r, v = _leapfrog(r0, v0, E.SUBSTEPS, E.DT)
            back = torch.autograd.grad((r, v), (r0, v0), (p["bar_r"][:, s], p["bar_v"][:, s]))
            parts.append((r.detach(), v.detach(), *back))
        o = dict(zip(("r", "v", "bar_r0", "bar_v0"), (torch.cat(x, dim=1) for x in zip(*parts))))
    elif what == "solve":
        parts = []
        for s in _blocks(case["n"], 1 << 18):
            a = p["A"][:, :, s].permute(2, 0, 1)
            a = 0.5 * (a + a.mT)
            inv = torch.linalg.inv(a)
            inv = inv + inv @ (torch.eye(6, dtype=torch.float64, device=DEVICE) - a @ inv)   # one refinement
            x = (inv * p["b"][:, s].T[:, None, :]).sum(-1)
            lam = (inv * p["bar_x"][:, s].T[:, None, :]).sum(-1)
            outer = lam[:, :, None] * x[:, None, :]
            parts.append((x.T, (-0.5 * (outer + outer.mT)).permute(1, 2, 0), lam.T))
        o = dict(zip(("x", "bar_A", "bar_b"), (torch.cat(x, dim=-1).contiguous() for x in zip(*parts))))
    elif what == "matmul":
        o = {name: torch.empty(16, 16, case["n"], dtype=torch.float64, device=DEVICE) for name in ("C", "bar_A", "bar_B")}
        for s in _blocks(case["n"], 1 << 16):
            a, b, c = (p[k][:, :, s].permute(2, 0, 1).contiguous() for k in ("A", "B", "bar_C"))
            o["C"][:, :, s] = torch.bmm(a, b).permute(1, 2, 0)
            o["bar_A"][:, :, s] = torch.bmm(c, b.mT.contiguous()).permute(1, 2, 0)
            o["bar_B"][:, :, s] = torch.bmm(a.mT.contiguous(), c).permute(1, 2, 0)
    elif what == "chain":
        x = p["x"]
        t4 = torch.tanh(1.5 * torch.sin(torch.exp(x)) + 0.25)
        t6 = torch.sqrt(t4.abs() + 1.0).square() - x
        y = torch.exp(-t6.abs()) * x + t4
        o = {"y": y, "total": y.sum().reshape(1), "bins": _binned(p["key"], y, case["cells"])}
    elif what == "bins":
        key, x = p["key"].long(), p["x"]
        o = {"acc": _binned(key, x * x, case["cells"]), "bar_x": 2.0 * x * p["bar_acc"][key]}
    elif what == "nets":
        k, s = case["nets"], case["samples"]
        w = p["W"].reshape(k, E.NET_UNITS, 3).requires_grad_()
        x, y, mask = p["x"].reshape(k, s), p["y"].reshape(k, s), p["mask"].reshape(k, E.NET_UNITS)
        pred = torch.zeros_like(x)
        for h in range(E.NET_UNITS):
            act = torch.tanh(w[:, h, 0, None] * x + w[:, h, 1, None])
            pred = pred + mask[:, h, None] * w[:, h, 2, None] * act
        loss = (pred - y).square().sum(1)
        (bar_w,) = torch.autograd.grad(loss, w, p["bar_out"])
        o = {"out": loss.detach(), "bar_W": bar_w.reshape(-1)}
    elif what == "keyed":
        sums = p["x"].reshape(case["keys"], case["samples"]).sum(1)
        o = {"ordered": sums, "default": sums}
    else:
        x = p["x"]
        o = {"total": x.sum().reshape(1), "mean_sq": (x * x).mean().reshape(1), "low": x.min().reshape(1),
             "high": x.max().reshape(1), "ordered": x.sum().reshape(1)}
    if kind == "rows":
        o = {name: x.movedim(-1, 0).contiguous() for name, x in o.items()}
    return o
