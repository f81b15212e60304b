"""The work whose speed this repository watches, as calls of its public entry points.

A case is a dict of plain values with a "kind":

  advect    fidibench_amd.Upwind: `steps` upwind steps of a field that stays on
            the GPU.  time_block 1 is the class's default (one launch per step,
            as the reference steps), 0 the library's own split into fused passes.
  run       the same with the checksum the upwindCxx program prints at its end.
  forward   autograd.advect of a torch tensor without a gradient (a model
            evaluation, the run that makes a misfit's target).
  gradient  autograd.advect + autograd.misfit + backward: loss, dL/df0, dL/dv.
  filter    fidibench_amd.Filter: `steps` applications of a star stencil
            (laplacian's 2nd- and 4th-order shapes, as a diffusion step, which
            stays bounded), the output read back and its checksum.

Grids are n0 x n1 x n2 (n0 = 0: two axes).  A pass of advect, run and filter
continues from the state the pass before it left, as a simulation does.
"""
from __future__ import annotations

import math

import torch

import fidibench_amd
from fidibench_amd import _lib as L
from fidibench_amd import autograd, configs

SIZE = {"f64": 8, "f32": 4, "bf16": 2, "bf16sr": 2}
TORCH = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16,
         "bf16sr": torch.bfloat16}


def _case(name, kind, dtype, n, steps, **more):
    n0, n1, n2 = n
    return {"name": name, "kind": kind, "dtype": dtype, "n0": n0, "n1": n1, "n2": n2,
            "steps": steps, **more}


def listed():
    return [
        # A small box stepped by an interactive or coupled program: launches
        # and their latency are all there is.
        _case("small_default", "advect", "f64", (32, 24, 40), 10, time_block=1),
        # The same kind of call at an ordinary small size, split by the library.
        _case("cube96_auto", "advect", "f64", (96, 96, 96), 20, time_block=0),
        # What `upwindCxx` does with its default options: 128^3, 10 steps, checksum.
        _case("upwindCxx_default", "run", "f64", (128, 128, 128), 10, time_block=1),
        # The benchmark's headline: 512^3 in the reference's precision.
        _case("cube512_auto", "advect", "f64", (512, 512, 512), 20, time_block=0),
        # Single precision on a grid whose axes fit no tile.
        _case("ragged_f32_auto", "advect", "f32", (257, 300, 390), 25, time_block=0),
        # The mixed-precision run in its largest box, stochastically rounded.
        _case("cube1024_bf16sr", "advect", "bf16sr", (1024, 1024, 1024), 8, time_block=0),
        # One launch per step over a field far larger than the caches.
        _case("default_f32_large", "advect", "f32", (768, 512, 640), 4, time_block=1),
        # Upwind<2>: a plane, as a 2-D run of the reference class.
        _case("plane_2d", "advect", "f64", (0, 2000, 3000), 40, time_block=0),
        # A torch program evaluating the forward model.
        _case("torch_forward", "forward", "f64", (192, 200, 210), 30),
        # The misfit gradient at its test size, by the default method.
        _case("gradient_256", "gradient", "f64", (256, 256, 256), 50, method="shift", slots=0),
        # The checkpointed gradient with room for a few states only.
        _case("gradient_checkpoint", "gradient", "f32", (120, 161, 192), 40,
              method="checkpoint", slots=10),
        # The 4th-order Laplacian's stencil in 3-D, read back as laplacian does.
        _case("filter_3d", "filter", "f64", (160, 144, 150), 20, order=4),
    ]


# Cells x steps of the largest listed case, which no drawn one exceeds.
_MOST_UPDATES = 512 ** 3 * 20


def _grid(rng, lo, hi, nd):
    """An nd-axis grid of about exp(U(log lo, log hi)) cells, axes within a
    factor of four of each other, of any divisibility."""
    cells = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    skew = [rng.uniform(-0.5, 0.5) for _ in range(nd)]
    mean = sum(skew) / nd
    n = [max(4, round(cells ** (1.0 / nd) * 2.0 ** (s - mean))) for s in skew]
    if rng.random() < 0.3:  # a power of two along one axis, as many users choose
        k = rng.randrange(nd)
        n[k] = 2 ** max(2, round(math.log2(n[k])))
    return tuple(n) if nd == 3 else (0,) + tuple(n)


def draw(rng):
    kind = rng.choice(["advect", "advect", "advect", "plane", "run", "forward", "gradient",
                       "filter"])
    if kind == "advect":
        dtype = rng.choice(["f64", "f64", "f32", "bf16", "bf16sr"])
        n = _grid(rng, 2 ** 13, 2 ** 28, 3)
        steps = round(math.exp(rng.uniform(0.0, math.log(40))))
        c = _case("", kind, dtype, n, steps, time_block=rng.choice([0, 0, 1]))
    elif kind == "plane":
        n = _grid(rng, 2 ** 12, 2 ** 25, 2)
        c = _case("", "advect", rng.choice(["f64", "f64", "f32"]), n, rng.randint(5, 60),
                  time_block=rng.choice([0, 0, 1]))
    elif kind == "run":
        c = _case("", kind, rng.choice(["f64", "f64", "f32"]), _grid(rng, 2 ** 13, 2 ** 24, 3),
                  rng.randint(1, 20), time_block=rng.choice([0, 1]))
    elif kind == "forward":
        c = _case("", kind, rng.choice(["f64", "f32", "bf16"]), _grid(rng, 2 ** 13, 2 ** 25, 3),
                  rng.randint(2, 50))
    elif kind == "gradient":
        method = rng.choice(["shift", "shift", "checkpoint"])
        c = _case("", kind, rng.choice(["f64", "f32"]), _grid(rng, 2 ** 13, 2 ** 24, 3),
                  rng.randint(3, 50), method=method,
                  slots=rng.randint(2, 40) if method == "checkpoint" else 0)
    else:
        nd = rng.choice([2, 3])
        c = _case("", kind, "f64", _grid(rng, 2 ** 12, 2 ** 22, nd), rng.randint(1, 40),
                  order=rng.choice([2, 4]))
    c.pop("name")
    cells = max(1, c["n0"]) * c["n1"] * c["n2"]
    c["steps"] = max(1, min(c["steps"], _MOST_UPDATES // cells))
    return c


# ------------------------------------------------------------------ inputs

def _shape(case):
    return tuple(case[k] for k in ("n0", "n1", "n2") if case[k])


def _velocity(case, seed):
    """Seeded components of magnitude 0.1 to 1 and either sign."""
    n = len(_shape(case))
    u = [configs.uniform(seed + 1000, k) for k in range(2 * n)]
    return tuple((0.1 + 0.9 * u[k]) * (1.0 if u[n + k] < 0.5 else -1.0) for k in range(n))


def _dt(case, v):
    shape = _shape(case)
    return configs.cfl_dt(shape, v, (1.0,) * len(shape))


def _sphere(case):
    """A ball (disc) of radius 0.25 with 1 % noise: init_field's parameters."""
    return (0.5, 0.5, 0.5, 0.25, 0.01)


def _init(case, seed, dtype):
    """The initial field as a tensor, from the library's device generator."""
    shape = _shape(case)
    f = torch.empty(shape, dtype=TORCH[dtype], device="cuda")
    L.check(L.lib().fdb_init_field_dev(len(shape), L.u64s(shape), L.dbls((1.0,) * len(shape)),
                                       L.DTYPES[dtype], L.INIT_SPHERE, L.dbls(_sphere(case)), 5,
                                       seed, f.data_ptr(),
                                       torch.cuda.current_stream().cuda_stream))
    return f


def _stencil(case):
    """A diffusion step: 1 + 0.1 h^2 Laplacian, of 2nd or 4th order."""
    nd = len(_shape(case))
    taps = {1: 1.0} if case["order"] == 2 else {1: 16.0 / 12.0, 2: -1.0 / 12.0}
    centre = -2.0 if case["order"] == 2 else -30.0 / 12.0
    st = {(0,) * nd: 1.0 + 0.1 * nd * centre}
    for a in range(nd):
        for k, w in taps.items():
            for o in (k, -k):
                st[tuple(o if b == a else 0 for b in range(nd))] = 0.1 * w
    return st


def _filter_input(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.rand(_shape(case), generator=g, device="cuda", dtype=torch.float64)


class _View:
    """A handle's device buffer as torch sees it (__cuda_array_interface__).
    The tensor made from it holds this object, and so the handle, whose end
    would free the buffer."""

    def __init__(self, up, ptr, typestr):
        self.owner = up
        self.__cuda_array_interface__ = {"shape": up.numCells, "typestr": typestr,
                                         "data": (ptr, False), "version": 3}


def _field(state):
    """The handle's current field as a tensor (no copy); one view per buffer."""
    up, views = state["up"], state["views"]
    p = up.device_ptr()
    if p not in views:
        ts = {"f64": "<f8", "f32": "<f4"}.get(state["dtype"], "<i2")
        t = torch.as_tensor(_View(up, p, ts), device="cuda")
        views[p] = t.view(torch.bfloat16) if ts == "<i2" else t
    return views[p]


def prepare(case, seed):
    kind, shape = case["kind"], _shape(case)
    state = {"kind": kind, "dtype": case["dtype"], "steps": case["steps"]}
    if kind == "filter":
        flt = fidibench_amd.Filter(shape, [0.0] * len(shape), [1.0] * len(shape),
                                   _stencil(case))
        flt.setInData(_filter_input(case, seed).cpu().numpy())
        state["flt"] = flt
        return state
    v = _velocity(case, seed)
    state["dt"] = _dt(case, v)
    if kind in ("advect", "run"):
        up = fidibench_amd.Upwind(v, (1.0,) * len(shape), shape, dtype=case["dtype"])
        if case["time_block"] != 1:
            up.set_time_block(case["time_block"])
        up.init_field(L.INIT_SPHERE, _sphere(case), seed=seed)
        if case["dtype"] == "bf16sr":
            up.set_seed(seed)
        state.update(up=up, views={})
        return state
    state["f0"] = _init(case, seed, case["dtype"])
    state["v"] = torch.tensor(v, dtype=torch.float64)
    if kind == "gradient":
        state["method"] = case["method"]
        if case["slots"]:  # the working set (4 fields) and this many states
            state["max_bytes"] = (4 + case["slots"]) * state["f0"].numel() * SIZE[case["dtype"]]
        else:
            state["max_bytes"] = None
        state["target"] = _init(case, seed + 1, case["dtype"])
        state["f0"].requires_grad_(True)
        state["v"].requires_grad_(True)
    return state


def run(state):
    kind = state["kind"]
    if kind == "advect":
        state["up"].advect(state["steps"], state["dt"])
        return {"field": _field(state)}
    if kind == "run":
        state["up"].advect(state["steps"], state["dt"])
        return {"field": _field(state), "checksum": state["up"].checksum()}
    if kind == "forward":
        with torch.no_grad():
            return {"field": autograd.advect(state["f0"], state["v"], state["dt"],
                                             state["steps"])}
    if kind == "gradient":
        fT = autograd.advect(state["f0"], state["v"], state["dt"], state["steps"],
                             max_bytes=state["max_bytes"], method=state["method"])
        loss = autograd.misfit(fT, state["target"])
        df0, dv = torch.autograd.grad(loss, (state["f0"], state["v"]))
        return {"loss": loss.detach(), "df0": df0, "dv": dv}
    flt = state["flt"]
    flt.iterate(state["steps"])
    return {"output": flt.get_data("output"), "checksum": flt.computeCheckSum("output")}


def work(case):
    """Bytes: the field read once and written once (a gradient also reads the
    target and f0 again and writes dL/df0).  Flops: 9 per cell and upwind step
    (three differences, products and subtractions), 18 with the transpose
    step; two per stencil term."""
    cells = max(1, case["n0"]) * case["n1"] * case["n2"]
    size, nd = SIZE[case["dtype"]], len(_shape(case))
    if case["kind"] == "filter":
        terms = 1 + nd * (2 if case["order"] == 2 else 4)
        return {"bytes": 16 * cells, "flops": 2 * terms * cells * case["steps"]}
    if case["kind"] == "gradient":
        return {"bytes": 4 * size * cells, "flops": 2 * 3 * nd * cells * case["steps"]}
    return {"bytes": 2 * size * cells, "flops": 3 * nd * cells * case["steps"]}


# ------------------------------------------------- the same in 64 bits, in torch

def _upstream(f, ups):
    """The upwind neighbour's value along each axis."""
    return [torch.roll(f, -u, dims=j) for j, u in enumerate(ups)]


def _step(f, coef, ups):
    g = f.clone()
    for c, n in zip(coef, _upstream(f, ups)):
        g -= c * (n - f)
    return g


def exact(case, seed):
    kind, shape = case["kind"], _shape(case)
    if kind == "filter":
        x = _filter_input(case, seed)
        for _ in range(case["steps"]):
            y = torch.zeros_like(x)
            for off, w in sorted(_stencil(case).items()):
                y += w * _gather(x, off)
            x = y
        out = x.cpu()
        return {"output": out, "checksum": float(out.sum())}
    v = _velocity(case, seed)
    dt = _dt(case, v)
    ups = [1 if c < 0.0 else -1 for c in v]
    coef = [dt * c * u / (1.0 / n) for c, u, n in zip(v, ups, shape)]
    f = _init(case, seed, case["dtype"]).double()
    if kind != "gradient":
        for _ in range(case["steps"]):
            f = _step(f, coef, ups)
        if kind == "run":
            return {"field": f, "checksum": float(f.sum())}
        return {"field": f}
    states = []
    for _ in range(case["steps"]):
        states.append(f)
        f = _step(f, coef, ups)
    lam = f - _init(case, seed + 1, case["dtype"]).double()
    loss = 0.5 * (lam * lam).sum()
    dots = [0.0] * len(shape)
    for f in reversed(states):
        for j, n in enumerate(_upstream(f, ups)):
            dots[j] += float((lam * (n - f)).sum())
        lam = _step(lam, coef, [-u for u in ups])
    dv = [-(dt * u / (1.0 / n)) * d for u, n, d in zip(ups, shape, dots)]
    return {"loss": loss, "df0": lam, "dv": torch.tensor(dv, dtype=torch.float64)}


def _gather(x, off):
    """x at the neighbour `off` with the reference's unsigned wrap: index -k of
    an n-cell axis is (2^64 - k) mod n."""
    for a, o in enumerate(off):
        if o:
            n = x.shape[a]
            at = [(i + o) % n if i + o >= 0 else (2 ** 64 + i + o) % n for i in range(n)]
            x = x.index_select(a, torch.tensor(at, device=x.device))
    return x
