"""The timed cases: what a user of this framework has it do, through its public API.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)` another one
of the ranges they stand for.  Three kinds of calls:

* "plan": a time loop on a device-resident grid (`Plan.run`), the state left on the device
  for the program's next use.  A pass advances the state by `steps` physical steps, as one
  iteration of a simulation's outer loop does; its output is the whole padded array.
* "batch": many independent 2-D grids (`Batch.run`), then every grid downloaded, which is
  the only way a program gets at a batch's results.
* "host": the one-shot call on host arrays (`run`), which is what the reference's own
  launchers do: plan, upload, time loop, download.

Weights are uniform in (0, 1) and normalised to sum 1, grids uniform in [-1, 1), as in the
benchmark.  `exact` steps the same inputs with plain torch in 64 bits.
"""
import math

import numpy as np
import torch

import convstencil_amd as cs

# name -> (dimensions, radius, taps on the axes only)
STENCILS = {
    "1d1r": (1, 1, False),
    "1d2r": (1, 2, False),
    "star2d1r": (2, 1, True),
    "box2d1r": (2, 1, False),
    "star2d3r": (2, 3, True),
    "box2d3r": (2, 3, False),
    "star3d1r": (3, 1, True),
    "box3d1r": (3, 1, False),
}


def _taps(shape):
    """Tap offsets, row-major, slowest axis first."""
    ndim, r, star = STENCILS[shape]
    return [o for o in np.ndindex(*([2 * r + 1] * ndim)) if not star or sum(v != r for v in o) <= 1]


def _plan(name, shape, sizes, steps, precision="fp64", graph=False, halo="zero"):
    ndim = STENCILS[shape][0]
    n = [1] * (3 - ndim) + list(sizes)
    return {"name": name, "kind": "plan", "shape": shape, "nz": n[0], "ny": n[1], "nx": n[2], "steps": steps,
            "precision": precision, "graph": graph, "halo": halo}


def listed():
    return [
        # a small 2-D grid advanced a few steps, the size and step count of the smoke run: launch latency
        _plan("box2d1r_300x517", "box2d1r", [300, 517], 10),
        # the 1-D workload of the benchmark
        _plan("1d1r_1m", "1d1r", [1 << 20], 64),
        # an ordinary, ragged 2-D grid that fits the Infinity Cache, with an odd step count
        _plan("box2d1r_1531x2749", "box2d1r", [1531, 2749], 50),
        # the benchmark's headline workload: a large 2-D grid, captured in a graph
        _plan("box2d1r_10240", "box2d1r", [10240, 10240], 64, graph=True),
        # the benchmark's radius-3 workloads: the 13-point star and the 49-point box
        _plan("star2d3r_8192", "star2d3r", [8192, 8192], 64, graph=True),
        _plan("box2d3r_8192", "box2d3r", [8192, 8192], 64, graph=True),
        # the 49-point box in the split-precision form that trades accuracy for speed
        _plan("box2d3r_8192_fp16w3", "box2d3r", [8192, 8192], 64, precision="fp16w3", graph=True),
        # the reference programs' own kind of run: the 49 weights and a halo that is not zero
        _plan("box2d3r_5120_halo", "box2d3r", [5120, 5120], 20, halo="random"),
        # the benchmark's 3-D box, and the 3-D star on a ragged, smaller grid
        _plan("box3d1r_512", "box3d1r", [512, 512, 512], 32, graph=True),
        _plan("star3d1r_389x301x517", "star3d1r", [389, 301, 517], 40),
        # uneven grids with mixed stencils, sides log-uniform in [128, 2048], downloaded at the end
        {"name": "batch_24", "kind": "batch", "grids": 24, "steps": 500, "graph": True, "sides": 11},
        # one call on host arrays
        {"name": "host_box2d1r_2048", "kind": "host", "shape": "box2d1r", "nz": 1, "ny": 2048, "nx": 2048, "steps": 100,
         "halo": "zero"},
    ]


MOST_FLOPS = 4.0e11  # the largest listed case has 4.2e11
MOST_CELLS = 10240 * 10240


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plan"] * 8 + ["batch", "host"])
    if kind == "batch":
        return {"kind": "batch", "grids": rng.randint(8, 32), "steps": rng.randint(50, 500),
                "graph": rng.random() < 0.5, "sides": rng.randrange(1 << 20)}
    if kind == "host":
        shape = rng.choice(["box2d1r", "star2d1r", "box2d3r", "star2d3r"])
        sizes = [_size(rng, 64, 4096), _size(rng, 64, 4096)]
    else:
        shape = rng.choice(list(STENCILS))
        ndim = STENCILS[shape][0]
        lo, hi = {1: (1 << 12, 1 << 24), 2: (96, 10240), 3: (24, 640)}[ndim]
        sizes = [_size(rng, lo, hi) for _ in range(ndim)]
    while math.prod(sizes) > MOST_CELLS:
        k = max(range(len(sizes)), key=lambda i: sizes[i])
        sizes[k] = sizes[k] * 2 // 3 + 1
    per_step = 2.0 * len(_taps(shape)) * math.prod(sizes)
    steps = max(1, min(_size(rng, 4, 128), int(MOST_FLOPS / per_step)))
    halo = "random" if rng.random() < 0.2 else "zero"
    n = [1] * (3 - len(sizes)) + sizes
    if kind == "host":
        return {"kind": "host", "shape": shape, "nz": n[0], "ny": n[1], "nx": n[2], "steps": steps, "halo": halo}
    precision = rng.choice(["fp64", "fp64", "fp16w3", "bf16x3"]) if shape == "box2d3r" else "fp64"
    c = _plan("", shape, sizes, steps, precision=precision, graph=rng.random() < 0.5, halo=halo)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs from the seed

def _generator(seed, device="cpu"):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _weights(shape, seed):
    """One weight per tap, uniform in (0, 1), sum 1."""
    w = torch.rand(len(_taps(shape)), generator=_generator(seed), dtype=torch.float64).numpy()
    return w / w.sum()


def _dense(shape, w):
    ndim, r, _ = STENCILS[shape]
    cube = np.zeros((2 * r + 1,) * ndim)
    for o, v in zip(_taps(shape), w):
        cube[o] = v
    return cube.reshape(-1)


def _layout(case):
    ndim, r, _ = STENCILS[case["shape"]]
    # the reference's 2-D arrays have rows two cells longer than the halos need
    return cs.Layout.with_halo([case["nz"], case["ny"], case["nx"]][3 - ndim:], r,
                               2 if case["halo"] == "random" and ndim == 2 else 0)


def _interior(shape, v, n):
    """View of the interior of a padded array (numpy or torch) of interior sizes n."""
    r = STENCILS[shape][1]
    return v[tuple(slice(r, r + s) for s in n)]


def _sizes(case):
    return [case["nz"], case["ny"], case["nx"]][3 - STENCILS[case["shape"]][0]:]


def _ext(case):
    ndim, r, _ = STENCILS[case["shape"]]
    e = [s + 2 * r for s in _sizes(case)]
    if case["halo"] == "random" and ndim == 2:
        e[-1] += 2
    return e


def _device_interior(case, seed):
    """Interior cells of a zero-halo grid, made on the device."""
    x = torch.rand(_sizes(case), generator=_generator(seed, "cuda"), device="cuda", dtype=torch.float64)
    return x.mul_(2.0).sub_(1.0)


def _host_grid(shape, ext, n, halo, seed):
    """A padded host array: random everywhere, or only inside."""
    rng = np.random.default_rng(int(seed))
    if halo == "random":
        return rng.uniform(-1.0, 1.0, ext)
    a = np.zeros(ext)
    _interior(shape, a, n)[...] = rng.uniform(-1.0, 1.0, n)
    return a


def _batch_grids(case):
    """(shape, sides) of every grid of a batch."""
    rng = np.random.default_rng(case["sides"])
    sides = np.exp(rng.uniform(math.log(128), math.log(2048), (case["grids"], 2))).astype(int)
    shapes = rng.choice(["box2d1r", "star2d3r"], case["grids"])
    return [(str(s), [int(a), int(b)]) for s, (a, b) in zip(shapes, sides)]


# ------------------------------------------------------------------ the calls

class _Buffer:
    """One of a plan's device buffers, for torch to look at."""

    def __init__(self, plan, ptr, ext):
        self.plan = plan  # the buffer lives as long as its plan
        self.__cuda_array_interface__ = {"shape": tuple(ext), "typestr": "<f8", "data": (ptr, False), "version": 2}


def prepare(case, seed):
    if case["kind"] == "host":
        shape, n = case["shape"], _sizes(case)
        return {"kind": "host", "layout": _layout(case), "radius": STENCILS[shape][1],
                "weights": _dense(shape, _weights(shape, seed)), "steps": case["steps"],
                "x": _host_grid(shape, _ext(case), n, case["halo"], seed)}
    if case["kind"] == "batch":
        grids = _batch_grids(case)
        layouts = [cs.Layout.with_halo(n, STENCILS[s][1]) for s, n in grids]
        b = cs.Batch(layouts, [STENCILS[s][1] for s, _ in grids],
                     [_dense(s, _weights(s, seed + i)) for i, (s, _) in enumerate(grids)], use_graph=case["graph"])
        for i, (s, n) in enumerate(grids):
            b.upload(i, _host_grid(s, layouts[i].ext[1:], n, "zero", seed + i))
        return {"kind": "batch", "batch": b, "grids": len(grids), "steps": case["steps"]}
    shape = case["shape"]
    p = cs.Plan(_layout(case), STENCILS[shape][1], _dense(shape, _weights(shape, seed)), precision=case["precision"],
                use_graph=case["graph"])
    if case["halo"] == "random":
        p.upload(_host_grid(shape, _ext(case), _sizes(case), "random", seed))
    cur, other = p.device_buffers()
    views = {q: torch.as_tensor(_Buffer(p, q, _ext(case)), device="cuda") for q in (cur, other)}
    if case["halo"] == "zero":
        _interior(shape, views[cur], _sizes(case)).copy_(_device_interior(case, seed))
        torch.cuda.synchronize()  # the plan works on a stream of its own
    return {"kind": "plan", "plan": p, "views": views, "steps": case["steps"]}


def run(state):
    if state["kind"] == "host":
        return cs.run(state["layout"], state["radius"], state["weights"], state["x"], state["steps"])[0]
    if state["kind"] == "batch":
        state["batch"].run(state["steps"])
        return [state["batch"].download(i) for i in range(state["grids"])]
    state["plan"].run(state["steps"])
    return state["views"][state["plan"].device_buffers()[0]]


def work(case):
    """The grid read once and written once; one multiply-add per tap, cell and step."""
    grids = _batch_grids(case) if case["kind"] == "batch" else [(case["shape"], _sizes(case))]
    cells = sum(math.prod(n) for _, n in grids)
    flops = sum(2.0 * len(_taps(s)) * math.prod(n) for s, n in grids) * case["steps"]
    return {"bytes": 16.0 * cells, "flops": flops}


def _stepped(shape, w, a, n, steps):
    """`steps` steps of the padded array `a`: two buffers in turn, the second all zero at first, only the
    interior written."""
    b = torch.zeros_like(a)
    for _ in range(steps):
        out = _interior(shape, b, n)
        out.zero_()
        for o, v in zip(_taps(shape), w):
            out.add_(a[tuple(slice(k, k + s) for k, s in zip(o, n))], alpha=float(v))
        a, b = b, a
    return a


def exact(case, seed):
    if case["kind"] == "batch":
        got = []
        for i, (s, n) in enumerate(_batch_grids(case)):
            r = STENCILS[s][1]
            x = torch.from_numpy(_host_grid(s, [v + 2 * r for v in n], n, "zero", seed + i)).cuda()
            got.append(_stepped(s, _weights(s, seed + i), x, n, case["steps"]).reshape(-1).cpu().numpy())
        return got
    shape, n = case["shape"], _sizes(case)
    if case["kind"] == "host" or case["halo"] == "random":
        a = torch.from_numpy(_host_grid(shape, _ext(case), n, case["halo"], seed)).cuda()
    else:
        a = torch.zeros(_ext(case), device="cuda", dtype=torch.float64)
        _interior(shape, a, n).copy_(_device_interior(case, seed))
    a = _stepped(shape, _weights(shape, seed), a, n, case["steps"])
    return a.reshape(-1).cpu().numpy() if case["kind"] == "host" else a
