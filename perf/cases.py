"""Performance cases of the brick-stencil library: the calls a solver built on it makes.

Each case is one of

  steps    a time-stepping loop: ``sweeps`` of a 7/13/25-point star, the cond stencil or the
           125-point cube, on a ghost zone refreshed by its own copies ("separate"), by the sweep's
           own stores ("fused"), or on a wrapped box without ghosts ("none")
  apply    one stencil application, ``sweep``
  convert  ``copyToBrick`` of a padded array and ``copyFromBrick`` of another field: the way in and
           the way out of brick storage
  monitor  ``PeriodicGrid.stats`` and ``compare``: what a solver asks between steps
  batch    ``Batch.run`` of many independent boxes of mixed stencils and element types

Fields hold uniform values in [-1, 1) as the library's tests and benchmark use.  Star coefficients are
the symmetric normalised ones of ``Stencil.make``; the cube's are positive and sum to 1, so a long run
smooths the field and does not shrink it to nothing.
"""
import math
import random

import numpy as np
import torch

import bricklib_amd as bk
from bricklib_amd import batch as bkb

DTYPES = {"f64": (bk.BK_F64, torch.float64, "<f8"), "f32": (bk.BK_F32, torch.float32, "<f4"),
          "bf16": (bk.BK_BF16, torch.bfloat16, "<i2")}
STENCILS = ("7pt", "13pt", "25pt", "cond", "125pt")
FLOPS = {"7pt": 13, "13pt": 25, "25pt": 49, "cond": 13, "125pt": 249}
LAYOUT_EXTENTS = {0: (8, 8, 8), 1: (4, 8, 16), 2: (4, 8, 16)}  # (k, j, i) cells of a brick


def listed():
    return [
        # the library's benchmark: a 512^3 diffusion run in double, ghost refresh fused
        dict(name="steps 7pt f64 512", do="steps", stencil="7pt", dtype="f64", ni=64, nj=64, nk=64,
             sweeps=100, refresh="fused", graph=True),
        # a ragged production box in single, ghosts refreshed by their own copies
        dict(name="steps 7pt f32 ragged", do="steps", stencil="7pt", dtype="f32", ni=45, nj=27, nk=33,
             sweeps=25, refresh="separate", graph=True),
        # half-size storage on a wrapped box, queued without a graph
        dict(name="steps 7pt bf16 256", do="steps", stencil="7pt", dtype="bf16", ni=32, nj=32, nk=32,
             sweeps=20, refresh="none", graph=False),
        # a small box: the smallest request size of the serving workload, many steps
        dict(name="steps cond f64 32", do="steps", stencil="cond", dtype="f64", ni=4, nj=4, nk=4,
             sweeps=50, refresh="fused", graph=True),
        # higher-order operators
        dict(name="steps 13pt f64 ragged", do="steps", stencil="13pt", dtype="f64", ni=19, nj=50,
             nk=23, sweeps=8, refresh="none", graph=False),
        dict(name="steps 25pt f32 384", do="steps", stencil="25pt", dtype="f32", ni=48, nj=48, nk=48,
             sweeps=10, refresh="separate", graph=True),
        # the dense 5x5x5 operator: a large run, and one application to a small box
        dict(name="steps 125pt f64 256", do="steps", stencil="125pt", dtype="f64", ni=32, nj=32,
             nk=32, sweeps=10, refresh="none", graph=True),
        dict(name="apply 125pt f32 64", do="apply", stencil="125pt", dtype="f32", ni=8, nj=8, nk=8,
             layout=0, refresh="separate"),
        # the smallest call: one application to a 16^3 box
        dict(name="apply 7pt f64 16", do="apply", stencil="7pt", dtype="f64", ni=2, nj=2, nk=2,
             layout=0, refresh="separate"),
        # array in, array out, the array padded unevenly
        dict(name="convert f64 ragged", do="convert", dtype="f64", ni=50, nj=33, nk=39, pad_i=8,
             pad_j=3, pad_k=1),
        # residual and norms of a single-precision field against a double one
        dict(name="monitor f32 256", do="monitor", dtype="f32", reference="f64", ni=32, nj=32, nk=32),
        # the serving mix: boxes of 32..256 cells an edge, every stencil, up to 16 sweeps each
        dict(name="batch mixed 24", do="batch", requests=24, most=32, ticks=16, mix=7),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _box(rng, most_cells, di=8, dj=8, dk=8):
    """Bricks per axis of a ragged box, 16 to 512 cells an edge and at most most_cells cells."""
    while True:
        edge = math.exp(rng.uniform(math.log(16), math.log(400)))
        n = [max(1, min(512 // d, int(round(edge * math.exp(rng.uniform(-0.5, 0.5)) / d))))
             for d in (di, dj, dk)]
        if n[0] * n[1] * n[2] * di * dj * dk <= most_cells:
            return n


def draw(rng: random.Random):
    """One more case of the listed ones' kinds and ranges."""
    do = rng.choice(["steps"] * 6 + ["apply"] * 3 + ["convert", "monitor", "batch"])
    dtype = rng.choice(["f64", "f64", "f32", "f32", "bf16"])
    if do == "batch":
        return dict(do=do, requests=rng.randint(4, 32), most=rng.choice([8, 16, 24, 32]),
                    ticks=rng.choice([4, 8, 16]), mix=rng.randrange(1 << 20))
    if do == "convert":
        ni, nj, nk = _box(rng, 6 << 23)
        return dict(do=do, dtype=dtype, ni=ni, nj=nj, nk=nk, pad_i=rng.choice([0, 1, 4, 8]),
                    pad_j=rng.randint(0, 8), pad_k=rng.randint(0, 8))
    if do == "monitor":
        ni, nj, nk = _box(rng, 4 << 23)
        return dict(do=do, dtype=dtype, reference=rng.choice(["f64", dtype]), ni=ni, nj=nj, nk=nk)
    stencil = rng.choice(["7pt", "7pt", "13pt", "25pt", "cond", "125pt"])
    if do == "apply":
        layout = rng.choice([0, 0, 0, 0, 1, 2])
        bk_, bj, bi = LAYOUT_EXTENTS[layout]
        ni, nj, nk = _box(rng, (1 << 23 if stencil == "125pt" else 6 << 23), bi, bj, bk_)
        return dict(do=do, stencil=stencil, dtype=dtype, ni=ni, nj=nj, nk=nk, layout=layout,
                    refresh=rng.choice(["separate", "none"]))
    ni, nj, nk = _box(rng, (1 << 24 if stencil == "125pt" else 6 << 23))
    cells = ni * nj * nk * 512
    most = (1 << 31) // FLOPS[stencil] * 13 // cells  # updates, weighed by what each costs
    refresh = rng.choice(["separate", "none"] if stencil == "125pt" else
                         ["fused", "separate", "none"])
    return dict(do=do, stencil=stencil, dtype=dtype, ni=ni, nj=nj, nk=nk,
                sweeps=_log_int(rng, 1, max(1, min(100, most))), refresh=refresh,
                graph=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# fields
# ---------------------------------------------------------------------------
class _Memory:
    """Device memory of the library as torch sees it."""

    def __init__(self, buf, shape, typestr, ptr=None):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "version": 2,
                                         "data": (int(ptr if ptr is not None else buf.ptr), False)}


def _view(buf, shape, dtype, ptr=None):
    _, tdt, code = DTYPES[dtype]
    t = torch.as_tensor(_Memory(buf, shape, code, ptr), device="cuda")
    return t.view(tdt) if dtype == "bf16" else t


def _interior(t, g):
    """The interior bricks (nk, nj, ni, 512) of a field's bricks (nbricks, 512)."""
    ni, nj, nk = g.padded
    t = t.view(nk, nj, ni, 512)
    return t[1:-1, 1:-1, 1:-1] if g.ghost else t


def _to_bricks(x, layout=0):
    """A (k, j, i) array as bricks (nk, nj, ni, 512)."""
    ek, ej, ei = LAYOUT_EXTENTS[layout]
    nk, nj, ni = x.shape[0] // ek, x.shape[1] // ej, x.shape[2] // ei
    if layout == 2:  # rows of 16 split in two 8 x 8 vectors
        y = x.view(nk, ek, nj, ej, ni, 2, 8).permute(0, 2, 4, 1, 5, 3, 6)
    else:
        y = x.view(nk, ek, nj, ej, ni, ei).permute(0, 2, 4, 1, 3, 5)
    return y.reshape(nk, nj, ni, 512)


def _cells(case):
    ek, ej, ei = LAYOUT_EXTENTS[case.get("layout", 0)]
    return case["nk"] * ek, case["nj"] * ej, case["ni"] * ei


def _values(shape, seed, dtype):
    """Uniform values in [-1, 1), rounded to the element type."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    tdt = DTYPES[dtype][1]
    x = torch.rand(shape, generator=gen, device="cuda",
                   dtype=torch.float64 if dtype == "f64" else torch.float32)
    return x.mul_(2).sub_(1).to(tdt)


def _stencil(name, seed):
    st = bk.Stencil.make(name, seed=3 + seed % 1000)
    if name == "125pt":
        c = np.random.RandomState(seed % (1 << 31)).uniform(0.0, 1.0, 125)
        st.coeff = c / c.sum()
    return st


def _field(g, x, dtype, layout=0):
    """A field of the grid holding the (k, j, i) array x."""
    storage = g.field_storage(DTYPES[dtype][0])
    t = _view(storage.buf, (storage.chunks, 512), dtype)
    t.zero_()
    if x is not None:
        _interior(t, g).copy_(_to_bricks(x, layout))
    return bk.Brick(g.info, storage, 0), t


# ---------------------------------------------------------------------------
# a pass
# ---------------------------------------------------------------------------
def _mix(case):
    """The boxes of a batch: bricks per axis, stencil, element type, sweeps."""
    rng = random.Random(case["mix"])
    out = []
    for _ in range(case["requests"]):
        nb = tuple(_log_int(rng, 4, case["most"]) for _ in range(3))
        out.append((nb, rng.choice(STENCILS), rng.choice(["f64", "f32"]),
                    rng.randint(1, case["ticks"])))
    return out


def prepare(case, seed):
    do = case["do"]
    s = {"do": do, "case": case}
    if do == "batch":
        shapes = bkb.ShapeCache()
        s["reqs"], s["steps"], s["fields"] = [], [], {}
        for q, (nb, name, dtype, steps) in enumerate(_mix(case)):
            r = bkb.Request(q, nb, _stencil(name, seed + q), DTYPES[dtype][0], steps, seed + q)
            r.allocate(shapes)
            shape = (nb[2], nb[1], nb[0], 512)
            f0, f1 = (_view(f, shape, dtype) for f in (r.f0, r.f1))
            x = _values((nb[2] * 8, nb[1] * 8, nb[0] * 8), seed + q, dtype)
            f0.copy_(_to_bricks(x))
            s["fields"][r.f0.ptr], s["fields"][r.f1.ptr] = f0, f1
            s["reqs"].append(r)
            s["steps"].append(steps)
        s["batch"] = bkb.Batch(max_reqs=max(8, len(s["reqs"])))
        return s
    layout = case.get("layout", 0)
    ghost = 0 if case.get("refresh") == "none" else 1
    g = s["grid"] = bk.PeriodicGrid((case["ni"], case["nj"], case["nk"]), ghost=ghost, layout=layout)
    nk, nj, ni = _cells(case)
    dtype = case["dtype"]
    if do == "convert":
        pad = (case["pad_i"], case["pad_j"], case["pad_k"])
        full = (nk + 2 * (8 + pad[2]), nj + 2 * (8 + pad[1]), ni + 2 * (8 + pad[0]))
        n = full[0] * full[1] * full[2]
        size = DTYPES[dtype][1].itemsize
        s["dims"], s["pad"] = (ni, nj, nk), pad
        s["arr_in"], s["arr_out"] = bk.DeviceBuffer(n * size), bk.DeviceBuffer(n * size)
        _view(s["arr_in"], full, dtype).copy_(_values(full, seed, dtype))
        s["t_out"] = _view(s["arr_out"], full, dtype)
        s["t_out"].zero_()
        s["to"], s["t_to"] = _field(g, None, dtype)
        s["from"], _ = _field(g, _values((nk, nj, ni), seed + 1, dtype), dtype)
        return s
    x = _values((nk, nj, ni), seed, dtype)
    if do == "monitor":
        s["a"], _ = _field(g, x, dtype)
        y = x.to(torch.float64) * (1 + 1e-3 * _values((nk, nj, ni), seed + 1, "f64"))
        s["ref"], _ = _field(g, y.to(DTYPES[case["reference"]][1]), case["reference"])
        return s
    s["stencil"] = _stencil(case["stencil"], seed)
    s["a"], ta = _field(g, x, dtype, layout)
    s["b"], tb = _field(g, None, dtype)
    s["tensors"] = {s["a"].ptr: ta, s["b"].ptr: tb}
    if do == "apply" and ghost:
        g.ghost_refresh(s["a"])
    return s


def run(s):
    do, case = s["do"], s["case"]
    if do == "batch":
        for r, steps in zip(s["reqs"], s["steps"]):  # the boxes come again with as many sweeps
            r.done, r.steps = 0, steps
        s["batch"].run(s["reqs"], case["ticks"])
        return [s["fields"][r.result_ptr] for r in s["reqs"]]
    g = s["grid"]
    if do == "convert":
        bk.copyToBrick(s["dims"], s["pad"], (8, 8, 8), s["arr_in"], g.d_grid, s["to"])
        bk.copyFromBrick(s["dims"], s["pad"], (8, 8, 8), s["arr_out"], g.d_grid, s["from"])
        return [_interior(s["t_to"], g), s["t_out"]]
    if do == "monitor":
        d = g.compare(s["a"], s["ref"], floor=1e-2, atol=1e-6, rtol=5e-4)
        return [g.stats(s["a"]), d]
    if do == "apply":
        bk.sweep(s["stencil"], s["b"], s["a"], g)
        return _interior(s["tensors"][s["b"].ptr], g)
    res = bk.sweeps(s["stencil"], s["a"], s["b"], g, case["sweeps"], use_graph=case["graph"],
                    fused=case["refresh"] == "fused")
    if res is s["b"]:  # the next call goes on from this one's result
        s["a"], s["b"] = s["b"], s["a"]
    return _interior(s["tensors"][res.ptr], g)


# ---------------------------------------------------------------------------
# what a pass cannot do without, and its values in 64 bits
# ---------------------------------------------------------------------------
def _size(dtype):
    return DTYPES[dtype][1].itemsize


def work(case):
    do = case["do"]
    if do == "batch":
        nbytes = flops = 0
        for nb, name, dtype, steps in _mix(case):
            cells = nb[0] * nb[1] * nb[2] * 512
            nbytes += 2 * cells * _size(dtype)
            flops += cells * steps * FLOPS[name]
        return {"bytes": nbytes, "flops": flops}
    cells = math.prod(_cells(case))
    if do == "convert":
        return {"bytes": 4 * cells * _size(case["dtype"]), "flops": 0}
    if do == "monitor":
        return {"bytes": cells * (_size(case["dtype"]) + _size(case["reference"])),
                "flops": 12 * cells}
    return {"bytes": 2 * cells * _size(case["dtype"]),
            "flops": cells * case.get("sweeps", 1) * FLOPS[case["stencil"]]}


def _offsets(name):
    if name == "125pt":
        return [(di, dj, dk) for dk in range(-2, 3) for dj in range(-2, 3) for di in range(-2, 3)]
    out = [(0, 0, 0)]
    for r in range(1, {"7pt": 1, "cond": 1, "13pt": 2, "25pt": 4}[name] + 1):
        out += [(r, 0, 0), (-r, 0, 0), (0, r, 0), (0, -r, 0), (0, 0, r), (0, 0, -r)]
    return out


def _apply(x, name, st):
    y = x.clamp(min=0.0) if name == "cond" else x
    acc = torch.zeros_like(x)
    for (di, dj, dk), c in zip(_offsets(name), st.coeff):
        acc.add_(torch.roll(y, (-dk, -dj, -di), (0, 1, 2)), alpha=float(c))
    if name == "cond":
        acc = torch.where(x > st.theta, acc, -acc)
    return acc


def exact(case, seed):
    do = case["do"]
    if do == "batch":
        out = []
        for q, (nb, name, dtype, steps) in enumerate(_mix(case)):
            x = _values((nb[2] * 8, nb[1] * 8, nb[0] * 8), seed + q, dtype).double()
            st = _stencil(name, seed + q)
            for _ in range(steps):
                x = _apply(x, name, st)
            out.append(_to_bricks(x))
        return out
    nk, nj, ni = _cells(case)
    dtype = case["dtype"]
    if do == "convert":
        p = [8 + case["pad_k"], 8 + case["pad_j"], 8 + case["pad_i"]]
        full = tuple(n + 2 * q for n, q in zip((nk, nj, ni), p))
        inner = tuple(slice(q, q + n) for n, q in zip((nk, nj, ni), p))
        x = _values(full, seed, dtype).double()[inner].contiguous()
        arr = torch.zeros(full, dtype=torch.float64, device="cuda")
        arr[inner] = _values((nk, nj, ni), seed + 1, dtype).double()
        return [_to_bricks(x), arr]
    x = _values((nk, nj, ni), seed, dtype).double()
    if do == "monitor":
        y = x * (1 + 1e-3 * _values((nk, nj, ni), seed + 1, "f64"))
        y = y.to(DTYPES[case["reference"]][1]).double()
        d, r = (x - y).abs(), y.abs()
        sums = [float(x.sum()), float(x.square().sum()), float(x.abs().max())]
        rms = math.sqrt(float(d.square().sum()) / x.numel())
        return [np.array(sums), {
            "max_abs": float(d.max()), "max_rel": float((d / r.clamp(min=1e-2)).max()),
            "rms_rel": math.sqrt(float(d.square().sum()) / float(y.square().sum())),
            "rms_abs": rms, "bad": int((d > 1e-6 + 5e-4 * r).sum())}]
    if case["stencil"] == "cond" and dtype == "bf16" and case.get("sweeps", 1) > 1:
        return None  # the select turns 16-bit rounding into sign changes: no common value
    st = _stencil(case["stencil"], seed)
    for _ in range(case.get("sweeps", 1)):
        x = _apply(x, case["stencil"], st)
    return _to_bricks(x, case.get("layout", 0))
