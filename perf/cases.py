"""The work that a user of this framework has it do, as cases to be timed.

Each kind of case is one operation of the NArray path through the public
Python API (`phase`), or through the C-ABI (include/phhip.h) for the batches,
whose sums the Python API only hands out as lists:

  operators  (a + b.tile(rows, 1)) * c            Float32 / Float64
  checked    a * b + c, Int32: raises on overflow
  chunk      a strided or trimmed region gathered, and written into a zeroed
             array through a MutableView
  permute    a permuted rank-3 view made an array
  mask       z[x > t] = y
  reduce2d   a ProcView block, then sum and max in full, per row and per column
  slices     slices(axis).map(&.sum) and (&.max) of a rank-3 array
  heat       the explicit 5-point heat equation, with its energy
  batch      thousands of small arrays: add, sum and step-2 slice of each

Sizes run from those of the tests (tens of elements a side) to those of the
benchmark's configurations (BASELINE's 1024^2, 8192^2, 16384^2, 20000 arrays).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ph-core_amd"))
import phase  # noqa: E402
from phase.workloads import batched_shapes  # noqa: E402

SIZE = {"i32": 4, "f32": 4, "f64": 8, "bf16": 2}
_DT = {"i32": phase.DType.I32, "f32": phase.DType.F32, "f64": phase.DType.F64, "bf16": phase.DType.BF16}
_TYPESTR = {phase.DType.I32: "<i4", phase.DType.F32: "<f4", phase.DType.F64: "<f8", phase.DType.BF16: "<i2",
            phase.DType.Bool: "|b1"}
# range literals of views, and the indices that each selects of n
_RANGES = {
    "..": lambda n: range(n),
    "..2..": lambda n: range(0, n, 2),          # every other one (the batches' slices)
    "1..3..-1": lambda n: range(1, n, 3),       # BASELINE's strided view
    "..-2..": lambda n: range(n - 1, -1, -2),
    "1..-3": lambda n: range(1, n - 2),         # a border trimmed off
    "5..-2": lambda n: range(5, n - 1),
    "-1..0": lambda n: range(n - 1, -1, -1),    # an axis reversed
}


def listed():
    return [
        # BASELINE's broadcast configuration, as ph-core's operators write it
        {"name": "operators_f64_1024", "kind": "operators", "dtype": "f64", "rows": 1024, "cols": 1024},
        # the smallest calls: two checked operators on a small array
        {"name": "checked_i32_32x48", "kind": "checked", "rows": 32, "cols": 48},
        # BASELINE's strided view configuration (the benchmark's headline)
        {"name": "chunk_i32_8192", "kind": "chunk", "dtype": "i32", "rows": 8192, "cols": 8192,
         "row_range": "1..3..-1", "col_range": "..-2.."},
        # a border trimmed off an image-like array of odd sides, and pasted back
        {"name": "chunk_bf16_trim", "kind": "chunk", "dtype": "bf16", "rows": 6007, "cols": 4001,
         "row_range": "1..-3", "col_range": "5..-2"},
        # the last axis first, odd extents: a layout change
        {"name": "permute_f32_201", "kind": "permute", "dtype": "f32", "d0": 257, "d1": 1023, "d2": 515, "order": "201"},
        # a threshold replaced through a mask
        {"name": "mask_i32_ragged", "kind": "mask", "rows": 3001, "cols": 4003},
        # BASELINE's fused ProcView chain and reductions, and in BF16 storage on odd sides
        {"name": "reduce2d_f32_16384", "kind": "reduce2d", "dtype": "f32", "rows": 16384, "cols": 16384},
        {"name": "reduce2d_bf16_ragged", "kind": "reduce2d", "dtype": "bf16", "rows": 5003, "cols": 3001},
        # statistics along the middle axis of a rank-3 array
        {"name": "slices_f64_axis1", "kind": "slices", "dtype": "f64", "d0": 96, "d1": 1000, "d2": 515, "axis": 1},
        # BASELINE's heat run, and a grid of ordinary, odd size in Float64
        {"name": "heat_f32_8192", "kind": "heat", "dtype": "f32", "rows": 8192, "cols": 8192, "steps": 2000, "every": 100},
        {"name": "heat_f64_750x1111", "kind": "heat", "dtype": "f64", "rows": 750, "cols": 1111, "steps": 1000,
         "every": 100},
        # BASELINE's batch of uneven arrays
        {"name": "batch_20000", "kind": "batch", "arrays": 20000, "shapes_seed": 4},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["operators", "checked", "chunk", "permute", "mask", "reduce2d", "slices", "heat", "batch"])
    if kind == "batch":
        return {"kind": kind, "arrays": _log_int(rng, 16, 20000), "shapes_seed": rng.randrange(1000)}
    if kind in ("permute", "slices"):
        while True:
            d = [_log_int(rng, 8, 2048) for _ in range(3)]
            if d[0] * d[1] * d[2] <= 1 << 27:
                break
        c = {"kind": kind, "dtype": rng.choice(["i32", "f32", "f64"]), "d0": d[0], "d1": d[1], "d2": d[2]}
        if kind == "permute":
            c["order"] = rng.choice(["201", "120", "021", "102", "210"])
        else:
            c["axis"] = rng.randrange(3)
        return c
    hi = 16384 if kind in ("operators", "reduce2d") else 8192
    rows, cols = _log_int(rng, 32, hi), _log_int(rng, 32, hi)
    if kind in ("checked", "mask"):
        return {"kind": kind, "rows": rows, "cols": cols}
    if kind == "operators":
        return {"kind": kind, "dtype": rng.choice(["f32", "f64"]), "rows": rows, "cols": cols}
    if kind == "chunk":
        return {"kind": kind, "dtype": rng.choice(["i32", "f32", "f64", "bf16"]), "rows": rows, "cols": cols,
                "row_range": rng.choice(sorted(_RANGES)), "col_range": rng.choice(sorted(_RANGES))}
    if kind == "reduce2d":
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16"]), "rows": rows, "cols": cols}
    dtype = rng.choice(["f32", "f64"])
    steps = _log_int(rng, 20, 2000)
    if dtype == "f64":  # twice the time a step
        steps = max(20, min(steps, 2 ** 26 * 900 // (rows * cols)))
    return {"kind": kind, "dtype": dtype, "rows": rows, "cols": cols, "steps": steps, "every": rng.choice([0, 100])}


# ------------------------------------------------------------------ inputs
class _Shared:
    """An NArray's device buffer to torch, without a copy; keeps the array."""

    def __init__(self, a):
        self.array = a
        self.__cuda_array_interface__ = {"shape": tuple(a.shape), "typestr": _TYPESTR[a.dtype], "version": 3,
                                         "data": (a.device_ptr, False), "strides": None}


def _tensor(a):
    t = torch.as_tensor(_Shared(a), device="cuda")
    return t.view(torch.bfloat16) if a.dtype == phase.DType.BF16 else t


def _random(shape, dtype, seed, stream, a=-1.0, b=1.0):
    if dtype == "i32":
        a, b = -1000, 1000
    return phase.NArray.random(list(shape), _DT[dtype], seed=seed * 8 + stream, a=a, b=b)


def _bumps(case, seed):
    """A sum of 16 Gaussian bumps (Float64), as phase.workloads draws them."""
    rng = np.random.default_rng(seed)
    ny, nx = case["rows"], case["cols"]
    cy, cx = rng.uniform(0.1, 0.9, 16) * ny, rng.uniform(0.1, 0.9, 16) * nx
    sig, amp = rng.uniform(0.01, 0.05, 16) * max(ny, nx), rng.uniform(0.5, 2.0, 16)
    t = lambda v: torch.from_numpy(v)[:, None]  # noqa: E731
    fy = t(amp) * torch.exp(-(torch.arange(ny, dtype=torch.float64)[None] - t(cy)) ** 2 / (2 * t(sig) ** 2))
    fx = torch.exp(-(torch.arange(nx, dtype=torch.float64)[None] - t(cx)) ** 2 / (2 * t(sig) ** 2))
    u = torch.zeros((ny, nx), dtype=torch.float64, device="cuda")
    for k in range(16):
        u += fy[k].cuda()[:, None] * fx[k].cuda()[None, :]
    return u


class _Batch:
    """A batch handle of the C-ABI over torch buffers, tuned for its shapes."""

    def __init__(self, shapes, scalars, seed):
        lib = self.lib = ctypes.CDLL(os.path.join(phase.LIB_DIR, "libphhip.so"))
        lib.ph_batch_run.argtypes = [ctypes.c_void_p, ctypes.c_int32]
        lib.ph_batch_destroy.argtypes = [ctypes.c_void_p]
        n = len(shapes)
        ranks = np.array([len(s) for s in shapes], np.int32)
        flat = np.zeros((n, 3), np.int64)
        for k, s in enumerate(shapes):
            flat[k, :len(s)] = s
        sc = np.ascontiguousarray(scalars, np.float32)
        at = lambda v: ctypes.c_void_p(v.ctypes.data)  # noqa: E731
        self.handle = ctypes.c_void_p()
        null = ctypes.c_void_p()
        self._check(lib.ph_batch_create(ctypes.byref(self.handle), ctypes.c_int32(n), at(ranks), at(flat), null, at(sc),
                                        null, null, null))
        xy, z = ctypes.c_int64(), ctypes.c_int64()
        self.offsets = np.zeros(n, np.int64)
        self._check(lib.ph_batch_sizes(self.handle, ctypes.byref(xy), ctypes.byref(z), at(self.offsets), null))
        g = torch.Generator("cuda").manual_seed(seed)
        self.x = torch.rand(xy.value, generator=g, device="cuda") * 2 - 1
        self.y = torch.zeros(xy.value, device="cuda")
        self.z = torch.zeros(z.value, device="cuda")
        self.sums = torch.zeros(n, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        self._check(lib.ph_batch_bind(self.handle, *(ctypes.c_void_p(t.data_ptr()) for t in (self.x, self.y, self.z, self.sums))))
        self._check(lib.ph_batch_tune(self.handle, null, null, null))

    @staticmethod
    def _check(rc):
        if rc != 0:
            raise RuntimeError("batch call: status %d" % rc)

    def run(self):
        self._check(self.lib.ph_batch_run(self.handle, 0))

    def __del__(self):
        if getattr(self, "handle", None):
            self.lib.ph_batch_destroy(self.handle)


def prepare(case, seed):
    phase.init(0)
    kind = case["kind"]
    s = dict(case)
    if kind == "batch":
        shapes, scalars, _ = batched_shapes(case["arrays"], case["shapes_seed"])
        s["batch"] = _Batch(shapes, scalars, seed)
        return s
    if kind in ("permute", "slices"):
        s["x"] = _random((case["d0"], case["d1"], case["d2"]), case["dtype"], seed, 0)
        if kind == "permute":
            s["view"] = s["x"].view().permute(*(int(k) for k in case["order"]))
        return s
    shape = (case["rows"], case["cols"])
    if kind == "operators":
        s["a"], s["c"] = _random(shape, case["dtype"], seed, 0), _random(shape, case["dtype"], seed, 2)
        s["b"] = _random((1, shape[1]), case["dtype"], seed, 1).tile(shape[0], 1)
    elif kind == "checked":
        s["a"], s["b"], s["c"] = (_random(shape, "i32", seed, k) for k in range(3))
    elif kind == "mask":
        s["x"], s["y"], s["z"] = (_random(shape, "i32", seed, k) for k in range(3))
    elif kind == "chunk":
        if case["dtype"] == "i32":
            s["x"] = phase.NArray.random(list(shape), phase.DType.I32, seed=seed, dist="int31")
        else:
            s["x"] = _random(shape, case["dtype"], seed, 0)
        s["zero"] = phase.i32(0) if case["dtype"] == "i32" else phase.f64(0.0) if case["dtype"] == "f64" else phase.f32(0.0)
    elif kind == "reduce2d":
        s["x"] = phase.NArray.random(list(shape), _DT[case["dtype"]], seed=seed, dist="normal", a=0.0, b=1.0)
        s["block"] = s["x"].process(lambda v: (v + 4) ** 2 * 0.5 - v)
    else:
        u = _bumps(case, seed)
        s["u0"] = phase.NArray.empty(list(shape), _DT[case["dtype"]])
        _tensor(s["u0"]).copy_(u)
        torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "operators":
        return _tensor((s["a"] + s["b"]) * s["c"])
    if kind == "checked":
        return _tensor(s["a"] * s["b"] + s["c"])
    if kind == "chunk":
        region = (s["row_range"], s["col_range"])
        g = s["x"].view(*region).to_narr()
        z = phase.NArray.fill(s["x"].shape, s["zero"], s["x"].dtype)
        z.mutable_view(*region)[[]] = g
        return _tensor(g), _tensor(z)
    if kind == "permute":
        return _tensor(s["view"].to_narr())
    if kind == "mask":
        s["z"][s["x"] > 0] = s["y"]
        return _tensor(s["z"])
    if kind == "reduce2d":
        return _tensor(s["block"].reduce2d_all_device())
    if kind == "slices":
        return np.array(s["x"].slices_sum(s["axis"])), np.array(s["x"].slices_max(s["axis"]))
    if kind == "heat":
        u = s["u0"].clone()
        energy = phase.heat2d(u, 0.2, s["steps"], every=s["every"])
        return _tensor(u), np.array(energy)
    b = s["batch"]
    b.run()
    return b.y, b.z, b.sums


def work(case):
    kind = case["kind"]
    if kind == "batch":
        shapes, _, _ = batched_shapes(case["arrays"], case["shapes_seed"])
        n = sum(math.prod(s) for s in shapes)
        nz = sum(math.prod((d + 1) // 2 for d in s) for s in shapes)
        return {"bytes": 8 * n + 4 * nz, "flops": 2 * n}
    es = SIZE[case.get("dtype", "i32")]
    if kind in ("permute", "slices"):
        n = case["d0"] * case["d1"] * case["d2"]
        if kind == "permute":
            return {"bytes": 2 * es * n, "flops": 0}
        return {"bytes": es * n + 16 * case["d%d" % case["axis"]], "flops": 2 * n}
    rows, cols = case["rows"], case["cols"]
    n = rows * cols
    if kind == "operators":
        return {"bytes": (3 * n + cols) * es, "flops": 2 * n}
    if kind == "checked":
        return {"bytes": 16 * n, "flops": 2 * n}
    if kind == "mask":
        return {"bytes": 12 * n, "flops": n}
    if kind == "chunk":
        g = len(_RANGES[case["row_range"]](rows)) * len(_RANGES[case["col_range"]](cols))
        return {"bytes": (3 * g + n) * es, "flops": 0}
    if kind == "reduce2d":
        return {"bytes": n * es + 8 * (2 + 2 * rows + 2 * cols), "flops": 8 * n}
    return {"bytes": 2 * n * es, "flops": 7 * n * case["steps"]}


# ------------------------------------------------------------- 64-bit results
def _heat64(u, steps, every):
    p = torch.zeros((u.shape[0] + 2, u.shape[1] + 2), dtype=torch.float64, device=u.device)
    c = p[1:-1, 1:-1]
    c.copy_(u)
    d = torch.empty_like(u)
    energy = [float(c.sum())] if every else []
    for t in range(1, steps + 1):
        torch.add(p[:-2, 1:-1], p[2:, 1:-1], out=d)
        d += p[1:-1, :-2]
        d += p[1:-1, 2:]
        d.sub_(c, alpha=4)
        c.add_(d, alpha=0.2)
        if every and t % every == 0:
            energy.append(float(c.sum()))
    return c.contiguous(), np.array(energy)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("checked", "mask") or case.get("dtype") == "i32":
        return None
    s = prepare(case, seed)
    torch.cuda.synchronize()  # the arrays are filled on the library's stream
    if kind == "batch":
        b = s["batch"]
        shapes, scalars, _ = batched_shapes(case["arrays"], case["shapes_seed"])
        x = b.x.double().cpu().numpy()
        y, sums, z = np.zeros_like(x), [], []  # the padding between arrays stays zero
        for o, sh, add in zip(b.offsets, shapes, scalars):
            a = x[o:o + math.prod(sh)]
            y[o:o + a.size] = a + np.float64(add)
            sums.append(a.sum())
            z.append(a.reshape(sh)[(slice(None, None, 2),) * len(sh)].ravel())
        return y, np.concatenate(z), np.array(sums)
    if kind == "heat":
        u = _tensor(s["u0"]).double()
        return _heat64(u, case["steps"], case["every"])
    if kind == "operators":
        b = s["b"].to_narr().materialize()
        torch.cuda.synchronize()
        t = lambda v: _tensor(v).double()  # noqa: E731
        return (t(s["a"]) + t(b)) * t(s["c"])
    x = _tensor(s["x"]).double()
    if kind == "permute":
        return x.permute(*(int(k) for k in case["order"])).contiguous()
    if kind == "slices":
        others = [k for k in range(3) if k != case["axis"]]
        return x.sum(dim=others).cpu().numpy(), x.amax(dim=others).cpu().numpy()
    if kind == "reduce2d":
        f = (x + 4) ** 2 * 0.5 - x
        return torch.cat([f.sum().view(1), f.max().view(1), f.sum(1), f.amax(1), f.sum(0), f.amax(0)])
    i = torch.tensor(list(_RANGES[case["row_range"]](case["rows"])), device=x.device)
    j = torch.tensor(list(_RANGES[case["col_range"]](case["cols"])), device=x.device)
    g = x[i][:, j]
    z = torch.zeros_like(x)
    z[i[:, None], j[None, :]] = g
    return g, z
