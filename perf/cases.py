"""What is timed: static solves and their parts, through the entry points that a program calls.

Kinds of case and what each stands for:

* `static`  -- a whole `Static` solution on a resident model: reset, load steps with their Newton
  iterations, node results read back.  `part` says which structure: `cantilever` (a Beam_1 chain
  rolled up by a follower tip moment, the short latency-bound analyses), `riser` (a hanging Beam_1
  chain with seeded lateral loads, the marine analyses) or `plate` (a clamped Shell_1 plate under
  follower pressure).  `mixed` runs it in the mixed-precision mode.
* `newton`  -- a caller that drives its own Newton loop on a plate: begin a step, assemble / solve /
  update a few times, read the displacements, roll back.
* `btd`     -- a block-tridiagonal system on the caller's device buffers (no allocation).
* `band`    -- a band system on host arrays, the LAPACK-style call.
* `stream`  -- a batch of independent risers and plates through the request server, submitted,
  pumped to the end and taken.
"""
import ctypes
import math

import numpy as np
import torch

from giraffe_amd import abi, model as M, runtime as R


def listed():
    return [
        # the smallest analysis: a chain of twenty elements in four load steps, all latency
        {"name": "cantilever_20", "kind": "static", "part": "cantilever", "size": 20, "steps": 4, "mixed": False},
        # a hundred elements in twenty steps to the full circle, the usual roll-up check
        {"name": "cantilever_100", "kind": "static", "part": "cantilever", "size": 100, "steps": 20, "mixed": False},
        # a riser of ordinary length
        {"name": "riser_777", "kind": "static", "part": "riser", "size": 777, "steps": 10, "mixed": False},
        # the long catenary
        {"name": "riser_10000", "kind": "static", "part": "riser", "size": 10000, "steps": 10, "mixed": False},
        # a coarse plate, its mesh not a power of two
        {"name": "plate_13", "kind": "static", "part": "plate", "size": 13, "steps": 15, "mixed": False},
        # a plate of ordinary mesh in the mixed-precision mode
        {"name": "plate_32_mixed", "kind": "static", "part": "plate", "size": 32, "steps": 15, "mixed": True},
        # the fine plate of the benchmark
        {"name": "plate_64", "kind": "static", "part": "plate", "size": 64, "steps": 15, "mixed": False},
        # the largest mesh, three Newton iterations of a caller's own loop
        {"name": "newton_101", "kind": "newton", "size": 101, "iterations": 3},
        # a narrow system at an odd block size, and one of wide blocks
        {"name": "btd_12x900", "kind": "btd", "m": 12, "blocks": 900},
        {"name": "btd_31x131", "kind": "btd", "m": 31, "blocks": 131},
        # a band system called from host code
        {"name": "band_3001_97", "kind": "band", "n": 3001, "half_band": 97},
        # a stream of analyses sharing the device
        {"name": "stream_12", "kind": "stream", "risers": 9, "plates": 3, "largest_riser": 1500, "largest_plate": 40},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cantilever", "riser", "riser", "plate", "plate", "newton", "btd", "band", "stream"])
    if kind == "cantilever":
        return {"kind": "static", "part": kind, "size": _log_int(rng, 5, 120), "steps": rng.randint(4, 20),
                "mixed": False}
    if kind == "riser":
        return {"kind": "static", "part": kind, "size": _log_int(rng, 50, 10000), "steps": 10, "mixed": False}
    if kind == "plate":
        return {"kind": "static", "part": kind, "size": _log_int(rng, 6, 60), "steps": 15,
                "mixed": rng.random() < 0.3}
    if kind == "newton":
        return {"kind": "newton", "size": _log_int(rng, 6, 100), "iterations": rng.randint(1, 3)}
    if kind == "btd":
        m = rng.randint(1, 32)
        return {"kind": "btd", "m": m, "blocks": _log_int(rng, 8, min(8000, 131072 // (m * m)))}
    if kind == "band":
        return {"kind": "band", "n": _log_int(rng, 200, 6000), "half_band": _log_int(rng, 3, 190)}
    return {"kind": "stream", "risers": rng.randint(2, 9), "plates": rng.randint(1, 3),
            "largest_riser": _log_int(rng, 100, 1500), "largest_plate": rng.randint(16, 40)}


def _cantilever(size, steps, rng):
    """A tube of seeded section under the follower moment that closes 0.2 to 1 of a circle at full load."""
    De = rng.uniform(0.1, 0.3)
    return M.cantilever_rollup(n_elem=size, De=De, Di=0.9 * De, n_steps=steps,
                               turns=rng.uniform(0.8, 1.0) * min(1.0, steps / 20.0))[:2]


def _riser(size, steps, rng):
    """The long catenary's span and pipe, its weight, section and lateral loads seeded (the loads of
    a fine mesh smaller, as they stand for one load along the pipe)."""
    od = rng.uniform(0.28, 0.32)
    return M.catenary(n_elem=size, De=od, Di=od - 0.04, w=rng.uniform(1350.0, 1650.0),
                      sigma=500.0 * min(1.0, 1000.0 / size), seed=int(rng.integers(1 << 30)), n_steps=steps)[:2]


def _plate(size, steps, rng):
    """A plate of the serving stream's ranges: seeded thickness, deflection and imperfections."""
    t = rng.uniform(0.003, 0.008)
    p_max = 1.7e7 * (rng.uniform(10.0, 20.0) / 20.0) ** 3 * (t / 0.005) ** 4
    return M.shell_plate(nq=size, t=t, p_max=p_max, n_steps=steps, seed=int(rng.integers(1 << 30)))[:2]


_PARTS = {"cantilever": _cantilever, "riser": _riser, "plate": _plate}


def _blocks(case, seed):
    """Blocks A, B, C [blocks][m][m] with dominant diagonal blocks, and a right-hand side."""
    rng = np.random.default_rng(seed)
    m, n = case["m"], case["blocks"]
    A, B, C = (rng.normal(size=(n, m, m)) for _ in range(3))
    B += 4.0 * math.sqrt(m) * np.eye(m) + np.sign(rng.normal(size=(n, 1, 1))) * 0.5 * np.eye(m)
    A[0] = C[-1] = 0.0
    return A, B, C, rng.normal(size=n * m)


def _band(case, seed):
    """Rows [n][2 hb + 1] of a band matrix with a dominant diagonal, and a right-hand side."""
    rng = np.random.default_rng(seed)
    n, hb = case["n"], case["half_band"]
    rows = rng.normal(size=(n, 2 * hb + 1))
    rows[:, hb] += 3.0 * math.sqrt(2 * hb + 1)
    return rows, rng.normal(size=n)


def _spread(least, largest, count):
    """`count` sizes from `least` to `largest`, evenly in their logarithm."""
    least = min(least, largest)
    return [int(round(least * (largest / least) ** (i / max(1, count - 1)))) for i in range(count)]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "static":
        m, p = _PARTS[case["part"]](case["size"], case["steps"], rng)
        dm = R.DeviceModel(m, precision=abi.GF_PREC_MIXED if case["mixed"] else abi.GF_PREC_FP64)
        return {"kind": kind, "model": dm, "params": p}
    if kind == "newton":
        m, p = _plate(case["size"], 15, rng)
        return {"kind": kind, "model": R.DeviceModel(m), "iterations": case["iterations"]}
    if kind == "btd":
        A, B, C, b = (torch.from_numpy(v).cuda() for v in _blocks(case, seed))
        return {"kind": kind, "m": case["m"], "blocks": case["blocks"], "in": (A, B, C, b),
                "x": torch.empty_like(b), "info": torch.zeros(1, dtype=torch.int32, device=b.device)}
    if kind == "band":
        rows, b = _band(case, seed)
        return {"kind": kind, "rows": rows, "half_band": case["half_band"], "b": b}
    work = [_riser(e, 10, rng) for e in _spread(50, case["largest_riser"], case["risers"])]
    work += [_plate(q, 15, rng) for q in _spread(16, case["largest_plate"], case["plates"])]
    return {"kind": kind, "server": R.Server(max_inflight=16), "work": [(m, p) for m, p in work]}


def run(state):
    kind = state["kind"]
    if kind == "static":
        dm = state["model"]
        dm.reset()
        dm.static_solve(state["params"])
        return {"nodes": dm.nodes()}
    if kind == "newton":
        dm = state["model"]
        dm.set_window(0.0, 1.0)
        dm.begin_step(0.0, 0.2)
        for _ in range(state["iterations"]):
            dm.assemble()
            dm.solve()
            dm.update()
        d = dm.disp()
        dm.rollback()
        return {"disp": d}
    if kind == "btd":
        p = [ctypes.c_void_p(t.data_ptr()) for t in state["in"]]
        R.check(R.load().gf_btdsystem_noalloc(
            state["m"], state["blocks"], *p, ctypes.c_void_p(state["x"].data_ptr()),
            ctypes.c_void_p(state["info"].data_ptr()),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "gf_btdsystem_noalloc")
        return {"x": state["x"], "info": state["info"]}
    if kind == "band":
        x, fail = R.bandsystem(state["rows"], state["half_band"], state["b"])
        return {"x": x, "info": fail}
    server = state["server"]
    ids = [server.submit(m, p) for m, p in state["work"]]
    done = 0
    while done < len(ids):
        done += server.pump(2000)
    return [server.take(i)[2] for i in ids]


# One Newton iteration of a mesh, by its unknowns n and elements: the tangent's entries are written
# once and its factor read once; the factorisation of a plate costs about 400 n^1.5 operations over a
# nested dissection, that of a chain of 16-row blocks about 14/3 products of a block a row.
def _iteration(part, size):
    if part == "plate":
        n = 6.0 * (2 * size - 1) ** 2 - 3.0 * (size - 1) ** 2
        return {"bytes": 2 * size * size * 13044 + n * 31 * math.log2(max(n, 2.0)) * 8,
                "flops": 2 * size * size * 7e4 + 400.0 * n ** 1.5}
    n = 12.0 * size
    return {"bytes": size * 6108 + 3 * n * 16 * 8, "flops": size * 1.5e4 + (n / 16) * (14 / 3) * 2 * 16 ** 3}


def _solution(part, size, steps):
    """A load step takes about seven iterations of a plate or chain."""
    w = _iteration(part, size)
    return {k: 7 * steps * v for k, v in w.items()}


def work(case):
    kind = case["kind"]
    if kind == "static":
        return _solution(case["part"], case["size"], case["steps"])
    if kind == "newton":
        return {k: case["iterations"] * v for k, v in _iteration("plate", case["size"]).items()}
    if kind == "btd":
        m, n = float(case["m"]), float(case["blocks"])
        return {"bytes": 8 * (3 * n * m * m + 2 * n * m), "flops": n * (14 / 3) * 2 * m ** 3}
    if kind == "band":
        n, hb = float(case["n"]), float(case["half_band"])
        return {"bytes": 8 * (n * (2 * hb + 1) + 2 * n), "flops": 2 * n * hb * hb + 4 * n * hb}
    parts = [("riser", e, 10) for e in _spread(50, case["largest_riser"], case["risers"])]
    parts += [("plate", q, 15) for q in _spread(16, case["largest_plate"], case["plates"])]
    each = [_solution(*p) for p in parts]
    return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}


def exact(case, seed):
    """The linear systems' solutions: block elimination from the first row to the last, and a dense solve.
    A static solution has no closed form over these inputs."""
    if case["kind"] == "btd":
        A, B, C, b = _blocks(case, seed)
        n, m = case["blocks"], case["m"]
        b = b.reshape(n, m)
        Y, z = np.zeros((n, m, m)), np.zeros((n, m))
        for i in range(n):
            D = B[i] - A[i] @ Y[i - 1] if i else B[i]
            f = b[i] - A[i] @ z[i - 1] if i else b[i]
            s = np.linalg.solve(D, np.concatenate([C[i], f[:, None]], 1))
            Y[i], z[i] = s[:, :m], s[:, m]
        x = z.copy()
        for i in range(n - 2, -1, -1):
            x[i] -= Y[i] @ x[i + 1]
        return {"x": x.reshape(-1), "info": None}
    if case["kind"] == "band":
        rows, b = _band(case, seed)
        n, hb = case["n"], case["half_band"]
        A = np.zeros((n, n))
        for k in range(-hb, hb + 1):
            i = np.arange(max(0, -k), min(n, n - k))
            A[i, i + k] = rows[i, k + hb]
        return {"x": np.linalg.solve(A, b), "info": None}
    return None
