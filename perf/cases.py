"""What the performance of this library is measured on: products with a plan, plans made from a matrix, transposes.

A matrix is one of seven kinds, made on the GPU from the seed:

  uniform   `per_row` columns drawn uniformly in every row
  band      the same, drawn within `half` columns of the diagonal
  stencil   27 points on an nx x ny x nz grid; `coefs` "constant" (26 and -1: two distinct values) or "variable"
            (a coefficient of its own for every entry, as a material that varies gives)
  blocks    64 entries a row, a share of them in dense aligned 8 x 8 blocks near the diagonal, the rest uniform
  power     row lengths with the tail of Zipf(1.6), clipped at 4096, 7 in 10 columns around a place of the row's own
            while there is room there
  mixed     a share of the runs of 128 rows are strips (32 consecutive columns sliding along the diagonal), the
            other rows as in "power"

Repeats are drawn again once and dropped after that, so rows are a little ragged; a transpose takes the matrix with
its repeats, as an assembly leaves them, and the number of entries is then the same for every seed.

One of four things is done with it:

  product    y = A x with a plan in hand: what a solver or a ranking iteration does hundreds of times
  plan       a matrix that lives in device memory -> plan (extraction, decisions, layouts) -> first y
  surface    a matrix in host memory -> partition -> plan -> y: the call sequence of the reference's driver
  transpose  csr2csc of a matrix in device memory (the step of A^T x, and of every column-wise pass)
"""
import math

import numpy as np
import torch

import matxtractt_amd as mx

DEVICE = "cuda:0"
BYTES_MAX = 4.1e8  # the largest listed case's


def listed():
    return [
        # the smallest: one launch, a matrix of a megabyte (a coarse grid of a multigrid cycle, a small circuit)
        dict(name="product_small_f64", op="product", kind="uniform", dtype="f64", rows=4096, cols=4096, per_row=16, tau_c=0.0, tau_r=0.0),
        # clustered coupling with a random background, all of it in the memory-side cache
        dict(name="product_blocks_f64", op="product", kind="blocks", dtype="f64", rows=65536, share=0.4, tau_c=0.5, tau_r=0.25),
        # a finite-difference operator with constant coefficients: two distinct values
        dict(name="product_stencil_f64", op="product", kind="stencil", dtype="f64", nx=100, ny=100, nz=100, coefs="constant", tau_c=0.0, tau_r=0.0),
        # the same operator where the material varies, on a grid of odd sides: every value its own
        dict(name="product_coefs_f64", op="product", kind="stencil", dtype="f64", nx=97, ny=89, nz=83, coefs="variable", tau_c=0.0, tau_r=0.0),
        # a rectangular matrix with a few long rows and many short ones (least squares, incidence), odd sizes
        dict(name="product_rect_f64", op="product", kind="power", dtype="f64", rows=700001, cols=412345, tau_c=0.0, tau_r=0.0),
        # a web or social graph in half precision: a ranking iteration
        dict(name="product_power_f16", op="product", kind="power", dtype="f16", rows=1048576, cols=1048576, tau_c=0.0, tau_r=0.0),
        # the largest: dense strips beside power-law rows, the hybrid of matrix cores and slices
        dict(name="product_mixed_f16", op="product", kind="mixed", dtype="f16", rows=4194304, share=0.2, tau_c=1.0, tau_r=1.0),
        # an unstructured mesh numbered for a small bandwidth, ordinary in every respect, half precision
        dict(name="product_band_f16", op="product", kind="band", dtype="f16", rows=250007, cols=250007, per_row=40, half=3000, tau_c=0.0, tau_r=0.0),
        # a hybrid plan from a matrix that a GPU program has just assembled, and its first product
        dict(name="plan_mixed_f16", op="plan", kind="mixed", dtype="f16", rows=1048576, share=0.2, tau_c=1.0, tau_r=1.0),
        # the same for a mesh operator whose whole matrix is the CSR part (nothing is extracted)
        dict(name="plan_coefs_f64", op="plan", kind="stencil", dtype="f64", nx=61, ny=67, nz=71, coefs="variable", tau_c=0.0, tau_r=0.0),
        # the reference driver's sequence with its usual fractions, from host arrays
        dict(name="surface_blocks_f64", op="surface", kind="blocks", dtype="f64", rows=65536, share=0.4, tau_c=0.5, tau_r=0.25),
        # csr2csc in device memory
        dict(name="transpose_power_f64", op="transpose", kind="power", dtype="f64", rows=700001, cols=412345, tau_c=0.0, tau_r=0.0),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    op = rng.choice(["product"] * 7 + ["plan"] * 2 + ["surface", "transpose"])
    kind = rng.choice(["uniform", "band", "stencil", "blocks", "power", "power", "mixed"])
    dtype = rng.choice(["f64", "f16"])
    value = 8 if dtype == "f64" else 2
    # entries: products over the whole range; what is made once per matrix from a hundred thousand on
    most = BYTES_MAX * 0.9 / (value + 4 + (value * 2 + 4) / 10)
    nnz = _log(rng, 6e4, most) if op == "product" else _log(rng, 1e5, min(most, 1.6e7 if op != "surface" else 6e6))
    case = dict(op=op, kind=kind, dtype=dtype)
    tau = rng.choice([(0.0, 0.0), (0.5, 0.25), (1.0, 1.0)]) if kind in ("blocks", "mixed") else rng.choice([(0.0, 0.0), (0.0, 0.0), (0.5, 0.25)])
    if kind in ("uniform", "band"):
        per_row = int(_log(rng, 5, 80))
        rows = max(1000, int(nnz / per_row))
        cols = max(1000, int(rows * _log(rng, 0.5, 2.0))) if kind == "uniform" else rows
        case.update(rows=rows, cols=cols, per_row=per_row)
        if kind == "band":
            case.update(half=int(_log(rng, 100, max(200, min(20000, cols / 4)))))
    elif kind == "stencil":
        side = (nnz / 27) ** (1 / 3)
        nx, ny = max(6, int(side * rng.uniform(0.8, 1.2))), max(6, int(side * rng.uniform(0.8, 1.2)))
        case.update(nx=nx, ny=ny, nz=max(6, int(nnz / 27 / nx / ny)), coefs=rng.choice(["constant", "variable"]))
    elif kind == "blocks":
        case.update(rows=max(1024, int(nnz / 64)), share=round(rng.uniform(0.1, 0.7), 3))
    elif kind == "power":
        rows = max(4000, int(nnz / 10))
        case.update(rows=rows, cols=max(4000, int(rows * _log(rng, 0.5, 2.0))))
    else:
        share = round(rng.uniform(0.05, 0.4), 3)
        case.update(rows=max(4000, int(nnz / (10 + 22 * share))), share=share)
    case.update(tau_c=tau[0], tau_r=tau[1])
    return case


# ---- matrices -----------------------------------------------------------------------------------------------

def _length_scale(longest, mean):
    """s such that min(max(floor(s * U^(-1/0.6)), 1), longest) has this mean."""
    k = np.arange(1, longest + 1, dtype=np.float64)
    lo, hi = 1e-9, float(longest)
    for _ in range(60):
        mid = 0.5 * (lo + hi)
        lo, hi = (mid, hi) if np.minimum(1.0, (mid / k) ** 0.6).sum() < mean else (lo, mid)
    return 0.5 * (lo + hi)


def _power_entries(row_ids, cols, g):
    longest = max(1, min(4096, cols // 2))
    # (the quantiles of the law in random order: the same lengths for every seed, at other rows)
    u = (torch.randperm(row_ids.numel(), generator=g, device=DEVICE).double() + 0.5) / row_ids.numel()
    length = (_length_scale(longest, 10.0) * u ** (-1 / 0.6)).clamp(1, longest).long()
    centre = torch.randint(0, cols, (row_ids.numel(),), generator=g, device=DEVICE)
    r = row_ids.repeat_interleave(length)
    near = centre.repeat_interleave(length) + torch.randint(-512, 513, r.shape, generator=g, device=DEVICE)
    far = torch.randint(0, cols, r.shape, generator=g, device=DEVICE)
    c = torch.where(torch.rand(r.shape, generator=g, device=DEVICE) < 0.7, near.clamp(0, cols - 1), far)
    return r, c


def _entries(case, g):
    """(rows, cols, row of every entry, column of every entry), in any order, repeats allowed."""
    kind = case["kind"]
    if kind == "uniform":
        r = torch.arange(case["rows"], device=DEVICE).repeat_interleave(case["per_row"])
        return case["rows"], case["cols"], r, torch.randint(0, case["cols"], r.shape, generator=g, device=DEVICE)
    if kind == "band":
        r = torch.arange(case["rows"], device=DEVICE).repeat_interleave(case["per_row"])
        c = r + torch.randint(-case["half"], case["half"] + 1, r.shape, generator=g, device=DEVICE)
        return case["rows"], case["cols"], r, c.clamp(0, case["cols"] - 1)
    if kind == "blocks":
        n = case["rows"]
        nb = n // 8
        at = torch.arange(8 * nb, device=DEVICE)[torch.rand(8 * nb, generator=g, device=DEVICE) < case["share"]] // 8
        to = (at + torch.randint(-128, 128, at.shape, generator=g, device=DEVICE)).clamp(0, nb - 1)
        place = torch.unique(at * nb + to)
        at, to = torch.div(place, nb, rounding_mode="floor"), place % nb
        i = torch.arange(8, device=DEVICE)
        r = (8 * at[:, None, None] + i[None, :, None]).expand(-1, 8, 8).reshape(-1)
        c = (8 * to[:, None, None] + i[None, None, :]).expand(-1, 8, 8).reshape(-1)
        rest = (64 - torch.bincount(r, minlength=n)).clamp_min(0)
        rr = torch.arange(n, device=DEVICE).repeat_interleave(rest)
        return n, n, torch.cat((r, rr)), torch.cat((c, torch.randint(0, n, rr.shape, generator=g, device=DEVICE)))
    if kind == "power":
        return (case["rows"], case["cols"]) + _power_entries(torch.arange(case["rows"], device=DEVICE), case["cols"], g)
    n = case["rows"]  # mixed
    runs = n // 128  # (the rows of a last, shorter run are never a strip)
    strip = torch.zeros(runs + 1, dtype=torch.bool, device=DEVICE)
    strip[torch.randperm(runs, generator=g, device=DEVICE)[:round(case["share"] * runs)]] = True
    off = torch.randint(-32, 33, (runs + 1,), generator=g, device=DEVICE)
    row = torch.arange(n, device=DEVICE)
    in_strip = strip[row // 128]
    sr = row[in_strip]
    first = (8 * (sr // 8 + off[sr // 128])).clamp(0, (n - 32) // 8 * 8)
    r, c = _power_entries(row[~in_strip], n, g)
    sc = (first[:, None] + torch.arange(32, device=DEVICE)[None, :]).reshape(-1)
    return n, n, torch.cat((r, sr.repeat_interleave(32))), torch.cat((c, sc))


def _matrix(case, g):
    """(rowPtr, colInd, val, cols) in device memory; every row lists its columns in ascending order."""
    dtype = torch.float64 if case["dtype"] == "f64" else torch.float16
    if case["kind"] == "stencil":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        n = rows = cols = nx * ny * nz
        at = torch.arange(n, device=DEVICE)
        x, y, z = at % nx, at // nx % ny, at // (nx * ny)
        near = [(dx, dy, dz) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]
        c = torch.stack([at + dx + nx * (dy + ny * dz) for dx, dy, dz in near], 1)
        inside = torch.stack([(x + dx >= 0) & (x + dx < nx) & (y + dy >= 0) & (y + dy < ny) & (z + dz >= 0) & (z + dz < nz)
                              for dx, dy, dz in near], 1)
        v = torch.full(c.shape, -1.0, dtype=torch.float64, device=DEVICE)
        if case["coefs"] == "variable":
            v = -0.5 - torch.rand(c.shape, generator=g, device=DEVICE, dtype=torch.float64)
        v[:, 13] *= -26.0
        counts, ci, va = inside.sum(1), c[inside], v[inside]
    else:
        rows, cols, r, c = _entries(case, g)
        key = torch.sort(r * cols + c)[0]
        again = torch.zeros(key.shape, dtype=torch.bool, device=DEVICE)
        again[1:] = key[1:] == key[:-1]
        other = torch.randint(0, cols, key.shape, generator=g, device=DEVICE)
        key = torch.where(again, key - key % cols + other, key)
        key = torch.sort(key)[0] if case["op"] == "transpose" else torch.unique(key)
        r, ci = torch.div(key, cols, rounding_mode="floor"), key % cols
        counts = torch.bincount(r, minlength=rows)
        va = 2.0 * torch.rand(ci.shape, generator=g, device=DEVICE, dtype=torch.float64 if case["dtype"] == "f64" else torch.float32) - 1.0
    rp = torch.zeros(rows + 1, dtype=torch.int32, device=DEVICE)
    rp[1:] = torch.cumsum(counts, 0)
    return rp, ci.to(torch.int32), va.to(dtype), cols


# ---- what is measured -----------------------------------------------------------------------------------------

def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    rp, ci, va, cols = _matrix(case, g)
    x = (2.0 * torch.rand(cols, generator=g, device=DEVICE, dtype=torch.float64) - 1.0).to(va.dtype)
    tau = (case["tau_c"], case["tau_r"])
    state = {"op": case["op"], "tau": tau, "x": x, "cols": cols}
    if case["op"] == "product":
        state["plan"] = mx.Plan.from_device(rp, ci, va, cols, *tau)
        state["y"] = torch.empty(rp.numel() - 1, dtype=va.dtype, device=DEVICE)
    elif case["op"] == "surface":
        state["A"] = mx.Csr(rp.numel() - 1, cols, rp.cpu().numpy(), ci.cpu().numpy(), va.cpu().numpy())
    else:
        state["A"] = (rp, ci, va)
    return state


def run(state):
    op = state["op"]
    if op == "product":
        return state["plan"].spmv(state["x"], state["y"])
    if op == "plan":
        return mx.Plan.from_device(*state["A"], state["cols"], *state["tau"]).spmv(state["x"])
    if op == "surface":
        return mx.Plan(mx.Partition(state["A"], *state["tau"], device=None)).spmv(state["x"])
    rp, ci, va = state["A"]
    return mx.transpose_device(rp, ci, va, state["cols"])


def _shape(case):
    """(rows, cols, entries) that the case's recipe gives, closely."""
    kind = case["kind"]
    if kind == "stencil":
        n = case["nx"] * case["ny"] * case["nz"]
        return n, n, (3 * case["nx"] - 2) * (3 * case["ny"] - 2) * (3 * case["nz"] - 2)
    rows, cols = case["rows"], case.get("cols", case["rows"])
    if kind in ("uniform", "band"):
        return rows, cols, rows * case["per_row"]
    if kind == "blocks":
        return rows, cols, 64 * rows
    share = case.get("share", 0.0)
    return rows, cols, int(rows * (10 * (1 - share) + 32 * share))


def work(case):
    rows, cols, nnz = _shape(case)
    value = 8 if case["dtype"] == "f64" else 2
    matrix = nnz * (value + 4) + 4 * (rows + 1)
    if case["op"] == "transpose":  # in once, out once
        return {"bytes": matrix + nnz * (value + 4) + 4 * (cols + 1), "flops": 0}
    return {"bytes": matrix + value * (cols + rows), "flops": 2 * nnz}


def tolerance(case):
    if case["op"] == "transpose":
        return "exact"
    # about four times what the product differs by from sums in binary64 (binary16: the rounding of y), and from
    # sums of the same products in a random order (binary64: more in rows of thousands of entries)
    if case["dtype"] == "f16":
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 6e-15, "max": 5e-13} if case["kind"] in ("power", "mixed") else {"rel": 1.3e-15, "max": 1e-14}
