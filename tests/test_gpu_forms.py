"""GPU tests of the forms of the CSR part that a plan makes and picks on the device: value dictionaries,
offset patterns, row windows.  Against the host's layouts where they exist, against the oracle otherwise."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _exact(ora, A, x):
    """The oracle's y on integer data: the sums are exact in the accumulator (below 2^24), rounded once to the value type."""
    y = ora.spmv_f64(A.val, A.rowPtr, A.colInd, x) if x.dtype == np.float64 else ora.spmv_f16_f32acc(A.val, A.rowPtr, A.colInd, x)[0]
    return np.asarray(y).astype(x.dtype)


def _diagonals(mx, rng, rows, cols, offs, dtype, few, holes=0.0):
    """Rows with the column offsets `offs` where they lie inside the matrix, some of them missing; integer values."""
    r = np.repeat(np.arange(rows), len(offs))
    c = r + np.tile(offs, rows)
    ok = (c >= 0) & (c < cols) & (rng.random(r.size) >= holes)
    r, c = r[ok], c[ok]
    ptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=rows))]).astype(np.int32)
    val = rng.choice([-3, -1, 1, 2], r.size) if few else rng.integers(1, 400, r.size) * rng.choice([-1, 1], r.size)
    return mx.Csr(rows, cols, ptr, c.astype(np.int32), val.astype(dtype))


@pytest.mark.parametrize("dtype", [np.float64, np.float16])
@pytest.mark.parametrize("few", [False, True])
@pytest.mark.parametrize("rows,cols,offs", [
    (1024, 1024, [0]),                                   # one offset, whole chunks
    (1025, 1025, [-1, 0, 1]),                            # one row beyond them
    (1151, 1300, [-130, -1, 0, 1, 130]),                 # more columns than rows
    (5000, 3000, [-2500, -7, 3, 64]),                    # fewer: the last rows have few entries or none
    (30011, 30011, list(range(-32, 32))),                # as many offsets as a chunk may have
    (30011, 30011, list(range(-32, 33))),                # one more: another form takes the matrix
    (40000, 40000, sorted({dx + 20 * (dy + 50 * dz) for dx in (-1, 0, 1) for dy in (-1, 0, 1) for dz in (-1, 0, 1)})),
    (270000, 270000, [-700, -3, -2, 0, 2, 3, 700]),      # more than 2048 chunks of binary64 rows, a wave each
    (270000, 270000, list(range(-6, 6))),                # ... a list of more than one round: two or four waves a chunk
    (5001, 5001, list(range(0, 16, 2))),                 # as long a list as one wave takes, a row beyond whole chunks
    (5001, 5001, list(range(0, 18, 2))),                 # one more
    (1100, 1100, list(range(-30, 30))),                  # a small matrix with a long list: row tiles are the faster ones
])
def test_offset_form(mx, ora, dtype, few, rows, cols, offs):
    """Matrices whose rows repeat a pattern of column offsets: the product from both routes equals the oracle's
    (integers: every sum is exact), entries kept or streamed, over an old y and with every chunk's edges outside x; a
    row's sum is not touched by an infinite x that the row does not name."""
    import torch
    rng = np.random.default_rng(rows + len(offs))
    A = _diagonals(mx, rng, rows, cols, np.array(offs), dtype, few, holes=0.05 if len(offs) > 8 else 0.0)
    small = few or dtype == np.float64
    x = rng.integers(-2, 3, cols).astype(dtype) if small else rng.choice([-1, 0, 0, 0, 0, 0, 0, 0, 0, 1], cols).astype(dtype)
    long = 48 if dtype == np.float16 else 40
    takes = len(offs) <= 64 and (len(offs) <= long or rows >= 30000)
    xd = torch.from_numpy(x).cuda()
    dev = [torch.from_numpy(a).cuda() for a in (A.rowPtr, A.colInd, A.val)]
    ref = _exact(ora, A, x)
    P = mx.Partition(A, 0.0, 0.0)
    arrays = None
    for plan in (mx.Plan(P), mx.Plan.from_device(*dev, cols, 0.0, 0.0), mx.Plan.from_device(*dev, cols, 0.0, 0.0, mx.MX_PLAN_STREAM)):
        assert (plan.info["csr_variant"] == 3) == takes, plan.info
        if takes:
            assert (plan.info["csr_value_dict"] > 0) == (few and A.nnz >= 65536)
            assert arrays is None or plan.arrays() == arrays
            arrays = plan.arrays()
        y = torch.full((rows,), 7.0, dtype=xd.dtype, device="cuda")
        plan.spmv(xd, y)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), ref)
    if takes:  # x and y at any element, as row tiles take them
        xo, yo = torch.zeros(cols + 1, dtype=xd.dtype, device="cuda")[1:], torch.full((rows + 1,), 7.0, dtype=xd.dtype, device="cuda")
        xo.copy_(xd)
        plan.spmv(xo, yo[1:])
        assert np.array_equal(yo.cpu().numpy(), np.concatenate([[7], ref]).astype(dtype))
    bad = x.copy()
    bad[[0, cols // 2, cols - 1]] = np.inf
    touched = np.zeros(rows, bool)
    touched[np.repeat(np.arange(rows), np.diff(A.rowPtr))[~np.isfinite(bad[A.colInd])]] = True
    got = plan.spmv(torch.from_numpy(bad).cuda()).cpu().numpy()
    assert np.array_equal(~np.isfinite(got), touched)


@pytest.mark.parametrize("dtype", [np.float64, np.float16])
@pytest.mark.parametrize("what", ["twice", "minus zero", "any order"])
def test_matrices_the_offset_form_leaves_or_takes(mx, ora, dtype, what):
    """A column named twice or a stored -0.0 sends the matrix to another form; rows in any order do not."""
    import torch
    rng = np.random.default_rng(8)
    A = _diagonals(mx, rng, 4000, 4000, np.array([-50, -1, 0, 1, 50]), dtype, False)
    ci, va = A.colInd.copy(), A.val.copy()
    p = A.rowPtr[2000]
    if what == "twice":
        ci[p] = ci[p + 1]
    elif what == "minus zero":
        va[p] = -0.0
    else:
        for r in range(0, 4000, 3):
            s = slice(A.rowPtr[r], A.rowPtr[r + 1])
            o = rng.permutation(s.stop - s.start)
            ci[s], va[s] = ci[s][o], va[s][o]
    B = mx.Csr(4000, 4000, A.rowPtr, ci, va)
    x = rng.integers(-1, 2, 4000).astype(dtype)
    ref = _exact(ora, B, x)
    plan = mx.Plan.from_device(*(torch.from_numpy(a).cuda() for a in (B.rowPtr, B.colInd, B.val)), 4000, 0.0, 0.0)
    assert (plan.info["csr_variant"] == 3) == (what == "any order")
    got = plan.spmv(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("dtype", [np.float64, np.float16])
@pytest.mark.parametrize("values", [1, 2, 254, 255, 256, 300, 3000])
def test_value_dictionary_of_a_device_layout(mx, dtype, values):
    """The values of a slice layout made on the device are numbered as the host numbers them, up to 255 of them
    (the last of them met late, the pattern of all ones among them) and none beyond."""
    rng = np.random.default_rng(values)
    rows, cols = 3000, 70000
    ptr = np.concatenate([[0], np.cumsum(rng.integers(20, 60, rows))]).astype(np.int32)
    bits = np.uint64 if dtype == np.float64 else np.uint16
    pool = rng.choice(60000, values, replace=False).astype(bits) + bits(1)
    pool[0] = bits(2 ** (8 * np.dtype(bits).itemsize) - 1)
    at = rng.integers(0, max(values - 1, 1), ptr[-1])
    at[-1] = values - 1
    A = mx.Csr(rows, cols, ptr, rng.integers(0, cols, ptr[-1]).astype(np.int32), pool[at].view(dtype))
    H, D = mx.slice_layout(A, nCU=256), mx.slice_layout(A, nCU=256, device=True)
    assert (H["nDict"] > 0) == (len(np.unique(at)) <= 255)
    assert H["nDict"] == D["nDict"]
    for k in ("ecode", "dict", "eval"):
        assert np.array_equal(H[k].view(np.uint8), D[k].view(np.uint8)), k


def test_memory_kept_between_calls_is_bounded_and_given_back(mx):
    """Plans made and dropped one after the other, from two threads with streams of their own, leave products
    right while the library keeps what they gave back; release_memory() returns that to the device.  (These plans are far smaller than
    what the library may keep: the bound itself is looked at in the next test and in tests/test_memory.py.)"""
    import threading

    import torch
    rng = np.random.default_rng(3)
    mats = []
    for rows in (20000, 90000):
        ptr = (np.arange(rows + 1) * 12).astype(np.int32)
        mats.append(mx.Csr(rows, rows, ptr, rng.integers(0, rows, ptr[-1]).astype(np.int32), rng.integers(-3, 4, ptr[-1]).astype(np.float64)))
    wrong = []

    def work(A, seed):
        g = np.random.default_rng(seed)
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            dev = [torch.from_numpy(a).cuda() for a in (A.rowPtr, A.colInd, A.val)]
            for k in range(12):
                x = g.integers(-2, 3, A.cols).astype(np.float64)
                want = np.add.reduceat(A.val * x[A.colInd], A.rowPtr[:-1])
                s.synchronize()
                plan = mx.Plan.from_device(*dev, A.cols, *((0.0, 0.0) if k % 2 else (0.5, 0.25)))
                y = plan.spmv(torch.from_numpy(x).cuda())
                plan.close()                     # while the product may still run
                t = mx.transpose_device(*dev, A.cols)
                if not np.array_equal(y.cpu().numpy(), want):
                    wrong.append((seed, k))
                if int(t[0][-1]) != A.nnz:
                    wrong.append((seed, k, "transpose"))
    threads = [threading.Thread(target=work, args=(A, i)) for i, A in enumerate(mats)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    free0, total = torch.cuda.mem_get_info()
    mx.release_memory()
    free1 = torch.cuda.mem_get_info()[0]
    assert free0 + (16 << 20) <= free1 <= free0 + total // 128 + (64 << 20)
    mx.release_memory()
    assert torch.cuda.mem_get_info()[0] == free1


def test_memory_of_destroyed_plans_is_bounded(mx):
    """Plans of more than 1/128 of the device's memory, alive side by side and then destroyed: what the library keeps of
    them stays within that bound, and release_memory() gives back what it kept."""
    import torch
    rows, offs = 6000000, torch.arange(-4, 4, device="cuda", dtype=torch.int32) * 1000
    r = torch.arange(rows, device="cuda", dtype=torch.int32)
    c = r[:, None] + offs[None, :]
    ok = (c >= 0) & (c < rows)
    ptr = torch.zeros(rows + 1, dtype=torch.int32, device="cuda")
    ptr[1:] = torch.cumsum(ok.sum(1), 0)
    c = c[ok]
    v = torch.rand(c.numel(), dtype=torch.float64, device="cuda")
    del ok, r
    slack = 64 << 20  # (of the runtime's own)

    def free():
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        return torch.cuda.mem_get_info()[0]

    mx.Plan.from_device(ptr, c, v, rows, 0.0, 0.0).close()  # (code objects and the like are there from here on)
    mx.release_memory()
    total, before = torch.cuda.mem_get_info()[1], free()
    plans = []
    while before - free() < total // 128 + (1 << 30):
        plans.append(mx.Plan.from_device(ptr, c, v, rows, 0.0, 0.0))
        assert len(plans) < 32
    for p in plans:
        p.close()
    kept = before - free()
    assert 256 << 20 < kept <= total // 128 + slack, kept
    mx.release_memory()
    assert before - free() <= slack


@pytest.mark.parametrize("dtype", [np.float64, np.float16])
@pytest.mark.parametrize("lens", [
    [511, 512, 513, 1, 0, 1535, 1536, 1537, 2, 2047, 2048, 2049, 3],  # a workgroup's share of short rows, the first long class
    [4095, 4096, 4097, 7, 8191, 8192, 0, 5, 512, 512, 512, 512],      # the other two classes
    [20, 8193, 3000, 1, 700, 0, 0, 9],                                # a row that no workgroup has room for
    [1] * 1536 + [512] * 4 + [1] * 511 + [513] + [0] * 40 + [2] * 700,
    [0] * 20000 + [3] + [0] * 9000 + [600, 0, 2] + [0] * 40000,       # nearly all rows empty
], ids=["short", "long", "beyond", "packed", "empty"])
def test_rows_put_in_order(mx, dtype, lens):
    """Split, tile encoding and slice layout made on the device from rows in any order that name columns twice, with
    rows at the edges of what a workgroup puts in order: byte for byte the host's."""
    import torch
    rng = np.random.default_rng(len(lens))
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n, cols = int(ptr[-1]), 9000
    A = mx.Csr(len(lens), cols, ptr, rng.integers(0, cols, n).astype(np.int32), (rng.integers(1, 2000, n) / 64.0).astype(dtype))
    rp, ci, va = (torch.from_numpy(a).cuda() for a in (A.rowPtr, A.colInd, A.val))
    for tau in [(0.5, 0.25), (1.0, 1.0), (0.1, 0.02)]:
        P = mx.Partition(A, *tau)
        dc, dr, sel = mx.select_device(rp, ci, cols, *tau)
        got = mx.split_device(rp, ci, va, cols, sel, dc, dr)
        T = mx.tiles_device(got[0], got[1], got[2], sel["dCols"])
        pairs = list(zip(got, ("ddRowPtr", "ddColInd", "ddVal", "cdRowPtr", "cdColInd", "cdVal")))
        pairs += [(T[k], k) for k in ("chunkPtr", "sparse_AToX_index", "fragPtr", "fragBit", "tcVal")]
        for g, name in pairs:
            want = np.ascontiguousarray(getattr(P, name))
            assert np.array_equal(g.cpu().numpy().view(np.uint8), want.view(np.uint8)), (tau, name)
        P.close()
    H, D = mx.slice_layout(A, nCU=16), mx.slice_layout(A, nCU=16, device=True)
    for k in ("chunkEnd", "segPtr", "segIdx", "rowInfo", "ecol", "eval"):
        assert np.array_equal(H[k].view(np.uint8), D[k].view(np.uint8)), k


@pytest.mark.parametrize("dtype", [np.float64, np.float16])
@pytest.mark.parametrize("rows,cols,half,far", [
    (40000, 40000, 300, 0),      # nothing outside the windows
    (40001, 40000, 300, 300),    # one row beyond whole chunks; a few rows that reach elsewhere
    (65600, 30011, 900, 2000),   # fewer columns, an odd number: the last windows end at the end of x
    (40007, 90005, 2000, 40007), # more columns; an entry outside for every row
])
def test_window_form(mx, ora, dtype, rows, cols, half, far):
    """Matrices whose neighbouring rows reach into one window of x, with entries outside it, chunks taken apart for a
    row with many of those, empty rows and whole empty chunks, rows in any order that name a column twice: the product
    from both routes equals the oracle's (integers: every sum is exact), entries kept or streamed, with x at any element;
    a row's sum is not touched by an infinite x that the row does not name."""
    import torch
    rng = np.random.default_rng(rows + far)
    lens = rng.integers(14, 21, rows)
    lens[5], lens[640:704], lens[1000:1003], lens[-1] = 90, 0, 0, 1
    r = np.repeat(np.arange(rows), lens)
    c = np.clip(r * cols // rows + rng.integers(-half, half + 1, r.size), 0, cols - 1)
    lo = np.concatenate([[0], np.cumsum(lens)])
    for i in rng.choice(rows, far, replace=False) if far else []:
        if lens[i] > 1:
            c[lo[i] + rng.integers(0, lens[i])] = rng.integers(0, cols)
    if far:
        c[lo[2000]:lo[2000] + 12] = rng.integers(0, cols, 12)   # more than a lane takes beside its window
    c[lo[3000] + 1] = c[lo[3000]]
    val = rng.integers(1, 4, r.size) * rng.choice([-1, 1], r.size)
    if dtype == np.float64:
        val = val * rng.integers(1, 1000, r.size)  # (few distinct binary64 values would send it to another form)
    A = mx.Csr(rows, cols, lo.astype(np.int32), c.astype(np.int32), val.astype(dtype))
    x = rng.integers(-2, 3, cols).astype(dtype)
    ref = _exact(ora, A, x)
    dev = [torch.from_numpy(a).cuda() for a in (A.rowPtr, A.colInd, A.val)]
    xd = torch.zeros(cols + 1, dtype=torch.from_numpy(x).dtype, device="cuda")[1:]  # not at a multiple of 16 bytes
    xd.copy_(torch.from_numpy(x))
    arrays = None
    for plan in (mx.Plan(mx.Partition(A, 0.0, 0.0)), mx.Plan.from_device(*dev, cols, 0.0, 0.0),
                 mx.Plan.from_device(*dev, cols, 0.0, 0.0, mx.MX_PLAN_STREAM)):
        assert plan.info["csr_variant"] == 4 and plan.info["csr_main_kernel"] == 3, plan.info
        got = plan.arrays()
        assert len(got["windows.apart"]) > 0 or not far
        assert arrays is None or got == arrays
        arrays = got
        y = torch.full((rows,), 7.0, dtype=xd.dtype, device="cuda")
        plan.spmv(xd, y)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), ref)
    bad = x.copy()
    bad[[0, cols // 2, cols - 1]] = np.inf
    touched = np.zeros(rows, bool)
    touched[r[~np.isfinite(bad[A.colInd])]] = True
    got = plan.spmv(torch.from_numpy(bad).cuda()).cpu().numpy()
    assert np.array_equal(~np.isfinite(got), touched)


@pytest.mark.parametrize("dtype", [np.float64, np.float16])
@pytest.mark.parametrize("form", ["offsets", "windows"])
def test_forms_in_a_captured_graph(mx, dtype, form):
    """A product of either form, by mx_spmv and by mx_spmv_static, recorded into a graph: replays with a new x in the same place,
    eager work between them, give what the eager product gives."""
    import torch
    rng = np.random.default_rng(4)
    rows, per = 40000, 18
    if form == "offsets":
        A = _diagonals(mx, rng, rows, rows, np.arange(-9, 9) * 3, dtype, False)
    else:
        c = np.clip(np.repeat(np.arange(rows), per) + rng.integers(-300, 301, rows * per), 0, rows - 1)
        A = mx.Csr(rows, rows, (np.arange(rows + 1) * per).astype(np.int32), c.astype(np.int32), rng.standard_normal(rows * per).astype(dtype))
    plan = mx.Plan(mx.Partition(A, 0.0, 0.0))
    assert plan.info["csr_variant"] == (3 if form == "offsets" else 4)
    x = torch.zeros(rows, dtype=torch.float64 if dtype == np.float64 else torch.float16, device="cuda")
    y, ys = torch.empty_like(x), torch.empty_like(x)
    plan.spmv(x, y)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.spmv(x, y)
        plan.spmv_static(x, ys)
    for k in range(4):
        x.copy_(torch.from_numpy(rng.standard_normal(rows).astype(dtype)))
        graph.replay()
        torch.cuda.synchronize()
        want = plan.spmv(x)
        assert torch.equal(y, want) and torch.equal(ys, want), k
        x.mul_(2)
        torch.cuda.synchronize()
