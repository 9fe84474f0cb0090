"""GPU tests of what a plan's layout decides on the device, against the host's decisions at the edges of the rules."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAMES = ("wgDesc", "waveDesc", "chunkEnd", "segPtr", "segIdx", "rowInfo", "lightInfo", "heavyInfo", "ecol", "eval", "ecode", "dict")
SCALARS = ("nWG", "S", "sliceCols", "waves", "stepEntries", "batchEntries", "cap", "chunks", "batches", "vrows", "nLight", "nHeavy", "lightSegs", "nDict")


def _same_layout(mx, A, ncu):
    H, D = mx.slice_layout(A, nCU=ncu), mx.slice_layout(A, nCU=ncu, device=True)
    for k in SCALARS:
        assert H[k] == D[k], (k, H[k], D[k])
    for k in NAMES:
        assert H[k].shape == D[k].shape and np.array_equal(H[k].view(np.uint8), D[k].view(np.uint8)), k
    return H


@pytest.mark.parametrize("dtype,rows,cols,lengths,ncu", [
    (np.float64, 64, 16384, [64], 7),                       # one chunk
    (np.float64, 65, 16384, [64, 70], 7),                   # two, one of a single virtual row
    (np.float64, 30000, 16384, [3], 7),                     # chunks of one length only: every workgroup filled to one level
    (np.float64, 30000, 16385, [1, 2, 3, 90], 7),           # a second slice with a column of its own
    (np.float16, 40000, 65536, list(range(1, 60)), 256),    # a length to a handful of chunks: few of each, and more workgroups than that
    (np.float16, 200000, 400000, [1, 1, 1, 2, 40], 256),
    (np.float64, 600000, 30000, [1, 2], 1),                 # workgroups full of chunks (4096) before the others: the limit binds
    (np.float64, 150000, 16000, [1, 5, 9], 1500),           # more workgroups in a slice than its wave keeps in LDS
    (np.float16, 150000, 65000, [7], 1024),                 # as many as it keeps there
])
def test_chunks_are_dealt_as_on_the_host(mx, dtype, rows, cols, lengths, ncu):
    rng = np.random.default_rng(rows + cols)
    lens = rng.choice(lengths, rows)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    A = mx.Csr(rows, cols, ptr, rng.integers(0, cols, ptr[-1]).astype(np.int32), rng.uniform(-1, 1, ptr[-1]).astype(dtype))
    H = _same_layout(mx, A, ncu)
    assert H["chunks"] >= rows // 64


@pytest.mark.parametrize("dtype,lens,cols", [
    (np.float64, [5000] * 9, 40000),                            # rows of several tiles, runs that tiles begin in, cut at the cap
    (np.float64, [1024, 1023, 1, 1024, 0, 0, 2048, 512, 512], 60000),    # rows that end with a tile, and one entry off
    (np.float64, [64, 0, 64, 1, 63, 128, 960, 0] * 6, 16384),   # ... with a word; one slice
    (np.float16, [9000] + [3] * 4000, 140000),
    (np.float64, [0] * 500 + [4159] + [0] * 9000 + [1], 20000), # mostly rows without entries; a last tile of one word
    (np.float16, [1] * 70000, 300000),                          # a virtual row to an entry
])
@pytest.mark.parametrize("order", ["ascending", "any"])
def test_virtual_rows_are_cut_as_on_the_host(mx, dtype, lens, cols, order):
    rng = np.random.default_rng(len(lens) + cols)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    col = rng.integers(0, cols, ptr[-1]).astype(np.int32)
    if order == "ascending":
        for r in np.nonzero(lens)[0] if len(lens) < 5000 else []:
            col[ptr[r]:ptr[r + 1]].sort()
    A = mx.Csr(len(lens), cols, ptr, col, rng.integers(-9, 10, ptr[-1]).astype(dtype))
    _same_layout(mx, A, 7)


@pytest.mark.parametrize("dtype,most", [(np.float64, 15), (np.float64, 16), (np.float64, 17), (np.float16, 17), (np.float64, 64), (np.float64, 65), (np.float16, 3000)])
def test_rows_of_many_virtual_rows(mx, dtype, most):
    """The list of a row's virtual rows by the row's own thread (up to 16 of them) or by its wave: a virtual row to an entry, rows without, short and long
    lists side by side, long ones at both ends of a wave and in the last row."""
    per = 16384 if dtype == np.float64 else 65536
    lens = np.array(([0, 1, most, 2, most - 1] + [3] * 57 + [most, most] + [0] * 63 + [most]) * 3)
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    slices = min(most, 60)
    col = np.concatenate([np.sort(np.arange(n) % slices * per + np.arange(n) // slices) for n in lens]).astype(np.int32)
    A = mx.Csr(lens.size, slices * per, ptr, col, np.random.default_rng(most).uniform(-1, 1, ptr[-1]).astype(dtype))
    H = _same_layout(mx, A, 30)
    assert np.diff(H["segPtr"]).max() >= min(most, 60)


def _fused_case(name, rng):
    """(matrix, whether the one-launch form takes it when it is asked for)"""
    def m(lens, col, cols, dtype=np.float64):
        ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        row = np.repeat(np.arange(len(lens)), lens)
        return len(lens), cols, ptr, np.asarray(col(row), np.int32), rng.uniform(-1, 1, ptr[-1]).astype(dtype)
    anywhere = lambda cols: (lambda row: rng.integers(0, cols, row.size))
    few = lambda rows: rng.integers(0, 9, rows)
    if name == "fewer groups than XCDs":
        return m(np.full(7 * 256, 16), anywhere(16384), 16384), False
    if name == "a group each":
        return m(np.full(8 * 256, 32), lambda row: np.arange(row.size) % 8 * 16384 + rng.integers(0, 16384, row.size), 131072), True
    if name == "a row more":
        return m(np.full(8 * 256 + 1, 32), lambda row: np.arange(row.size) % 8 * 16384 + rng.integers(0, 16384, row.size), 131072), True
    if name == "all entries in the last rows":
        lens = np.zeros(20000, int)
        lens[-300:] = 200
        return m(lens, anywhere(40000), 40000), None
    if name == "eight places":
        lens = few(20000)
        lens[7000] = 4000
        return m(lens, lambda row: np.where(row == 7000, rng.integers(0, 8, row.size) * 16384, rng.integers(0, 130000, row.size)), 131072), False
    if name == "eight places, no more":
        lens = few(20000)
        lens[7000] = 8
        return m(lens, lambda row: np.where(row == 7000, np.arange(row.size) % 8 * 16384, rng.integers(0, 130000, row.size)), 131072), True
    if name == "nine places":
        lens = few(20000)
        lens[7000] = 9
        return m(lens, lambda row: np.where(row == 7000, np.arange(row.size) % 9 * 16384, rng.integers(0, 140000, row.size)), 9 * 16384), False
    if name == "more slices than workgroups of an XCD":
        return m(np.full(100000, 6), anywhere(33 * 65536), 33 * 65536, np.float16), False
    if name == "as many":
        return m(np.full(100000, 6), anywhere(32 * 65536), 32 * 65536, np.float16), True
    if name == "a small part":
        return m(few(60000), lambda row: np.where(rng.random(row.size) < 1e-4, 70000, 0) + rng.integers(0, 60000, row.size), 140000, np.float16), True
    if name == "too many chunks for a workgroup":
        return m(np.full(1700000, 1), anywhere(60000), 60000, np.float16), False
    if name == "as many as it may have":
        return m(np.full(1500000, 1), anywhere(60000), 60000, np.float16), True
    if name.startswith("virtual rows"):
        return m(np.full(int(name.split()[-1]), 9), anywhere(16384), 16384), True
    assert name == "repeats"
    return m(few(30000), lambda row: row // 300 * 100, 30000), True


@pytest.mark.parametrize("name", ["fewer groups than XCDs", "a group each", "a row more", "all entries in the last rows", "eight places", "eight places, no more",
                                  "nine places", "more slices than workgroups of an XCD", "as many", "a small part", "too many chunks for a workgroup",
                                  "as many as it may have", "repeats", "virtual rows 16383", "virtual rows 16384"])
def test_one_launch_plan_is_the_hosts(mx, monkeypatch, name):
    """The one-launch form planned on the device (from 16384 virtual rows on) and on the host: taken or refused alike, and every array the same."""
    import torch
    rng = np.random.default_rng(len(name))
    (rows, cols, ptr, col, val), takes = _fused_case(name, rng)
    A = mx.Csr(rows, cols, ptr, col, val)
    flags = mx.MX_PLAN_CSR_SLICES | mx.MX_PLAN_FUSE
    D = mx.Plan.from_device_csr(*(torch.from_numpy(a).cuda() for a in (ptr, col, val)), cols, flags)
    P = mx.Partition(A, 0.0, 0.0)
    monkeypatch.setenv("MX_LAYOUT", "host")
    H = mx.Plan(P, flags)
    monkeypatch.delenv("MX_LAYOUT")
    assert H.info["csr_variant"] == D.info["csr_variant"] == 1
    assert H.info["csr_fused"] == D.info["csr_fused"], H.info
    assert takes is None or bool(D.info["csr_fused"]) == takes
    assert H.arrays() == D.arrays()
    x = torch.from_numpy(rng.integers(-2, 3, cols).astype(val.dtype)).cuda()
    assert bool((H.spmv(x) == D.spmv(x)).all())


@pytest.mark.parametrize("rows,cols", [(8191, 8192), (8193, 8191), (20000, 3), (3, 20000), (5000, 40000), (1, 1)])
@pytest.mark.parametrize("tau", [(1.0, 1.0), (0.6, 0.2)])
def test_lines_by_count_are_the_hosts(mx, rows, cols, tau):
    """Columns and rows ordered by count on the device: counts of one digit and of two (columns that every row names, a row of 4100
    entries), ties, lines without entries, and as many lines as a tile has, one fewer and one more."""
    rng = np.random.default_rng(rows + cols)
    lens = rng.integers(0, 7, rows)
    lens[rng.integers(0, rows, 2)] = min(cols, 4100)
    row = np.repeat(np.arange(rows), lens)
    col = np.where(rng.random(row.size) < 0.5, rng.integers(0, min(cols, 5), row.size), rng.integers(0, cols, row.size))
    ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    A = mx.Csr(rows, cols, ptr, col.astype(np.int32), rng.integers(-9, 10, row.size).astype(np.float64))
    D, H = mx.Partition(A, *tau, device=True), mx.Partition(A, *tau, device=False)
    for k in ("dCols", "dRows", "nnzColD", "nnzRowD"):
        assert getattr(D, k) == getattr(H, k), k
    for k in ("descColId", "rId", "ddRowPtr", "ddColInd", "cdRowPtr", "cdColInd", "chunkPtr", "fragPtr", "sparse_AToX_index"):
        assert np.array_equal(getattr(D, k), getattr(H, k)), k
