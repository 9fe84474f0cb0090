"""GPU tests of mx_transpose_device's routes (buckets of output lines, crowded buckets, radix sort) at the edges of their tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(mx, ptr, ind, val, inner):
    import torch
    ptr, ind = ptr.astype(np.int32), ind.astype(np.int32)
    got = mx.transpose_device(*(torch.from_numpy(a).cuda() for a in (ptr, ind, val)), inner)
    order = np.argsort(ind, kind="stable")
    want = (np.concatenate([[0], np.cumsum(np.bincount(ind, minlength=inner))]).astype(np.int32),
            np.repeat(np.arange(ptr.size - 1, dtype=np.int32), np.diff(ptr))[order], val[order])
    for g, w in zip(got, want):
        assert np.array_equal(g.cpu().numpy().view(np.uint8), w.view(np.uint8))


def _matrix(rng, outer, nnz, dtype):
    ptr = np.sort(np.concatenate([[0, nnz], rng.integers(0, nnz + 1, outer - 1)]))
    return ptr, rng.integers(-9, 10, nnz).astype(dtype)


@pytest.mark.parametrize("dtype", [np.float64, np.float16])
@pytest.mark.parametrize("outer,inner,nnz", [
    (1, 1, 1), (5, 1, 8191), (300, 2, 8192), (300, 63, 8193), (9, 64, 16385), (9, 65, 4097),   # tiles; one line to a bucket, two
    (50, 2047, 300000), (50, 2048, 300000), (50, 2049, 300000),
    (20000, 64 * 2048, 70000), (50, 64 * 2048 + 1, 70000),    # as many lines as 64 buckets hold, one more
    (100, 2048 * 2048, 9000), (100, 2048 * 2048 + 1, 9000),   # ... as all of them hold; the radix sort
    (200000, 3000, 64 * 6800 + 1), (7, 100003, 3000000), (900000, 100003, 3000000), (60000, 300, 2000000),
])
def test_transpose_at_the_edges(mx, dtype, outer, inner, nnz):
    rng = np.random.default_rng(outer + inner + nnz)
    ptr, val = _matrix(rng, outer, nnz, dtype)
    _check(mx, ptr, rng.integers(0, inner, nnz), val, inner)


@pytest.mark.parametrize("share", [0.005, 0.015, 0.02, 0.07, 0.5, 1.0])
def test_transpose_of_crowded_lines(mx, share):
    """Many entries in one line: a bucket of two and of three rounds (0.5 and 1.5 %), one that its tiles' own workgroups put in order."""
    rng = np.random.default_rng(5)
    outer, inner, nnz = 30000, 40000, 1000000
    ptr, val = _matrix(rng, outer, nnz, np.float64)
    ind = np.where(rng.random(nnz) < share, 123, rng.integers(0, inner, nnz))
    _check(mx, ptr, ind, val, inner)


@pytest.mark.parametrize("dtype", [np.float64, np.float16])
@pytest.mark.parametrize("inner,nnz,crowds", [
    (40, 1023, []), (40, 1024, []),                               # from 1024 entries on by buckets
    (1, 24576, []), (1, 24577, []), (1, 90000, []),               # one bucket of one line: as many as its workgroup takes, one more
    (64, 700000, [(0, 24576)]), (64, 700000, [(0, 24577)]), (64, 700000, [(63, 40961)]),  # a line to a bucket; the first and the last of them
    (40000, 1000000, [(0, 50000)]), (40000, 1000000, [(39999, 50000), (39998, 9), (0, 26000), (1, 40000)]),  # several lines of a bucket
    (4000, 500000, [(500 * k, 25000) for k in range(8)]), (4000, 500000, [(440 * k, 25000) for k in range(9)]),  # eight crowded buckets, nine
    (4000, 1200000, [(440 * k, 110000) for k in range(9)]),       # nine that are too many for one workgroup each: the radix sort
    (10, 3000000, []),                                            # ... without counting
])
def test_transpose_of_crowded_buckets(mx, dtype, inner, nnz, crowds):
    """Buckets by their own workgroup, by workgroups for their tiles, and the radix sort, on both sides of the lines between them.  crowds: (line, entries)"""
    rng = np.random.default_rng(inner + nnz + len(crowds))
    ptr, val = _matrix(rng, 700, nnz, dtype)
    ind, places, at = np.empty(nnz, int), rng.permutation(nnz), 0
    for line, n in crowds:
        ind[places[at:at + n]] = line
        at += n
    named = {line for line, _ in crowds} if inner < 100 else set()  # (a crowd of exactly so many)
    ind[places[at:]] = rng.choice([c for c in range(inner) if c not in named], nnz - at)
    _check(mx, ptr, ind, val, inner)


def test_transpose_refuses_an_index_before_it_writes(mx):
    import ctypes

    import torch
    from matxtractt_amd import _lib
    nnz, inner = 20000, 500
    ptr = torch.arange(0, nnz + 1, 10, dtype=torch.int32, device="cuda")
    for bad in (inner, -1):
        ind = torch.randint(0, inner, (nnz,), dtype=torch.int32, device="cuda")
        ind[nnz - 1] = bad
        val = torch.ones(nnz, dtype=torch.float64, device="cuda")
        out = [torch.full((n,), 7, dtype=t, device="cuda") for n, t in ((inner + 1, torch.int32), (nnz, torch.int32), (nnz, torch.float64))]
        torch.cuda.synchronize()
        rc = _lib.load().mx_transpose_device(mx.MX_F64, ptr.numel() - 1, inner, nnz, *(ctypes.c_void_p(t.data_ptr()) for t in (ptr, ind, val, *out)), None)
        assert rc != 0 and all(bool((t == 7).all()) for t in out)
