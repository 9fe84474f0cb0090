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
