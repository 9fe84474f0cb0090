"""GPU tests of the forms of the CSR part that a plan makes and picks on the device: value dictionaries,
offset patterns, row windows.  Against the host's layouts where they exist, against the oracle otherwise."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mx():
    import matxtractt_amd as m
    assert m.device_count() > 0, "libmatxtract_hip.so sees no HIP device"
    return m


@pytest.fixture(scope="module")
def ora():
    from oracle import mx_oracle
    return mx_oracle


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
