"""cmag_sort_by_key takes 9- or 10-bit digits for keys of 17 to 20 bits up to
2^21 keys, if its scratch holds their tables, and scans up to 2^17 counts in one
launch: the stable argsort on both sides of every line, whatever the scratch's
size and alignment."""
import numpy as np
import pytest
import torch

from cmag_amd import _lib as L

pytestmark = pytest.mark.gpu


def least_bytes(n):
    """what 8-bit digits take: key bits outside 17..20 choose them"""
    return int(L.lib().cmag_sort_scratch_bytes(n, 16))


def check(n, bits, nbytes, offset=0):
    rng = np.random.default_rng(n + bits)
    # few distinct keys and many, both ends of the range among them
    keys = rng.integers(0, 1 << bits, n, dtype=np.uint32) if n % 2 else \
        rng.choice(np.array([0, 1, (1 << bits) - 1, 1 << (bits - 1), 255, 256, 511, 512], np.uint32), n)
    vals = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    k = torch.as_tensor(keys.view(np.int32), device="cuda")
    v = torch.as_tensor(vals.view(np.int32), device="cuda")
    scratch = torch.empty(nbytes + offset, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    L.call("cmag_sort_by_key", k.data_ptr(), v.data_ptr(), n, bits, scratch.data_ptr() + offset, nbytes, None)
    torch.cuda.synchronize()
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(k.cpu().numpy().view(np.uint32), keys[order])
    assert np.array_equal(v.cpu().numpy().view(np.uint32), vals[order])


@pytest.mark.parametrize("bits", [16, 17, 18, 19, 20, 21])
@pytest.mark.parametrize("n", [2, 255, 4097, 65535, (1 << 18) - 1, (1 << 18) + 1, (1 << 21) - 1, 1 << 21, (1 << 21) + 1])
def test_stable_argsort(device, n, bits):
    full = int(L.lib().cmag_sort_scratch_bytes(n, bits))
    assert full >= least_bytes(n)
    check(n, bits, full)
    if full > least_bytes(n):
        check(n, bits, least_bytes(n))
        check(n, bits, full - 1)
    check(n, bits, full, offset=4)


def test_too_small_scratch_is_refused(device):
    n = 5000
    k = torch.zeros(n, dtype=torch.int32, device="cuda")
    s = torch.empty(least_bytes(n), dtype=torch.uint8, device="cuda")
    with pytest.raises(Exception):
        L.call("cmag_sort_by_key", k.data_ptr(), k.data_ptr(), n, 18, s.data_ptr(), least_bytes(n) - 1, None)
