"""The small kernels around the prefill attention at the sizes where their tiles
end: the K smoothing mean against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host, note

pytestmark = pytest.mark.gpu


# tiles of 1024 rows, four in a ring, 16 running sums: both sides of each
@pytest.mark.parametrize("n", [1, 15, 17, 1023, 1024, 1025, 2048, 3079, 4096, 5121, 8192])
@pytest.mark.parametrize("offset", [0, 1])
def test_kmean_bit_exact(lk, oracle, n, offset):
    rng = np.random.default_rng(n)
    K = rng.standard_normal((n, 512)).astype(np.float16).view(np.uint16)
    buf = torch.empty(n * 512 + 8, dtype=torch.int16, device="cuda")
    kc = buf[offset:offset + n * 512]                     # offset 1: an address that is a multiple of 2 bytes only
    kc.copy_(dev(K.view(np.int16).reshape(-1)))
    cm = torch.full((512,), float("nan"), device="cuda")
    note(f"pf_kmean n={n} offset={offset}")
    lk.pf_kmean(kc, n, cm)
    torch.cuda.synchronize()
    want = oracle.pf_kmean(K.reshape(-1), n)
    assert np.array_equal(host(cm).view(np.uint32), np.asarray(want, np.float32).reshape(-1).view(np.uint32))
