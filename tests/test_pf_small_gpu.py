"""The small kernels around the prefill attention at the sizes where their tiles
end, against the oracle, bit for bit: the K smoothing mean and the standalone
planar Q8_1."""
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


# 64 blocks per workgroup, two per lane; ld and the address decide the 16-byte
# path (ld % 4, offset % 4 floats); all-zero, tiny and huge blocks
@pytest.mark.parametrize("rows,kb,pad,offset", [(1, 1, 0, 0), (3, 8, 4, 0), (5, 33, 0, 4), (2, 64, 0, 0), (3, 65, 8, 0),
                                                (2, 130, 0, 0), (4, 64, 1, 0), (3, 9, 0, 1)])
def test_quant_rows_bit_exact(lk, oracle, rows, kb, pad, offset):
    rng = np.random.default_rng(rows * 1000 + kb)
    ld = kb * 32 + pad
    X = rng.standard_normal((rows, ld)).astype(np.float32)
    X[0, :32] = 0.0
    X[-1, kb * 32 - 32:kb * 32] *= np.float32(1e-30)
    X[rows // 2, kb * 32 - 20] = 3e30
    buf = torch.empty(rows * ld + 8, device="cuda")
    x = buf[offset:offset + rows * ld]
    x.copy_(dev(X.reshape(-1)))
    qs = torch.zeros(rows, kb * 32, dtype=torch.int8, device="cuda")
    sc = torch.zeros(rows, kb, 2, device="cuda")
    note(f"pf_quant_rows rows={rows} kb={kb} pad={pad} offset={offset}")
    lk.pf_quant_rows(x, rows, ld, kb, qs, sc)
    torch.cuda.synchronize()
    wq, ws = oracle.pf_quant_rows(X, rows, ld, kb)
    assert np.array_equal(host(qs), np.asarray(wq).reshape(rows, kb * 32))
    assert np.array_equal(host(sc).view(np.uint32), np.asarray(ws, np.float32).reshape(rows, kb, 2).view(np.uint32))
