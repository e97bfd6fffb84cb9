"""The small kernels around the prefill attention at the sizes where their tiles
end, against the oracle, bit for bit: the K smoothing mean and the standalone
planar Q8_1; and the merge of many split-K parts."""
import numpy as np
import pytest
import torch

from gpu_util import dev, host, note

pytestmark = pytest.mark.gpu


# tiles of 1024 rows, four in a ring, 16 running sums, up to 128 rows without
# tiles: both sides of each
@pytest.mark.parametrize("n", [1, 15, 17, 128, 129, 145, 1023, 1024, 1025, 2048, 3079, 4096, 5121, 8192])
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


# up to 14336 blocks one value per lane; above, 64 blocks per workgroup, two per
# lane: 64 of one row, or 8 of 8 rows, where ld and the address allow 16 bytes (ld
# % 4, offset % 4 floats); all-zero, tiny and huge blocks
@pytest.mark.parametrize("rows,kb,pad,offset", [(1, 1, 0, 0), (3, 8, 4, 0), (5, 33, 0, 4), (2, 64, 0, 0), (3, 65, 8, 0),
                                                (2, 130, 0, 0), (4, 64, 1, 0), (3, 9, 0, 1), (2001, 8, 0, 0),
                                                (1600, 9, 4, 0), (447, 33, 0, 4), (225, 64, 0, 0), (113, 128, 8, 0),
                                                (222, 65, 0, 0), (16385, 1, 0, 0), (225, 64, 1, 0), (2001, 8, 0, 1), (224, 64, 0, 0), (14336, 1, 0, 0),
                                                (14337, 1, 0, 0)])
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


def _both_forms(lk, X):
    """The planes of X, repeated to more blocks than the one-value form is chosen for,
    by 16-byte loads, and by single values (an address off by 4 bytes)."""
    X = np.tile(X, (14336 // (X.size // 32) + 1, 1))
    rows, ld = X.shape
    out = []
    for offset in (0, 1):
        buf = torch.empty(rows * ld + 8, device="cuda")
        x = buf[offset:offset + rows * ld]
        x.copy_(dev(X.reshape(-1)))
        qs = torch.full((rows, ld), 77, dtype=torch.int8, device="cuda")
        sc = torch.zeros(rows, ld // 32, 2, device="cuda")
        note(f"pf_quant_rows special values, offset={offset}")
        lk.pf_quant_rows(x, rows, ld, ld // 32, qs, sc)
        torch.cuda.synchronize()
        out.append((host(qs), host(sc)))
    return out


# NaN and infinities: the two forms give the same bytes and scales; a block of
# NaN alone has a NaN scale.
def test_quant_rows_nan_and_infinite_blocks(lk):
    rng = np.random.default_rng(5)
    X = rng.standard_normal((6, 4 * 32)).astype(np.float32)
    X[0, :32] = np.nan
    X[1, 40] = np.nan
    X[2, 64:96] = np.inf
    X[3, 100], X[3, 101] = np.inf, -np.inf
    X[4, :32], X[4, 7] = np.nan, np.inf
    X[5, 32:64] = np.float32(3.4e38) * np.sign(X[5, 32:64])
    (q4, s4), (q1, s1) = _both_forms(lk, X)
    assert np.isnan(s1[0, 0, 0])
    assert np.array_equal(q4, q1)
    assert np.array_equal(s4, s1, equal_nan=True)


# Blocks whose maximum is a subnormal of 1 to 200 units: below 64 of them d = am /
# 127 rounds to zero, and the quotients are infinite.
def test_quant_rows_smallest_subnormals(lk):
    rng = np.random.default_rng(6)
    X = np.empty((200, 2 * 32), np.float32)
    for r in range(200):
        u = rng.integers(0, r + 2, 64).astype(np.uint32)
        u[[3, 40]] = r + 1
        X[r] = (u | (rng.integers(0, 2, 64).astype(np.uint32) << 31)).view(np.float32)
    (q4, s4), (q1, s1) = _both_forms(lk, X)
    assert np.array_equal(s4.view(np.uint32), s1.view(np.uint32))
    assert np.array_equal(q4, q1)


# more than 8 parts per block take the wide merge: part counts off its two
# eights, ragged last blocks, both outputs.  2e-3 of the largest output is the
# bound every prefill case here is held to: p rounded to fp16 (2^-11 each) on
# rows of a few thousand keys.
@pytest.mark.parametrize("m,P,tiles", [(1, 640, 1), (5, 2100, 2), (77, 1500, 1), (130, 3000, 3), (64, 4000, 1)])
def test_combine_many_parts(lk, oracle, m, P, tiles):
    from gpu_util import dev_h
    K, V, Q = oracle.mt_prefill_case(99 + m, m, P, 0.0, False)
    kc, vc, qh = dev_h(K), dev_h(V), dev_h(Q)
    try:
        lk.pf_split_override(tiles)
        items = lk.pf_plan_items(m, P, 0, 0, False)
        assert max(sum(1 for i in items if i[0] == q) for q in {i[0] for i in items}) > 8
        outs = []
        note(f"pf_attn many parts m={m} P={P} tiles={tiles}")
        for _ in range(2):
            o = torch.full((m, 2048), float("nan"), device="cuda")
            aqs = torch.zeros(m, 2048, dtype=torch.int8, device="cuda")
            asc = torch.zeros(m, 64, 2, device="cuda")
            lk.pf_attn_q81(qh, m, P, kc, vc, o, aqs, asc)
            torch.cuda.synchronize()
            outs.append((host(o), host(aqs), host(asc)))
    finally:
        lk.pf_split_override(0)
    for a, b in zip(*outs):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), "run-to-run bit-identical"
    rows = np.array(sorted({0, m // 2, m - 1}), np.int32)
    ref = oracle.pf_ref(Q, m, P, K, V, rows=rows)
    assert oracle.rel_err(outs[0][0][rows], ref[rows]) <= 2e-3
    q, sc = oracle.pf_quant_rows(outs[0][0], m, 2048, 64)
    assert np.array_equal(outs[0][1], q) and np.array_equal(outs[0][2].view(np.uint32), sc.view(np.uint32))


# A last block of at most 16 or 32 rows runs only the query blocks that hold
# rows.  The same rows inside a chunk of whole blocks go through the full tile:
# the same key tiles in the same order (unsplit), so every output is the same
# bits.  The chunk's further queries are zero, as the kernel takes rows that are
# not there: a query whose weights pass 2^15 makes its wave raise every running
# maximum whose weights passed 2^14, so other neighbours could move a rounding.
@pytest.mark.parametrize("m", [1, 15, 16, 17, 32, 33, 65, 80, 81, 96, 97])
@pytest.mark.parametrize("P,near,sink", [(0, 1024, 1), (700, 64, 1), (1999, 128, 0)])
@pytest.mark.parametrize("int8", [True, False])
def test_short_last_block_is_bit_identical(lk, m, P, near, sink, int8):
    full = (m + 63) // 64 * 64
    S, ks = P + full, lk.kstride_for(P + full)
    g = torch.Generator(device="cuda").manual_seed(m + P)
    qh = (torch.randn(full, 2048, device="cuda", generator=g) / 4).half()
    qh[m:] = 0
    kc = torch.randn(S, 512, device="cuda", generator=g).half()
    kc[S // 3] *= 12                                      # a late large key: the running maximum has to move
    vc = torch.randn(S, 512, device="cuda", generator=g).half()
    k8 = torch.empty(S, 512, dtype=torch.int8, device="cuda")
    ksc = torch.empty(8, ks, device="cuda")
    lk.pf_k8(kc, 0, S, None, ks, k8, ksc)
    q8 = torch.empty(full, 2048, dtype=torch.int8, device="cuda")
    qsc, qcs = torch.empty(full, 32, device="cuda"), torch.empty(full, 32, device="cuda")
    lk.pf_q8(qh, full, None, q8, qsc, qcs)

    def run(rows, given):
        o = torch.full((full, 2048), 7.0, device="cuda")
        aqs = torch.full((full, 2048), 7, dtype=torch.int8, device="cuda")
        asc = torch.full((full, 64, 2), 7.0, device="cuda")
        note(f"short last block m={rows} P={P} near={near} sink={sink} int8={int8} q8 given={given}")
        if int8:
            q = (q8, qsc, qcs) if given else (None, None, None)
            lk.pf_attn8_q81(*q, qh, rows, P, k8, ksc, ks, kc, vc, near, sink, o, aqs, asc)
        else:
            lk.pf_attn_q81(qh, rows, P, kc, vc, o, aqs, asc)
        torch.cuda.synchronize()
        return o, aqs, asc

    lk.pf_split_override(-1)
    lk.pf_pair_override(-1)
    try:
        for given in (False, True) if int8 else (False,):
            for a, b in zip(run(m, given), run(full, given)):
                assert torch.equal(a[:m].view(torch.uint8), b[:m].view(torch.uint8))
                assert bool((a[m:] == 7).all())           # nothing past the chunk's rows is written
    finally:
        lk.pf_split_override(0)
        lk.pf_pair_override(0)


# Asking for the Q8_1 planes changes no row: the key-range cuts are those of the
# chunk, for both score types, on chunks of few blocks whose plan splits.
@pytest.mark.parametrize("m,P", [(5, 30000), (77, 3000), (77, 30011), (300, 9000), (700, 700)])
@pytest.mark.parametrize("int8", [True, False])
def test_rows_do_not_depend_on_the_planes(lk, m, P, int8):
    S, ks = P + m, lk.kstride_for(P + m)
    g = torch.Generator(device="cuda").manual_seed(m + P)
    qh = (torch.randn(m, 2048, device="cuda", generator=g) / 4).half()
    kc = torch.randn(S, 512, device="cuda", generator=g).half()
    vc = torch.randn(S, 512, device="cuda", generator=g).half()
    assert lk.pf_plan_items(m, P, 1024, 1, int8)
    o1, o2 = (torch.full((m, 2048), float("nan"), device="cuda") for _ in range(2))
    aqs = torch.empty(m, 2048, dtype=torch.int8, device="cuda")
    asc = torch.empty(m, 64, 2, device="cuda")
    note(f"rows with and without planes m={m} P={P} int8={int8}")
    if int8:
        k8 = torch.empty(S, 512, dtype=torch.int8, device="cuda")
        ksc = torch.empty(8, ks, device="cuda")
        lk.pf_k8(kc, 0, S, None, ks, k8, ksc)
        lk.pf_attn8(None, None, None, qh, m, P, k8, ksc, ks, kc, vc, 1024, 1, o1)
        lk.pf_attn8_q81(None, None, None, qh, m, P, k8, ksc, ks, kc, vc, 1024, 1, o2, aqs, asc)
    else:
        lk.pf_attn(qh, m, P, kc, vc, o1)
        lk.pf_attn_q81(qh, m, P, kc, vc, o2, aqs, asc)
    torch.cuda.synchronize()
    assert torch.equal(o1.view(torch.int32), o2.view(torch.int32))
    qs, sc = torch.empty_like(aqs), torch.empty_like(asc)
    lk.pf_quant_rows(o1, m, 2048, 64, qs, sc)
    torch.cuda.synchronize()
    assert torch.equal(qs, aqs) and torch.equal(sc.view(torch.int32), asc.view(torch.int32))


# The merge adds the parts in part order, four a pass, whatever their number: the
# same recurrence on the partials that the launch left in the caller's workspace
# gives the same bits.  One tile per part; part counts on both sides of the wide
# merge's line and of its eights.
@pytest.mark.parametrize("m,P,parts", [(5, 120, [2]), (64, 128, [3]), (5, 500, [8]), (5, 570, [9]), (5, 1010, [16]),
                                       (20, 1060, [17]), (77, 2112, [34, 35]), (40, 2960, [47]), (1, 4095, [64])])
def test_merge_is_the_part_order_recurrence(lk, m, P, parts):
    S = P + m
    g = torch.Generator(device="cuda").manual_seed(m + P)
    qh = (torch.randn(m, 2048, device="cuda", generator=g) / 2).half()
    kc = torch.randn(S, 512, device="cuda", generator=g).half()
    vc = torch.randn(S, 512, device="cuda", generator=g).half()
    o = torch.full((m, 2048), float("nan"), device="cuda")
    aqs = torch.empty(m, 2048, dtype=torch.int8, device="cuda")
    asc = torch.empty(m, 64, 2, device="cuda")
    work = torch.zeros(lk.pf_part_bytes() // 4, device="cuda")
    note(f"merge order m={m} P={P} parts={parts}")
    try:
        lk.pf_split_override(1)
        items = lk.pf_plan_items(m, P, 0, 0, False)
        assert [sum(1 for i in items if i[0] == q) for q in range((m + 63) // 64)] == parts
        lk.pf_attn_ws(qh, m, P, kc, vc, o, aqs, asc, work)
        torch.cuda.synchronize()
    finally:
        lk.pf_split_override(0)
    ACC, SLOT = 4 * 16 * 64 * 4, 4 * 16 * 64 * 4 + 4 * 64 * 2
    for qt in {i[0] for i in items}:
        slots = [i[3] for i in sorted(items) if i[0] == qt]
        if slots == [-1]:
            continue
        rows = min(64, m - 64 * qt)
        recs = work[slots[0] * 8 * SLOT:(slots[0] + len(slots)) * 8 * SLOT].view(len(slots), 8, SLOT)
        acc = recs[:, :, :ACC].reshape(-1, 8, 4, 16, 64, 4).permute(0, 1, 2, 4, 3, 5).reshape(-1, 8, 4, 64, 64)
        ml = recs[:, :, ACC:].reshape(-1, 8, 4, 64, 2)
        M = torch.full((8, 4, 64), -float("inf"), device="cuda")
        L, A = torch.zeros_like(M), torch.zeros(8, 4, 64, 64, device="cuda")
        for p0 in range(0, len(slots), 4):
            one = range(p0, min(p0 + 4, len(slots)))
            Mn = M
            for p in one:
                Mn = torch.maximum(Mn, ml[p, ..., 0])
            r = torch.exp2(M - Mn)
            L, A = L * r, A * r.unsqueeze(-1)
            for p in one:
                w = torch.exp2(ml[p, ..., 0] - Mn)
                L, A = L + ml[p, ..., 1] * w, A + acc[p] * w.unsqueeze(-1)
            M = Mn
        want = (A * (1.0 / L).unsqueeze(-1)).permute(2, 0, 1, 3).reshape(64, 2048)[:rows]
        assert torch.equal(o[64 * qt:64 * qt + rows].view(torch.int32), want.contiguous().view(torch.int32)), len(slots)
