"""The K-quants' wide matrix-core kernel (wide_plan in csrc/plan.h; each test holds its shapes to that rule): ragged rows and
tokens, a last token block of at most 64, whole and split k (slices of several super-blocks, the last one shorter), against
the int8 oracle on sampled rows (tier 1: the same integer products, another f32 summation order); row and column views and the
fused epilogue against the plain call bit for bit; non-finite scales and activations."""
import numpy as np
import pytest

from conftest import random_blocks
from oracle import epilogue as EP
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TYPES = [O.Q4_K, O.Q5_K, O.Q6_K]
# split into slices of 2 super-blocks, the last one short (65 tokens: one narrow block); the same over a ragged last block; whole k
# of a ragged last block and of a narrow one; 4 slices of 4 and 14
SPLIT, WHOLE = (8240, 65, 3328), (6640, 1100, 1024)
SHAPES = [SPLIT, WHOLE, (11040, 128, 2560), (1440, 700, 3328), (7040, 1030, 1024), (14336, 128, 4096), (4096, 512, 14336)]


def weights(dt, m, k, seed):
    if dt != O.Q5_K:
        return random_blocks(dt, m, k, seed)
    w = np.random.default_rng(seed).integers(0, 256, (m, k // 256, 176), dtype=np.uint8)
    for at, lo, hi in ((0, 2e-5, 8e-5), (2, 1e-4, 5e-4)):
        w[:, :, at:at + 2] = np.random.default_rng(at).uniform(lo, hi, (m, k // 256)).astype(np.float16).view(np.uint8).reshape(m, -1, 2)
    return np.ascontiguousarray(w.reshape(m, -1))


def sampled_rows(m):
    """Whole 16-row bands: the first, a middle and the last tiles."""
    rows = np.unique(np.r_[0:32, 96:160, m - m % 128 - 16:m])[:208]
    return rows[:len(rows) // 16 * 16]


def close(oracle, dt, w, a, c, rows):
    n, k = a.shape
    ws = np.ascontiguousarray(w[rows])
    ref = oracle.mm_int8(dt, ws, a, len(rows), n, k)
    _, sa = oracle.mm_ref(dt, ws, a, len(rows), n, k)
    return np.abs(c[:, rows] - ref) <= 1e-3 * np.abs(ref) + 1e-5 * sa


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dt", TYPES)
def test_wide_tiles(hip, oracle, plans, dt, m, n, k):
    from qxotic_amd.jam import JAM, Segment
    assert plans.wide(dt, k, m, n)[0]
    w = weights(dt, m, k, m + n)
    a = oracle.outliers(n + k, (n, k))
    c = np.full((n, m + 3), -3.0, np.float32)
    assert hip.pin(Segment.of(w), dt, k, m) == JAM.OK, hip.last_error()
    try:
        st = hip.mm(Segment.of(w), 0, dt, k, Segment.of(a), 0, JAM.F32, k, Segment.of(c), 0, JAM.F32, m + 3, m, n, k)
        assert st == JAM.OK, hip.last_error()
    finally:
        hip.evict(Segment.of(w))
    assert (c[:, m:] == -3.0).all() and np.isfinite(c).all()
    ok = close(oracle, dt, w, a, c, sampled_rows(m))
    assert ok.all(), (O.NAMES[dt], m, n, k, int((~ok).sum()))


@pytest.mark.parametrize("m,n,k", [SPLIT, WHOLE])
@pytest.mark.parametrize("dt", TYPES)
def test_wide_views_and_epilogue(hip, oracle, plans, dt, m, n, k):
    """Rows 96.. and the first k columns of a larger pinned tensor give the bits of a tensor that is just these; bias and residual
    are the f32 operations after the plain result, whole and behind the K slices' sum."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    assert plans.wide(dt, k, m, n)[0]
    r0, ldw = 96, k + 512
    big = weights(dt, m + r0 + 40, ldw, 31 + m)
    view, small = big[r0:], np.ascontiguousarray(big[r0:r0 + m, :O.row_bytes(dt, k)])
    a = torch.from_numpy(oracle.outliers(n + k + 1, (n, k))).cuda()
    rng = np.random.default_rng(m + n)
    bias, c0 = rng.standard_normal(m).astype(np.float32), rng.standard_normal((n, m)).astype(np.float32)
    db = torch.from_numpy(bias).cuda()
    plain, sliced = torch.zeros((n, m), device="cuda"), torch.ones((n, m), device="cuda")
    fused = torch.from_numpy(c0).cuda()
    for t, ld, rows in ((big, ldw, m + r0 + 40), (small, k, m)):
        assert hip.pin(Segment.of(t), dt, ld, rows) == JAM.OK, hip.last_error()
    try:
        torch.cuda.synchronize()
        assert hip.mm_device(Segment.of(small), dt, k, a.data_ptr(), k, plain.data_ptr(), m, m, n, k) == JAM.OK
        assert hip.mm_device(Segment.of(view), dt, ldw, a.data_ptr(), k, sliced.data_ptr(), m, m, n, k) == JAM.OK, hip.last_error()
        assert hip.mm_device_ex(Segment.of(view), dt, ldw, a.data_ptr(), k, fused.data_ptr(), m, m, n, k, db.data_ptr(), True) == JAM.OK
        hip.synchronize()
    finally:
        hip.evict(Segment.of(big))
        hip.evict(Segment.of(small))
    assert torch.equal(plain, sliced)
    p = plain.cpu().numpy()
    rows = sampled_rows(m)
    assert close(oracle, dt, small, a.cpu().numpy(), p, rows).all()
    want = EP.add_in_place(c0, EP.add_row_bias(p, bias))
    assert np.array_equal(fused.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("m,n,k", [SPLIT, WHOLE])
@pytest.mark.parametrize("dt", TYPES)
def test_wide_non_finite(hip, oracle, plans, dt, m, n, k):
    """An infinite or NaN block scale or activation shows in its own row or token, where the oracle's result is not finite either,
    and changes no bit of any other."""
    from qxotic_amd.jam import JAM, Segment
    assert plans.wide(dt, k, m, n)[0]
    w = weights(dt, m, k, 7 + m)
    a = oracle.outliers(n + k + 2, (n, k))
    at = 208 if dt == O.Q6_K else 0   # the super-block's d
    bad_w, bad_a = w.copy(), a.copy()
    blocks = bad_w.reshape(m, k // 256, -1)
    for row, sb, d in ((5, 0, np.inf), (130, k // 256 - 1, np.nan), (m - 1, 1, -np.inf)):
        blocks[row, sb, at:at + 2] = np.array([d], np.float16).view(np.uint8)
    bad_a[3, 17], bad_a[n - 1, k - 1] = np.nan, np.inf
    out = []
    for ww, aa in ((w, a), (bad_w, bad_a)):
        c = np.zeros((n, m), np.float32)
        assert hip.pin(Segment.of(ww), dt, k, m) == JAM.OK, hip.last_error()
        try:
            st = hip.mm(Segment.of(ww), 0, dt, k, Segment.of(aa), 0, JAM.F32, k, Segment.of(c), 0, JAM.F32, m, m, n, k)
            assert st == JAM.OK, hip.last_error()
        finally:
            hip.evict(Segment.of(ww))
        out.append(c)
    rows, toks = np.setdiff1d(np.arange(m), [5, 130, m - 1]), np.setdiff1d(np.arange(n), [3, n - 1])
    clean, bad = out
    assert np.array_equal(clean[np.ix_(toks, rows)].view(np.uint32), bad[np.ix_(toks, rows)].view(np.uint32))
    sample = np.r_[0:16, 128:144, m - 16:m]
    ref = oracle.mm_int8(dt, np.ascontiguousarray(bad_w[sample]), bad_a, len(sample), n, k)
    assert np.array_equal(np.isfinite(bad[:, sample]), np.isfinite(ref))
