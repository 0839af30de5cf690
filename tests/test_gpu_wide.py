"""The K-quants' wide matrix-core kernel (more than 64 tokens, enough 128 x 128 tiles): ragged rows and tokens, a last token
block of at most 64, whole and split k, against the int8 oracle on sampled rows (tier 1: the same integer products,
another f32 summation order)."""
import numpy as np
import pytest

from conftest import random_blocks
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(12288, 65, 256), (12304, 128, 512), (5232, 1030, 256), (14336, 320, 512), (8208, 513, 1024),
                                   (4096, 257, 2816), (1040, 1000, 768)])
@pytest.mark.parametrize("dt", [O.Q4_K, O.Q5_K, O.Q6_K])
def test_wide_tiles(hip, oracle, dt, m, n, k):
    from qxotic_amd.jam import JAM, Segment
    if dt == O.Q5_K:
        w = np.random.default_rng(7).integers(0, 256, (m, k // 256, 176), dtype=np.uint8)
        for at, lo, hi in ((0, 2e-5, 8e-5), (2, 1e-4, 5e-4)):
            w[:, :, at:at + 2] = np.random.default_rng(at).uniform(lo, hi, (m, k // 256)).astype(np.float16).view(np.uint8).reshape(m, -1, 2)
        w = np.ascontiguousarray(w.reshape(m, -1))
    else:
        w = random_blocks(dt, m, k, m + n)
    a = oracle.outliers(n + k, (n, k))
    c = np.full((n, m + 3), -3.0, np.float32)
    assert hip.pin(Segment.of(w), dt, k, m) == JAM.OK, hip.last_error()
    try:
        st = hip.mm(Segment.of(w), 0, dt, k, Segment.of(a), 0, JAM.F32, k, Segment.of(c), 0, JAM.F32, m + 3, m, n, k)
        assert st == JAM.OK, hip.last_error()
    finally:
        hip.evict(Segment.of(w))
    assert (c[:, m:] == -3.0).all() and np.isfinite(c).all()
    rows = np.unique(np.r_[0:32, 96:160, m - m % 128 - 16:m])[:208]   # whole 16-row bands; the first, a middle and the last tiles
    rows = rows[:len(rows) // 16 * 16]
    ws = np.ascontiguousarray(w[rows])
    ref = oracle.mm_int8(dt, ws, a, len(rows), n, k)
    _, sa = oracle.mm_ref(dt, ws, a, len(rows), n, k)
    ok = np.abs(c[:, rows] - ref) <= 1e-3 * np.abs(ref) + 1e-5 * sa
    assert ok.all(), (O.NAMES[dt], m, n, k, int((~ok).sum()))
