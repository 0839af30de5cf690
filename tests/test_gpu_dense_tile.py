"""Short dense matrices (a router's few rows): the one-tile-per-workgroup GEMM whose waves split k (n > 8; F32, and
BF16 where its activations are not rounded) and the GEMV that gives each row a workgroup (n <= 8), at the edges
of their tiles (16 and 32 rows or tokens), runs (32 and 64 elements of k, 8 waves) and dispatch.

Bound: any summation order of k exact products in f32 errs by at most (k - 1)·2^-24·sum|w*a| to first order; the
bias and the residual round once each."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 9, 1), (8, 512, 544), (15, 16, 63), (16, 17, 64), (17, 31, 65), (32, 512, 2880), (33, 33, 511), (64, 300, 1000),
          (600, 40, 96), (256, 1, 2880), (257, 2, 100), (3, 4, 1024), (32, 8, 31), (31, 5, 2881), (2048, 64, 33),
          (6200, 16, 70), (6200, 17, 70), (4100, 5, 4099)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dt", [O.F32, O.BF16])
def test_short_dense(hip, dt, m, n, k):
    import torch
    from qxotic_amd.jam import JAM, Segment
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    w32 = rng.standard_normal((m, k)).astype(np.float32)
    a = rng.standard_normal((n, k)).astype(np.float32)
    bias, c0 = rng.standard_normal(m).astype(np.float32), rng.standard_normal((n, m)).astype(np.float32)
    if dt == O.BF16:
        wt = torch.from_numpy(w32).bfloat16()
        w, w64 = wt.view(torch.uint8).numpy(), wt.double().numpy()
        rounds = (n >= 8 and k % 2 == 0) or k % 32 == 0   # jam.c:622-652
        x64 = (torch.from_numpy(a).bfloat16().double().numpy()) if rounds else a.astype(np.float64)
    elif dt == O.F16:
        wt = w32.astype(np.float16)
        w, w64, x64 = wt, wt.astype(np.float64), a.astype(np.float64)
    else:
        w, w64, x64 = w32, w32.astype(np.float64), a.astype(np.float64)
    ref, bound = x64 @ w64.T, (k + 2) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64).T)
    assert hip.pin(Segment.of(w), dt, k, m) == JAM.OK, hip.last_error()
    try:
        for lda in (k, k + 5):   # aligned rows and rows that no 16-byte load may take
            xa = np.full((n, lda), np.nan, np.float32)
            xa[:, :k] = a
            dev = lambda v: torch.from_numpy(v).to("cuda")   # noqa: E731
            da, db, dc, de = dev(xa), dev(bias), dev(np.full((n, m + 3), -7.0, np.float32)), dev(c0.copy())
            torch.cuda.synchronize()
            assert hip.mm_device(Segment.of(w), dt, k, da.data_ptr(), lda, dc.data_ptr(), m + 3, m, n, k) == JAM.OK
            assert hip.mm_device_ex(Segment.of(w), dt, k, da.data_ptr(), lda, de.data_ptr(), m, m, n, k, db.data_ptr(),
                                    True) == JAM.OK
            hip.synchronize()
            got, fused = dc.cpu().numpy(), de.cpu().numpy()
            assert (np.abs(got[:, :m] - ref) <= bound).all(), (dt, m, n, k, lda)
            assert (got[:, m:] == -7.0).all()
            whole = c0 + ref + bias
            assert (np.abs(fused - whole) <= bound + 2.0 ** -23 * (np.abs(ref) + np.abs(bias) + np.abs(c0))).all()
    finally:
        hip.evict(Segment.of(w))


# a workgroup per row whose activations fill the 64 KB of LDS, and one row beside that
@pytest.mark.parametrize("m,n,k", [(128, 8, 2048), (256, 4, 4096), (1, 5, 2048), (255, 3, 4001)])
@pytest.mark.parametrize("dt", [O.F32, O.F16, O.BF16])
def test_row_split_full_lds(hip, dt, m, n, k):
    test_short_dense(hip, dt, m, n, k)


# staged GEMM, 64 of k per stage; whole, split and masked last stages, ragged edges: 128 x 64 tiles, then 256 x 128 ones (dense_big
# in csrc/plan.h), the first two rows of each of these with whole k, the others with slices, the last of them shorter
TILES = [(4096, 1024, 64), (3870, 1000, 100), (257, 129, 8200), (8192, 513, 36), (2048, 65, 4100), (4224, 512, 330),
         # the activation prep's two forms at their limits, its grid padded and not
         (64, 256, 2040), (64, 257, 2040), (64, 320, 1024), (64, 321, 1024), (33, 72, 3000), (64, 469, 2050), (16, 9, 2048)]
BIG = {O.F16: [(8192, 1000, 100), (6144, 700, 330), (8400, 65, 778), (6144, 129, 778), (8192, 1000, 64)],
       O.BF16: [(4224, 1000, 520), (6144, 700, 520), (5000, 65, 3000), (12000, 129, 778)]}


@pytest.mark.parametrize("dt,m,n,k,big", [(dt, *s, False) for dt in BIG for s in TILES] + [(dt, *s, True) for dt in BIG for s in BIG[dt]])
def test_dense_wide_tiles(hip, plans, dt, m, n, k, big):
    """Rows 24.. and the first k columns of a pinned tensor with NaN past them, bias and residual. F16 products are exact in f32, x
    kept to 22 bits; any order of k sums errs by at most (k + 2)·2^-24·sum|w*a| and the dropped remainder of x by 2^-22 of it.
    BF16 activations are rounded first, products exact. The bias and the residual round once each."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    assert bool(plans.lib.q_big(dt, m, k, n)) == big
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = (torch.randn((m + 40, k + 24), generator=g, device="cuda") * 0.02).to(torch.float16 if dt == O.F16 else torch.bfloat16)
    w[:, k:] = float("nan")   # the pinned rows go on past k
    w[:24], w[24 + m:] = float("nan"), float("nan")
    host = w.view(torch.uint8).cpu().numpy()
    a = torch.randn((n, k), generator=g, device="cuda")
    bias, c0 = torch.randn(m, generator=g, device="cuda"), torch.randn((n, m), generator=g, device="cuda")
    c, fused = torch.full((n, m + 1), -7.0, device="cuda"), c0.clone()
    torch.cuda.synchronize()
    assert hip.pin(Segment.of(host), dt, k + 24, m + 40) == JAM.OK, hip.last_error()
    try:
        view = Segment.of(host[24:])
        assert hip.mm_device(view, dt, k + 24, a.data_ptr(), k, c.data_ptr(), m + 1, m, n, k) == JAM.OK, hip.last_error()
        assert hip.mm_device_ex(view, dt, k + 24, a.data_ptr(), k, fused.data_ptr(), m, m, n, k, bias.data_ptr(), True) == JAM.OK
        hip.synchronize()
    finally:
        hip.evict(Segment.of(host))
    x = a.double() if dt == O.F16 else a.bfloat16().double()
    w64 = w[24:24 + m, :k].double()
    bound, ref = ((k + 2) * 2.0 ** -24 + 2.0 ** -22) * (x.abs() @ w64.abs().T), x @ w64.T
    assert ((c[:, :m].double() - ref).abs() <= bound).all()
    assert (c[:, m:] == -7.0).all()
    slack = 2.0 ** -23 * (ref.abs() + bias.abs() + c0.abs())
    assert ((fused.double() - (ref + bias.double() + c0.double())).abs() <= bound + slack).all()


@pytest.mark.parametrize("dt,m,n,k", [(O.F16, 8400, 65, 778), (O.F16, 8192, 1000, 100), (O.BF16, 5000, 65, 3000), (O.BF16, 4224, 1000, 520)])
def test_big_tiles_non_finite(hip, plans, dt, m, n, k):
    """Infinities and NaN stay in their own row or token and change no bit of any other."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    assert plans.lib.q_big(dt, m, k, n)
    g = torch.Generator(device="cuda").manual_seed(m + n)
    w = (torch.randn((m, k), generator=g, device="cuda") * 0.02 + 0.001).to(torch.float16 if dt == O.F16 else torch.bfloat16)
    a = torch.randn((n, k), generator=g, device="cuda")
    bad_w, bad_a = w.clone(), a.clone()
    bad_w[7, 3], bad_w[m - 1, k - 1], bad_a[2, 5], bad_a[n - 1, k - 1] = float("nan"), float("inf"), float("inf"), float("nan")
    out = []
    for ww, aa in ((w, a), (bad_w, bad_a)):
        host, c = ww.view(torch.uint8).cpu().numpy(), torch.zeros((n, m), device="cuda")
        torch.cuda.synchronize()
        assert hip.pin(Segment.of(host), dt, k, m) == JAM.OK, hip.last_error()
        try:
            assert hip.mm_device(Segment.of(host), dt, k, aa.data_ptr(), k, c.data_ptr(), m, m, n, k) == JAM.OK
            hip.synchronize()
        finally:
            hip.evict(Segment.of(host))
        out.append(c)
    clean, bad = out
    hit = torch.zeros((n, m), dtype=torch.bool, device="cuda")
    hit[[2, n - 1]], hit[:, [7, m - 1]] = True, True
    assert not torch.isfinite(bad[hit]).any()
    assert torch.equal(clean[~hit], bad[~hit])
