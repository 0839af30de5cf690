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


# n past 64 with enough tiles: 256 x 128 workgroups, 64 of k per stage; whole, split and masked last stages, ragged edges
@pytest.mark.parametrize("m,n,k", [(4096, 1024, 64), (3870, 1000, 100), (257, 129, 8200), (8192, 513, 36), (2048, 65, 4100), (4224, 512, 330)])
@pytest.mark.parametrize("dt", [O.F16, O.BF16])
def test_dense_wide_tiles(hip, dt, m, n, k):
    """F16 products are exact in f32, x kept to 22 bits; any order of k sums errs by at most (k + 2)·2^-24·sum|w*a| and the
    dropped remainder of x by 2^-22 of it. BF16 activations are rounded first, products exact."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    w = (torch.randn((m, k + 24), generator=g, device="cuda") * 0.02).to(torch.float16 if dt == O.F16 else torch.bfloat16)
    w[:, k:] = float("nan")   # the pinned rows go on past k
    host = w.view(torch.uint8).cpu().numpy()
    a = torch.randn((n, k), generator=g, device="cuda")
    c = torch.full((n, m + 1), -7.0, device="cuda")
    torch.cuda.synchronize()
    assert hip.pin(Segment.of(host), dt, k + 24, m) == JAM.OK, hip.last_error()
    try:
        assert hip.mm_device(Segment.of(host), dt, k + 24, a.data_ptr(), k, c.data_ptr(), m + 1, m, n, k) == JAM.OK
        hip.synchronize()
        x = a.double() if dt == O.F16 else a.bfloat16().double()
        w64 = w[:, :k].double()
        bound = ((k + 2) * 2.0 ** -24 + 2.0 ** -22) * (x.abs() @ w64.abs().T)
        assert ((c[:, :m].double() - x @ w64.T).abs() <= bound).all()
        assert (c[:, m:] == -7.0).all()
    finally:
        hip.evict(Segment.of(host))
