"""MXFP4 on the scaled matrix cores (n >= 8, jam's int8 activations): extreme codes, exponents from 0 to past the kernel's
limit, edges of its tiles (32 and 64 rows per wave, 64 tokens), stages (128 of k) and K split, against the operation in 64
bits.

Bound: block sums are exact, so an output of B blocks carries at most one rounding per block, one per group of 8 blocks and
one per K slice (16 at the most here), each of at most 2^-24·sum|w*q| over the block terms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def blocks(rng, m, k, lo, hi, extreme):
    b = rng.integers(0, 256, (m, k // 32, 17), dtype=np.uint8)
    if extreme:   # largest codes, mixed signs
        b[:, :, 1:] = rng.choice(np.array([0x77, 0x7F, 0xF7, 0xFF], np.uint8), (m, k // 32, 16))
    e0 = rng.integers(lo, hi + 1, (m, 1))   # a row's blocks within the 14 binades the kernel is given
    b[:, :, 0] = np.clip(e0 + rng.integers(0, 7, (m, k // 32)), lo, hi)
    return np.ascontiguousarray(b.reshape(m, -1))


# 64-row waves over whole 64-token tiles, no half tile in the last round, several stages: the last one full and short
FULL = [(1024, 4096, 288), (1024, 4090, 416)]
# m in whole bands of 16: the last m % 16 rows of a call are a float dot on another kernel
SHAPES = [(16, 9, 32), (32, 64, 96), (48, 65, 128), (96, 33, 160), (128, 40, 256), (160, 130, 288), (528, 77, 416), (544, 1920, 288),
          (2880, 545, 96), (512, 31, 4096), (144, 8, 2880), *FULL]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("lo,hi,extreme", [(110, 126, False), (110, 126, True), (0, 14, False), (225, 238, False), (232, 254, False)])
def test_mx4_exact_blocks(hip, oracle, plans, monkeypatch, m, n, k, lo, hi, extreme):
    from qxotic_amd.jam import JAM, Segment
    rt, tiles, _, _ = plans.mx4(m, k, n)
    assert (m, n, k) not in FULL or (rt, plans.lib.q_tail(tiles, 256)) == (2, 0)
    monkeypatch.setenv("JAM_HIP_MMA_MIN_N", "8")
    rng = np.random.default_rng(m + 31 * n + 977 * k + lo)
    w = blocks(rng, m, k, lo, hi, extreme)
    a = oracle.normal(m + n, (n, k)) * np.float32(2.0 ** -100 if lo > 200 else 1.0)
    if extreme:
        a = np.where(rng.random((n, k)) < 0.5, np.float32(3.0), np.float32(-3.0)) * np.where(rng.random((n, k)) < 0.9, 1, 0).astype(np.float32)
    a = np.ascontiguousarray(a, dtype=np.float32)
    c = np.full((n, m + 5), -7.0, np.float32)
    st = hip.mm(Segment.of(w), 0, JAM.MXFP4, k, Segment.of(a), 0, JAM.F32, k, Segment.of(c), 0, JAM.F32, m + 5, m, n, k)
    assert st == JAM.OK, hip.last_error()
    # the operation in 64 bits: F2 codes and scales (their own f32 arithmetic, jam_kernels_q4k_avx512.c:25-37), exact sums
    x = a.reshape(n, k // 32, 32)
    top = np.abs(x).max(-1)
    with np.errstate(divide="ignore"):
        inv = np.where(top > 0, np.float32(127) / top, np.float32(0))
    q = (np.rint(x * inv[..., None]).clip(-128, 127) * (top / np.float32(127)).astype(np.float64)[..., None]).reshape(n, k)
    wb = w.reshape(m, -1, 17)
    code = np.concatenate([wb[:, :, 1:] & 15, wb[:, :, 1:] >> 4], -1)
    mags = np.array([0, 1, 2, 3, 4, 6, 8, 12.0])
    kv = (np.concatenate([mags, -mags])[code] * np.exp2(wb[:, :, :1].astype(np.float64) - 128)).reshape(m, k)
    ref, mag, nb = q @ kv.T, np.abs(q) @ np.abs(kv).T, k / 32
    # results below f32's normal range round in steps of 2^-149
    bound = 2.0 ** -24 * (9 / 8 * nb + 16) * mag + (9 / 8 * nb + 16) * 2.0 ** -150
    err = np.abs(c[:, :m].astype(np.float64) - ref)
    assert (err <= bound).all(), (m, n, k, float((err / bound).max()))
    assert (c[:, m:] == -7.0).all()


def test_mx4_noalloc_takes_no_unused_scratch(hip, oracle):
    """5760 tokens on waves of 64 rows, whose k is never split: 50 MB of activations, inside the static 64 MiB without the 24 MB
    of partial sums that two K slices would add."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    m, n, k = 512, 5760, 4096
    w = blocks(np.random.default_rng(5), m, k, 110, 126, False)
    a = torch.from_numpy(oracle.normal(6, (n, k))).cuda()
    c, ref = torch.zeros((n, m), device="cuda"), torch.ones((n, m), device="cuda")
    assert hip.pin(Segment.of(w), JAM.MXFP4, k, m) == JAM.OK, hip.last_error()
    try:
        torch.cuda.synchronize()
        assert hip.mm_device(Segment.of(w), JAM.MXFP4, k, a.data_ptr(), k, ref.data_ptr(), m, m, n, k) == JAM.OK
        st = hip.mm_device_noalloc(Segment.of(w), JAM.MXFP4, k, a.data_ptr(), k, c.data_ptr(), m, m, n, k)
        assert st == JAM.OK, hip.last_error()
        hip.synchronize()
        assert torch.equal(c, ref)
    finally:
        hip.evict(Segment.of(w))
