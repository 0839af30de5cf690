"""GPU parity: the HIP path through the C-ABI (libjamhip.so) against the pinned oracle.

Tier 1 (same int8 semantics, f32 order differs): |gpu - oracle_int8| <= 1e-3*|oracle| + 1e-5*sumAbs.
Tier 2 (jam's own bound, PRECISION.md:20-26): |gpu - float_ref| <= 1e-2*sumAbs + 1e-3, and the same
bound against libjam itself when oracle/_ref is present.
Activation quantization is checked bit for bit.
"""
import sys

import numpy as np
import pytest

from conftest import adversarial_activations, parity_report
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(104, 1024), (100, 512), (70, 256), (64, 768)]   # JamBackendParityTest.java:204-252
MMA_TYPES = O.QUANT_TYPES + (O.Q5_K, O.NVFP4, O.Q1_0)       # the types the matrix-core GEMM covers
NS = [1, 2, 3, 4, 7, 8, 13, 16, 17, 32, 33, 64, 100]


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def bits(x):
    return np.ascontiguousarray(x).view(np.uint32)


def tier1(got, ref, sa):
    return np.abs(got - ref) <= 1e-3 * np.abs(ref) + 1e-5 * sa


def run_mm(hip, dt, w, a, m, n, k, ldw=None, lda=None, ldc=None, out=None):
    from qxotic_amd.jam import JAM, Segment
    ldw = ldw or k
    lda = lda or a.shape[-1]
    ldc = ldc or m
    c = out if out is not None else np.zeros((n, ldc), np.float32)
    st = hip.mm(Segment.of(w), 0, dt, ldw, Segment.of(a), 0, JAM.F32, lda, Segment.of(c), 0, JAM.F32, ldc, m, n, k)
    assert st == JAM.OK, hip.last_error()
    return c


# ----------------------------------------------------------------------------- activation quantizers
@pytest.mark.parametrize("flavour", [1, 2])
def test_quantizer_bit_exact(hip, oracle, flavour):
    import torch
    say(f"quantizer flavour {flavour}")
    x = np.concatenate([adversarial_activations(4096), oracle.outliers(11, (64, 4096)), oracle.normal(12, (8, 4096))])
    n, k = x.shape
    a = torch.from_numpy(x).cuda()
    q = torch.empty((n, k), dtype=torch.int8, device="cuda")
    d = torch.empty((n, k // 32), dtype=torch.float32, device="cuda")
    s = torch.empty((n, k // (32 if flavour == 1 else 16)), dtype=torch.float32, device="cuda")
    assert hip.quantize_device(flavour, a.data_ptr(), k, n, k, q.data_ptr(), d.data_ptr(), s.data_ptr()) == 0
    assert hip.synchronize() == 0
    qo, do, so = (oracle.quant_f1 if flavour == 1 else oracle.quant_f2)(x)
    assert np.array_equal(q.cpu().numpy(), qo)
    assert np.array_equal(bits(d.cpu().numpy()), bits(do))
    assert np.array_equal(bits(s.cpu().numpy()), bits(so))


def test_quantizer_bit_exact_prefill_size(hip, oracle):
    """Config 4's activations at full size (512 x 14336, 1% +-20 outliers), F2."""
    import torch
    x = oracle.outliers(0x5A11C0DE ^ 4, (512, 14336))
    n, k = x.shape
    a = torch.from_numpy(x).cuda()
    q = torch.empty((n, k), dtype=torch.int8, device="cuda")
    d = torch.empty((n, k // 32), dtype=torch.float32, device="cuda")
    s = torch.empty((n, k // 16), dtype=torch.float32, device="cuda")
    assert hip.quantize_device(2, a.data_ptr(), k, n, k, q.data_ptr(), d.data_ptr(), s.data_ptr()) == 0
    hip.synchronize()
    qo, do, so = oracle.quant_f2(x)
    assert np.array_equal(q.cpu().numpy(), qo)
    assert np.array_equal(bits(d.cpu().numpy()), bits(do))
    assert np.array_equal(bits(s.cpu().numpy()), bits(so))


# ------------------------------------------------------------------------------------- matmul parity
@pytest.mark.parametrize("dt", O.QUANT_TYPES)
def test_mm_parity_shapes(hip, oracle, dt):
    for (m, k) in SHAPES:
        if k % O.BLOCK[dt][0]:
            continue
        w = oracle.quantize(dt, oracle.normal(0x5A11C0DE ^ (m * 31 + k + dt), (m, k), 0.0, 0.02))
        for n in NS:
            say(f"mm {O.NAMES[dt]} m={m} n={n} k={k}")
            # tier 1 on config 4's activation mix (1% +-20 outliers stress the per-32 scales)
            a = oracle.outliers(1000 + n, (n, k))
            got = run_mm(hip, dt, w, a, m, n, k)
            ref = oracle.mm_int8(dt, w, a, m, n, k)
            _, sa = oracle.mm_ref(dt, w, a, m, n, k)
            ok = tier1(got, ref, sa)
            assert ok.all(), (O.NAMES[dt], m, n, k, float(np.max(np.abs(got - ref) / (np.abs(ref) + 1e-30))))
            # tier 2, jam's own bound, holds for the N(0,1) activations it was written for: an outlier
            # inflates its block's int8 step 20x, which jam's CPU path shares (PRECISION.md:8-26)
            a = oracle.normal(2000 + n, (n, k))
            got = run_mm(hip, dt, w, a, m, n, k)
            fref, sa = oracle.mm_ref(dt, w, a, m, n, k)
            assert tier1(got, oracle.mm_int8(dt, w, a, m, n, k), sa).all()
            assert (np.abs(got - fref) <= 1e-2 * sa + 1e-3).all(), (O.NAMES[dt], m, n, k)


@pytest.mark.parametrize("dt", MMA_TYPES)
def test_matrix_cores_and_f2_at_few_tokens(hip, oracle, dt, monkeypatch):
    """Both n >= 8 paths at the token counts where the routing threshold (weight size and k dependent)
    hands over: JAM_HIP_MMA_MIN_N forces the matrix cores (8) or the F2 decode kernel (huge) on the same
    inputs; both meet the tier-1 bound."""
    for (m, k) in SHAPES[:2]:
        if k % O.BLOCK[dt][0]:
            continue
        w = oracle.quantize(dt, oracle.normal(0x7E57 ^ (m * 31 + k + dt), (m, k), 0.0, 0.02))
        for n in (8, 9, 13, 16, 17, 24, 32):
            a = oracle.outliers(3000 + n, (n, k))
            ref = oracle.mm_int8(dt, w, a, m, n, k)
            _, sa = oracle.mm_ref(dt, w, a, m, n, k)
            for force in ("8", "100000"):
                monkeypatch.setenv("JAM_HIP_MMA_MIN_N", force)
                say(f"few tokens {O.NAMES[dt]} m={m} n={n} k={k} mma_min_n={force}")
                got = run_mm(hip, dt, w, a, m, n, k)
                assert tier1(got, ref, sa).all(), (O.NAMES[dt], m, n, k, force)


@pytest.mark.parametrize("dt", O.QUANT_TYPES)
def test_mm_matches_golden_libjam(hip, dt):
    """Against libjam's own outputs committed as fixtures (PRECISION.md bound plus the tier-1 bound
    relative to libjam's own answer)."""
    from pathlib import Path
    g = np.load(Path(__file__).resolve().parent / "golden" / "jam_golden.npz")
    w, a = g[f"mm_{O.NAMES[dt]}_w"], g["mm_a"]
    m, k = 32, 512
    for n in (1, 3, 7, 8, 13, 16):
        say(f"golden {O.NAMES[dt]} n={n}")
        got = run_mm(hip, dt, w, a[:n].copy(), m, n, k)
        want = g[f"mm_{O.NAMES[dt]}_n{n}"]
        scale = np.abs(want).max()
        assert (np.abs(got - want) <= 1e-3 * np.abs(want) + 1e-4 * scale).all(), (O.NAMES[dt], n)


@pytest.mark.parametrize("dt", O.QUANT_TYPES)
def test_layout_metamorphic(hip, oracle, dt):
    """ldw > k (padding bytes 0xA5), lda > k, ldc > m gap untouched, rerun bit-identical
    (jam_test.c:272-353)."""
    be = O.BLOCK[dt][0]
    m, k = 48, 512
    ldw = k + 2 * max(be, 256)
    wfull = oracle.quantize(dt, oracle.normal(5, (m, ldw), 0.0, 0.02))
    rb = O.row_bytes(dt, k)
    wpad = wfull.copy()
    wpad[:, rb:] = 0xA5
    for n in (1, 5, 8, 20):
        say(f"layout {O.NAMES[dt]} n={n}")
        a = np.full((n, k + 40), 7.0, np.float32)
        a[:, :k] = oracle.normal(6 + n, (n, k))
        ldc = m + 9
        c = np.full((n, ldc), -12345.0, np.float32)
        run_mm(hip, dt, wpad, a, m, n, k, ldw=ldw, lda=k + 40, ldc=ldc, out=c)
        assert (c[:, m:] == -12345.0).all()
        ref = run_mm(hip, dt, np.ascontiguousarray(wfull[:, :rb]), np.ascontiguousarray(a[:, :k]), m, n, k)
        assert np.array_equal(bits(c[:, :m]), bits(ref[:, :m]))
        again = run_mm(hip, dt, wpad, a, m, n, k, ldw=ldw, lda=k + 40)
        assert np.array_equal(bits(again[:, :m]), bits(c[:, :m]))


@pytest.mark.parametrize("dt", O.QUANT_TYPES)
def test_pinned_matches_staged_and_slices(hip, oracle, dt):
    """Pinned (device-resident) weights give the staged answer bit for bit, also for row slices at
    non-zero offsets into one stacked tensor (the MoE expert pattern, GptOss.java:677-684)."""
    from qxotic_amd.jam import JAM, Segment
    experts, rows, k = 4, 64, 512
    w = oracle.quantize(dt, oracle.normal(17, (experts * rows, k), 0.0, 0.02))
    rb = O.row_bytes(dt, k)
    a = oracle.normal(18, (9, k))
    staged = [run_mm(hip, dt, np.ascontiguousarray(w[e * rows:(e + 1) * rows]), a[:n], rows, n, k)
              for e in range(experts) for n in (1, 9)]
    assert hip.pin(Segment.of(w), dt, k, experts * rows) == JAM.OK, hip.last_error()
    try:
        i = 0
        for e in range(experts):
            for n in (1, 9):
                say(f"pinned {O.NAMES[dt]} expert={e} n={n}")
                c = np.zeros((n, rows), np.float32)
                st = hip.mm(Segment.of(w), e * rows * rb, dt, k, Segment.of(a), 0, JAM.F32, k, Segment.of(c), 0,
                            JAM.F32, rows, rows, n, k)
                assert st == JAM.OK
                assert np.array_equal(bits(c), bits(staged[i]))
                i += 1
    finally:
        assert hip.evict(Segment.of(w)) == JAM.OK


def test_status_codes(hip, oracle):
    from qxotic_amd.jam import JAM, Segment, IllegalArgumentError, IndexOutOfBoundsError
    w = oracle.quantize(O.Q8_0, oracle.normal(1, (32, 64), 0.0, 0.02))
    a = oracle.normal(2, (2, 64))
    c = np.zeros((2, 32), np.float32)
    W, A, R = Segment.of(w), Segment.of(a), Segment.of(c)
    assert hip.mm(W, 0, JAM.Q8_0, 64, A, 0, JAM.F32, 64, R, 0, JAM.F32, 32, 32, 2, 64) == JAM.OK
    assert hip.mm(W, 0, JAM.Q8_0, 64, A, 0, JAM.F32, 64, R, 0, JAM.F32, 32, 0, 2, 64) == JAM.EINVAL
    assert hip.mm(W, 0, JAM.Q8_0, 32, A, 0, JAM.F32, 64, R, 0, JAM.F32, 32, 32, 2, 64) == JAM.EINVAL   # ldw < k
    assert hip.mm(W, 0, JAM.Q8_0, 64, A, 0, JAM.F32, 64, R, 0, JAM.F32, 16, 32, 2, 64) == JAM.EINVAL   # ldc < m
    assert hip.mm(W, 0, JAM.Q5_K, 256, A, 0, JAM.F32, 64, R, 0, JAM.F32, 32, 1, 1, 64) != JAM.OK
    assert hip.mm(W, 0, JAM.Q8_0, 64, A, 0, JAM.F16, 64, R, 0, JAM.F32, 32, 32, 1, 64) == JAM.EUNSUPPORTED
    assert hip.mm(W, 0, JAM.Q8_0, 48, A, 0, JAM.F32, 48, R, 0, JAM.F32, 32, 16, 1, 48) == JAM.EUNSUPPORTED
    with pytest.raises(IllegalArgumentError):
        hip.mm(Segment.heap([0]), 0, JAM.Q8_0, 64, A, 0, JAM.F32, 64, R, 0, JAM.F32, 32, 32, 2, 64)
    with pytest.raises(IndexOutOfBoundsError):
        hip.mm(W, 34, JAM.Q8_0, 64, A, 0, JAM.F32, 64, R, 0, JAM.F32, 32, 32, 2, 64)


# ------------------------------------------------------------------------------- BASELINE full sizes
FULL = [(O.Q4_K, 14336, 4096, 1), (O.Q6_K, 4096, 14336, 1), (O.Q8_0, 4096, 4096, 1),
        (O.Q4_0, 14336, 4096, 4), (O.Q4_0, 4096, 14336, 8), (O.MXFP4, 2880, 2880, 3)]


@pytest.mark.parametrize("dt,m,k,n", FULL)
def test_full_size_decode(hip, oracle, dt, m, k, n):
    say(f"full {O.NAMES[dt]} {m}x{k} n={n}")
    w = oracle.quantize(dt, oracle.normal(0x5A11C0DE ^ dt, (m, k), 0.0, 0.02))
    a = oracle.normal(0x5A11C0DE ^ 99, (n, k))
    got = run_mm(hip, dt, w, a, m, n, k)
    ref = oracle.mm_int8(dt, w, a, m, n, k)
    _, sa = oracle.mm_ref(dt, w, a, m, n, k)
    cfg = {(O.Q8_0, 4096, 4096): "config1 ", (O.Q4_K, 14336, 4096): "config3 ", (O.Q6_K, 4096, 14336): "config3 "}
    parity_report(f"{cfg.get((dt, m, k), '')}{O.NAMES[dt]} {m}x{k} M={n}", got, ref, sa)
    assert tier1(got, ref, sa).all()


@pytest.mark.parametrize("dt", O.QUANT_TYPES)
def test_decode_workgroup_shapes(hip, oracle, dt):
    """One-token decode workgroups sized to the row band: 3, 6 and 7 items of 8 groups per band (k = 5120,
    11008, 14336: 6, 6 and 7 waves) and small grids (4 waves), beside two tokens on the 8-wave kernel."""
    for (m, k) in [(72, 5120), (40, 11008), (24, 14336), (200, 4096)]:
        w = oracle.quantize(dt, oracle.normal(0x5A11C0DE ^ (k + dt), (m, k), 0.0, 0.02))
        for n in (1, 2):
            say(f"decode workgroups {O.NAMES[dt]} m={m} n={n} k={k}")
            a = oracle.outliers(4000 + n, (n, k))
            got = run_mm(hip, dt, w, a, m, n, k)
            ref = oracle.mm_int8(dt, w, a, m, n, k)
            _, sa = oracle.mm_ref(dt, w, a, m, n, k)
            assert tier1(got, ref, sa).all(), (O.NAMES[dt], m, n, k)


@pytest.mark.parametrize("dt", [O.Q4_0, O.Q8_0])
def test_matrix_core_block_scale_spread(hip, oracle, dt):
    """Q4_0 / Q8_0 on the matrix cores fold each block's fp16 scale into the weight operand through a per-row
    power of two: block scales 2^-20 .. 2^6 apart inside a group, a row whose blocks are all tiny, a
    zero block, and a partial last group (k = 800) must all meet the tier-1 bound row by row."""
    m, k, n = 64, 800, 40
    rng = np.random.default_rng(0x5CA1E ^ dt)
    x = oracle.normal(0x5CA1E + dt, (m, k), 0.0, 0.02)
    factor = np.exp2(rng.choice([-20.0, -8.0, 0.0, 6.0], size=(m, k // 32)))
    factor[5, :] = 2.0 ** -22        # a row of tiny blocks only
    factor[9, 3] = 0.0               # a zero block
    w = oracle.quantize(dt, (x * np.repeat(factor, 32, axis=1)).astype(np.float32))
    a = oracle.outliers(77 + dt, (n, k))
    say(f"block-scale spread {O.NAMES[dt]} m={m} n={n} k={k}")
    got = run_mm(hip, dt, w, a, m, n, k)
    ref = oracle.mm_int8(dt, w, a, m, n, k)
    _, sa = oracle.mm_ref(dt, w, a, m, n, k)
    ok = tier1(got, ref, sa)
    assert ok.all(), (O.NAMES[dt], np.argwhere(~ok)[:4].tolist())


@pytest.mark.parametrize("dt", O.QUANT_TYPES)
def test_split_k_decode(hip, oracle, dt):
    """From k = 8192 on the decode kernels split K into 4096-element slices and sum the slices' partial
    results in slice order: a partial last slice (for the 32-element types also a partial last group), F1
    quantized in the kernel (n < 8), F1 from the quantized copy (rows not 16-byte aligned), F2 tiles (n >= 8
    where the matrix cores do not take the call), ldc gap untouched, rerun bit-identical."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    be = O.BLOCK[dt][0]
    m, k = 80, (9024 if be == 32 else 9216)
    w = oracle.quantize(dt, oracle.normal(0x5A11C0DE ^ 0x5C ^ dt, (m, k), 0.0, 0.02))
    for n in (1, 4, 7, 8, 13):
        say(f"split-k {O.NAMES[dt]} m={m} n={n} k={k}")
        a = oracle.outliers(3000 + n, (n, k))
        got = run_mm(hip, dt, w, a, m, n, k, ldc=m + 3)
        assert (got[:, m:] == 0.0).all()
        ref = oracle.mm_int8(dt, w, a, m, n, k)
        _, sa = oracle.mm_ref(dt, w, a, m, n, k)
        ok = tier1(got[:, :m], ref, sa)
        assert ok.all(), (O.NAMES[dt], n, float(np.max(np.abs(got[:, :m] - ref) / (np.abs(ref) + 1e-30))))
        assert np.array_equal(bits(run_mm(hip, dt, w, a, m, n, k, ldc=m + 3)), bits(got))
    # device path with lda = k + 1: the kernel cannot load the rows as 16-byte pieces and reads the F1 copy
    assert hip.pin(Segment.of(w), dt, k, m) == JAM.OK, hip.last_error()
    try:
        n = 3
        say(f"split-k {O.NAMES[dt]} unaligned rows n={n}")
        a = oracle.normal(3100, (n, k))
        a_pad = np.zeros((n, k + 1), np.float32)
        a_pad[:, :k] = a
        a_dev = torch.from_numpy(a_pad).cuda()
        c_dev = torch.zeros((n, m), dtype=torch.float32, device="cuda")
        st = hip.mm_device(Segment.of(w), dt, k, a_dev.data_ptr(), k + 1, c_dev.data_ptr(), m, m, n, k)
        assert st == JAM.OK, hip.last_error()
        hip.synchronize()
        ref = oracle.mm_int8(dt, w, a, m, n, k)
        _, sa = oracle.mm_ref(dt, w, a, m, n, k)
        assert tier1(c_dev.cpu().numpy(), ref, sa).all()
    finally:
        assert hip.evict(Segment.of(w)) == JAM.OK


@pytest.mark.parametrize("dt", O.ALL_QUANT_TYPES)
def test_past_k_65536(hip, oracle, dt):
    """jam takes any k. One token past k = 65536 (the most one row band holds) splits K into 32768-element
    slices summed in slice order; 2..7 tokens take 4096-element slices, 8 and more the F2 path the matrix cores
    decline to (their prep holds k <= 65536). A partial last slice (for the types with blocks below 256 also a
    partial last group), F1 quantized in the kernel and, with rows that are not 16-byte aligned, read from the
    quantized copy; ldc gap untouched, rerun bit-identical."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    be = O.BLOCK[dt][0]
    m, k = 48, 65536 + 8192 + (be if be < 256 else 256)
    w = oracle.quantize(dt, oracle.normal(0x5A11C0DE ^ 0x6B ^ dt, (m, k), 0.0, 0.02))
    for n in (1, 3, 8, 17):
        a = oracle.outliers(3200 + 16 * dt + n, (n, k))
        say(f"past k 65536: {O.NAMES[dt]} m={m} n={n} k={k}")
        got = run_mm(hip, dt, w, a, m, n, k, ldc=m + 3)
        assert (got[:, m:] == 0.0).all()
        ref = oracle.mm_int8(dt, w, a, m, n, k)
        _, sa = oracle.mm_ref(dt, w, a, m, n, k)
        ok = tier1(got[:, :m], ref, sa)
        assert ok.all(), (O.NAMES[dt], n, float(np.max(np.abs(got[:, :m] - ref) / (np.abs(ref) + 1e-30))))
        assert np.array_equal(bits(run_mm(hip, dt, w, a, m, n, k, ldc=m + 3)), bits(got))
    a = oracle.outliers(3200 + 16 * dt + 1, (1, k))
    ref = oracle.mm_int8(dt, w, a, m, 1, k)
    _, sa = oracle.mm_ref(dt, w, a, m, 1, k)
    assert hip.pin(Segment.of(w), dt, k, m) == JAM.OK, hip.last_error()
    try:
        a_pad = np.zeros((1, k + 1), np.float32)
        a_pad[:, :k] = a
        a_dev = torch.from_numpy(a_pad).cuda()
        c_dev = torch.zeros((1, m), dtype=torch.float32, device="cuda")
        st = hip.mm_device(Segment.of(w), dt, k, a_dev.data_ptr(), k + 1, c_dev.data_ptr(), m, m, 1, k)
        assert st == JAM.OK, hip.last_error()
        hip.synchronize()
        assert tier1(c_dev.cpu().numpy(), ref, sa).all()
    finally:
        assert hip.evict(Segment.of(w)) == JAM.OK


@pytest.mark.parametrize("dt", O.ALL_QUANT_TYPES)
def test_decode_fused_prologue_matches_quantized_copy(hip, oracle, dt):
    """1..7 tokens: rows the kernel can load as 16-byte pieces are quantized in each workgroup's prologue (MXFP4
    and NVFP4 with one token: into f16 pairs for the hardware e2m1 conversion and v_dot2), rows that are not
    (lda = k + 1) come from the F1 copy through the int8 dot products. Both give jam's integer block sums, so the outputs are
    bit-identical: a partial last group, the k = 14336 one-band workgroups (split K from two tokens on) and a
    small 4-wave grid."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    be = O.BLOCK[dt][0]
    for (m, k) in [(200, 2880 if 2880 % be == 0 else 2816), (96, 14336), (520, 4096)]:
        w = oracle.quantize(dt, oracle.normal(0x5A11C0DE ^ 0xF1 ^ dt ^ k, (m, k), 0.0, 0.02))
        assert hip.pin(Segment.of(w), dt, k, m) == JAM.OK, hip.last_error()
        try:
            for n in (1, 3, 7):
                say(f"fused vs copy {O.NAMES[dt]} m={m} n={n} k={k}")
                a = oracle.outliers(3200 + k + n, (n, k))
                outs = []
                for lda in (k, k + 1):
                    a_pad = np.zeros((n, lda), np.float32)
                    a_pad[:, :k] = a
                    a_dev = torch.from_numpy(a_pad).cuda()
                    c_dev = torch.zeros((n, m), dtype=torch.float32, device="cuda")
                    st = hip.mm_device(Segment.of(w), dt, k, a_dev.data_ptr(), lda, c_dev.data_ptr(), m, m, n, k)
                    assert st == JAM.OK, hip.last_error()
                    hip.synchronize()
                    outs.append(c_dev.cpu().numpy())
                assert np.array_equal(bits(outs[0]), bits(outs[1])), (O.NAMES[dt], m, n, k)
                ref = oracle.mm_int8(dt, w, a, m, n, k)
                _, sa = oracle.mm_ref(dt, w, a, m, n, k)
                assert tier1(outs[0], ref, sa).all()
        finally:
            assert hip.evict(Segment.of(w)) == JAM.OK


# ------------------------------------------------------------------------------------ prefill GEMM
PREFILL = [(O.Q4_K, 14336, 4096), (O.Q6_K, 4096, 14336), (O.Q5_K, 14336, 4096), (O.NVFP4, 14336, 4096),
           (O.Q1_0, 14336, 4096)]


@pytest.mark.parametrize("dt,m,k", PREFILL)
def test_prefill_full_size(hip, oracle, dt, m, k):
    """Config 4 (M=512, 1% +-20 outliers) at full size on the MFMA GEMM. The oracle checks a seeded sample of
    192 rows against all 512 tokens; the whole output is checked for rerun bit-identity and finiteness."""
    n = 512
    say(f"prefill {O.NAMES[dt]} {m}x{k} n={n}")
    w = oracle.quantize(dt, oracle.normal(0x5A11C0DE ^ 4 ^ dt, (m, k), 0.0, 0.02))
    a = oracle.outliers(0x5A11C0DE ^ 4, (n, k))
    got = run_mm(hip, dt, w, a, m, n, k)
    again = run_mm(hip, dt, w, a, m, n, k)
    assert np.isfinite(got).all()
    assert np.array_equal(bits(got), bits(again))
    rows = np.sort(np.random.default_rng(dt).choice(m, 192, replace=False))
    ws = np.ascontiguousarray(w[rows])
    ref = oracle.mm_int8(dt, ws, a, len(rows), n, k)
    _, sa = oracle.mm_ref(dt, ws, a, len(rows), n, k)
    parity_report(f"config4 {O.NAMES[dt]} {m}x{k} M={n} (192 sampled rows)", got[:, rows], ref, sa)
    ok = tier1(got[:, rows], ref, sa)
    assert ok.all(), (int((~ok).sum()), float(np.max(np.abs(got[:, rows] - ref) / (np.abs(ref) + 1e-30))))


@pytest.mark.parametrize("dt", MMA_TYPES)
def test_prefill_ragged_shapes(hip, oracle, dt):
    """GEMM edge tiles: m not a multiple of the row tile (and of 16: float-dot tail), n not a multiple of the
    token tile, k with a partial 256-element chunk for the 32-element block types."""
    be = O.BLOCK[dt][0]
    for (m, n, k) in [(200, 37, 512), (130, 64, 1024), (47, 96, 256 if be == 256 else 288), (16, 33, 2304)]:
        if k % be:
            continue
        say(f"ragged {O.NAMES[dt]} m={m} n={n} k={k}")
        w = oracle.quantize(dt, oracle.normal(m + n + k, (m, k), 0.0, 0.02))
        a = oracle.outliers(m * n, (n, k))
        got = run_mm(hip, dt, w, a, m, n, k)
        ref = oracle.mm_int8(dt, w, a, m, n, k)
        _, sa = oracle.mm_ref(dt, w, a, m, n, k)
        assert tier1(got, ref, sa).all(), (O.NAMES[dt], m, n, k)


@pytest.mark.parametrize("dt", [O.Q4_K, O.Q5_K, O.Q6_K, O.MXFP4, O.NVFP4, O.Q8_0, O.Q4_0, O.Q1_0])
def test_prefill_tail_split_tiles(hip, oracle, plans, dt):
    """Grids whose last partial round of tiles runs as half tiles: 1024 rows x 65 slot blocks give 65 tiles per
    XCD (MXFP4, 256 rows a tile: 33), one of them split into two 32-token workgroups. Every token's result equals that
    of the n = 4096 grid (64 and 32 tiles per XCD, none split) bit for bit, and a row sample meets tier 1. n = 4150
    leaves the second half of the last slot block partly valid, n = 4110 leaves it empty."""
    m, k = 1024, 256
    for n, tail in ((4096, 0), (4110, 1), (4150, 1)):
        tiles = plans.mx4(m, k, n)[1] if dt == O.MXFP4 else m // 128 * -(-n // 64)
        assert plans.lib.q_tail(tiles, 256) == tail and not plans.wide(dt, k, m, n)[0]
    w = oracle.quantize(dt, oracle.normal(0x7A11 ^ dt, (m, k), 0.0, 0.02))
    a = oracle.outliers(0x7A12, (4150, k))
    base = run_mm(hip, dt, w, np.ascontiguousarray(a[:4096]), m, 4096, k)
    rows = np.sort(np.random.default_rng(dt + 7).choice(m, 48, replace=False))
    ws = np.ascontiguousarray(w[rows])
    for n in (4150, 4110):
        say(f"tail split {O.NAMES[dt]} m={m} n={n} k={k}")
        an = np.ascontiguousarray(a[:n])
        got = run_mm(hip, dt, w, an, m, n, k)
        assert np.array_equal(bits(got[:4096]), bits(base)), (O.NAMES[dt], n)
        ref = oracle.mm_int8(dt, ws, an, len(rows), n, k)
        _, sa = oracle.mm_ref(dt, ws, an, len(rows), n, k)
        ok = tier1(got[:, rows], ref, sa)
        assert ok.all(), (O.NAMES[dt], n, int((~ok).sum()))


@pytest.mark.parametrize("dt", MMA_TYPES)
def test_prefill_error_floor(hip, oracle, dt):
    """The GEMM stays at its arithmetic's error floor, far inside tier 1: max |gpu - oracle| / sum|w*a| <= 2e-6
    over 160 tokens of N(0,1) activations with a per-token offset in [-1, 1] (an offset token's super-block
    sums cancel against the min term, the case that exposes a wrong activation element). One activation
    element off by one f16 ulp of its hi + lo split moves an output by about 1e-5 of sum|w*a|."""
    m, n, k = 96, 160, 2048
    say(f"error floor {O.NAMES[dt]} m={m} n={n} k={k}")
    w = oracle.quantize(dt, oracle.normal(0xF100 ^ dt, (m, k), 0.0, 0.02))
    a = oracle.normal(0xF101, (n, k)) + np.linspace(-1.0, 1.0, n, dtype=np.float32)[:, None]
    a = np.ascontiguousarray(a, dtype=np.float32)
    got = run_mm(hip, dt, w, a, m, n, k)
    ref = oracle.mm_int8(dt, w, a, m, n, k)
    _, sa = oracle.mm_ref(dt, w, a, m, n, k)
    rel = np.abs(got - ref) / sa
    worst = np.unravel_index(int(np.argmax(rel)), rel.shape)
    assert rel.max() <= 2e-6, (O.NAMES[dt], float(rel.max()), worst)


@pytest.mark.parametrize("dt", O.ALL_QUANT_TYPES)
def test_pinned_column_slice(hip, oracle, dt, monkeypatch):
    """A pinned tensor read with ldw > k (the first k elements of each ldw-element row, jam.c:551): the device
    copy holds whole rows, the kernels read its first k / 256 groups. Decode (F1, in-kernel and from the
    quantized copy), the F2 decode kernel, the matrix cores and the grouped matmul give the staged call's bits
    (staging copies only the k columns), and tier 1 against the oracle."""
    import torch
    from qxotic_amd.jam import JAM, Segment
    be = O.BLOCK[dt][0]
    m, k = 64, 768 if be < 256 else 512
    ldw = k + 256
    w = oracle.quantize(dt, oracle.normal(0x51CE ^ dt, (m, ldw), 0.0, 0.02))
    assert hip.pin(Segment.of(w), dt, ldw, m) == JAM.OK, hip.last_error()
    try:
        for n, force in ((1, None), (3, None), (12, "100000"), (40, "8")):
            monkeypatch.delenv("JAM_HIP_MMA_MIN_N", raising=False)
            if force:
                monkeypatch.setenv("JAM_HIP_MMA_MIN_N", force)
            say(f"pinned column slice {O.NAMES[dt]} m={m} k={k} ldw={ldw} n={n}")
            a = oracle.outliers(0x51CF + n, (n, k))
            got = run_mm(hip, dt, w, a, m, n, k, ldw=ldw)
            ref = oracle.mm_int8(dt, w, a, m, n, k, ldw=ldw)
            _, sa = oracle.mm_ref(dt, w, a, m, n, k, ldw=ldw)
            assert tier1(got, ref, sa).all(), (O.NAMES[dt], n)
            staged = run_mm(hip, dt, np.ascontiguousarray(w[:, :O.row_bytes(dt, k)]), a, m, n, k)
            assert np.array_equal(bits(got), bits(staged)), (O.NAMES[dt], n)
        monkeypatch.delenv("JAM_HIP_MMA_MIN_N", raising=False)
        if dt in O.QUANT_TYPES:   # grouped: two experts of 32 rows of the pinned tensor, ldw > k
            counts = [20, 2]
            a = oracle.outliers(0x51D0, (22, k))
            a_d = torch.from_numpy(a).cuda()
            c = torch.zeros((22, 32), dtype=torch.float32, device="cuda")
            cnt = torch.from_numpy(np.array(counts, np.int32)).cuda()
            say(f"pinned column slice grouped {O.NAMES[dt]}")
            assert hip.mm_grouped(Segment.of(w), dt, ldw, 32, 2, cnt.data_ptr(), a_d.data_ptr(), k, c.data_ptr(), 32,
                                  k, 22, None) == JAM.OK, hip.last_error()
            hip.synchronize()
            got = c.cpu().numpy()
            for e, (o, nr) in enumerate(((0, 20), (20, 2))):
                we = np.ascontiguousarray(w[32 * e:32 * e + 32])
                ae = np.ascontiguousarray(a[o:o + nr])
                ref = oracle.mm_int8(dt, we, ae, 32, nr, k, ldw=ldw)
                _, sa = oracle.mm_ref(dt, we, ae, 32, nr, k, ldw=ldw)
                assert tier1(got[o:o + nr], ref, sa).all(), (O.NAMES[dt], e)
    finally:
        assert hip.evict(Segment.of(w)) == JAM.OK
