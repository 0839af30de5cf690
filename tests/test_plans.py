"""The rules that choose a kernel and its K slices (csrc/plan.h), on the CPU: at sizes where both kernels were measured the
rule takes the faster one, over the whole range it stays within what the kernels and the scratch can hold."""
import pytest

from oracle import oracle as O

# (type, m, k, n, the wide kernel is the faster one), measured with prep and reduce; every pair differs by 4% or more
WIDE = [(O.Q4_K, 14336, 4096, 512, True), (O.Q4_K, 14336, 4096, 2048, True), (O.Q4_K, 14336, 4096, 128, True),
        (O.Q4_K, 14336, 4096, 260, False), (O.Q4_K, 14336, 4096, 576, False), (O.Q4_K, 28672, 4096, 128, False),
        (O.Q4_K, 28672, 4096, 260, False), (O.Q4_K, 16384, 1024, 65, False), (O.Q4_K, 128256, 1024, 160, False),
        (O.Q4_K, 128256, 1024, 96, True), (O.Q4_K, 4096, 14336, 1024, False), (O.Q4_K, 4096, 14336, 384, True),
        (O.Q5_K, 14336, 4096, 260, False), (O.Q5_K, 14336, 4096, 576, False), (O.Q5_K, 8192, 4096, 576, False),
        (O.Q5_K, 14336, 4096, 512, True), (O.Q6_K, 4096, 14336, 512, True), (O.Q6_K, 14336, 4096, 129, False),
        (O.Q6_K, 12288, 4096, 260, False), (O.Q6_K, 12288, 4096, 160, False), (O.Q6_K, 8192, 4096, 384, False),
        (O.Q6_K, 4096, 4096, 160, False), (O.Q6_K, 16384, 1024, 160, False), (O.Q6_K, 4096, 14336, 129, False),
        (O.Q6_K, 14336, 4096, 512, True)]


@pytest.mark.parametrize("dt,m,k,n,wide", WIDE)
def test_wide_where_it_is_faster(plans, dt, m, k, n, wide):
    assert plans.wide(dt, k, m, n)[0] == wide


@pytest.mark.parametrize("dt", [O.Q4_K, O.Q5_K, O.Q6_K])
def test_wide_slices(plans, dt):
    """Whole super-blocks that cover k, none of the slices empty, and no more scratch than the 64 MiB of an allocation-free
    call unless the other kernel's slices take it too."""
    for m in (1, 128, 129, 1000, 4096, 14336, 128256):
        for nsb in (1, 2, 5, 16, 56):
            for n in (65, 128, 129, 200, 512, 4150):
                wide, ns, per = plans.wide(dt, 256 * nsb, m, n)
                if not wide:
                    continue
                assert (ns, per) == (1, 0) or (per * (ns - 1) < nsb <= per * ns)
                other = plans.split((m + 127) // 128 * ((n + 63) // 64), nsb)[0]
                assert ns <= max(1, other) or ns * n * m * 4 <= 60 << 20
    assert not any(plans.wide(dt, 4096, 14336, n)[0] for n in (1, 9, 64))
    assert not plans.wide(O.Q8_0, 4096, 14336, 512)[0]


def test_wide_offsets_fit_32_bits(plans):
    """The wide kernel reads token slot t of block b (up to 10: the next super-block's first stage) at the 32-bit offset
    b * 64 * slots + 16 * t from its super-block: longer calls stay with the other kernel."""
    most = max(n for n in (1 << 16, 1 << 20, (1 << 22) - 64, 1 << 22, (1 << 22) + 1, 5 << 20, 1 << 23, 1 << 24)
               if plans.wide(O.Q6_K, 256, 512, n)[0])
    assert 11 * 64 * ((most + 63) // 64 * 64) < 1 << 32


def test_mx4_plan(plans):
    """64-row waves never split k; 32-row waves split it like the other types, whole super-blocks that cover it."""
    for m in (16, 511, 512, 2880, 14336):
        for k in (32, 4096, 4128, 14336):
            for n in (9, 64, 128, 512, 5120):
                rt, tiles, ns, per = plans.mx4(m, k, n)
                assert tiles == -(-m // (128 * rt)) * -(-n // 64)
                nsb = -(-k // 256)
                if rt == 2:
                    assert (ns, per) == (1, 0)
                else:
                    assert [ns, per] == plans.split(tiles, nsb) and ((ns, per) == (1, 0) or per * (ns - 1) < nsb <= per * ns)
    assert plans.mx4(14336, 4096, 512)[0] == 2 and plans.mx4(14336, 4096, 64)[0] == 1 and plans.mx4(4096, 14336, 512)[0] == 1


# (type, m, k, n, the 256 x 128 tiles are faster), both measured over the same prep and K slices; 4% or more apart
BIG = [(O.F16, 14336, 4096, 512, True), (O.F16, 14336, 4096, 65, True), (O.F16, 6144, 4096, 80, True), (O.F16, 4096, 14336, 129, True),
       (O.F16, 8192, 4096, 1024, True), (O.F16, 257, 4096, 128, False), (O.F16, 256, 4096, 512, False), (O.F16, 1000, 1024, 256, False),
       (O.F16, 4096, 128, 512, False), (O.F16, 32, 2880, 512, False), (O.F16, 128, 4096, 256, False), (O.F16, 512, 8192, 128, False),
       (O.BF16, 14336, 4096, 512, True), (O.BF16, 14336, 4096, 128, True), (O.BF16, 2048, 14336, 192, True),
       (O.BF16, 256, 4096, 512, False), (O.BF16, 257, 4096, 96, False), (O.BF16, 32, 2880, 512, False), (O.BF16, 512, 8192, 384, False),
       (O.BF16, 18910, 192, 881, False), (O.F16, 50000, 768, 512, True)]


@pytest.mark.parametrize("dt,m,k,n,big", BIG)
def test_big_dense_tiles_where_they_are_faster(plans, dt, m, k, n, big):
    assert bool(plans.lib.q_big(dt, m, k, n)) == big


def test_big_dense_tiles_never_for_few_tokens(plans):
    assert not any(plans.lib.q_big(dt, m, k, n) for dt in (O.F16, O.BF16) for m in (32, 4096, 200000) for k in (64, 14336)
                   for n in (2, 9, 64))


def test_dense_prep_grid(plans):
    """Every group of 8 tokens and every run of 8 elements has a workgroup, and the workgroups of a group (x, x + gridDim.x, ... in
    launch order, dealt to the 8 XCDs in turn) meet on one XCD once there are groups for all."""
    for n in (2, 9, 64, 65, 72, 136, 197, 300, 469, 512, 1000, 4150):
        for kp in (64, 512, 2048, 2880, 14336):
            x, y = plans.prep_grid(n, kp)
            groups = -(-n // 8)
            assert groups <= x < groups + 8 and 1 <= y <= max(1, -(-kp // 512))
            assert groups <= 8 or len({(x * i) % 8 for i in range(y)}) == 1


@pytest.mark.parametrize("dt,k,n,few", [(O.F16, 4096, 9, False), (O.F16, 4096, 64, False), (O.F16, 14336, 9, False), (O.F16, 1024, 9, True),
                                        (O.F16, 1024, 128, True), (O.F16, 512, 192, True), (O.F16, 2000, 64, True), (O.F16, 2048, 256, False),
                                        (O.F16, 1024, 1024, False), (O.BF16, 1024, 128, True), (O.BF16, 4096, 64, False),
                                        (O.BF16, 14336, 9, False), (O.BF16, 2048, 1024, False)])
def test_dense_prep_form_that_is_faster(plans, dt, k, n, few):
    assert bool(plans.lib.q_few(dt, k, n)) == few


@pytest.mark.parametrize("m,n,big", [(14336, 5, False), (14336, 16, False), (32000, 9, False), (14336, 17, True), (512, 512, True),
                                     (2048, 96, True), (2048, 64, False), (256, 512, False), (32, 512, False)])
def test_f32_tile_that_is_faster(plans, m, n, big):
    assert bool(plans.lib.q_tile32(m, n)) == big


def test_dense_pitch(plans):
    """A row fits and starts on 256 bytes; rows of 4096 bytes and more lie an odd number of 256 bytes apart, at most 1/16 further
    than before that rule; shorter rows take no more memory than their 256-byte pieces."""
    for b in [1, 2, 255, 256, 257, 512, 1024, 2048, 3841, 4095, 4096, 4097, 5760, 8192, 11520, 16384, 28672, 57344, 1 << 33]:
        p, even = plans.lib.q_pitch(b), -(-b // 256) * 256
        assert p >= b and p % 256 == 0
        if even < 4096:
            assert p == even
        else:
            assert p // 256 % 2 == 1 and p - even <= min(256, even // 16)
