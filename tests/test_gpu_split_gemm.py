"""fp32 products on the three-way bf16 split (gemm_split_kernel) against
float64: the slab counts its pipeline treats apart (one to four slabs of 16 k,
the k tail, the sign changes every 16 slabs), partial tiles of each
configuration, values that overflow or are not finite, and the mean of its
error over a long contraction."""

import pytest
import torch

from torchsplinekan_amd import _C, _lib

pytestmark = pytest.mark.gpu


def _operands(M, N, K, ta, tb, seed=0):
    g = torch.Generator().manual_seed(seed)
    A = torch.randn(*((K, M) if ta else (M, K)), generator=g)
    B = torch.randn(*((N, K) if tb else (K, N)), generator=g)
    return (A.t() if ta else A), (B.t() if tb else B)


def _check(A, B, adds=None):
    got = _C.matmul(A.cuda(), B.cuda()).cpu().double()
    want = A.double() @ B.double()
    adds = A.shape[1] / 16 if adds is None else adds
    # one rounding per add (a slab's, K / 16 of them), at most 16 in a slab's
    # chain (six MFMAs, each two truncating steps, and the dropped products), of
    # 2^-24 of the sum of magnitudes
    bound = (adds + 16) * 2.0 ** -24 * (A.double().abs() @ B.double().abs())
    assert bool(((got - want).abs() <= bound).all())
    # Normwise: adds to a sum that grows with their square root, each off by at
    # most 2^-24 / sqrt(3) rms of it, make sqrt(adds / 2) of that (1.4e-7 at
    # K = 530); a slab's last MFMA truncates its own sum (2^-23 / sqrt(3) of it,
    # whatever K) and the earlier ones at most half as much more.  An operand
    # without its lo part costs 2e-6, a missing mid times mid product 6e-7.
    rel = 2.0 ** -24 / 3 ** 0.5 * ((adds / 2) ** 0.5 + 2 * 1.5)
    assert float((got - want).norm() / want.norm()) <= rel


@pytest.mark.parametrize("tile", ["256", "128", "256x64"])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False), (False, False), (True, True)])
def test_every_part_product_decides(tile, ta, tb):
    """Sums in which all but one of the six part products cancel: 2^-20 from
    lo times hi, hi times lo or mid times mid, 2^-10 from mid times hi or hi
    times mid, 1 from hi times hi.  A row holds one such sum, in one 8-k half of
    one of 18 slabs (either side of the change of sign), and is zero elsewhere;
    every value is exact."""
    e10, e20 = 2.0 ** -10, 2.0 ** -20
    sums = [([1 + e10 + e20, -(1 + e10)], [1, 1]), ([1, -1], [1 + e10 + e20, 1 + e10]),
            ([1 + e10, -1, -1], [1 + e10, 1, 2 * e10]), ([1 + e10, -1], [1, 1]),
            ([1, -1], [1 + e10, 1]), ([1], [1])]
    slabs, N = 18, 64
    for a, b in sums:
        A, B = torch.zeros(2 * slabs, 16 * slabs), torch.zeros(16 * slabs, N)
        want = sum(u * v for u, v in zip(a, b))
        for r in range(2 * slabs):
            for i, (u, v) in enumerate(zip(a, b)):
                k = 8 * r + (3 * r + i) % 8
                A[r, k], B[k] = u, v
        A = A.t().contiguous().t() if ta else A
        B = B.t().contiguous().t() if tb else B
        with _lib.route("gemm_tile", _lib.GEMM_TILES[tile]):
            got = _C.matmul(A.cuda(), B.cuda()).cpu()
        assert bool((got == want).all())


@pytest.mark.parametrize("tile", ["256", "128", "256x64"])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False), (False, False), (True, True)])
@pytest.mark.parametrize("K", [17, 32, 33, 47, 64, 79, 257, 272, 530])
def test_slab_counts_and_tails(tile, ta, tb, K):
    M, N = 129, 64 if tile == "256x64" else 131
    with _lib.route("gemm_tile", _lib.GEMM_TILES[tile]):
        _check(*_operands(M, N, K, ta, tb, seed=K))


@pytest.mark.parametrize("shape", [(17, 17, 40), (255, 257, 48), (257, 63, 100), (1000, 301, 77)])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
def test_partial_tiles(shape, ta, tb):
    _check(*_operands(*shape, ta, tb, seed=sum(shape)))


@pytest.mark.parametrize("tile", ["256", "128", "256x64"])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
def test_non_finite_and_overflowing_values(tile, ta, tb):
    """What fp32 arithmetic gives: infinities keep their sign, NaN stays NaN,
    and a value whose parts overflow bf16 still has its product."""
    M, N, K = 40, 40, 100
    A, B = _operands(M, N, K, ta, tb)
    B = B.abs() + 0.25
    A, B = A.clone(), B.clone()
    A[3, 5], A[7, 90] = float("inf"), -float("inf")
    A[11, 2] = float("nan")
    A[20] = 0.0
    A[20, 7] = 3.4028234e38
    B[7, 1] = 0.5
    with _lib.route("gemm_tile", _lib.GEMM_TILES[tile]):
        got = _C.matmul(A.cuda(), B.cuda()).cpu()
    assert bool((got[3] == float("inf")).all()) and bool((got[7] == -float("inf")).all())
    assert bool(got[11].isnan().all())
    want = (A[20:21].double() @ B.double()).float()[0]    # one term a value: exact
    assert torch.equal(got[20], want)
    rest = [i for i in range(M) if i not in (3, 7, 11, 20)]
    err = (got[rest].double() - A[rest].double() @ B.double()).abs()
    assert bool((err <= (K + 8) * 2.0 ** -24 * (A[rest].double().abs() @ B.double().abs())).all())


@pytest.mark.parametrize("tile", ["256", "128", "256x64"])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False), (False, False), (True, True)])
@pytest.mark.parametrize("power", [-109, -112, -120, -128, -140, -146])
def test_operands_below_the_split_parts(tile, ta, tb, power):
    """An operand below 2^-110 would have low parts past bf16's last bit 2^-133
    (none left at 2^-134); with a large other operand its products are
    ordinary numbers, and they keep fp32's accuracy: as whole operands, and as
    one value, in the first or the last slab."""
    M, N, K = 70, 40, 100
    A, B = _operands(M, N, K, ta, tb, seed=-power)
    small = (A.double() * 2.0 ** power).float()
    with _lib.route("gemm_tile", _lib.GEMM_TILES[tile]):
        _check(small, B * 2.0 ** 60)
        _check(A * 2.0 ** 60, (B.double() * 2.0 ** power).float())
        for k in (3, K - 1):
            one = A.clone()
            one[9], B2 = 0.0, B.clone()
            one[9, k] = small[9, k]
            B2[k] = B[k] * 2.0 ** 60
            got = _C.matmul(one.cuda(), B2.cuda())[9].cpu().double()
            want = small[9, k].double() * B2[k].double()
            # one product: the last MFMA truncates (2^-23), the five before it at
            # 2^-8 of that or less, the dropped parts 2^-26
            assert bool(((got - want).abs() <= 1.25 * 2.0 ** -23 * want.abs()).all())


@pytest.mark.parametrize("tile", ["256", "128", "256x64"])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
@pytest.mark.parametrize("pa,pb", [(-64, -60), (46, 45), (100, 18), (18, 100), (115, 3), (126, -40)])
def test_small_and_large_products(tile, ta, tb, pa, pb):
    """Products near both ends of fp32's range (those whose scaled sums or
    parts overflow are evaluated in plain fp32)."""
    A, B = _operands(70, 40, 100, ta, tb, seed=pa)
    with _lib.route("gemm_tile", _lib.GEMM_TILES[tile]):
        # (plain fp32 adds one product at a time)
        _check(A.clamp(-1.9, 1.9) * 2.0 ** pa, B * 2.0 ** pb, None if pa < 0 else 100)


@pytest.mark.parametrize("tile", ["256", "128", "256x64"])
@pytest.mark.parametrize("K", [40, 256, 257, 400, 513, 1000])
def test_zero_sums_are_positive(tile, K):
    """Rows of zeros give +0, whichever sign the sums end with (outputs large
    enough that K is not split)."""
    M, N = 2304, 64 if tile == "256x64" else 2304
    A, B = _operands(M, N, K, False, True, seed=K)
    A[::2] = 0.0
    with _lib.route("gemm_tile", _lib.GEMM_TILES[tile]):
        got = _C.matmul(A.cuda(), B.cuda())[::2]
    assert not bool(got.any()) and not bool(got.signbit().any())


def test_error_has_no_mean():
    """The MFMA's rounding towards minus infinity must not add up: over 65536
    output values the mean error lies within five standard errors plus a
    hundredth of the truncation's own mean (-3e-8 of a term's rms per slab,
    K / 16 slabs, were it left in)."""
    M = N = 256
    K = 16384
    A, B = _operands(M, N, K, False, True, seed=1)
    with _lib.route("gemm_tile", 0):
        err = _C.matmul(A.cuda(), B.cuda()).cpu().double() - A.double() @ B.double()
    limit = 5 * float(err.std()) / (M * N) ** 0.5 + 0.01 * 3e-8 * (K / 16)
    assert abs(float(err.mean())) < limit


@pytest.mark.parametrize("kcont_a,kcont_b", [(True, False), (True, True), (False, False),
                                             (False, True)])
def test_leading_dimension_past_a_buffer_resource(kcont_a, kcont_b):
    """256 rows of 2.2 million columns, or 16 of 34 million, span more than 2^31
    bytes: the loads with 64-bit addresses."""
    M, N, K = 300, 70, 40
    A, B = _operands(M, N, K, not kcont_a, kcont_b, seed=5)
    if kcont_a:
        wide = torch.empty(M, 2_200_000, device="cuda")[:, :K]
    else:
        wide = torch.empty(K, 34_000_000, device="cuda")[:, :M].t()
    wide.copy_(A)
    with _lib.route("gemm_tile", 0):    # 256 rows
        got = _C.matmul(wide, B.cuda())
        assert torch.equal(got, _C.matmul(A.cuda(), B.cuda()))
        _check(wide.cpu(), B)
        # the wide operand on the other side
        assert torch.equal(_C.matmul(B.cuda().t(), wide.t()),
                           _C.matmul(B.cuda().t(), A.cuda().t()))


def test_long_sums_of_samples():
    """A parameter product of 65536 samples with a mean, large enough to fill
    the chip unsplit.  A running sum rounds once per slab of 16, each rounding
    at most half an ulp of it, uniform up to that: 2^-24 / sqrt(3) rms of the
    running sum, which grows evenly, so a chain of L / 16 slabs is off by
    2^-24 / 3 * sqrt(L / 16) of its end (1.3e-6 for all 65536 samples) and s
    slices' sums by 1 / sqrt(s) of theirs: 1.6e-7 for eight, 2^-24 on top for
    the slabs' own chains and the adds of the slices."""
    M, N, K = 1024, 14336, 65536
    g = torch.Generator(device="cuda").manual_seed(2)
    A = torch.rand(K, M, device="cuda", generator=g)
    B = torch.rand(K, N, device="cuda", generator=g)
    got = _C.matmul(A.t(), B)[:, ::112].double()
    want = A.double().t() @ B[:, ::112].double()
    assert float((got - want).norm() / want.norm()) < 1.6e-7 + 2.0 ** -24
