"""The split GEMM's forms and cuts: products whose tiles fill whole rounds of one form and leave a
rest for another, K tails and odd K-tile counts in every form, all against float64, with the same
bits from every layout of A and B and every group order."""
import numpy as np
import pytest
import torch

from oracle import fp64
from piton_amd.runtime import mi355x as rt

pytestmark = pytest.mark.gpu


def _run(a, b, a_t, b_t, pad, group=8):
    M, K = a.shape
    N = b.shape[1]

    def store(x, t):
        x = x.t() if t else x
        s = torch.full((x.shape[0] + 1, x.shape[1] + pad), float("nan"), device="cuda")
        s[:-1, :x.shape[1]] = x
        return s, (1, s.shape[1]) if t else (s.shape[1], 1)

    (sa, st_a), (sb, st_b) = store(a, a_t), store(b, b_t)
    c = torch.full((M + 1, N + 3), -7.0, device="cuda")
    rt.matmul(sa, sb, c, M, N, K, *st_a, *st_b, N + 3, 1, group)
    names = [x["kernel"] for x in rt.last_launches()]
    assert (c[M:] == -7.0).all() and (c[:, N:] == -7.0).all()
    return c[:M, :N].contiguous(), names


# one launch per form, and cuts by rows and by columns; K tails, odd and even K-tile counts, fewer
# K tiles than waves
@pytest.mark.parametrize("M,N,K,launches", [(2500, 3000, 68, 1), (3000, 3200, 132, 1), (1100, 1800, 1000, 1),
                                            (700, 300, 44, 1), (33, 65, 4, 1), (2560, 2560, 2560, 2),
                                            (300, 4000, 3000, 2), (4000, 300, 3000, 2), (1, 1, 100, 1),
                                            (2049, 2177, 96, 1), (1344, 1976, 1600, 1)])
def test_forms_and_cuts(M, N, K, launches):
    """Every element within the float32 bound (K + 2) 2^-24 sum |a| |b| of float64; rows, columns
    and the padding (NaN) around them never reach C; all layouts and group orders agree bit for
    bit (the padding keeps every layout on the split kernel: 16-byte columns)."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a, b = (torch.rand(s, device="cuda", generator=g) * 2 - 1 for s in ((M, K), (K, N)))
    base, names = _run(a, b, False, False, 4)
    assert all(n.startswith("gemm_split_kernel") for n in names), names
    if rt.device_info()["cu_count"] == 256:
        assert len(names) == launches, names
    rows = np.unique(np.r_[0, M - 1, np.random.default_rng(1).integers(0, M, 200)])
    an, bn = a.cpu().numpy()[rows].astype(np.float64), b.cpu().numpy().astype(np.float64)
    bound = (K + 2) * 2.0 ** -24 * (np.abs(an) @ np.abs(bn))
    assert not (np.abs(base.cpu().numpy()[rows] - an @ bn) > bound).any()
    for a_t, b_t in ((True, False), (False, True), (True, True)):
        if (K % 4 or N % 4 or M % 4) and (a_t or b_t):
            continue
        got, names = _run(a, b, a_t, b_t, 4)
        assert all(n.startswith("gemm_split_kernel") for n in names), (a_t, b_t, names)
        assert torch.equal(got, base), (a_t, b_t, names)
    assert torch.equal(_run(a, b, False, False, 3)[0], base)  # rows off the 16-byte boundaries
    for group in (1, 3, 2 ** 31 - 1):
        assert torch.equal(_run(a, b, False, False, 4, group)[0], base)


@pytest.mark.parametrize("M,N,tiles", [(96, 160, 1), (96, 160, 5), (2049, 2177, 2), (600, 1100, 9)])
def test_every_k_tail(M, N, tiles):
    """All 31 lengths of the partial K tile (up to 16 values, or more, to the two lane halves), with NaN
    after A's and B's rows: dyadic inputs, every sum exact, so float64's bits."""
    g = torch.Generator(device="cuda").manual_seed(M + tiles)
    for rem in range(1, 32):
        K = 32 * tiles + rem
        a, b = (torch.randint(-4, 5, s, device="cuda", generator=g).float() / 4 for s in ((M, K), (K, N)))
        want = (a.double() @ b.double()).float()
        for a_t, b_t, pad in ((False, False, 4), (False, False, 3), (True, False, 4), (False, True, 4 - K % 4)):
            got, names = _run(a, b, a_t, b_t, pad)
            assert torch.equal(got, want), (K, a_t, b_t, names)


# the partial sums per element that the waves over K kept for these sizes: fewer than 1024 tiles of
# 64 x 64 have four, fewer than 2048 two
SUMS = [(1971, 654, 1280, 4), (1115, 2752, 354, 4), (2945, 960, 231, 4), (2112, 1664, 704, 4), (1024, 3353, 712, 4),
        (3897, 2060, 594, 2), (2873, 2880, 620, 2), (3689, 2240, 2410, 2), (2578, 3130, 129, 2)]


@pytest.mark.parametrize("M,N,K,sums", SUMS)
def test_partial_sums_per_element(M, N, K, sums):
    """Every form keeps at least `sums` interleaved partial sums, so the error against float64 is
    that of sums so long: no larger than 1.1 times (the rounding errors are random: the relative
    2-norm over 64 x N elements varies by 2 %) the error of the same sums formed one product after
    another in float32; and four sums are the bits of four waves over K, which a product of 64 rows
    has."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.rand(s, device="cuda", generator=g) * 2 - 1 for s in ((M, K), (K, N)))
    got, names = _run(a, b, False, False, 4)
    for name in names:  # gemm_split_kernel<.., .., waves over K, .., .., .., sums per wave>
        values = name.rstrip(">").split(", ")
        assert int(values[2]) * int(values[-1]) >= sums, names
    rows = a[:64]
    if sums == 4:
        few, few_names = _run(rows, b, False, False, 4)
        assert all(", 4, A_" in n for n in few_names), few_names
        assert torch.equal(got[:64], few), (names, few_names)
    part = torch.zeros((sums, 64, N), device="cuda")
    for k in range(K):  # product by product, K tiles of 32 dealt to the sums
        part[k // 32 % sums] += rows[:, k, None] * b[k]
    chain = part[0]
    for p in part[1:]:
        chain = chain + p
    want = rows.double() @ b.double()
    err, ref = ((x.double() - want).norm().item() for x in (got[:64], chain))
    assert err <= 1.1 * ref, (err, ref, names)


@pytest.mark.parametrize("M,N,K,tail", [(1344, 1976, 1600, False), (829, 3476, 1632, False), (1000, 1000, 1632, True),
                                        (1344, 1976, 1604, True)])
def test_zero_tiles_pad_odd_counts(M, N, K, tail):
    """64 x 64 tiles, more than two to a CU, and no K tail: every wave takes its K tiles in pairs,
    the last one of an odd count beside a tile of zeros; others take it ahead of the loop. Dyadic
    inputs with NaN around them: float64's bits."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randint(-4, 5, s, device="cuda", generator=g).float() / 4 for s in ((M, K), (K, N)))
    got, (name, *_) = _run(a, b, False, False, 4)
    assert torch.equal(got, (a.double() @ b.double()).float())
    if rt.device_info()["cu_count"] == 256:
        assert name == f"gemm_split_kernel<2, 2, 4, A_ROW16, false, {str(tail).lower()}, 1>"


@pytest.mark.parametrize("M,N,K", [(900, 1500, 260), (1767, 896, 256), (2176, 512, 308), (1000, 1800, 700)])
def test_matmul_linear_and_dense_take_the_same_form(M, N, K):
    """One planner for the three entries: the same product gets the same launches and bits from each."""
    g = torch.Generator(device="cuda").manual_seed(M)
    a, b = (torch.rand(s, device="cuda", generator=g) * 2 - 1 for s in ((M, K), (K, N)))
    c, y, z = (torch.full((M, N), -7.0, device="cuda") for _ in range(3))
    names = []
    for call in (lambda: rt.matmul(a, b, c, M, N, K, K, 1, N, 1, N, 1, 8),
                 lambda: rt.linear(a, K, b, None, None, 0, y, N, M, N, K),
                 lambda: rt.dense(a, b, None, z, M, N, K, add_bias=False)):
        call()
        names.append([x["kernel"] for x in rt.last_launches()])
    assert names[0] == names[1] == names[2], names
    assert torch.equal(c, y) and torch.equal(c, z)


@pytest.mark.parametrize("M,N,K", [(3324, 1664, 384), (1971, 654, 1280), (4032, 3072, 1000)])
def test_forms_of_slow_rounds_are_left(M, N, K):
    """B column-major with many 32 x 32 tiles of one wave, and a third round of 64 x 64 tiles of one wave,
    take longer than whole rounds of another form, which the planner takes instead."""
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = (torch.randint(-4, 5, s, device="cuda", generator=g).float() / 4 for s in ((M, K), (K, N)))
    got, names = _run(a, b, False, True, 4)
    assert torch.equal(got, (a.double() @ b.double()).float())
    if rt.device_info()["cu_count"] == 256:
        slow = "<2, 2, 1," if M == 4032 else "<1, 1, 1,"
        assert all(slow not in n for n in names), names


# whole 128 x 128 tiles in generations that are part full: the split kernel's and the direct kernel's
# times lie closest together here
@pytest.mark.parametrize("M,N,K", [(768, 7936, 256), (1280, 5120, 256), (5888, 1024, 256), (5888, 2560, 128),
                                   (1664, 3840, 256), (2688, 6144, 128)])
def test_whole_tiles_take_one_kernel_in_every_layout(M, N, K):
    """The choice between the split and the direct kernel depends on the sizes alone, so A and B stored
    either way give the same bits."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a, b = (torch.rand(s, device="cuda", generator=g) * 2 - 1 for s in ((M, K), (K, N)))
    base, names = _run(a, b, False, False, 4)
    family = {n.partition("<")[0] for n in names}
    for a_t, b_t in ((True, False), (False, True), (True, True)):
        got, names = _run(a, b, a_t, b_t, 4)
        assert {n.partition("<")[0] for n in names} == family, (a_t, b_t, names)
        assert torch.equal(got, base), (a_t, b_t, names)
