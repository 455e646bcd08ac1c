"""The dense entry's routes: layers that the fused chain takes (K even, K and N up to 256) on the split
kernel with four partial sums, of the others up to 64 rows with K a multiple of 256 on the small-row
kernel and the rest on the split kernel in any form, each against float64 around the lines between."""
import numpy as np
import pytest
import torch

from piton_amd.runtime import mi355x as rt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,kernel", [
    (100, 256, 256, "gemm_split_kernel"), (100, 257, 256, "gemm_split_kernel"), (100, 256, 258, "gemm_split_kernel"),
    (100, 64, 255, "gemm_split_kernel"), (1, 10, 32, "gemm_split_kernel"), (64, 257, 256, "gemm_small_m_kernel"),
    (65, 257, 256, "gemm_split_kernel"), (1, 10, 512, "gemm_small_m_kernel"), (17, 33, 1280, "gemm_small_m_kernel"),
    (64, 300, 260, "gemm_split_kernel"), (2000, 1000, 784, "gemm_split_kernel"), (1, 1, 257, "gemm_split_kernel")])
@pytest.mark.parametrize("add_bias,relu", [(True, True), (False, False)])
def test_dense_routes(M, N, K, kernel, add_bias, relu):
    """Each element within (K + 3) 2^-24 (sum |x| |w| + |b|) of float64; nothing past Y is written."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, w, b = (torch.rand(s, device="cuda", generator=g) * 2 - 1 for s in ((M, K), (K, N), (N,)))
    y = torch.full((M * N + 64,), -7.0, device="cuda")
    pred = torch.full((M,), -1, dtype=torch.int32, device="cuda")
    rt.dense(x, w, b if add_bias else None, y, M, N, K, add_bias=add_bias, relu=relu, argmax_out=pred, n_classes=N)
    launches = [l["kernel"] for l in rt.last_launches()]
    assert launches[0].startswith(kernel) and launches[-1].startswith("argmax_rows"), launches
    assert (y[M * N:] == -7.0).all()
    got = y[:M * N].view(M, N).cpu().numpy()
    xn, wn, bn = (t.cpu().numpy().astype(np.float64) for t in (x, w, b))
    bn = bn if add_bias else 0 * bn
    ref = xn @ wn + bn
    bound = (K + 3) * 2.0 ** -24 * (np.abs(xn) @ np.abs(wn) + np.abs(bn))
    ref = np.maximum(ref, 0) if relu else ref
    assert not (np.abs(got - ref) > bound).any()
    np.testing.assert_array_equal(pred.cpu().numpy(), got.argmax(1))


@pytest.mark.parametrize("M", [1, 128, 333])
@pytest.mark.parametrize("sizes", [(64, 128, 128, 256), (100, 30, 2, 7), (256, 256, 256, 256), (34, 224, 190, 33)])
def test_fused_chain_adds_as_the_dense_launches(M, sizes):
    """mlp3_kernel and the dense entry's split kernel keep the same four partial sums over K, with
    and without a partial K tile and whichever tile size the rows get: the same logits bit for bit."""
    g = torch.Generator(device="cuda").manual_seed(M + sum(sizes))
    rand = lambda *s: torch.rand(s, device="cuda", generator=g) * 2 - 1  # noqa: E731
    x = rand(M, sizes[0])
    w = [rand(k, n) for k, n in zip(sizes[:-1], sizes[1:])]
    b = [rand(n) for n in sizes[1:]]
    logits = torch.full((M, sizes[3]), -7.0, device="cuda")
    rt.mlp3(x, M, w[0], b[0], w[1], b[1], w[2], b[2], logits, None, 1)
    assert [l["kernel"] for l in rt.last_launches()] == ["mlp3_kernel"]
    h = x
    for i in range(3):
        y = torch.full((M, sizes[i + 1]), -7.0, device="cuda")
        rt.dense(h, w[i], b[i], y, M, sizes[i + 1], sizes[i], relu=i < 2)
        assert [l["kernel"].startswith("gemm_split_kernel") for l in rt.last_launches()] == [True]
        h = y
    assert torch.equal(logits, h)


@pytest.mark.parametrize("M,N,K", [(65, 33, 40), (2048, 768, 256), (700, 1000, 100), (2500, 3000, 68),
                                   (4000, 300, 2000), (300, 4000, 3000), (4096, 4096, 64)])
def test_linear_residual_in_place(M, N, K):
    """bias, ReLU and a residual that is the output itself, rows N + 5 apart, in the split kernel's
    forms (ragged tiles, one and four waves over K, cuts by rows and by columns) and the direct
    kernel: within (K + 4) 2^-24 (sum |x| |w| + |b| + |r|) of float64, the padding untouched."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    rand = lambda *s: torch.rand(s, device="cuda", generator=g) * 2 - 1  # noqa: E731
    x, w, b, y = rand(M, K), rand(K, N), rand(N), rand(M, N + 5)
    y0 = y.clone()
    rt.linear(x, K, w, b, y, N + 5, y, N + 5, M, N, K, relu=True)
    assert torch.equal(y[:, N:], y0[:, N:])
    rows = torch.from_numpy(np.unique(np.r_[0, M - 1, np.random.default_rng(1).integers(0, M, 200)])).cuda()
    xd, wd, bd, rd = x[rows].double(), w.double(), b.double(), y0[rows, :N].double()
    ref = torch.relu(xd @ wd + bd) + rd
    bound = (K + 4) * 2.0 ** -24 * (xd.abs() @ wd.abs() + bd.abs() + rd.abs())
    assert not ((y[rows, :N].double() - ref).abs() > bound).any()
