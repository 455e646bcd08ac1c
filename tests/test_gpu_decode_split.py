"""Decode attention over a cache of several chunks (16384 / head_dim keys each): against float64
at the edges of the chunks, against the unsplit kernel, and with a chunk whose keys are all
masked by -inf."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import fp64
from piton_amd.runtime import mi355x as rt

pytestmark = pytest.mark.gpu


def _cache(B, H, n, dh, pad, seed):
    """q [B, H, dh] and position-major k, v [n, B, H, dh + pad]."""
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((B, H, dh)).astype(np.float32),
            *(rng.standard_normal((n, B, H, dh + pad)).astype(np.float32) for _ in range(2)))


def _args(q, k, v, out, scale):
    n, B, H, row = k.shape
    dh = q.shape[2]
    return q, k, v, out, scale, H * dh, dh, H * row, row, B * H * row, H * row, row, B * H * row, H * dh, dh, n, B, H, dh


def _split(q, k, v, scale):
    tq, tk, tv = (torch.from_numpy(t).cuda() for t in (q, k, v))
    out = torch.full(tq.shape, -9.0, device="cuda")
    rt.attn_decode(*_args(tq, tk, tv, out, scale))
    parts = rt.last_launches()[0]["grid"][0] // (q.shape[0] * q.shape[1])
    return out.cpu().numpy(), parts, (tq, tk, tv)


def _fp64(q, k, v, scale):
    dh = q.shape[2]
    return fp64.attention_reference(q[:, :, None], k.transpose(1, 2, 0, 3)[..., :dh], v.transpose(1, 2, 0, 3)[..., :dh],
                                    False, scale)[:, :, 0]


@pytest.mark.parametrize("dh,n,pad", [(64, 257, 0), (64, 512, 0), (64, 513, 4), (64, 767, 1), (64, 8192, 0), (128, 128, 0),
                                      (128, 129, 0), (128, 8192, 0), (32, 513, 0), (32, 1025, 1), (16, 1100, 0)])
def test_chunk_edges(dh, n, pad):
    """Unsplit and split results are float32 sums of the same n products in another order: both
    within the float32 bound of float64 (1e-5 relative Frobenius), so within twice it of each
    other."""
    q, k, v = _cache(2, 3, n, dh, pad, dh + n)
    scale = dh ** -0.5
    got, parts, (tq, tk, tv) = _split(q, k, v, scale)
    assert parts == -(-n // (16384 // max(dh, 32)))
    ref = _fp64(q, k, v, scale)
    assert fp64.rel_fro(got, ref) <= 1e-5
    # the entry without a workspace: the unsplit kernel
    one = torch.empty_like(tq)
    a = _args(tq, tk, tv, one, scale)
    rt._call("piton_mi355x_attn_decode", *(rt._ptr(t) for t in a[:4]), float(scale), *a[5:], rt._stream())
    assert fp64.rel_fro(one.cpu().numpy(), got) <= 2e-5
    # as many floats as the split needs, and not one less
    need = ctypes.c_int64()
    rt._call("piton_mi355x_attn_decode_workspace", n, 2, 3, dh, ctypes.byref(need))
    assert need.value == (6 * parts * (max(dh, 32) + 2) if parts > 1 else 0)
    if parts > 1:
        ws = torch.full((need.value + 64,), -7.0, device="cuda")
        rt._call("piton_mi355x_attn_decode_split", *(rt._ptr(t) for t in a[:4]), float(scale), *a[5:], rt._ptr(ws),
                 need.value, rt._stream())
        np.testing.assert_array_equal(one.cpu().numpy(), got)
        assert (ws[need.value:] == -7.0).all()
        rt._call("piton_mi355x_attn_decode_split", *(rt._ptr(t) for t in a[:4]), float(scale), *a[5:], rt._ptr(ws),
                 need.value - 1, rt._stream())
        assert len(rt.last_launches()) == 1


def test_masked_and_infinite_keys():
    """A whole chunk of -inf scores weighs nothing; a row of -inf scores alone is NaN; an infinite V
    in the last key counts once whatever the chunk's padding repeats."""
    q, k, v = _cache(1, 3, 600, 64, 0, 5)
    q = np.abs(q) + np.float32(0.1)  # with positive q, a key of -inf scores -inf
    k[256:512, :, 0] = -np.inf       # head 0: the second chunk
    k[:, :, 1] = -np.inf             # head 1: every key
    v[599, :, 2, 7] = np.inf         # head 2
    got, parts, _ = _split(q, k, v, 0.125)
    assert parts == 3
    keep = np.r_[0:256, 512:600]
    assert fp64.rel_fro(got[:, 0], _fp64(q[:, :1], k[keep][:, :, :1], v[keep][:, :, :1], 0.125)[:, 0]) <= 1e-5
    assert np.isnan(got[:, 1]).all()
    assert np.isposinf(got[0, 2, 7]) and np.isfinite(np.delete(got[0, 2], 7)).all()


def _past_nan(B, H, n, dh, pad):
    """A cache of n + 70 rows, the last 70 and the padding NaN, and float64's result over the first n."""
    q, k, v = _cache(B, H, n + 70, dh, pad, dh + n + B)
    ref = _fp64(q, k[:n], v[:n], 0.3)
    for x in (k, v):
        x[n:] = np.nan
        x[..., dh:] = np.nan
    tq, tk, tv = (torch.from_numpy(x).cuda() for x in (q, k, v))
    out = torch.full((B + 1, H, dh), -9.0, device="cuda")
    a = list(_args(tq, tk, tv, out, 0.3))
    a[15] = n
    rt.attn_decode(*a)
    assert (out[B:] == -9.0).all()
    return out[:B].cpu().numpy(), ref, [x["kernel"] for x in rt.last_launches()]


@pytest.mark.parametrize("dh", [16, 32, 64, 128])
@pytest.mark.parametrize("pad", [0, 1])
def test_every_row_count(dh, pad):
    """One chunk: the kernels of 1, 2, 4, 8 and 16 rows per thread at the edges of their keys."""
    per = 1024 // max(dh, 32)
    for rows, kernel in ((1, 1), (2, 2), (3, 4), (4, 4), (5, 8), (8, 8), (9, 16), (16, 16)):
        for n in sorted({(rows - 1) * per + 1, rows * per - 1, rows * per}):
            got, ref, names = _past_nan(2, 3, n, dh, pad)
            assert len(names) == 1 and f", {kernel}, 1>" in names[0], (n, names)
            assert fp64.rel_fro(got, ref) <= 1e-5, n


@pytest.mark.parametrize("dh", [16, 32, 64, 128])
def test_the_chunk_is_the_librarys(dh):
    chunk = rt._decode_chunk(dh)
    assert chunk == 16384 // max(dh, 32)
    assert [rt._decode_floats(n, 2, 3, dh) > 0 for n in (1, chunk, chunk + 1, 8192, 8193)] == [0, 0, 1, 1, 0]


@pytest.mark.parametrize("dh", [32, 64, 128])
@pytest.mark.parametrize("pad", [0, 3])
def test_many_heads_take_several_chunks_in_one_workgroup(dh, pad):
    """Two heads per CU and more: up to three chunks' keys in one launch, four split as before."""
    B, H, chunk = 2 * rt.device_info()["cu_count"] // 8, 8, 16384 // dh
    g = torch.Generator(device="cuda").manual_seed(dh + pad)
    q = torch.randn((B, H, dh), device="cuda", generator=g)
    k, v = (torch.randn((3 * chunk + 2, B, H, dh + pad), device="cuda", generator=g) for _ in range(2))
    out = torch.empty_like(q)
    for n in (chunk + 1, chunk + chunk // 2, 2 * chunk, 2 * chunk + 1, 3 * chunk - 1, 3 * chunk, 3 * chunk + 1):
        tail = k[n:].clone(), v[n:].clone()
        k[n:], v[n:] = float("nan"), float("nan")
        a = list(_args(q, k, v, out, 0.3))
        a[15] = n
        rt.attn_decode(*a)
        assert len(rt.last_launches()) == (1 if n <= 3 * chunk else 2), n
        k[n:], v[n:] = tail
        p = torch.softmax((k[:n, ..., :dh].double() * q.double()).sum(-1) * 0.3, 0)
        ref = (p[..., None] * v[:n, ..., :dh].double()).sum(0)
        assert ((out.double() - ref).norm() / ref.norm()).item() <= 1e-5, n


@pytest.mark.parametrize("dh,n", [(64, 600), (128, 300), (32, 1100)])
def test_large_values_of_keys_without_weight(dh, n):
    """Finite values near the largest float whose keys have a weight of 0, or next to it, beside the
    others: their chunk's own sum would overflow, the result is float64's within the float32 bound."""
    q, k, v = _cache(1, 2, n, dh, 0, dh + n)
    chunk = 16384 // dh
    q[...], k[...] = 1, 0
    k[:chunk, :, 0] = -dh * 0.5   # head 0: the first chunk's weights underflow
    k[:chunk, :, 1] = -2.0        # head 1: they are 2^-(2 dh log2 e) and smaller, and count
    v[:chunk] = np.float32(1e37) * np.sign(v[:chunk])
    v[:chunk, :, 1] *= np.float32(1e-20)
    got, parts, _ = _split(q, k, v, 1.0)
    assert parts > 1
    ref = _fp64(q, k, v, 1.0)
    assert np.isfinite(got).all()
    for h in range(2):
        assert fp64.rel_fro(got[:, h], ref[:, h]) <= 1e-5, h


def test_captured_calls_replay():
    """The workspace of a captured call belongs to the graph: replays with eager calls of other
    shapes between them give the eager bits."""
    q, k, v = _cache(2, 4, 1000, 64, 0, 8)
    want, _, (tq, tk, tv) = _split(q, k, v, 0.125)
    out = torch.empty_like(tq)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        rt.attn_decode(*_args(tq, tk, tv, out, 0.125))
    for n in (700, 5000, 300):
        out.zero_()
        g.replay()
        np.testing.assert_array_equal(out.cpu().numpy(), want)
        _split(*_cache(3, 4, n, 64, 0, n), 0.125)
