"""The attention forward's pipelined kernel over head dims 32 / 64 / 128 and both K layouts ([N, D]
and [D, N]) against the general kernel: the two run the same blocks, products and merge, so every
form gives the general kernel's bits; and against float64."""
import numpy as np
import pytest
import torch

from oracle import fp64
from piton_amd.runtime import mi355x as rt

pytestmark = pytest.mark.gpu


def _rows(t, ld):
    """t [H, R, C] stored with rows ld floats apart, NaN between them."""
    s = torch.full((t.shape[0], t.shape[1], ld), float("nan"), device="cuda")
    s[:, :, : t.shape[2]] = t
    return s


def _run(q, k, v, causal, dn, kpad, vpad, misalign):
    """misalign: the output one float off a 16-byte boundary, which the pipelined kernel refuses."""
    H, N, D = q.shape
    ts = _rows(k.transpose(1, 2) if dn else k, (N if dn else D) + kpad)
    vs = _rows(v, D + vpad)
    buf = torch.full((H * N * D + 8,), -3.0, device="cuda")
    out = buf[4 + misalign:]
    s_kh, ldk = ts[0].numel(), ts.shape[2]
    rt.attn_fwd(q, ts, vs, out, D ** -0.5, N * D, D, s_kh, 1 if dn else ldk, ldk if dn else 1, vs[0].numel(), D + vpad,
                N * D, D, N, H, D, causal)
    name = rt.last_launches()[0]["kernel"]
    host = buf.cpu()
    lo = 4 + misalign
    assert (host[:lo] == -3.0).all() and (host[lo + H * N * D:] == -3.0).all()
    return host[lo:lo + H * N * D].reshape(H, N, D).numpy(), name


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("H,N,causal", [(2, 1, True), (3, 31, False), (2, 33, True), (1, 160, False), (8, 257, True),
                                        (20, 1000, False), (40, 1056, True)])
def test_every_form_gives_the_general_kernels_bits(D, H, N, causal):
    g = torch.Generator(device="cuda").manual_seed(N + D)
    q, k, v = (torch.randn((H, N, D), device="cuda", generator=g) for _ in range(3))
    want, name = _run(q, k, v, causal, False, 0, 0, 1)
    assert name.startswith("attn_fwd_kernel_f32")
    ref = fp64.attention_reference(*(t[:2].cpu().numpy() for t in (q, k, v)), causal)
    assert fp64.rel_fro(want[:2], ref) <= 1e-5
    for dn, kpad, vpad in ((False, 0, 0), (False, 4, 8), (True, 0, 0), (True, 5, 4), (True, 2, 0)):
        got, name = _run(q, k, v, causal, dn, kpad, vpad, 0)
        assert name.startswith("attn_fwd_fast_dn<" if dn else "attn_fwd_fast<"), name
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
