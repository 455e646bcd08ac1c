"""Row softmax past 16K columns against float64: the 1024-thread register kernels at the ends of
their ranges and the two-pass kernel past 64K columns, aligned and not, with the special rows."""
import numpy as np
import pytest
import torch

from oracle import fp64
from piton_amd.runtime import mi355x as rt

pytestmark = pytest.mark.gpu
NEG_NAN = np.array(0xFFC00000, np.uint32).view(np.float32)


@pytest.mark.parametrize("n,in_pad,out_pad", [(16385, 0, 0), (32768, 0, 0), (32765, 3, 3), (32769, 0, 0), (50000, 0, 1),
                                              (65532, 4, 0), (65533, 0, 0), (65536, 0, 0), (65537, 0, 0), (70001, 2, 2),
                                              (100000, 0, 0), (131073, 0, 6)])
def test_long_rows(n, in_pad, out_pad):
    """Float32 sums of n positive terms in any order: within 1e-5 of float64 (relative Frobenius).
    +inf, +NaN and all -inf rows are NaN; -inf and -NaN entries are exactly 0; columns past n
    stay untouched; a row whose maximum comes last rescales every earlier partial sum."""
    rng = np.random.default_rng(n)
    x = (rng.standard_normal((8, n + in_pad)) * 4).astype(np.float32)
    x[1, n // 2] = np.inf
    x[2, : n - 1] = -np.inf
    x[3, :n] = -np.inf
    x[4, n // 3] = np.nan
    x[5, [0, n - 1]] = NEG_NAN, -np.inf
    x[6, :n] = np.sort(x[6, :n])
    x[7, :n] -= np.float32(3e38)  # far below 0, where a sum referenced to 0 would vanish
    out = torch.full((8, n + out_pad), -5.0, device="cuda")
    rt.softmax(out, torch.from_numpy(x).cuda(), n + in_pad, n + out_pad, n, 8, 1 << 18)
    got = out.cpu().numpy()
    assert (got[:, n:] == -5.0).all()
    got = got[:, :n]
    assert np.isnan(got[[1, 3, 4]]).all()
    assert got[2, n - 1] == 1 and (got[2, : n - 1] == 0).all()
    assert got[5, 0] == 0 and got[5, n - 1] == 0
    x = x[:, :n].copy()
    x[5, 0] = -np.inf
    fin = [0, 5, 6, 7]
    assert fp64.rel_fro(got[fin], fp64.softmax(x[fin])) <= 1e-5


@pytest.mark.parametrize("n", [50001, 80000])
def test_in_place(n):
    x = np.random.default_rng(n).standard_normal((5, n)).astype(np.float32)
    t = torch.from_numpy(x).cuda()
    rt.softmax(t, t, n, n, n, 5, 1 << 18)
    assert fp64.rel_fro(t.cpu().numpy(), fp64.softmax(x)) <= 1e-5
