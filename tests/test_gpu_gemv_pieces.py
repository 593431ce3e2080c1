"""ikv_mul_mat_f32 where k is not a multiple of 1024 and n_out or k no multiple
of the GEMM's: rows of 16-byte pieces, and the form for any row, against a
64-bit product."""
import pytest
import torch

import ikv
from ikv import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 4, 7, 252, 256, 260, 380, 384, 512, 516, 768, 1020, 1028, 2044, 3076])
@pytest.mark.parametrize("n_out,m", [(1, 1), (5, 1), (1024, 1), (67, 3), (300, 28)])
def test_rows(dev, k, n_out, m):
    # one piece up to several rounds of 1024 columns, remainders in each; an
    # output is a sum of k products, 2^-24 (k + 1) of the sum of their sizes
    # bounds a correct one's error, and 2^-23 of the result the residual's
    w = torch.from_numpy(synth.normal(20 + k, (n_out, k), 0.02)).to(dev)
    x = torch.from_numpy(synth.normal(21 + k, (m, k), 1.0)).to(dev)
    r = torch.from_numpy(synth.normal(22 + k, (m, n_out), 1.0)).to(dev)
    ref = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    # a NaN past the operands' ends must not be read into a result
    for shift in (0, 1):  # 16-byte aligned, and not
        wb = torch.full((n_out * k + 9,), float("nan"), device=dev)
        xb = torch.full((m * k + 9,), float("nan"), device=dev)
        ws = wb[shift:shift + n_out * k].view(n_out, k).copy_(w)
        xs = xb[shift:shift + m * k].view(m, k).copy_(x)
        got = torch.full((m, n_out), float("nan"), device=dev)
        ikv.mul_mat(ws, xs if m > 1 else xs[0], out=got if m > 1 else got[0])
        assert bool(((got.double() - ref).abs() <= 2.0 ** -24 * (k + 1) * size).all())
        ikv.mul_mat(ws, xs if m > 1 else xs[0], out=got if m > 1 else got[0],
                    residual=r if m > 1 else r[0])
        want = ref + r.double()
        assert bool(((got.double() - want).abs() <=
                     2.0 ** -24 * (k + 1) * size + 2.0 ** -23 * want.abs()).all())
