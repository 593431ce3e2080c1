"""RMS norms whose scale lies on a float rounding midpoint, where the parallel
sums cannot tell which way the reference's index-order sum rounds and the
kernels take that sum instead; and the head-row kernel's sizes."""
import numpy as np
import pytest
import torch

import ikv
import oracle
from ikv import synth

pytestmark = pytest.mark.gpu

EPS = np.float32(1e-6)


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def midpoint_rows(dim, n, seed):
    """n rows whose sum of squares puts the scale within a few 2^-53 of the
    midpoint of two floats: three elements of falling size, in places that
    move, take up what is missing from the wanted sum."""
    x = synth.normal(seed, (n, dim))
    for i, row in enumerate(x):
        at = [(7 * i + 13 * j) % dim for j in range(3)]
        row[at] = 0
        sq = (row * row).astype(np.float64)
        t = 1.0 / np.sqrt((sq.sum() + 1.5) / dim + np.float64(EPS))
        f = np.float32(t)
        mid = 0.5 * (np.float64(f) + np.float64(np.nextafter(f, np.float32(np.inf))))
        want = (1.0 / (mid * mid) - np.float64(EPS)) * dim
        for j in at:
            left = max(want - (row * row).astype(np.float64).sum(), 0.0)
            v = np.float32(np.sqrt(left))
            row[j] = v if np.float64(v * v) <= left else np.nextafter(v, np.float32(0))
    S = (x * x).astype(np.float64).sum(axis=1)
    t = 1.0 / np.sqrt(S / dim + np.float64(EPS))
    f = t.astype(np.float32)
    nb = np.where(t >= f, np.nextafter(f, np.float32(np.inf)), np.nextafter(f, np.float32(0)))
    margin = np.abs(0.5 * (f.astype(np.float64) + nb.astype(np.float64)) - t) / t
    window = 2 * (0.5 * (dim - 1) + 8) * 2.0 ** -53  # the least any of the kernels has
    assert (margin < window).all()
    return x


@pytest.mark.parametrize("dim", [256, 768, 1024, 1280, 1536, 1792, 2048, 2304, 3072, 3328, 4096, 8192])
def test_midpoint_rows_long(dev, dim):
    x, w = midpoint_rows(dim, 9, 900 + dim), synth.normal(901, (dim,))
    got = ikv.rms_norm(torch.from_numpy(x).to(dev), torch.from_numpy(w).to(dev), float(EPS))
    assert np.array_equal(bits(got.cpu().numpy()), bits(oracle.rms_norm(x, w, float(EPS))))


@pytest.mark.parametrize("tokens,heads,dim", [
    (1, 1, 64), (1, 3, 128), (5, 3, 256), (33, 12, 64),        # one row set per wave, ragged
    (2731, 12, 64), (1367, 12, 128), (1640, 5, 256),           # four sets, the last wave ragged
])
def test_head_rows_with_midpoint_rows_among_them(dev, tokens, heads, dim):
    x = synth.normal(910 + tokens, (tokens * heads, dim))
    n = min(len(x), 24)
    x[np.linspace(0, len(x) - 1, n).astype(int)] = midpoint_rows(dim, n, 911 + dim)
    x = x.reshape(tokens, heads, dim)
    w = synth.normal(912, (dim,))
    pos = synth.uniform_ints(913, tokens, 512)
    th = oracle.rope_theta_table(1e6, dim, 512)
    s, c = (torch.from_numpy(t).to(dev) for t in ikv.rope_sincos_table(th))
    xd, wd, pd = (torch.from_numpy(t).to(dev) for t in (x, w, pos))
    want = oracle.rope_neox(oracle.rms_norm(x, w, float(EPS)), pos, th)
    got = ikv.qk_norm_rope(xd, wd, pd, float(EPS), s, c)
    assert np.array_equal(bits(got.cpu().numpy()), bits(want))
    assert np.array_equal(bits(ikv.rope_neox(xd, pd, s, c).cpu().numpy()),
                          bits(oracle.rope_neox(x, pos, th)))
    ikv.qk_norm_rope(xd, wd, pd, float(EPS), s, c, out=xd)  # in place
    assert np.array_equal(bits(xd.cpu().numpy()), bits(want))
    # a position outside the table: zero rows and the status bit, nothing else
    bad = pos.copy()
    bad[tokens // 2] = 512
    status = torch.zeros(1, dtype=torch.int32, device=dev)
    got = ikv.rope_neox(torch.from_numpy(x).to(dev), torch.from_numpy(bad).to(dev), s, c,
                        status=status).cpu().numpy()
    assert status.item() == ikv.STATUS_POSITION
    ref = oracle.rope_neox(x, pos, th)
    ref[tokens // 2] = 0
    assert np.array_equal(bits(got), bits(ref))


def test_midpoint_norm_folded_into_the_gemv(dev):
    # the projections' folded norm takes the index-order sum too
    k = 1024
    x = midpoint_rows(k, 1, 930)[0]
    nw, w = synth.normal(931, (k,)), [synth.normal(932 + i, (n, k), 0.02) for i, n in enumerate((64, 32, 32))]
    xd, nd = torch.from_numpy(x).to(dev), torch.from_numpy(nw).to(dev)
    wd = [torch.from_numpy(t).to(dev) for t in w]
    folded = ikv.gemv3(*wd, xd, norm_w=nd, eps=float(EPS))
    plain = ikv.gemv3(*wd, torch.from_numpy(oracle.rms_norm(x[None], nw, float(EPS))[0]).to(dev))
    assert all(torch.equal(a, b) for a, b in zip(folded, plain))
