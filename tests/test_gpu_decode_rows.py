"""The folded decode of generic heads (decode_rows_kernel, attn_generic.hip)
at the edges of its lanes, keys and splits: one lane group per key with part
of its lanes past the head, one key, a split's last keys, 1 to 8 query heads
per KV head; the folded qk-norm + RoPE and append against the separate
kernels, contiguous and paged; and a new token that has no place.

Bars: against float64, 1e-5 absolute + 1e-4 relative, the generic path's;
between the folded and the separate forms, and for appended rows, bitwise.
"""
import numpy as np
import pytest

import ikv
import oracle
from ikv import synth
from test_gpu_norm_rows import EPS, midpoint_rows

pytestmark = pytest.mark.gpu


def dev_t(a, dev):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dev)


def host(t):
    import torch
    torch.cuda.synchronize()
    return t.cpu().numpy()


def bits(t):
    return host(t).view(np.uint32)


def attend64(q, k, v):
    """softmax(q k^T / sqrt(D)) v in float64, GQA."""
    (n_head, D), n_kv_heads = q.shape, k.shape[1]
    g = n_head // n_kv_heads
    out = np.empty((n_head, D))
    for h in range(n_head):
        s = k[:, h // g].astype(np.float64) @ q[h].astype(np.float64) / np.sqrt(D)
        p = np.exp(s - s.max())
        out[h] = (p / p.sum()) @ v[:, h // g].astype(np.float64)
    return out


@pytest.mark.parametrize("D,Hq,Hkv,n_kv", [
    (4, 3, 1, 1), (20, 5, 5, 65), (60, 14, 2, 300), (64, 12, 4, 64), (64, 21, 3, 4100),
    (68, 6, 2, 63), (124, 15, 5, 129), (128, 6, 2, 1000), (132, 7, 1, 31), (256, 16, 2, 97),
    (252, 10, 2, 2049), (64, 18, 2, 200),  # the last from here: not folded
    # merges of 1, of 16 n and of 256 splits, dims past a workgroup's threads
    (30, 6, 2, 3), (300, 3, 1, 2048), (300, 6, 2, 2100), (512, 2, 1, 16384), (96, 9, 1, 16400)])
def test_rows_at_the_edges(dev, D, Hq, Hkv, n_kv):
    seed = 7100 + D + n_kv
    k, v = synth.normal(seed, (n_kv, Hkv, D)), synth.normal(seed + 1, (n_kv, Hkv, D))
    q = synth.normal(seed + 2, (Hq, D))
    ref = attend64(q, k, v)
    plain = host(ikv.attn_decode(dev_t(q, dev), dev_t(k, dev), dev_t(v, dev), n_kv))
    assert np.all(np.abs(plain - ref) <= 1e-5 + 1e-4 * np.abs(ref))
    # the last row given apart, behind a cache row that would change the result
    kc, vc = k.copy(), v.copy()
    kc[-1], vc[-1] = 50.0, 50.0
    kd, vd = dev_t(kc, dev), dev_t(vc, dev)
    got = host(ikv.attn_decode(dev_t(q, dev), kd, vd, n_kv, k_new=dev_t(k[-1], dev),
                               v_new=dev_t(v[-1], dev)))
    assert np.array_equal(got.view(np.uint32), plain.view(np.uint32))
    assert np.array_equal(bits(kd), k.view(np.uint32)) and np.array_equal(bits(vd), v.view(np.uint32))


@pytest.mark.parametrize("D,Hq,Hkv,n_kv,bt,pos", [
    (64, 12, 4, 2500, 0, 2499), (64, 7, 1, 1, 64, 0), (80, 6, 2, 130, 0, 129),
    (128, 6, 2, 191, 64, 190), (256, 10, 2, 65, 64, 64),
    (64, 6, 2, 70, 0, 4000), (64, 6, 2, 70, 64, -1)])  # the last two: no such position
def test_folded_norm_rope_and_append_equal_the_separate_kernels(dev, D, Hq, Hkv, n_kv, bt, pos):
    import torch
    seed = 7300 + D + n_kv
    sn, cs = ikv.rope_sincos_table(oracle.rope_theta_table(1e6, D, 4000))
    sn, cs = dev_t(sn, dev), dev_t(cs, dev)
    w_q, w_k = (dev_t(1 + 0.3 * synth.normal(seed + i, (D,)), dev) for i in range(2))
    rows = n_kv if not bt else (-(-n_kv // bt) + 2) * bt
    k0, v0 = synth.normal(seed + 2, (rows, Hkv, D)), synth.normal(seed + 3, (rows, Hkv, D))
    q, kn, vn = (dev_t(synth.normal(seed + 4 + i, (h, D)), dev) for i, h in enumerate((Hq, Hkv, Hkv)))
    p = torch.tensor([pos], dtype=torch.int32, device=dev)
    table = torch.tensor(np.random.default_rng(seed).permutation(max(rows // max(bt, 1), 1))[
        :-(-n_kv // bt) if bt else 1].astype(np.int32), device=dev)
    seen = []
    for fold in (True, False):
        k, v = dev_t(k0, dev), dev_t(v0, dev)
        st = torch.zeros(1, dtype=torch.int32, device=dev)
        if fold:
            args = (w_q, w_k, 1e-6, p, sn, cs)
            out = (ikv.attn_decode_rope_paged(q, kn, vn, k, v, table, bt, n_kv, *args, status=st)
                   if bt else ikv.attn_decode_rope(q, kn, vn, k, v, n_kv, *args, status=st))
        else:
            qr = ikv.qk_norm_rope(q[None], w_q, p, 1e-6, sn, cs, status=st)[0]
            kr = ikv.qk_norm_rope(kn[None], w_k, p, 1e-6, sn, cs, status=st)[0]
            out = (ikv.attn_decode_paged(qr, k, v, table, bt, n_kv, k_new=kr, v_new=vn)
                   if bt else ikv.attn_decode(qr, k, v, n_kv, k_new=kr, v_new=vn))
        seen.append([bits(out), bits(k), bits(v), host(st)])
    for a, b in zip(*seen):
        assert np.array_equal(a, b)


def test_a_new_token_without_a_block_is_dropped_and_reported(dev):
    """The new token's table entry names no block: nothing is written, the
    status says so, and the other keys are read as before."""
    import torch
    D, Hq, Hkv, bt, n_kv = 64, 6, 2, 64, 65
    k0, v0 = synth.normal(7500, (2 * bt, Hkv, D)), synth.normal(7501, (2 * bt, Hkv, D))
    q, kn, vn = (synth.normal(7502 + i, (h, D)) for i, h in enumerate((Hq, Hkv, Hkv)))
    k, v = dev_t(k0, dev), dev_t(v0, dev)
    table = torch.tensor([1, 2], dtype=torch.int32, device=dev)
    st = torch.zeros(1, dtype=torch.int32, device=dev)
    ikv.attn_decode_paged(dev_t(q, dev), k, v, table, bt, n_kv, k_new=dev_t(kn, dev),
                          v_new=dev_t(vn, dev), status=st)
    assert host(st)[0] == 2
    assert np.array_equal(bits(k), k0.view(np.uint32)) and np.array_equal(bits(v), v0.view(np.uint32))


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 12, 4), (64, 8, 1), (128, 10, 2), (128, 6, 2), (256, 10, 2)])
@pytest.mark.parametrize("which", ["all", "first", "last", "key"])
def test_rows_in_doubt_take_the_index_order_sum(dev, D, Hq, Hkv, which):
    """New q and k rows whose norm scale lies on a float rounding midpoint: all
    of them, one query row in the first or the last lane group, or the key row.
    The folded step gives the separate kernels' bits, and the appended key the
    oracle's."""
    import torch
    n_kv, pos = 130, 129
    seed = 7600 + D + Hq
    th = oracle.rope_theta_table(1e6, D, 200)
    sn, cs = (dev_t(t, dev) for t in ikv.rope_sincos_table(th))
    w_q, w_k = (1 + 0.3 * synth.normal(seed + i, (D,)) for i in range(2))
    k0, v0 = synth.normal(seed + 2, (n_kv, Hkv, D)), synth.normal(seed + 3, (n_kv, Hkv, D))
    q, kn, vn = (synth.normal(seed + 4 + i, (h, D)) for i, h in enumerate((Hq, Hkv, Hkv)))
    hard = midpoint_rows(D, Hq + Hkv, seed + 8)
    G = Hq // Hkv
    if which == "all":
        q, kn = hard[:Hq].copy(), hard[Hq:].copy()
    elif which == "first":
        q[::G] = hard[:Hkv]
    elif which == "last":
        q[G - 1::G] = hard[:Hkv]
    else:
        kn = hard[Hq:].copy()
    p = torch.tensor([pos], dtype=torch.int32, device=dev)
    wq_d, wk_d = dev_t(w_q, dev), dev_t(w_k, dev)
    k, v = dev_t(k0, dev), dev_t(v0, dev)
    out = ikv.attn_decode_rope(dev_t(q, dev), dev_t(kn, dev), dev_t(vn, dev), k, v, n_kv, wq_d, wk_d,
                               float(EPS), p, sn, cs)
    k2, v2 = dev_t(k0, dev), dev_t(v0, dev)
    qr = ikv.qk_norm_rope(dev_t(q, dev)[None], wq_d, p, float(EPS), sn, cs)[0]
    kr = ikv.qk_norm_rope(dev_t(kn, dev)[None], wk_d, p, float(EPS), sn, cs)[0]
    out2 = ikv.attn_decode(qr, k2, v2, n_kv, k_new=kr, v_new=dev_t(vn, dev))
    assert np.array_equal(bits(out), bits(out2))
    assert np.array_equal(bits(k), bits(k2)) and np.array_equal(bits(v), bits(v2))
    want = oracle.rope_neox(oracle.rms_norm(kn[None].astype(np.float32), w_k.astype(np.float32), float(EPS)),
                            np.array([pos], np.int32), th)
    assert np.array_equal(bits(k)[pos], np.ascontiguousarray(want[0], np.float32).view(np.uint32))
