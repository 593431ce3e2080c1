"""The bf16-piece product (gemm_bf16x3.hip) behind ikv_mul_mat_f32 and
ikv_gemm_nt_f32: every tile shape at ragged sizes and K splits against a
64-bit product, no farther from it than the F32 MFMA kernel; infinities, NaNs
and magnitudes that its bf16 pieces cannot carry."""
import ctypes

import pytest
import torch

import ikv
from ikv import synth

pytestmark = pytest.mark.gpu

F32_TILES, PIECE_TILES = range(5), range(5, 9)


def dev_t(seed, shape, std, dev):
    return torch.from_numpy(synth.normal(seed, shape, std)).to(dev)


def tile(code, split, w, x, residual=None, out=None):
    n, k = w.shape
    m = x.shape[0]
    if out is None:
        out = torch.full((m, n), float("nan"), device=w.device)
    ws = torch.zeros((16 << 10) + (16 << 20), dtype=torch.uint8, device=w.device)
    rc = ikv.load_bench().ikv_bench_gemm_nt_tile_f32(
        w.data_ptr(), x.data_ptr(), out.data_ptr(), n, k, m,
        None if residual is None else residual.data_ptr(), code, split, ws.data_ptr(), ws.numel(),
        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    assert not ws[:16 << 10].any()  # every tile counter back at 0
    return out


def rel(a, ref):
    return float((a.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize("code", PIECE_TILES)
@pytest.mark.parametrize("n_out,k,m", [(64, 64, 1), (192, 64, 33), (320, 192, 129), (256, 1600, 77)])
def test_every_shape_and_split(dev, code, n_out, k, m):
    # one step per K group up to 25 64-column ones, ranges that do not divide,
    # tiles past n_out and m; residual in place. An output is a sum of k
    # products: 2^-24 sqrt(k) of the row's norm bounds a correct one's error
    w, x = dev_t(10 + m, (n_out, k), 0.02, dev), dev_t(11 + m, (m, k), 1.0, dev)
    r = dev_t(12 + m, (m, n_out), 1.0, dev)
    ref = x.double() @ w.double().t()
    scale = x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None]
    for split in (1, 2, 3, 8):
        if split > k // 64:
            continue
        got = tile(code, split, w, x)
        assert bool(((got.double() - ref).abs() <= 2.0 ** -24 * k ** 0.5 * scale).all()), split
        assert torch.equal(got, tile(code, split, w, x))
        buf = r.clone()
        tile(code, split, w, x, residual=buf, out=buf)
        assert torch.equal(buf, got + r), split


@pytest.mark.parametrize("k", [64, 1024, 4096])
def test_no_farther_from_64_bits_than_f32(dev, k):
    w, x = dev_t(20, (256, k), 0.02, dev), dev_t(21, (256, k), 1.0, dev)
    ref = x.double() @ w.double().t()
    f32 = rel(tile(1, 1, w, x), ref)
    for code in PIECE_TILES:
        assert rel(tile(code, 1, w, x), ref) <= f32


@pytest.mark.parametrize("code", PIECE_TILES)
@pytest.mark.parametrize("split", [1, 2])
def test_values_the_pieces_cannot_carry(dev, code, split):
    # what the F32 kernel gives, for rows with an infinity, a NaN, a float
    # above bf16's largest, and for products near the bottom of F32's range
    n_out, k, m = 256, 256, 128
    w, x = dev_t(30, (n_out, k), 0.02, dev), dev_t(31, (m, k), 1.0, dev)
    x[3, 7], x[40, 200], x[70, 0] = float("inf"), float("nan"), 3.4e38
    x[100, 5], w[9, 5] = float("-inf"), 0.0
    want, got = tile(0, split, w, x), tile(code, split, w, x)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    ok = want.isfinite()
    ok[70] = False  # (3.4e38 * w: its own scale)
    assert rel(got[ok], (x.double() @ w.double().t())[ok]) < 1e-6
    assert rel(got[70], x[70].double() @ w.double().t()) < 1e-6
    for ex in (-60, -85, -115):  # every product above the smallest normal float
        xs, ws = x.nan_to_num(0, 0, 0).clamp(-4, 4) * 2.0 ** ex, w * 2.0 ** max(-60, -120 - ex)
        ref = xs.double() @ ws.double().t()
        assert rel(tile(code, split, ws, xs), ref) <= 1.01 * rel(tile(0, split, ws, xs), ref) + 1e-7, ex
    z = tile(code, split, torch.zeros_like(w), x.nan_to_num(0, 0, 0))
    assert not z.any()


@pytest.mark.parametrize("n_out,k,m", [(2048, 1024, 2048), (4096, 4096, 777), (4096, 4096, 128),
                                       (1024, 3072, 777), (768, 1024, 4096)])
def test_the_plan_takes_it_for_large_products(dev, n_out, k, m):
    code, split = ctypes.c_int(), ctypes.c_int()
    assert ikv.load_bench().ikv_bench_gemm_choice(n_out, k, m, ctypes.byref(code),
                                                  ctypes.byref(split)) == 0
    assert code.value in PIECE_TILES
    w, x = dev_t(40, (n_out, k), 0.02, dev), dev_t(41, (m, k), 1.0, dev)
    assert torch.equal(ikv.mul_mat(w, x), tile(code.value, split.value, w, x))


@pytest.mark.parametrize("code", PIECE_TILES)
@pytest.mark.parametrize("split", [1, 2])
def test_small_floats_keep_their_bits_beside_ordinary_ones(dev, code, split):
    # a float below 2^-109 has bits that no bf16 piece holds: one such token
    # among ordinary ones, one such weight row, one such element in a row, and
    # whole operands of them against large ones. Row by row and column by
    # column no farther from 64 bits than the F32 kernel's sums can be:
    # 2^-24 sqrt(k) of |x| |w|, and what a denormal result rounds by
    n_out, k, m = 256, 256, 128
    w0, x0 = dev_t(50, (n_out, k), 0.02, dev), dev_t(51, (m, k), 1.0, dev)

    def check(x, w, what):
        got = tile(code, split, w, x).double()
        xd, wd = x.double(), w.double()
        bar = 2.0 ** -24 * k ** 0.5 * xd.norm(dim=1)[:, None] * wd.norm(dim=1)[None] + k * 2.0 ** -149
        assert bool(((got - xd @ wd.t()).abs() <= bar).all()), what

    for ex in (-109, -112, -115, -122, -126, -132, -140):
        x, w = x0.clone(), w0.clone()
        x[77] *= 2.0 ** ex
        check(x, w0, ("token", ex))
        w[200] *= 2.0 ** (ex + 6)
        check(x0, w, ("weight row", ex))
        # (the row's other products are zero)
        x = x0.clone()
        x[5] = 0
        x[5, 200] = 1.2345678 * 2.0 ** ex
        check(x, w0 * 2.0 ** 60, ("element", ex))
        x, w = x0 * 2.0 ** ex, w0 * 2.0 ** min(100, -ex - 30)
        check(x, w, ("against large", ex))
        check(w[:m] * 1.0, (x0 * 2.0 ** ex).repeat(2, 1), ("large against", ex))
    # products that are denormal or next to it, of floats that are not
    x, w = x0.clone(), w0 * 2.0 ** -60
    x[::3] *= 2.0 ** -60
    check(x, w, "denormal sums")


def test_a_split_the_f32_plan_does_not_ask_for_needs_no_workspace(dev):
    # captured on a stream that never ran such a product, so without a
    # workspace: the product runs unsplit, as it did on the F32 kernel; one
    # that the F32 plan splits as well is refused, and the capture goes on
    lib = ikv.load_bench()
    hip = ctypes.CDLL("libamdhip64.so")

    def plan(name, n_out, k, m):
        code, split = ctypes.c_int(), ctypes.c_int()
        assert getattr(lib, name)(n_out, k, m, ctypes.byref(code), ctypes.byref(split)) == 0
        return code.value, split.value

    n_out, k, m = 4096, 4096, 128
    assert plan("ikv_bench_gemm_plan", n_out, k, m)[1] == 1
    assert plan("ikv_bench_gemm_choice", n_out, k, m)[1] > 1
    assert plan("ikv_bench_gemm_plan", 1024, 2048, 128)[1] > 1
    w, x = dev_t(60, (n_out, k), 0.02, dev), dev_t(61, (m, k), 1.0, dev)
    w2, x2 = dev_t(62, (1024, 2048), 0.02, dev), dev_t(63, (128, 2048), 1.0, dev)
    out, out2 = torch.empty(m, n_out, device=dev), torch.zeros(128, 1024, device=dev)
    eager = ikv.mul_mat(w, x)
    raw = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(raw)) == 0
    side = torch.cuda.ExternalStream(raw.value)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        ikv.mul_mat(w, x, out=out)
        with pytest.raises(RuntimeError):
            ikv.mul_mat(w2, x2, out=out2)
        ikv.mul_mat(w, x, out=out)
    scale = x.double().norm(dim=1)[:, None] * w.double().norm(dim=1)[None]
    ref = x.double() @ w.double().t()
    first = None
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert bool(((out.double() - ref).abs() <= 2.0 ** -24 * k ** 0.5 * scale).all())
        first = out.clone() if first is None else first
        assert torch.equal(out, first)
    assert rel(eager, ref) <= rel(out, ref) * 1.5 and not out2.any()
    del g
    assert hip.hipStreamDestroy(raw) == 0
