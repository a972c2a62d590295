"""GPU parity of the training step's FP8 linear (tg_linear_fwd, tg_linear_bwd,
tg_linear_bwd_kept) on the extents and types that no block divides: bit for bit
the general path's result, that is quantize_fp8 of zero-padded f32 copies and
scaled_matmul (bf16 values widen to f32 exactly, so the bytes are the same)."""
import pytest
import torch
import torch.nn.functional as F

import _tglib as L
import fp8
import gemm_tiles as G

pytestmark = pytest.mark.gpu

BF, F32 = torch.bfloat16, torch.float32


def _pad(x, r, c):
    x = x.float()
    return F.pad(x, (0, c - x.shape[1], 0, r - x.shape[0])).contiguous()


def _general(a, b, g):
    """y, da, db (bf16) through padded copies, separate quantizers and row-major scales."""
    (M, K), N = a.shape, b.shape[1]
    mp, np_ = -(-M // 128) * 128, -(-N // 128) * 128
    u8 = torch.uint8
    ap, bp, gp = _pad(a, mp, K), _pad(b, K, np_), _pad(g, mp, np_)

    def mm(x, y):            # x (R, C), y (S, C) quantized along C
        return fp8.scaled_matmul(x[0].view(u8), x[1], y[0].view(u8), y[1])

    def rows(x):
        return fp8.quantize_fp8(x)

    def cols(x):             # of x.T: the row quantizer on the transposed copy
        return fp8.quantize_fp8(x.t().contiguous())

    y = mm(rows(ap), cols(bp))[:M, :N]
    da = mm(rows(gp), rows(bp))[:M]
    db = mm(cols(ap), cols(gp))[:, :N]
    return y, da, db


def _inputs(dev, M, K, N, adt, bdt, seed=0, off=0):
    gen = torch.Generator(device=dev).manual_seed(seed + M + K + N)

    def make(r, c, std, dt):
        buf = torch.zeros(r * c + off, dtype=dt, device=dev)
        buf[off:] = (torch.randn(r * c, generator=gen, device=dev) * std).to(dt)
        return buf[off:].reshape(r, c)

    return make(M, K, 1.0, adt), make(K, N, 0.02, bdt), make(M, N, 1e-3, BF)


# tile edges (128), one row or column past and short of them, odd widths, a
# single row and a single column; every pairing of types
@pytest.mark.parametrize("adt,bdt", [(BF, BF), (F32, F32), (F32, BF), (BF, F32)])
@pytest.mark.parametrize("M,K,N", [(1, 128, 1), (127, 128, 130), (129, 384, 257), (300, 256, 128), (128, 128, 1001),
                                   (256, 384, 256), (1000, 640, 520)])
def test_linear_same_bits_as_general_path(dev, M, K, N, adt, bdt):
    a, b, g = _inputs(dev, M, K, N, adt, bdt)
    a.requires_grad_()
    b.requires_grad_()
    y = fp8.block_scaled_matmul(a, b)
    da, db = torch.autograd.grad(y, (a, b), g)
    assert (da.dtype, db.dtype) == (adt, bdt)
    ry, rda, rdb = _general(a.detach(), b.detach(), g)
    assert torch.equal(y, ry) and torch.equal(da, rda.to(adt)) and torch.equal(db, rdb.to(bdt))
    assert torch.equal(fp8._fp8_forward(a.detach(), b.detach(), 128), ry)


@pytest.mark.parametrize("M,K,N", sorted(G.LINEAR_F32))
def test_f32_linear_on_every_tile(dev, M, K, N):
    """The f32 gradients hold the bf16 results, on each tile that a linear's dX and dW take."""
    a, b, g = _inputs(dev, M, K, N, F32, F32)
    da, db = fp8._linear_bwd(a, b, g)
    _, rda, rdb = _general(a, b, g)
    assert torch.equal(da, rda.float()) and torch.equal(db, rdb.float())


@pytest.mark.parametrize("M,N", [(130, 257), (128, 256)])
def test_linear_bwd_from_element_aligned_operands(dev, M, N):
    """tg_linear_bwd takes operands at any element address (odd bf16 offsets included)."""
    a, b, g = _inputs(dev, M, 256, N, BF, BF, off=1)
    da, db = fp8._linear_bwd(a, b, g)
    _, rda, rdb = _general(a, b, g)
    assert torch.equal(da, rda) and torch.equal(db, rdb)


def test_linear_bwd_one_gradient(dev):
    a, b, g = _inputs(dev, 200, 256, 136, BF, F32)
    _, rda, rdb = _general(a, b, g)
    M, K, N = 200, 256, 136
    ws_bytes = L.lib().tg_linear_bwd_workspace(M, N, K)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    for want in ("da", "db"):
        out = torch.full((M, K) if want == "da" else (K, N), 7.0, dtype=BF if want == "da" else F32, device=dev)
        L.check(L.lib().tg_linear_bwd(L.ptr(a), 0, L.ptr(b), 1, L.ptr(g), 0, L.ptr(out) if want == "da" else None,
                                      L.ptr(out) if want == "db" else None, M, N, K, L.ptr(ws), ws_bytes,
                                      L.stream_of(a)))
        assert torch.equal(out, rda if want == "da" else rdb.float())


@pytest.mark.parametrize("dt", [BF, F32])
def test_linear_non_finite_rows_ragged(dev, dt):
    """A NaN and an infinity in a and g: the same positions as the general path."""
    a, b, g = _inputs(dev, 140, 256, 200, dt, dt)
    a[3, 5], a[139, 255], g[7, 199], g[131, 0] = float("nan"), float("inf"), float("nan"), float("-inf")
    da, db = fp8._linear_bwd(a, b, g)
    ry, rda, rdb = _general(a, b, g)
    y = fp8._fp8_forward(a, b, 128)
    for got, ref in ((y, ry), (da, rda), (db, rdb)):
        ok = (got.float() == ref.float()) | (torch.isnan(got.float()) & torch.isnan(ref.float()))
        assert bool(ok.all())


@pytest.mark.parametrize("cols", [1, 3, 130, 2304])
def test_quantize_cols_f32_same_bits_as_rows_of_the_transpose(dev, cols):
    gen = torch.Generator(device=dev).manual_seed(cols)
    x = torch.randn((384, cols), generator=gen, device=dev)
    q, s = fp8.quantize_fp8(x, transpose=True)
    rq, rs = fp8.quantize_fp8(x.t().contiguous())
    assert torch.equal(q.view(torch.uint8), rq.view(torch.uint8)) and torch.equal(s, rs)


@pytest.mark.parametrize("off", [1, 2, 8])
def test_frozen_input_takes_weights_and_gradients_at_any_element(dev, off):
    """Only dW wanted: b and g may start at any element of a flat buffer."""
    M, K, N = 128, 256, 384
    a, b, g = _inputs(dev, M, K, N, BF, BF)

    def at(x):
        flat = torch.empty(x.numel() + off, dtype=x.dtype, device=dev)
        flat[off:].copy_(x.reshape(-1))
        return flat[off:].view(x.shape)

    grads = []
    for bb, gg in ((b, g), (at(b), at(g))):
        w = bb.detach().requires_grad_()
        y = fp8.block_scaled_matmul(a, w)
        y.backward(gg)
        grads.append((y.detach(), w.grad))
    assert torch.equal(grads[0][0], grads[1][0]) and torch.equal(grads[0][1], grads[1][1])
    # beside f32 activations too
    assert torch.equal(fp8._fp8_forward(a.float(), at(b), 128), fp8._fp8_forward(a.float(), b, 128))


# rows of more columns than the ragged kernels' 32-bit offsets reach (2^26), and a column of so many rows (2^29) that
# its tiles pass a 1-D grid: element loads, the bytes of the separate quantizers
def test_quantize_cols_of_very_wide_unaligned_rows(dev):
    cols = (1 << 26) + 3
    x = torch.empty((128, cols), dtype=BF, device=dev).normal_(generator=torch.Generator(device=dev).manual_seed(5))
    q, s = fp8.quantize_fp8(x, transpose=True)
    for c in (0, (1 << 25) + 61, cols - 1024):
        rq, rs = fp8.quantize_fp8(x[:, c:c + 1024].t().contiguous())
        assert torch.equal(q[c:c + 1024].view(torch.uint8), rq.view(torch.uint8)) and torch.equal(s[c:c + 1024], rs)


def test_quantize_cols_of_one_very_long_f32_column(dev):
    x = torch.empty(((1 << 29) + 128, 1), device=dev).normal_(generator=torch.Generator(device=dev).manual_seed(6))
    q, s = fp8.quantize_fp8(x, transpose=True)
    rq, rs = fp8.quantize_fp8(x.reshape(1, -1))
    assert torch.equal(q.view(torch.uint8), rq.view(torch.uint8)) and torch.equal(s, rs)


def test_linear_over_a_very_long_contraction(dev):
    """K past 2^26 in f32, one token and one output: y, da and db against the row quantizers and the GEMM."""
    K = (1 << 26) + 128
    gen = torch.Generator(device=dev).manual_seed(7)
    a, b = (torch.empty(s, device=dev).normal_(generator=gen).requires_grad_() for s in ((1, K), (K, 1)))
    y = fp8.block_scaled_matmul(a, b)
    qa, qb = fp8.quantize_fp8(a.detach()), fp8.quantize_fp8(b.detach().reshape(1, K))
    assert torch.equal(y, fp8.scaled_matmul(qa[0], qa[1], qb[0], qb[1]))
    da, db = torch.autograd.grad(y, (a, b), torch.full((1, 1), 0.5, dtype=BF, device=dev))
    # one value to a block: its code is 448, its scale |value| / 448, so the products are the values themselves
    for got, v in ((da, b), (db, a)):
        want = 0.5 * v.detach().reshape(got.shape)
        assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs()).all())
