"""GPU parity of the head's path where the vocabulary is no multiple of 8 (rows
start at any even address): the packs, the bf16 GEMM's stores, the split-K of
the straight-through backward and the capped cross entropy on rows whose
gradient rows are aligned otherwise."""
import numpy as np
import pytest
import torch

import _tglib as L
import fp8
import losses
from helpers import bf16_bits, maxabs_rel, to_dev
from oracle import bf16 as ob
from oracle import fp8_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("transpose", [0, 1])
@pytest.mark.parametrize("rows,cols,off", [(1, 1, 1), (3, 9, 0), (130, 257, 1), (64, 2049, 3), (129, 8200, 2),
                                           (257, 8200, 0), (2, 16391, 1)])
def test_pack_any_even_address(dev, transpose, rows, cols, off):
    """x at an element offset `off` of its allocation, an output pitch of whole
    16-byte pieces: the bits of x, zeros past each row and nothing past y."""
    rng = np.random.default_rng(rows + cols + off)
    want = ob.randn_bf16(rng, (rows, cols))
    buf = torch.zeros(rows * cols + 16, dtype=torch.bfloat16, device=dev)
    x = buf[off:off + rows * cols]
    x.copy_(to_dev(want.reshape(-1), dev))
    want = want.T if transpose else want
    out_rows, width = want.shape
    pitch = -(-width // 64) * 64
    y = torch.full((out_rows * pitch + 64,), 7.0, dtype=torch.bfloat16, device=dev)
    L.check(L.lib().tg_pack_bf16(L.ptr(x), L.TG_DTYPE_BF16, rows, cols, transpose, L.ptr(y), pitch, L.stream_of(x)))
    got = bf16_bits(y[:out_rows * pitch].reshape(out_rows, pitch))
    assert np.array_equal(got[:, :width], want) and np.all(got[:, width:] == 0)
    assert bool((y[out_rows * pitch:] == 7.0).all())


# rows of fewer than 1024 output pieces, packed piece by piece over all rows, up to the edge (8120 -> 1016 pieces; 8184 -> 1024)
@pytest.mark.parametrize("rows,cols,off", [(1, 64, 0), (7782, 64, 1), (5000, 65, 0), (300, 1, 1), (4, 8120, 1), (4, 8184, 1),
                                           (1025, 1023, 0)])
def test_pack_narrow_rows(dev, rows, cols, off):
    test_pack_any_even_address(dev, 0, rows, cols, off)


@pytest.mark.parametrize("M,N,off", [(3, 1, 0), (64, 127, 0), (65, 129, 1), (300, 258, 0), (257, 513, 1)])
def test_gemm_bf16_ragged_rows_of_c(dev, M, N, off):
    """Output rows of any length and any even address: exact integer products,
    and nothing written before or past C."""
    K = 128
    a = ((np.arange(M)[:, None] * 3 + np.arange(K)) % 5 - 2).astype(np.float32)
    b = ((np.arange(N)[:, None] * 5 + 2 * np.arange(K)) % 7 - 3).astype(np.float32)
    ta, tb = to_dev(ob.f32_to_bf16(a), dev), to_dev(ob.f32_to_bf16(b), dev)
    buf = torch.full((M * N + 32,), 9.0, dtype=torch.bfloat16, device=dev)
    c = buf[8 + off:8 + off + M * N]
    L.check(L.lib().tg_gemm_bf16_nt(L.ptr(ta), L.ptr(tb), L.ptr(c), M, N, K, L.stream_of(ta)))
    assert np.array_equal(bf16_bits(c.reshape(M, N)), ob.f32_to_bf16((a @ b.T).astype(np.float32)))
    assert bool((buf[:8 + off] == 9.0).all()) and bool((buf[8 + off + M * N:] == 9.0).all())


# a wave's share of a row: 8, 16, 32 and 64 lanes to a row, one and two values left over, rows that end inside a batch
# of eight stores, and rows that start on a word and between two
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("M", [1, 17, 66, 130])
def test_gemm_bf16_narrow_rows_of_c(dev, M, off):
    K = 64
    for N in (1, 2, 3, 14, 15, 17, 18, 31, 33, 34, 63, 66, 97, 98, 113, 127, 129, 130, 131, 145, 161, 191, 194, 254, 290):
        a = ((np.arange(M)[:, None] * 3 + np.arange(K)) % 5 - 2).astype(np.float32)
        b = ((np.arange(N)[:, None] * 5 + 2 * np.arange(K)) % 7 - 3).astype(np.float32)
        ta, tb = to_dev(ob.f32_to_bf16(a), dev), to_dev(ob.f32_to_bf16(b), dev)
        buf = torch.full((M * N + 32,), 9.0, dtype=torch.bfloat16, device=dev)
        c = buf[8 + off:8 + off + M * N]
        L.check(L.lib().tg_gemm_bf16_nt(L.ptr(ta), L.ptr(tb), L.ptr(c), M, N, K, L.stream_of(ta)))
        assert np.array_equal(bf16_bits(c.reshape(M, N)), ob.f32_to_bf16((a @ b.T).astype(np.float32))), N
        assert bool((buf[:8 + off] == 9.0).all()) and bool((buf[8 + off + M * N:] == 9.0).all()), N


# 192-wide tiles (few of them) at their edges, and 256-wide ones (a whole round);
# 2, 6 and 10 slices of the four-stage ring
@pytest.mark.parametrize("M,N,K", [(1, 192, 64), (255, 191, 64), (256, 200, 192), (257, 193, 192), (130, 384, 320),
                                   (300, 576, 64), (4096, 4096, 64), (4090, 4089, 64)])
def test_gemm_bf16_tile_widths(dev, M, N, K):
    """Exact integer products, every value of C written and nothing past it."""
    a = ((np.arange(M)[:, None] * 3 + np.arange(K)) % 5 - 2).astype(np.float32)
    b = ((np.arange(N)[:, None] * 5 + 2 * np.arange(K)) % 7 - 3).astype(np.float32)
    ta, tb = to_dev(ob.f32_to_bf16(a), dev), to_dev(ob.f32_to_bf16(b), dev)
    buf = torch.full((M * N + 64,), 0.5, dtype=torch.bfloat16, device=dev)
    L.check(L.lib().tg_gemm_bf16_nt(L.ptr(ta), L.ptr(tb), L.ptr(buf), M, N, K, L.stream_of(ta)))
    assert np.array_equal(bf16_bits(buf[:M * N].reshape(M, N)), ob.f32_to_bf16((a @ b.T).astype(np.float32)))
    assert bool((buf[M * N:] == 0.5).all())


# dX contracts N, dW contracts M: each splits where its 256 x 256 tiles are few
# and the contraction long (down to 16 slices of 32 per split, a last split shorter)
@pytest.mark.parametrize("M,K,N", [(33, 256, 5001), (2049, 128, 72), (700, 384, 1025), (4100, 256, 264),
                                   (1024, 128, 1024)])
def test_bf16_backward_split_contractions(dev, M, K, N):
    rng = np.random.default_rng(M + N)
    a = ob.randn_bf16(rng, (M, K))
    b = ob.randn_bf16(rng, (K, N), std=0.02)
    g = ob.randn_bf16(rng, (M, N), std=1e-3)
    ta, tb, tg = to_dev(a, dev), to_dev(b, dev), to_dev(g, dev)
    da, db = fp8._bf16_backward(ta, tb, tg)
    again = fp8._bf16_backward(ta, tb, tg)
    assert torch.equal(da, again[0]) and torch.equal(db, again[1])
    rda, rdb = fp8_ref.fp8_backward_bf16(a, b, g)
    sda, sdb = fp8_ref.fp8_backward_bf16(a & 0x7FFF, b & 0x7FFF, g & 0x7FFF)
    for got, ref, s, k in ((da, rda, sda, N), (db, rdb, sdb, M)):
        assert maxabs_rel(got, ref) <= 1e-2
        # one bf16 rounding and an fp32 accumulation over k terms
        bound = np.abs(ref) * 2.0 ** -8 + k * 2.0 ** -23 * s
        assert np.all(np.abs(got.float().cpu().numpy().astype(np.float64) - ref) <= bound)


@pytest.mark.parametrize("cap", [15.0, 40.0])
@pytest.mark.parametrize("R,V", [(4, 50257), (3, 9), (2, 4097)])
def test_xent_rows_offset_from_their_gradient(dev, cap, R, V):
    """Logits one row into an odd-width buffer: they start 2 bytes off the
    gradient's alignment, and give the values of an aligned copy to f32 rounding."""
    g = torch.Generator(device=dev).manual_seed(V)
    buf = (torch.randn((R + 1, V), generator=g, device=dev) * 4).to(torch.bfloat16)
    tgt = torch.randint(0, V, (R,), generator=g, device=dev)
    tgt[0], tgt[-1] = 0, V - 1
    outs = []
    for l in (buf[1:].detach(), buf[1:].clone()):
        l.requires_grad_(True)
        nll, lse = losses.capped_cross_entropy_rows(l.detach(), tgt, cap)
        loss = losses.capped_cross_entropy(l, tgt, cap)
        (dl,) = torch.autograd.grad(loss, (l,))
        outs.append((nll, lse, dl.float()))
    for x, y in zip(*outs):
        # f32 sums of up to V terms in another order, and one bf16 rounding that they may move
        assert bool(((x - y).abs() <= 2.0 ** -8 * y.abs() + 1e-5 * y.abs().max()).all())
