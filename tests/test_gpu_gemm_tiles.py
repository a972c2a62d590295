"""The FP8 GEMM's tile choice changes no bit: every kernel adds a K block's
product in the same order, so an output element is the same whichever tile
computes it.  Each tile is run on shapes of its own (gemm_tiles.py;
test_gemm_tile_choice.py holds them to it) against launches of 32 x 64 tiles;
and a row range of one operand is multiplied alone and as part of taller
launches, at the edges of the 32- and 64-row tiles above all."""
import pytest
import torch

import _tglib as L
import fp8
import gemm_tiles as G

pytestmark = pytest.mark.gpu

ROWS = (1, 31, 32, 33, 65, 129, 255, 500, 1100, 2050)


def _operands(dev, M, N, K, bn):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a, b = (torch.randn(s, generator=g, device=dev).to(torch.float8_e4m3fn).view(torch.uint8) for s in ((M, K), (N, K)))
    sa = torch.rand((M, K // 128), generator=g, device=dev) + 0.5
    sb = torch.rand((N if bn == 1 else -(-N // 128), K // 128), generator=g, device=dev) + 0.5
    return a, sa, b, sb


@pytest.mark.parametrize("bn", [1, 128])
@pytest.mark.parametrize("N,K", [(8, 128), (63, 384), (97, 256), (200, 1280), (1001, 640), (2304, 1152), (3080, 256)])
def test_gemm_bits_do_not_depend_on_the_tile(dev, N, K, bn):
    M = 4100
    a, sa, b, sb = _operands(dev, M, N, K, bn)
    whole = fp8.scaled_matmul(a, sa, b, sb, b_scale_bn=bn)
    whole32 = fp8.scaled_matmul(a, sa, b, sb, b_scale_bn=bn, out_dtype=torch.float32)
    assert torch.equal(whole, whole32.to(torch.bfloat16))
    for m in ROWS:
        part = fp8.scaled_matmul(a[:m], sa[:m], b, sb, b_scale_bn=bn)
        assert torch.equal(part, whole[:m]), m
    m = 777
    part32 = fp8.scaled_matmul(a[M - m:], sa[M - m:], b, sb, b_scale_bn=bn, out_dtype=torch.float32)
    assert torch.equal(part32, whole32[M - m:])
    # the bar of the f32 output against float64 (5e-5 of the largest value: the MFMA's own block sums)
    ad = a.view(torch.float8_e4m3fn).double() * sa.double().repeat_interleave(128, 1)
    bd = b.view(torch.float8_e4m3fn).double() * sb.double().repeat_interleave(bn, 0)[:N].repeat_interleave(128, 1)
    ref = ad @ bd.t().contiguous()
    assert float((whole32.double() - ref).abs().max()) <= 5e-5 * float(ref.abs().max())


def test_gemm_writes_nothing_past_c(dev):
    """Guard bytes after C stay, for widths that end inside a tile and a 16-byte piece."""
    for M, N, K in ((33, 65, 256), (70, 104, 384), (129, 1001, 128), (300, 72, 256)):
        a, sa, b, sb = _operands(dev, M, N, K, 1)
        buf = torch.full((M * N + 64,), 5.0, dtype=torch.bfloat16, device=dev)
        L.check(L.lib().tg_gemm_fp8_nt(a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), 1, buf.data_ptr(), 0,
                                       M, N, K, 128, L.stream_of(a)))
        assert torch.equal(buf[:M * N].reshape(M, N), fp8.scaled_matmul(a, sa, b, sb))
        assert bool((buf[M * N:] == 5.0).all())


@pytest.mark.parametrize("bn", [1, 128])
@pytest.mark.parametrize("M,N,K,km", [c for t in sorted(G.GEMM) for c in G.GEMM[t]])
def test_every_tile_gives_the_bits_of_the_smallest(dev, M, N, K, km, bn):
    """bf16 and f32 outputs of a launch against those of 256 x 512 pieces on 32 x 64 tiles, 64 rows of it against
    float64, and nothing written past C."""
    a, sa, b, sb = _operands(dev, M, N, K, bn)
    fn = L.lib().tg_gemm_fp8_nt_km if km else L.lib().tg_gemm_fp8_nt
    la, lb = (x.t().contiguous() if km else x for x in (sa, sb))
    outs = []
    for code, dt in ((L.TG_DTYPE_BF16, torch.bfloat16), (L.TG_DTYPE_F32, torch.float32)):
        buf = torch.full((M * N + 64,), 5.0, dtype=dt, device=dev)
        L.check(fn(a.data_ptr(), la.data_ptr(), b.data_ptr(), lb.data_ptr(), bn, buf.data_ptr(), code, M, N, K, 128,
                   L.stream_of(a)))
        assert bool((buf[M * N:] == 5.0).all())
        outs.append(buf[:M * N].reshape(M, N))
    c16, c32 = outs
    assert torch.equal(c16, c32.to(torch.bfloat16))
    assert G.tile_of(256, 512, K, False, f32=True) == (32, 64)
    for m in range(0, M, 256):
        for n in range(0, N, 512):
            part = fp8.scaled_matmul(a[m:m + 256], sa[m:m + 256], b[n:n + 512], sb[n // bn:-(-(n + 512) // bn)],
                                     b_scale_bn=bn, out_dtype=torch.float32)
            assert torch.equal(part, c32[m:m + 256, n:n + 512]), (m, n)
    rows = torch.linspace(0, M - 1, 64, device=dev).long()
    ad = a[rows].view(torch.float8_e4m3fn).double() * sa[rows].double().repeat_interleave(128, 1)
    bd = b.view(torch.float8_e4m3fn).double() * sb.double().repeat_interleave(bn, 0)[:N].repeat_interleave(128, 1)
    ref = ad @ bd.t().contiguous()
    assert float((c32[rows].double() - ref).abs().max()) <= 5e-5 * float(ref.abs().max())
