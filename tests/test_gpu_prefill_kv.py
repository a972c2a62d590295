"""tg_prefill_kv: a prompt's k and v in the caches, bit for bit the strided copies."""
import pytest
import torch

import _tglib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,S,Dh", [(1, 1, 1, 1, 8), (1, 5, 3, 7, 128), (3, 17, 4, 17, 32), (2, 130, 18, 256, 128)])
def test_prefill_kv(dev, B, T, H, S, Dh):
    g = torch.Generator(device=dev).manual_seed(B + T + H + Dh)
    qkv = torch.randn((B * T, 3 * H * Dh), generator=g, device=dev).to(torch.bfloat16)
    kc, vc = (torch.full((B + 1, H, S, Dh), 3.0, dtype=torch.bfloat16, device=dev) for _ in range(2))
    L.check(L.lib().tg_prefill_kv(qkv.data_ptr(), kc.data_ptr(), vc.data_ptr(), B, T, H, S, Dh, L.stream_of(qkv)))
    _, k, v = qkv.reshape(B, T, 3, H, Dh).permute(2, 0, 3, 1, 4).unbind(0)
    for c, want in ((kc, k), (vc, v)):
        assert torch.equal(c[:B, :, :T], want)
        assert bool((c[B:] == 3.0).all()) and bool((c[:B, :, T:] == 3.0).all())   # nothing else is written
