"""The bf16 window launch in both tile orders: windows up to half of the
sequence (an eighth of the tiles per XCD) and past it (deepest tiles first), for
KV head counts that divide 8, are multiples of it, or neither."""
import pytest
import torch

import hba_amd
from hba_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,d", [(4, 2, 64), (6, 3, 64), (8, 8, 128), (1, 1, 128)])
def test_window_launch_in_both_tile_orders(Hq, Hkv, d):
    n, S, scale, dev = 704, 3, d ** -0.5, torch.device("cuda")
    g = torch.Generator().manual_seed(d + Hkv)
    q, k, v = (torch.randn(1, n, h, d, generator=g).bfloat16().cuda() for h in (Hq, Hkv, Hkv))
    qg, kg = (torch.full((h,), 1.5, device="cuda") for h in (Hq, Hkv))
    cos, sin = hba_amd.rope_tables(n, d, 10000.0, dev)
    kc, kr, vt = ops.prep_keys(k, v, kg, 1e-6, cos, sin)
    none = torch.zeros(1, Hkv, n, dtype=torch.int32, device="cuda")

    def window(W):
        out, ws = ops.attn_buffers(q, Hkv)
        return ops.attn_window_(q, qg, kg, 1e-6, kr, vt, cos, sin, 0, W, scale, out, ws)
    for W in (1, n // 2, n // 2 + 1, n - 1, n):
        f = [x.float() for x in (q, kc, kr, vt)]
        ref = ops.attn_fwd(f[0], qg, kg, 1e-6, *f[1:], cos, sin, none[..., None], none, 0, W, scale)
        # rows of norm 1.5 sqrt(d) rounded to bf16: 2^-9 * 2.25 sqrt(d) in a logit at most
        assert (window(W).float() - ref).abs().max() <= 2.25 * d ** 0.5 * 2 ** -8 * ref.abs().max(), W
    assert torch.equal(window(n), window(2 ** 63 - 1))        # longer than any sequence
