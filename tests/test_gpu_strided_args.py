"""Ops on non-contiguous arguments, several of one shape in a call: slices of
one packed tensor give what contiguous copies of them give, bit for bit."""
import pytest
import torch

import hba_amd
from hba_amd import ops

pytestmark = pytest.mark.gpu

EPS = 1e-6


def _packed(*ts):
    """Views of the tensors in one packed tensor, none of them contiguous."""
    out = torch.stack(ts, -2).unbind(-2)
    assert not any(t.is_contiguous() for t in out)
    return out


def _rows(n, Hkv, d, dt, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(1, n, h, d, generator=g).to(dt).cuda() for h in (3 * Hkv, Hkv, Hkv)]


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_append_of_slices_of_one_tensor(dt):
    Bd, Hkv, d = 3, 2, 64
    g = torch.Generator().manual_seed(1)
    k, v = (torch.randn(Bd, Hkv, d, generator=g).to(dt).cuda() for _ in range(2))
    gain = torch.full((Hkv,), 1.5, device="cuda")
    cos, sin = hba_amd.rope_tables(64, d, 10000.0, torch.device("cuda"))
    table = torch.arange(Bd, dtype=torch.int32, device="cuda")[:, None]
    probes, proj = torch.randn(Hkv, 2, d, device="cuda"), torch.randn(Hkv, d, d, device="cuda")

    def run(op, k, v):
        pages = [torch.zeros(Bd, Hkv, 64 * d, dtype=dt, device="cuda") for _ in range(3)]
        lens = torch.tensor([5, 0, 62], dtype=torch.int32, device="cuda")
        if op is ops.kv_append:
            op(k, v, gain, EPS, cos, sin, table, lens + 1, *pages)
        else:
            op(k, v, gain, EPS, cos, sin, table, lens, *pages, probes, proj,
               torch.zeros(Bd, Hkv, 2, d, dtype=dt, device="cuda"), torch.ones(65, device="cuda"),
               torch.zeros(Bd, device="cuda"))
        return pages
    for op in (ops.kv_append, ops.kv_append_advance):
        for a, b in zip(run(op, k, v), run(op, *_packed(k, v))):
            assert a.any() and torch.equal(a, b)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_attention_of_slices_of_one_tensor(dt):
    n, Hkv, d, S, W, scale = 256, 2, 64, 4, 64, 0.125
    q, k, v = _rows(n, Hkv, d, dt, 2)
    qg, kg = (torch.full((h,), 1.5, device="cuda") for h in (3 * Hkv, Hkv))
    cos, sin = hba_amd.rope_tables(n, d, 10000.0, torch.device("cuda"))
    kc, kr, vt = ops.prep_keys(k, v, kg, EPS, cos, sin)
    idx = torch.full((1, Hkv, n, 2), -1, dtype=torch.int32, device="cuda")
    idx[:, :, 192:, 0] = 1
    cnt = (idx >= 0).sum(-1).to(torch.int32)

    def run(kc, kr, vt):
        outs = [ops.attn_fwd(q, qg, kg, EPS, kc, kr, vt, cos, sin, idx, cnt, S, W, scale)]
        if dt == torch.bfloat16:
            out, ws = ops.attn_buffers(q, Hkv)
            ops.attn_window_(q, qg, kg, EPS, kr, vt, cos, sin, S, W, scale, out, ws)
            outs.append(ops.attn_routed_(q, qg, kg, EPS, kc, vt, idx, cnt, S, scale, out, ws))
        return outs
    for a, b in zip(run(kc, kr, vt), run(*_packed(kc, kr), _packed(vt, vt)[0])):
        assert torch.equal(a, b)
