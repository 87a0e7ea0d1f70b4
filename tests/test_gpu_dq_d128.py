"""The bf16 query gradient at head dim 128 (16-query workgroups of 8 row
tiles): group sizes that fill and split a row tile, ragged last workgroups,
sinks from none to a block, the fixed and the running softmax shift."""
import math
import os

import pytest
import torch

import hba_amd
from hba_amd import ops
from test_gpu_f32_attn import _grads, _inputs, _unique

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,Hq,Hkv,S,W,k,gain", [
    (64, 1, 1, 0, 1, 1, 1.5),
    (320, 7, 1, 4, 100, 3, 1.5),
    (192, 16, 1, 64, 64, 3, 1.5),      # one query per row tile
    (448, 10, 2, 17, 1000, 6, 1.5),    # 3 queries per row tile; a window past the sequence
    (320, 8, 2, 4, 70, 5, 9.0),        # logits past the fixed shift's bound
])
def test_query_gradient_d128(n, Hq, Hkv, S, W, k, gain):
    d, dev = 128, torch.device("cuda")
    q, kx, v, gq, gk, idx, cnt = _inputs(n, Hq, Hkv, d, S, W, k)
    gq, gk = gq * (gain / 1.5), gk
    q, kx, v = (t.bfloat16() for t in (q, kx, v))
    idx = _unique(idx, n)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(5)).bfloat16()
    cos, sin = hba_amd.rope_tables(n, d, 10000.0, dev)
    scale = 1.0 / math.sqrt(d)
    t = [x.to(dev) for x in (q, kx, v, gq, gk, idx, cnt, dout)]
    kc, kr, vt = ops.prep_keys(t[1], t[2], t[4], 1e-6, cos, sin)
    out = ops.attn_fwd(t[0], t[3], t[4], 1e-6, kc, kr, vt, cos, sin, t[5], t[6], S, W, scale)
    run = lambda: ops.attn_bwd(t[0], t[1], t[2], kc, kr, t[3], t[4], 1e-6, cos, sin, t[5], t[6], out, t[7], S, W, scale)
    got = run()
    os.environ["HBA_BWD_DQ_KERNEL"] = "pair"
    try:
        pair = run()
    finally:
        del os.environ["HBA_BWD_DQ_KERNEL"]
    ref = _grads(q, kx, v, gq, gk, idx, cnt, dout, S, W, scale, cos.cpu().double(), sin.cpu().double())
    # bf16 rows and keys: an error of 2^-9 |q| |k| scale in a logit, about 1 %
    # of a probability at gains of 1.5, six times that at 9; the gains' sums
    # over all rows cancel (see the oracle gates of the backward)
    f = gain / 1.5
    for name, a, b, r, tol in zip(("dq", "dk", "dv", "dgq", "dgk"), got, pair, ref, (2e-2, 2e-2, 1e-2, 6e-2, 6e-2)):
        big = max(r.abs().max().item(), 0.05)
        assert (a.cpu().double() - r).abs().max().item() <= tol * f * big, name
        assert (a.double() - b.double()).abs().max().item() <= tol * f * big, name
