"""The fp32 union attention (forward) at the edges of its tiles: group sizes
that fill, split and overflow a 16-column tile, pick lists of one and of
several 64-pick chunks, repeated and invalid picks, sinks past the first
block, windows of one key and of the whole sequence, and keys that are not
finite outside a query's union."""
import math

import pytest
import torch

import hba_amd
from hba_amd import ops

pytestmark = pytest.mark.gpu

#       n   Hq Hkv  d   S    W   k
SHAPES = [
    (64, 2, 2, 64, 0, 1, 1),           # one block, no routed blocks, a window of one key
    (192, 7, 1, 64, 4, 64, 3),         # 2 queries per tile, the last tile's rows past n idle
    (320, 14, 2, 64, 4, 100, 5),
    (320, 4, 4, 64, 64, 64, 5),        # 16 queries per tile: 80 picks, two chunks
    (256, 16, 1, 128, 20, 70, 4),      # a full tile of one query
    (256, 40, 2, 64, 4, 64, 4),        # 20 heads per KV head: two chunks of 10
    (384, 6, 2, 128, 130, 33, 6),      # sinks past block 1; 32-key units
    (320, 5, 1, 64, 4, 1000, 70),      # a window past the sequence; more picks than a chunk
]


def _inputs(n, Hq, Hkv, d, S, W, k, seed=0):
    g = torch.Generator().manual_seed(seed)
    q, kx, v = (torch.randn(2, n, h, d, generator=g) for h in (Hq, Hkv, Hkv))
    gq, gk = (1.5 + 0.1 * torch.randn(h, generator=g) for h in (Hq, Hkv))
    nb = n // 64
    idx = torch.randint(-1, nb + 1, (2, Hkv, n, k), generator=g).to(torch.int32)   # some out of range
    blocks = torch.rand(2, Hkv, n, nb, generator=g).argsort(-1)[..., :k].to(torch.int32)
    idx[..., :blocks.shape[-1]] = torch.where(torch.rand(blocks.shape, generator=g) < 0.8, blocks,
                                              idx[..., :blocks.shape[-1]])
    cnt = torch.randint(-1, k + 2, (2, Hkv, n), generator=g).to(torch.int32)
    return q, kx, v, gq, gk, idx, cnt


def _reference(q, kc, kr, v, gq, eps, cos, sin, idx, cnt, S, W, scale):
    """Dense masked softmax in 64 bits; a block picked twice counts twice."""
    B, n, Hq, d = q.shape
    G = Hq // kc.shape[1]
    x = q.double()
    x = x / x.pow(2).mean(-1, keepdim=True).clamp_min(eps).sqrt() * gq.double()[:, None]
    rot = torch.cat((-x[..., d // 2:], x[..., :d // 2]), -1)
    xr = x * cos.double()[:n, None] + rot * sin.double()[:n, None]
    i, j = torch.arange(n)[:, None], torch.arange(n)[None, :]
    sink, win = (j < S) & (j <= i), (j >= S) & (j <= i) & (j > i - W)
    out = torch.empty(q.shape, dtype=torch.float64)
    nb = n // 64
    for b in range(B):
        for h in range(Hq):
            g = h // G
            mult = torch.zeros(n, nb, dtype=torch.float64)
            ok = (torch.arange(idx.shape[-1]) < cnt[b, g][:, None]) & (idx[b, g] >= 1) & (idx[b, g] < nb)
            mult.scatter_add_(1, idx[b, g].long().clamp(0, nb - 1), ok.double())
            mult = mult.repeat_interleave(64, 1) * (j >= S)
            s = torch.stack((x[b, :, h] @ kc[b, g].double().T, xr[b, :, h] @ kr[b, g].double().T,
                             x[b, :, h] @ kc[b, g].double().T)) * scale
            wgt = torch.stack((sink.double(), win.double(), mult))
            s = torch.where(wgt > 0, s, torch.full_like(s, -math.inf))
            p = (s - s.amax((0, 2), keepdim=True)).exp() * wgt
            vv = torch.where(wgt.sum((0, 1))[:, None] > 0, v[b, :, g].double(), torch.zeros(()).double())
            out[b, :, h] = (p.sum(0) / p.sum((0, 2))[:, None]) @ vv
    return out


def _run(q, kx, v, gq, gk, idx, cnt, S, W):
    n, d = q.shape[1], q.shape[3]
    dev = torch.device("cuda")
    cos, sin = hba_amd.rope_tables(n, d, 10000.0, dev)
    kc, kr, vt = ops.prep_keys(kx.to(dev), v.to(dev), gk.to(dev), 1e-6, cos, sin)
    scale = 1.0 / math.sqrt(d)
    out = ops.attn_fwd(q.to(dev), gq.to(dev), gk.to(dev), 1e-6, kc, kr, vt, cos, sin, idx.to(dev), cnt.to(dev), S, W,
                       scale)
    return out.cpu(), kc.cpu(), kr.cpu(), cos.cpu(), sin.cpu(), scale


@pytest.mark.parametrize("shape", SHAPES)
def test_forward_against_64_bits(shape):
    n, Hq, Hkv, d, S, W, k = shape
    q, kx, v, gq, gk, idx, cnt = _inputs(*shape)
    out, kc, kr, cos, sin, scale = _run(q, kx, v, gq, gk, idx, cnt, S, W)
    ref = _reference(q, kc, kr, v, gq, 1e-6, cos, sin, idx, cnt, S, W, scale)
    # a logit is a sum of d products of rows of norm 1.5 sqrt(d), scaled by
    # d^-0.5: an error of about 2^-24 sqrt(d) * 2.25 sqrt(d) <= 2^-24 * 290 in
    # the exponent at most, 1.7e-5 of a value (in practice a tenth)
    assert (out.double() - ref).norm() <= 2e-6 * ref.norm()
    assert (out.double() - ref).abs().max() <= 1.7e-5 * ref.abs().max()


def test_keys_outside_the_union_are_not_read_into_it():
    """An infinite or NaN value row reaches the queries that attend it, and no
    other query of the same tile."""
    n, Hq, Hkv, d, S, W, k = shape = (320, 7, 1, 64, 4, 64, 2)
    q, kx, v, gq, gk, idx, cnt = _inputs(*shape)
    idx[:] = 0
    cnt[:] = 0
    idx[:, :, 201, 0], cnt[:, :, 201] = 1, 1        # query 201 alone picks block 1
    v[:, 70], v[:, 210] = math.inf, math.nan
    out, kc, kr, cos, sin, scale = _run(q, kx, v, gq, gk, idx, cnt, S, W)
    i = torch.arange(n)
    inf = ((i >= 70) & (i < 70 + W)) | (i == 201)
    nan = (i >= 210) & (i < 210 + W)
    assert (out[:, inf] == math.inf).all() and out[:, nan].isnan().all()
    clean = ~(inf | nan)
    ref = _reference(q, kc, kr, torch.nan_to_num(v, 0.0, 0.0, 0.0), gq, 1e-6, cos, sin, idx, cnt, S, W, scale)
    assert (out[:, clean].double() - ref[:, clean]).norm() <= 2e-6 * ref[:, clean].norm()
