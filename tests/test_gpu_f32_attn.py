"""The fp32 union attention (forward and backward) at the edges of its tiles: group sizes
that fill, split and overflow a 16-column tile, pick lists of one and of
several 64-pick chunks, repeated and invalid picks, sinks past the first
block, windows of one key and of the whole sequence, and keys that are not
finite outside a query's union."""
import ctypes
import math

import pytest
import torch

import hba_amd
from hba_amd import _lib, ops

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


def _norm_rope(x, gain, eps, cos, sin):
    d = x.shape[-1]
    x = x / x.pow(2).mean(-1, keepdim=True).clamp_min(eps).sqrt() * gain[:, None]
    rot = torch.cat((-x[..., d // 2:], x[..., :d // 2]), -1)
    return x, x * cos[:, None] + rot * sin[:, None]


def _unique(idx, n):
    """Repeated picks of a row become out-of-range ones."""
    for t in range(1, idx.shape[-1]):
        idx[..., t][(idx[..., :t] == idx[..., t:t + 1]).any(-1)] = n // 64
    return idx


def _grads(q, kx, v, gq, gk, idx, cnt, dout, S, W, scale, cos, sin):
    """64-bit gradients of q, k, v and the gains."""
    B, n, Hq, d = q.shape
    G, nb = Hq // kx.shape[2], n // 64
    leaf = [t.double().requires_grad_(True) for t in (q, kx, v, gq, gk)]
    x, xr = _norm_rope(leaf[0], leaf[3], 1e-6, cos, sin)
    y, yr = _norm_rope(leaf[1], leaf[4], 1e-6, cos, sin)
    i, j = torch.arange(n)[:, None], torch.arange(n)[None, :]
    sink, win = (j < S) & (j <= i), (j >= S) & (j <= i) & (j > i - W)
    ok = (torch.arange(idx.shape[-1]) < cnt[..., None]) & (idx >= 1) & (idx < nb)
    routed = torch.zeros(B, kx.shape[2], n, nb).scatter_add_(-1, idx.long().clamp(0, nb - 1), ok.float()) > 0
    routed = routed.repeat_interleave(64, -1) & (j >= S)
    total = 0.0
    for b in range(B):
        for h in range(Hq):
            g = h // G
            s = torch.cat((x[b, :, h] @ y[b, :, g].T, xr[b, :, h] @ yr[b, :, g].T), -1) * scale
            # a key in the window and in a routed block counts in both frames
            s = torch.cat((s, s[:, :n]), -1)
            p = s.masked_fill(~torch.cat((sink, win, routed[b, g]), -1), -math.inf).softmax(-1)
            o = (p[:, :n] + p[:, n:2 * n] + p[:, 2 * n:]) @ leaf[2][b, :, g]
            total = total + (o * dout[b, :, h].double()).sum()
    return torch.autograd.grad(total, leaf)


def _run_bwd(q, kx, v, gq, gk, idx, cnt, dout, S, W):
    dev = torch.device("cuda")
    n, d = q.shape[1], q.shape[3]
    cos, sin = hba_amd.rope_tables(n, d, 10000.0, dev)
    scale = 1.0 / math.sqrt(d)
    t = [x.to(dev) for x in (q, kx, v, gq, gk, idx, cnt, dout)]
    kc, kr, vt = ops.prep_keys(t[1], t[2], t[4], 1e-6, cos, sin)
    out = ops.attn_fwd(t[0], t[3], t[4], 1e-6, kc, kr, vt, cos, sin, t[5], t[6], S, W, scale)
    got = ops.attn_bwd(t[0], t[1], t[2], kc, kr, t[3], t[4], 1e-6, cos, sin, t[5], t[6], out, t[7], S, W, scale)
    return [x.cpu() for x in got], scale, cos.cpu().double(), sin.cpu().double()


#           n    Hq Hkv  d   S   W   k
BWD_SHAPES = [s for s in SHAPES if s[4] <= 64 and s[6] <= 64 and s[1] // s[2] <= 16] + [
    (832, 3, 1, 64, 17, 300, 4),       # 5 queries per tile, two sink waves, 13 ranges of 64 rows
    (2112, 2, 1, 64, 4, 130, 3),       # 17 ranges of 128 rows, the last one ragged
    (4608, 2, 2, 64, 4, 70, 3),        # one head per KV head, 18 ranges of 256 rows
]


@pytest.mark.parametrize("shape", BWD_SHAPES)
def test_backward_against_64_bits(shape):
    n, Hq, Hkv, d, S, W, k = shape
    q, kx, v, gq, gk, idx, cnt = _inputs(*shape)
    if n > 1024:
        q, kx, v, idx, cnt = q[:1], kx[:1], v[:1], idx[:1], cnt[:1]
    idx = _unique(idx, n)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(5))
    got, scale, cos, sin = _run_bwd(q, kx, v, gq, gk, idx, cnt, dout, S, W)
    ref = _grads(q, kx, v, gq, gk, idx, cnt, dout, S, W, scale, cos, sin)
    # p carries the logits' error of 1.7e-5 at most (see above) and dS = p (dP
    # - D) cancels to about 1 / sqrt(keys) of its terms; a row with few keys
    # keeps the sums' 2^-24 sqrt(terms).  In practice a tenth of this
    for name, a, r in zip(("dq", "dk", "dv", "dgq", "dgk"), got, ref):
        # rows that attend a single key have dS = 0 but for the rounding of dP
        # - D, 2^-24 sqrt(d) |dO| |v| <= 1e-5 per element; the gains sum n rows
        floor = 1e-5 * math.sqrt(r.numel()) * (math.sqrt(n * Hq / Hkv) if r.dim() == 1 else 1.0)
        assert (a.double() - r).norm() <= 1e-5 * r.norm() + floor, name


def test_backward_rows_outside_the_union_are_not_read_into_it():
    """A NaN cotangent row reaches the keys it attends and a NaN key the
    queries that attend it, and nothing else of their tiles."""
    n, Hq, Hkv, d, S, W, k = shape = (320, 7, 1, 64, 4, 64, 2)
    q, kx, v, gq, gk, idx, cnt = _inputs(*shape)
    idx[:], cnt[:] = 0, 0
    idx[:, :, 201, 0], cnt[:, :, 201] = 1, 1        # query 201 alone picks block 1
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(5))
    bad = dout.clone()
    bad[:, 201] = math.nan
    got, scale, cos, sin = _run_bwd(q, kx, v, gq, gk, idx, cnt, bad, S, W)
    ref = _grads(q, kx, v, gq, gk, idx, cnt, dout.index_fill(1, torch.tensor([201]), 0.0), S, W, scale, cos, sin)
    j = torch.arange(n)
    hit = (j < S) | ((j > 201 - W) & (j <= 201)) | ((j >= 64) & (j < 128))
    for a, r, sel in ((got[0], ref[0], j == 201), (got[1], ref[1], hit), (got[2], ref[2], hit)):
        assert a[:, sel].isnan().all()
        assert (a[:, ~sel].double() - r[:, ~sel]).norm() <= 1e-5 * r.norm()
    kb = kx.clone()
    kb[:, 70] = math.nan                            # key 70: block 1, and the window of 70 .. 133
    got = _run_bwd(q, kb, v, gq, gk, idx, cnt, dout, S, W)[0]
    sel = ((j >= 70) & (j < 70 + W)) | (j == 201)
    assert got[0][:, sel].isnan().all() and got[0][:, ~sel].isfinite().all()


def test_backward_takes_rows_off_16_byte_boundaries():
    """Contiguous fp32 tensors that begin 4 bytes past a 16-byte boundary."""
    n, Hq, Hkv, d, S, W, k = shape = (192, 7, 1, 64, 4, 64, 3)
    q, kx, v, gq, gk, idx, cnt = _inputs(*shape)
    idx = _unique(idx, n)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(5))
    dev = torch.device("cuda")
    cos, sin = hba_amd.rope_tables(n, d, 10000.0, dev)
    t = [x.to(dev) for x in (q, kx, v, gq, gk, idx, cnt, dout)]
    kc, kr, vt = ops.prep_keys(t[1], t[2], t[4], 1e-6, cos, sin)
    out = ops.attn_fwd(t[0], t[3], t[4], 1e-6, kc, kr, vt, cos, sin, t[5], t[6], S, W, 0.125)

    def off(x):
        y = torch.empty(x.numel() + 1, dtype=x.dtype, device=dev)[1:].view(x.shape)
        return y.copy_(x)
    run = lambda f: ops.attn_bwd(f(t[0]), f(t[1]), f(t[2]), f(kc), f(kr), t[3], t[4], 1e-6, f(cos), f(sin), t[5], t[6],
                                 f(out), f(t[7]), S, W, 0.125)
    for a, b in zip(run(lambda x: x), run(off)):
        assert (a - b).norm() <= 1e-6 * a.norm()       # the atomic sums' order
    # the C entry, which takes them as they are
    for a, b in zip(_c_bwd(t, kc, kr, cos, sin, out, shape), _c_bwd([off(x) if x.dtype == torch.float32 else x for x in t],
                                                                    off(kc), off(kr), off(cos), off(sin), off(out), shape)):
        assert torch.equal(a, b)


def _c_bwd(t, kc, kr, cos, sin, out, shape, nbytes=None):
    """dq, dk and dv of hba_attn_bwd itself; gradients in memory aligned like the inputs."""
    n, Hq, Hkv, d, S, W, k = shape
    lib, dev, dt = _lib.lib(), kc.device, 0 if kc.dtype == torch.float32 else 1
    if nbytes is None:
        b = ctypes.c_size_t(0)
        assert lib.hba_attn_bwd_workspace_bytes(dt, t[0].shape[0], n, Hq, Hkv, d, ctypes.byref(b)) == 0
        nbytes = b.value
    g = [torch.full((x.numel() + 8,), math.nan, dtype=x.dtype, device=dev)
         [x.data_ptr() % 16 // x.element_size():][:x.numel()].view(x.shape) for x in t[:3]]
    gg = [torch.zeros(h, device=dev) for h in (Hq, Hkv)]
    ws = torch.full((nbytes,), 255, dtype=torch.uint8, device=dev)
    p = lambda x: None if x is None else x.data_ptr()
    st = lib.hba_attn_bwd(dt, p(t[0]), p(t[1]), p(t[2]), p(kc), p(kr), p(t[3]), p(t[4]), 1e-6, p(cos), p(sin), p(t[5]),
                          p(t[6]), p(out), p(t[7]), t[0].shape[0], n, Hq, Hkv, d, S, W, 64, k, 0.125, p(ws), nbytes,
                          *(p(x) for x in g + gg), torch.cuda.current_stream().cuda_stream)
    assert st == 0
    return g


def _bwd_args(shape, dev, dt=torch.float32, gains=True):
    n, Hq, Hkv, d, S, W, k = shape
    q, kx, v, gq, gk, idx, cnt = (x[:1] if x.dim() > 1 else x for x in _inputs(*shape))
    q, kx, v = (x.to(dt) for x in (q, kx, v))
    idx = _unique(idx, n)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(5)).to(dt)
    cos, sin = hba_amd.rope_tables(n, d, 10000.0, dev)
    t = [x.to(dev) for x in (q, kx, v, gq, gk, idx, cnt, dout)]
    if not gains:
        t[3] = t[4] = None
    kc, kr, vt = ops.prep_keys(t[1], t[2], t[4], 1e-6, cos, sin)
    out = ops.attn_fwd(t[0], t[3], t[4], 1e-6, kc, kr, vt, cos, sin, t[5], t[6], S, W, 0.125)
    return t, kc, kr, cos, sin, out


def test_backward_of_long_ranges_against_the_generic_kernels():
    """17 ranges of 512 rows: two passes over the picks of each.  More than 64
    picks per row, here unused ones, take the generic kernels."""
    n, Hq, Hkv, d, S, W, k = shape = (8448, 2, 1, 64, 17, 300, 3)
    t, kc, kr, cos, sin, out = _bwd_args(shape, torch.device("cuda"))
    run = lambda idx: ops.attn_bwd(t[0], t[1], t[2], kc, kr, t[3], t[4], 1e-6, cos, sin, idx, t[6].clamp(max=k), out,
                                   t[7], S, W, 0.125)
    gen = run(torch.nn.functional.pad(t[5], (0, 65 - k), value=-1))
    for name, a, b in zip(("dq", "dk", "dv"), run(t[5]), gen):
        assert (a - b).norm() <= 1e-5 * b.norm(), name      # the bound of the 64-bit test, for either side


#                                    n     Hq Hkv d   S   W    k
@pytest.mark.parametrize("gains", [True, False])
@pytest.mark.parametrize("shape", [(2112, 6, 2, 64, 20, 130, 3), (832, 2, 1, 128, 4, 1000, 5), (192, 7, 1, 64, 0, 64, 3)])
def test_backward_is_the_same_bits_from_run_to_run_and_with_any_workspace(shape, gains, monkeypatch):
    """dq, dk and dv of two runs, of a workspace with places for no, for three
    and for all ranges of query rows, and of the op when memory is out."""
    n, Hq, Hkv, d, S, W, k = shape
    dev = torch.device("cuda")
    t, kc, kr, cos, sin, out = _bwd_args(shape, dev, gains=gains)
    lib, ws = _lib.lib(), {}
    for name in ("bytes", "full_bytes"):
        b = ctypes.c_size_t(0)
        assert getattr(lib, "hba_attn_bwd_workspace_" + name)(0, 1, n, Hq, Hkv, d, ctypes.byref(b)) == 0
        ws[name] = b.value
    place = Hkv * (n // 64 + 1) * 4 * (128 * d + 4)
    assert ws["full_bytes"] - ws["bytes"] == -(-n // (128 if n > 2048 else 64)) * place

    op = lambda: ops.attn_bwd(t[0], t[1], t[2], kc, kr, t[3], t[4], 1e-6, cos, sin, t[5], t[6], out, t[7], S, W, 0.125)[:3]
    want = op()
    assert all(x.isfinite().all() for x in want)
    empty, asked = torch.empty, []

    def out_of_memory(*a, **kw):
        if kw.get("dtype") == torch.uint8:
            asked.append(a[0])
            if a[0] == ws["full_bytes"]:
                raise torch.OutOfMemoryError("no room")
        return empty(*a, **kw)
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", out_of_memory)
        assert all(torch.equal(a, b) for a, b in zip(op(), want))
    assert asked == [ws["full_bytes"], ws["bytes"]]
    for nbytes in (ws["full_bytes"], ws["full_bytes"], ws["bytes"] + 3 * place + 64, ws["bytes"]):
        for name, a, b in zip(("dq", "dk", "dv"), _c_bwd(t, kc, kr, cos, sin, out, shape, nbytes), want):
            assert torch.equal(a, b), (name, nbytes)


@pytest.mark.parametrize("d", [64, 128])
def test_bf16_backward_takes_rows_off_16_byte_boundaries(d, monkeypatch):
    """Keys and values 8 bytes past a boundary: the C entry's query gradient by
    the kernel without 16-byte copies into LDS, the op's by the one with them."""
    n, Hq, Hkv, d, S, W, k = shape = (192, 7, 1, d, 4, 64, 3)
    dev = torch.device("cuda")
    t, kc, kr, cos, sin, out = _bwd_args(shape, dev, torch.bfloat16)

    def off(x):
        y = torch.empty(x.numel() + 4, dtype=x.dtype, device=dev)[4:].view(x.shape)
        return y.copy_(x)
    moved = [off(x) if x.dtype == torch.bfloat16 else x for x in t]
    run = lambda t, kc, kr: ops.attn_bwd(t[0], t[1], t[2], kc, kr, t[3], t[4], 1e-6, cos, sin, t[5], t[6], out, t[7], S, W,
                                         0.125)[0]
    assert torch.equal(run(t, kc, kr), run(moved, off(kc), off(kr)))
    got = _c_bwd(moved, off(kc), off(kr), cos, sin, out, shape)
    monkeypatch.setenv("HBA_BWD_DQ_KERNEL", "pair")
    pair = _c_bwd(t, kc, kr, cos, sin, out, shape)
    assert torch.equal(got[0], pair[0])
    for a, b in zip(got[1:], pair[1:]):      # fp32 sums in any order, stored in bf16
        assert (a.float() - b.float()).norm() <= 1e-2 * b.float().norm()
