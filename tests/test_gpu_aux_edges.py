"""The aux-KL where its kernels change over: candidate counts that fill one,
two and four register rows per lane of aux_rows and pass them, block counts
that are no multiple of 4 or 16, and several batch rows (the teacher's tile
order)."""
import math

import pytest
import torch

import hba_amd
from hba_amd import ops

pytestmark = pytest.mark.gpu


def _reference(q, gq, kc, S0, probes, proj, W, scale):
    """64-bit aux and its gradients into probes and proj.  q is QKNorm'd;
    S0's own values decide nothing here: the summaries are formed from kc."""
    B, n, Hq, d = q.shape
    Hkv, nb = kc.shape[1], n // 64
    G = Hq // Hkv
    x = q.double()
    x = x / x.pow(2).mean(-1, keepdim=True).clamp_min(1e-6).sqrt() * gq.double()[:, None]
    pr, pj = (t.double().requires_grad_(True) for t in (probes, proj))
    blk = torch.arange(nb, device=q.device)
    valid = max(0, n - (2 * 64 + W - 1)) * B * Hkv
    total, grads = 0.0, [torch.zeros_like(pr), torch.zeros_like(pj)]
    for b in range(B):
        for g in range(Hkv):
            kb = kc[b, g].double().view(nb, 64, d)
            att = (kb @ pr[g].T * d ** -0.5).softmax(1)
            S = torch.matmul(torch.matmul(att.transpose(1, 2), kb), pj[g])
            leaf = S.detach().requires_grad_(True)
            step = max(64, (1 << 26) // (n * G))
            for i0 in range(2 * 64 + W - 1, n, step):
                pos = torch.arange(i0, min(n, i0 + step), device=q.device)
                cand = (blk >= 1) & ((blk + 1) * 64 <= (pos - W + 1)[:, None])
                xs = x[b, pos, g * G:(g + 1) * G]
                s = (torch.matmul(xs, kc[b, g].double().T) * scale).view(len(pos), G, nb, 64).logsumexp(-1)
                p = s.masked_fill(~cand[:, None], -math.inf).softmax(-1).mean(1)
                raw = (xs.sum(1) @ leaf.reshape(-1, d).T).view(len(pos), nb, -1).amax(-1) * scale
                logp = raw.masked_fill(~cand, -math.inf).log_softmax(-1)
                term = -(p * torch.where(cand, logp, torch.zeros_like(logp))).sum() / valid
                grads_leaf = torch.autograd.grad(term, leaf)[0]
                leaf.grad = grads_leaf if leaf.grad is None else leaf.grad + grads_leaf
                total += float(term.detach())
            gp, gj = torch.autograd.grad(S, (pr, pj), leaf.grad)
            grads[0] += gp
            grads[1] += gj
    return total, grads


#  n (blocks * 64)   W   B  Hq Hkv  dtype
@pytest.mark.parametrize("nb,W,B,Hq,Hkv,dt", [
    (3, 64, 1, 2, 1, "f32"),            # one candidate block, for one query
    (37, 100, 2, 14, 2, "f32"),
    (37, 100, 2, 14, 2, "bf16"),        # stores of 4 blocks with a remainder
    (259, 64, 1, 2, 1, "bf16"),         # 257 candidates: 8 per lane
    (515, 64, 1, 1, 1, "f32"),          # 513: 16 per lane
    (1027, 64, 1, 1, 1, "bf16"),        # 1025: the passes over L
])
def test_aux_at_its_kernels_edges(nb, W, B, Hq, Hkv, dt):
    n, d, m = 64 * nb, 64, 4
    dev = torch.device("cuda")
    g = torch.Generator(dev).manual_seed(nb)
    t = torch.float32 if dt == "f32" else torch.bfloat16
    q = torch.randn(B, n, Hq, d, generator=g, device=dev).to(t)
    kx = torch.randn(B, n, Hkv, d, generator=g, device=dev).to(t)
    gq, gk = (1.5 + 0.1 * torch.randn(h, generator=g, device=dev) for h in (Hq, Hkv))
    probes = torch.randn(Hkv, m, d, generator=g, device=dev) * d ** -0.5
    proj = torch.eye(d, device=dev) + 0.02 * torch.randn(Hkv, d, d, generator=g, device=dev)
    cos, sin = hba_amd.rope_tables(n, d, 10000.0, dev)
    kc = ops.prep_keys(kx, kx, gk, 1e-6, cos, sin)[0]
    S0 = ops.summarize(kc, probes, proj)
    aux, dpr, dpj = ops.aux_kl(q, gq, gk, 1e-6, kc, S0, probes, proj, W, 1.0 / d, 1.0 / d, True)
    ref, grads = _reference(q, gq, kc, S0, probes, proj, W, 1.0 / d)
    # fp32: logits of |gq| |gk| <= 3.3 with errors of 2^-24 * 64 in the
    # exponents, and a slot chosen by scores that differ by less than the
    # error for about 1e-6 of the rows.  bf16: queries and summaries rounded
    # to 2^-9, and the slots whose scores differ by less than that
    rel = {"f32": (1e-5, 1e-3), "bf16": (1e-2, 1e-1)}[dt]
    assert abs(float(aux) - ref) <= rel[0] * abs(ref)
    for a, r in zip((dpr, dpj), grads):
        assert (a.double() - r).norm() <= rel[1] * r.norm()
