"""The fp32 flat selection at the edges of its split over waves: fewer
candidate blocks than waves, more query heads than waves, lists of 16, 32 and
64 entries, fewer candidates than picks, all slot counts."""
import numpy as np
import pytest
import torch

import hba_amd
import oracle.hba_oracle as O
from hba_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,W,Hq,Hkv,d,m,k", [
    (2, 64, 2, 1, 64, 4, 2),          # no candidates
    (4, 64, 7, 1, 64, 4, 4),          # two candidates for eight waves
    (21, 64, 20, 1, 64, 1, 16),       # 20 heads per KV head: three rounds of eight
    (40, 100, 4, 2, 64, 2, 17),       # lists of 32: four waves
    (70, 64, 3, 1, 128, 8, 32),
    (80, 64, 2, 2, 128, 4, 64),       # lists of 64: one wave per 64 queries
    (6, 64, 2, 1, 64, 8, 4),          # four candidates for eight waves
    (3, 64, 16, 1, 64, 1, 20),        # one candidate, sixteen heads: four waves
    (64, 64, 16, 16, 64, 1, 9),       # the chip full: one wave per 64 queries, lists of 16
    (64, 64, 16, 16, 64, 1, 20),      # and of 32
])
def test_flat_fp32_selection_is_exact(nb, W, Hq, Hkv, d, m, k):
    n, dev = 64 * nb, torch.device("cuda")
    g = torch.Generator().manual_seed(nb)
    q = torch.randn(2, n, Hq, d, generator=g)
    gain = 1.5 + 0.1 * torch.randn(Hq, generator=g)
    S0 = torch.randn(2, Hkv, nb, m, d, generator=g)
    S0[:, :, 5 % nb] = S0[:, :, 3 % nb]                 # equal scores: the lower block first
    scale = 1.0 / d
    idx, val, cnt, scores = ops.score_select_with_scores(q.to(dev), gain.to(dev), 1e-6, S0.to(dev), W, k, scale)
    plain = ops.score_select(q.to(dev), gain.to(dev), 1e-6, S0.to(dev), W, k, scale)
    assert torch.equal(idx, plain[0]) and torch.equal(val, plain[1]) and torch.equal(cnt, plain[2])
    x = ops.route_queries(q.to(dev), gain.to(dev), 1e-6, Hkv).cpu().numpy()     # [B, n, Hkv, d]
    rows = np.arange(n)
    for b in range(2):
        for h in range(Hkv):
            ref = O.block_scores(x[b, :, h], S0[b, h].numpy(), rows, scale, 64, W)
            got = scores[b, h].cpu().numpy()
            fin = np.isfinite(ref)
            assert np.array_equal(fin, np.isfinite(got)) and np.array_equal(ref[fin], got[fin])
            ti, tv, tc = O.topk(got, k)
            assert np.array_equal(ti, idx[b, h].cpu().numpy()) and np.array_equal(tc, cnt[b, h].cpu().numpy())
            assert np.array_equal(tv, val[b, h].cpu().numpy())
