"""Rows of more than 64 chunks (262144 columns): the row statistics come from several 64-chunk groups of one
wave, and the Gumbel merge takes more than one wave. Same oracles as the ordinary widths; chunk counts just
over one group, over two, and the widest row (256 chunks)."""

import pytest
import torch
from test_gpu_sampling import DEV, bf16_logits, check_warp_rows, ops, osm, probs_rows, run_warp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,top_p", [(262148, 0.9), (262148, 1.0), (530001, 0.9), (1048576, 0.8)])
def test_wide_warp_matches_oracle(V, top_p):
    lg = bf16_logits(2, V, 3.0, seed=V)
    check_warp_rows(run_warp(lg, V, 0.8, top_p), lg, V, 0.8, top_p)


@pytest.mark.parametrize("V,k", [(262148, 4), (530001, 16), (1048576, 16), (4096, 16), (4097, 1)])
def test_wide_gumbel_topk_matches_oracle(V, k):
    q = probs_rows(2, V, seed=k, zero_frac=0.5)
    qd = torch.zeros(2, (V + 3) // 4 * 4, device=DEV)
    qd[:, :V] = q.to(DEV)
    tok, lp = torch.zeros(2 * k, dtype=torch.int32, device=DEV), torch.zeros(2 * k, device=DEV)
    ops().gumbel_topk(qd, 2, V, k, 77, 5, tok, lp)
    for r in range(2):
        want, wlp, fragile = osm.gumbel_topk(q[r], k, osm.Stream(77, 5), r, 0)
        if not fragile:
            assert tok.view(2, k)[r].tolist() == want
            torch.testing.assert_close(lp.view(2, k)[r].cpu(), torch.tensor(wlp, dtype=torch.float32), rtol=1e-6, atol=1e-6)
