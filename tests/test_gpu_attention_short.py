"""Short contexts on the one-launch attention kernel, and the split of the shared superblocks over row tiles.

l_max decides the kernel: the same rows called with a larger l_max take the two launches (blocks past a row's
keys contribute nothing), and must come out with the same bits; a row may not depend on its neighbours either.
The values are pinned by the fp32 oracle: fp16 superblock outputs and a bf16 result, 2^-8 relative each step,
and P rounded to bf16 before P V (2^-9 of the largest |v|, under 5 here)."""

import random

import pytest
import torch

from oracle import kernels as ok

pytestmark = pytest.mark.gpu
DEV = "cuda"
CAP = 2048


def _case(m, heads, kvh, hd, L, seed):
    g = torch.Generator().manual_seed(seed)
    rng = random.Random(seed)
    q = torch.randn(m, heads, hd, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(kvh, CAP, hd, generator=g).to(torch.bfloat16) for _ in range(2))
    prefix, anc = [], []
    for t in range(m):
        d = 0 if t == 0 else min(rng.choice([0, 1, 5, 32]), L)
        prefix.append(L - d if t % 3 else rng.randint(1 if d == 0 else 0, L - d))
        anc.append(sorted(rng.sample(range(CAP), d)))
    return q, k, v, prefix, anc


def _call(case, rows, p_min, l_max, ws=None):
    from ssd import ops

    q, k, v, prefix, anc = case
    heads, hd, kvh, m = q.shape[1], q.shape[2], k.shape[0], len(rows)
    an = torch.zeros(m, 32, dtype=torch.int32)
    for i, t in enumerate(rows):
        an[i, :len(anc[t])] = torch.tensor(anc[t], dtype=torch.int32)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    ws = torch.zeros(ops.attn_workspace_floats(m, heads, hd, CAP), device=DEV) if ws is None else ws
    out = torch.full((m, heads * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    qd = q[rows].reshape(m, heads * hd).to(DEV)
    ops.tree_attention(qd, m, heads, kvh, hd, ops.kv_tile(k.to(DEV), "k"), ops.kv_tile(v.to(DEV), "v"), CAP,
                       i32([prefix[t] for t in rows]), i32([len(anc[t]) for t in rows]), an.to(DEV), p_min, l_max,
                       ws, out)
    return out.view(m, heads, hd).cpu()


# 48 q heads per kv head: three 16-row tiles; 64 rows at 8 kv heads: more workgroups than fit at once
@pytest.mark.parametrize("hd,heads,kvh,m", [(32, 8, 4, 5), (64, 32, 8, 25), (64, 48, 1, 3), (128, 32, 8, 9),
                                            (128, 64, 8, 40), (64, 32, 8, 64), (128, 32, 8, 64)])
@pytest.mark.parametrize("L", [1, 33, 64, 65, 255, 256, 257, 512, 513, 768, 1024, 1025])
def test_one_launch_matches_two(hd, heads, kvh, m, L):
    case = _case(m, heads, kvh, hd, L, seed=L + hd + m)
    rows = list(range(m))
    got = _call(case, rows, 0, L)
    assert torch.equal(got, _call(case, rows, 0, CAP))
    assert torch.equal(got, _call(case, rows, min(case[3]), L))
    some = [0, m - 1, m // 2]
    assert torch.equal(got[some], _call(case, some, 0, L))
    q, k, v, prefix, anc = case
    want = ok.tree_attention(q[some], k, v, [prefix[t] for t in some], [anc[t] for t in some]).float()
    assert ((got[some].float() - want).abs() <= 3 * 2 ** -8 * want.abs() + 2 ** -9 * 5).all()


@pytest.mark.parametrize("hd,heads,kvh", [(64, 32, 8), (128, 64, 8), (128, 8, 1)])
@pytest.mark.parametrize("m", [33, 40, 64])
@pytest.mark.parametrize("P", [520, 1100, 1900])
def test_tile_groups_leave_the_rows_alone(hd, heads, kvh, m, P):
    g = torch.Generator().manual_seed(P + m)
    rng = random.Random(P + m)
    q = torch.randn(m, heads, hd, generator=g).to(torch.bfloat16)
    k, v = (torch.randn(kvh, CAP, hd, generator=g).to(torch.bfloat16) for _ in range(2))
    case = (q, k, v, [P] * m, [sorted(rng.sample(range(P, CAP), 1 + t % 8)) for t in range(m)])
    got = _call(case, list(range(m)), P, P + 8)
    for t in (0, 1, m // 2, m - 1):
        assert torch.equal(got[t:t + 1], _call(case, [t], P, P + 8)), t


# the last row count of each kind that takes one launch; the next takes two
@pytest.mark.parametrize("hd,heads,kvh,L,last", [(32, 32, 8, 1024, 32), (32, 32, 16, 600, 16), (32, 32, 16, 512, 64),
                                                 (64, 32, 8, 1024, 32), (64, 32, 16, 512, 48), (64, 32, 8, 512, 96),
                                                 (128, 32, 8, 512, 32)])
def test_one_launch_only_while_its_workgroups_fit(hd, heads, kvh, L, last):
    """One launch keeps its records in LDS, two pass them through the workspace."""
    from ssd import ops

    for m in (last, last + 1):
        ws = torch.full((ops.attn_workspace_floats(m, heads, hd, CAP),), -7.0, device=DEV)
        _call(_case(m, heads, kvh, hd, L, seed=m), list(range(m)), 0, L, ws)
        assert bool((ws == -7.0).all()) == (m == last), m
