"""Decode projections whose X is staged through LDS (K = 2048, 4096, 8192): every plan and row count.

A row's bits may not depend on how many rows share the call (one to four 16-row column tiles, chunks of
64), and the products match the fp32 ones of the same operands: outputs round fp32 sums to bf16, so they may
land on the neighbouring value (2^-7 relative covers one step), plus 2e-3 for the order of the sums."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
SHAPES = [(3072, 2048), (2048, 2048), (6144, 2048), (6144, 4096), (4096, 4096), (10240, 8192), (8192, 8192),
          (8192, 2048)]


def _rand(*shape, seed, std=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("norm", [False, True])
def test_rows_do_not_depend_on_the_row_count(n, k, norm):
    from ssd import ops

    eps = 1e-5 if norm else 0.0
    x, w = _rand(80, k, seed=1), _rand(n, k, seed=2, std=0.02)
    wp = ops.pack_weight(w)
    ref = torch.zeros(80, n, dtype=torch.bfloat16, device=DEV)
    ops.gemm(x, 80, wp, n, k, ref, norm_eps=eps)
    # (8, 9, 17, 20, 21: where calls with the norm change between staged and direct)
    for m in (1, 8, 9, 15, 16, 17, 20, 21, 32, 33, 47, 49, 64, 65):
        out = torch.zeros(m, n, dtype=torch.bfloat16, device=DEV)
        ops.gemm(x, m, wp, n, k, out, norm_eps=eps)
        assert torch.equal(out, ref[:m]), m
    want = x.float() @ w.float().T
    if norm:
        want = want * torch.rsqrt(x.float().pow(2).mean(1, keepdim=True) + eps)
    torch.testing.assert_close(ref.float(), want, rtol=2 ** -7, atol=2e-3)


@pytest.mark.parametrize("n,k", SHAPES)
def test_residual_rows_do_not_depend_on_the_row_count(n, k):
    from ssd import ops

    x, w, h = _rand(64, k, seed=3), _rand(n, k, seed=4, std=0.02), _rand(64, n, seed=5)
    wp = ops.pack_weight(w, residual=True)
    part = torch.zeros(max(1, ops.residual_floats(64, n, k)), device=DEV)
    ref = h.clone()
    ops.gemm_residual(x, 64, wp, n, k, ref, part)
    for m in (1, 16, 17, 33, 48, 50):
        out = h.clone()
        ops.gemm_residual(x, m, wp, n, k, out, part)
        assert torch.equal(out[:m], ref[:m]) and torch.equal(out[m:], h[m:]), m
    # bf16(h + bf16(product)): one step of the product (2^-7 of it), one rounding of the sum (2^-8)
    p = (x.float() @ w.float().T).to(torch.bfloat16).float()
    want = h.float() + p
    assert ((ref.float() - want).abs() <= 2 ** -7 * p.abs() + 2 ** -8 * want.abs() + 2e-3).all()


@pytest.mark.parametrize("heads,kvh,hd,k", [(64, 8, 128, 8192), (32, 8, 128, 4096), (32, 8, 64, 2048)])
@pytest.mark.parametrize("norm", [True, False])
def test_qkv_rows_do_not_depend_on_the_row_count(heads, kvh, hd, k, norm):
    """The same through the q/k/v epilogue (RoPE, cache write) at the 70B, 8B and 1B shapes. A rotated value is
    bf16(bf16(a cos) + bf16(b sin)) of its pair's products, each within one bf16 step (2^-7): 2^-7 of |a| + |b|, as much
    again for the three roundings."""
    from ssd import ops
    from ssd.models.llama import qkv_row_map, rope_tables

    n, cap, top, eps = (heads + 2 * kvh) * hd, 128, 80, 1e-5 if norm else 0.0
    x, w = _rand(top, k, seed=6), _rand(n, k, seed=7, std=0.02)
    wp = ops.pack_weight(w, qkv_row_map(heads, kvh, hd))
    cos, sin = rope_tables(cap, hd, 500000.0, DEV)
    pos = (torch.arange(top, device=DEV) * 5 % 97).to(torch.int32)
    slot = (torch.arange(top, device=DEV) * 11 % 128).to(torch.int32)  # all different

    def run(m):
        q = torch.zeros(m, heads * hd, dtype=torch.bfloat16, device=DEV)
        kc, vt = (torch.zeros(kvh, cap * hd, dtype=torch.bfloat16, device=DEV) for _ in range(2))
        ops.qkv_rope(x, m, wp, k, heads, kvh, hd, cos, sin, pos, slot, q, kc, vt, cap, norm_eps=eps)
        at = slot[:m].long()
        return [q.view(m, heads, hd), ops.kv_untile(kc, cap, hd, "k")[:, at].transpose(0, 1),
                ops.kv_untile(vt, cap, hd, "v")[:, at].transpose(0, 1)]

    ref = run(top)
    for m in (1, 8, 17, 20, 33, 48, 49, 64):
        assert all(torch.equal(a, b[:m]) for a, b in zip(run(m), ref)), m
    p = x.float() @ w.float().T
    if norm:
        p = p * torch.rsqrt(x.float().pow(2).mean(1, keepdim=True) + eps)
    p = p.to(torch.bfloat16).float().view(top, heads + 2 * kvh, hd)
    c, s = (t[pos.long()].float()[:, None] for t in (cos, sin))
    lo, hi = p[..., :hd // 2], p[..., hd // 2:]
    rot = torch.cat([lo * c - hi * s, hi * c + lo * s], -1)
    room = (lo.abs() + hi.abs()).repeat(1, 1, 2) * 2 ** -6 + 4e-3
    for got, want, tol in ((ref[0], rot[:, :heads], room[:, :heads]), (ref[1], rot[:, heads:-kvh], room[:, heads:-kvh])):
        assert ((got.float() - want).abs() <= tol).all()
    torch.testing.assert_close(ref[2].float(), p[:, -kvh:], rtol=2 ** -7, atol=2e-3)
