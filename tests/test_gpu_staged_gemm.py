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
