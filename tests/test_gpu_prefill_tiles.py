"""Every tile shape of the prefill GEMM at its edges.

The shape is chosen from (M, N, K), so the same rows run on different shapes when M changes; every
output element is the same chain of MFMAs over k on all of them, so a row's bits must not change. One
plain call is also held against the fp32 product of the same operands (bounds beside it); the epilogues
have their own oracle tests in test_gpu_prefill.py.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(*shape, seed, std=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(torch.bfloat16)


def _qkv(heads, kv, hd, rows, pos0):
    from ssd.models.llama import rope_tables

    cap = (pos0 + rows + 63) // 64 * 64
    cos, sin = rope_tables(cap, hd, 500000.0, DEV)
    z = lambda: torch.zeros(kv, cap * hd, dtype=torch.bfloat16, device=DEV)
    return dict(heads=heads, kv_heads=kv, head_dim=hd, cos=cos, sin=sin, pos0=pos0, k_cache=z(), vt_cache=z(), max_len=cap)


def _run(epi, x, m, wp, grp, n, k, res, pos0=0, qkv_shape=None):
    """(out rows, K cache, V cache) of one call over the first m rows."""
    from ssd import ops

    cols = {"store": n, "swiglu": n // 2, "qkv": qkv_shape and qkv_shape[0] * qkv_shape[2]}[epi]
    out = torch.zeros(m, cols, dtype=torch.bfloat16, device=DEV)
    q = _qkv(*qkv_shape, m, pos0) if epi == "qkv" else None
    ops.prefill_gemm(x[:m], m, wp, grp, n, k, out, epi, residual=res[:m] if epi == "store" else None,
                     norm_eps=1e-5 if epi != "store" else 0.0, qkv=q)
    kv = ()
    if q is not None:
        kv = (ops.kv_untile(q["k_cache"], q["max_len"], q["head_dim"], "k")[:, pos0:pos0 + m],
              ops.kv_untile(q["vt_cache"], q["max_len"], q["head_dim"], "v")[:, pos0:pos0 + m])
    return (out, *kv)


# N, K and row counts around the tiles' 32 / 64 / 96 / 128 / 160 / 192 / 256 rows; wide N makes the large tiles the cheapest
@pytest.mark.parametrize("epi,n,k,qkv_shape", [("store", 4096, 4096, None), ("store", 200, 192, None),
                                               ("store", 28672, 256, None), ("swiglu", 28672, 512, None),
                                               ("swiglu", 1056, 2048, None), ("swiglu", 16384, 2048, None),
                                               ("qkv", 6144, 4096, (32, 8, 128)), ("qkv", 3072, 2048, (32, 8, 64)),
                                               ("qkv", 3072, 64, (32, 8, 64))])
def test_rows_have_the_same_bits_on_every_tile_shape(epi, n, k, qkv_shape):
    from ssd import ops

    top = 1100
    x, w = _rand(top, k, seed=1), _rand(n, k, seed=2, std=0.02)
    res = _rand(top, n, seed=3)
    grp = ops.weight_group(n, k)
    wp = ops.pack_weight(w)
    pos0 = 5 if qkv_shape else 0
    ref = _run(epi, x, top, wp, grp, n, k, res, pos0, qkv_shape)
    for m in (1, 31, 32, 33, 64, 65, 96, 127, 129, 161, 200, 257, 300, 350, 450, 513, 700, 900):
        got = _run(epi, x, m, wp, grp, n, k, res, pos0, qkv_shape)
        assert torch.equal(got[0], ref[0][:m]), (epi, m)
        for a, b in zip(got[1:], ref[1:]):
            assert torch.equal(a, b[:, :m]), (epi, m)
    if epi == "store":
        # bf16(residual + bf16(product)): the product may land on the neighbouring bf16 value (one step is at
        # most 2^-7 of it), the sum is then rounded (2^-8 of it); 1e-3 for the fp32 summation order
        p = (x.float() @ w.float().T).to(torch.bfloat16).float()
        want = res.float() + p
        assert ((ref[0].float() - want).abs() <= 2 ** -7 * p.abs() + 2 ** -8 * want.abs() + 1e-3).all()


# the 192-token shapes' plain and q/k/v write-outs, whose cheapest calls are longer ones
@pytest.mark.parametrize("epi,n,k,qkv_shape", [("store", 4096, 4096, None), ("qkv", 6144, 4096, (32, 8, 128))])
def test_long_calls_have_the_same_bits_on_every_tile_shape(epi, n, k, qkv_shape):
    from ssd import ops

    x, w = _rand(3000, k, seed=12), _rand(n, k, seed=13, std=0.02)
    res, grp, wp = _rand(3000, n, seed=14), ops.weight_group(n, k), ops.pack_weight(w)
    ref = _run(epi, x, 3000, wp, grp, n, k, res, 3, qkv_shape)
    for m in (1150, 1300, 1500, 1800, 2500):
        got = _run(epi, x, m, wp, grp, n, k, res, 3, qkv_shape)
        assert torch.equal(got[0], ref[0][:m]), (epi, m)
        for a, b in zip(got[1:], ref[1:]):
            assert torch.equal(a, b[:, :m]), (epi, m)


# k loops shorter than, equal to and just past the operand ring's depth (K / 64 = 1 .. 9), on the
# smallest tile (N = 64), tiles between, and on the largest (N = 28672, M = 4096: the cheapest from K = 192 on)
@pytest.mark.parametrize("m,n,k", [(m, n, k) for m, n in ((40, 64), (700, 640), (290, 16384), (190, 16384))
                                   for k in range(64, 577, 64)]
                         + [(4096, 28672, k) for k in (192, 256, 320)])
def test_short_k_loops_match_the_fp32_product(m, n, k):
    from ssd import ops

    x, w = _rand(m, k, seed=4), _rand(n, k, seed=5, std=0.1)
    out = torch.zeros(m, n, dtype=torch.bfloat16, device=DEV)
    ops.prefill_gemm(x, m, ops.pack_weight(w), ops.weight_group(n, k), n, k, out)
    want = x.float() @ w.float().T  # one bf16 rounding (2^-8 relative, 2^-9 from the nearest) of sums within 2e-3
    torch.testing.assert_close(out.float(), want, rtol=2 ** -8, atol=2e-3)


def test_rows_far_apart_equal_contiguous_rows():
    """A row stride of 2^27 elements does not fit the kernel's 32-bit lane offsets: such rows are run one by one."""
    from ssd import ops

    k, n, m = 256, 384, 3
    x, w = _rand(m, k, seed=6), _rand(n, k, seed=7, std=0.05)
    wp, grp = ops.pack_weight(w), ops.weight_group(n, k)
    far = torch.empty((m - 1) * (1 << 27) + k, dtype=torch.bfloat16, device=DEV).as_strided((m, k), (1 << 27, 1))
    far.copy_(x)
    res = _rand(m, n, seed=8)
    a, b = torch.zeros(m, n, dtype=torch.bfloat16, device=DEV), torch.zeros(m, n, dtype=torch.bfloat16, device=DEV)
    ops.prefill_gemm(x, m, wp, grp, n, k, a, residual=res)
    ops.prefill_gemm(far, m, wp, grp, n, k, b, residual=res)
    assert torch.equal(a, b)


@pytest.mark.parametrize("heads,kv,hd", [(32, 8, 128), (32, 8, 64), (6, 3, 128)])
def test_attention_rows_do_not_depend_on_the_tile(heads, kv, hd):
    """A call with many rows gives each wave 32 tokens, one with few 16, and a row's block is masked or not
    depending on its tile: the same rows in calls of other sizes and starts have the same bits."""
    from ssd import ops

    m = 128 * (32 // ((heads + 3) // 4)) + 70  # past the line between the two
    cap = (m + 63) // 64 * 64 + 64
    q = _rand(m, heads * hd, seed=9)
    k, v = _rand(kv, cap, hd, seed=10), _rand(kv, cap, hd, seed=11)
    k[:, m:] = float("nan")
    v[:, m:] = float("nan")
    kd, vd = ops.kv_tile(k, "k"), ops.kv_tile(v, "v")
    ref = torch.zeros(m, heads * hd, dtype=torch.bfloat16, device=DEV)
    ops.prefill_attention(q, m, 0, heads, kv, hd, kd, vd, cap, ref)
    assert torch.isfinite(ref.float()).all()
    for r0, n in ((0, 16), (0, 65), (37, 128), (64, 17), (100, 200), (m - 33, 33)):
        out = torch.zeros(n, heads * hd, dtype=torch.bfloat16, device=DEV)
        ops.prefill_attention(q[r0:r0 + n], n, r0, heads, kv, hd, kd, vd, cap, out)
        assert torch.equal(out, ref[r0:r0 + n]), (r0, n)


@pytest.mark.parametrize("heads,kv,hd", [(24, 8, 128), (32, 32, 128), (24, 8, 64), (32, 8, 128)])
@pytest.mark.parametrize("pos0", [2048, 2049, 5000])
def test_attention_rows_after_a_long_past_do_not_depend_on_the_tile(heads, kv, hd, pos0):
    """The row count from which a wave takes 32 rows depends on the heads' sharing and on the past as well: calls on
    both sides of each line, in rows, give a row the same bits."""
    from ssd import ops

    n_hg = heads // 4
    m = 512 // n_hg * 16 + 16
    cap = (pos0 + m + 63) // 64 * 64
    q = _rand(m, heads * hd, seed=15)
    k, v = ops.kv_tile(_rand(kv, cap, hd, seed=16), "k"), ops.kv_tile(_rand(kv, cap, hd, seed=17), "v")
    ref = torch.zeros(m, heads * hd, dtype=torch.bfloat16, device=DEV)
    ops.prefill_attention(q, m, pos0, heads, kv, hd, k, v, cap, ref)
    for n in (256 // n_hg * 16, 256 // n_hg * 16 + 1, m - 16, 70):
        out = torch.zeros(n, heads * hd, dtype=torch.bfloat16, device=DEV)
        ops.prefill_attention(q, n, pos0, heads, kv, hd, k, v, cap, out)
        assert torch.equal(out, ref[:n]), n
