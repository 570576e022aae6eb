"""SwiGLU of the prefill GEMM over every finite bf16 gate value.

The gate is rounded to bf16 before SiLU and SiLU's value to bf16 after it, so 65280 inputs are the whole function.
The prefill's must be the decode GEMM's bit for bit (a prompt's rows are no less exact on one path than on the
other), and both the 64-bit value rounded to bf16, except below -88.5, where 1 + exp(-x) leaves fp32's range and
the result is -0 instead of a value under 2e-37."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_every_bf16_gate_value_matches_decode_and_64_bits():
    from ssd import ops
    from ssd.models.llama import gate_up_row_map

    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = x[torch.isfinite(x.float())]
    m, k, inter = x.numel(), 64, 64
    rows = torch.zeros(m, k, dtype=torch.bfloat16)
    rows[:, 0], rows[:, 1] = x, 1
    w = torch.zeros(2 * inter, k, dtype=torch.bfloat16)
    w[:inter, 0] = 1  # every gate column is x, every up column 1
    w[inter:, 1] = 1
    grp = ops.weight_group(2 * inter, k)
    wp = ops.pack_weight(w.cuda(), gate_up_row_map(inter), group=grp)
    pre, dec = (torch.zeros(m, inter, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    ops.prefill_gemm(rows.cuda(), m, wp, grp, 2 * inter, k, pre, "swiglu")
    ops.gemm_swiglu(rows.cuda(), m, wp, inter, k, dec)
    pre, dec = pre.cpu(), dec.cpu()
    bits = lambda t: t.view(torch.int16)
    assert torch.equal(bits(pre), bits(dec)), x[(bits(pre) != bits(dec)).any(1)].tolist()
    want = x.double() / (1 + torch.exp(-x.double()))
    same = (pre == want.to(torch.bfloat16)[:, None]).all(1)
    assert same[x >= -88.5].all()
    assert ((pre.double() - want[:, None]).abs()[~same] < 2e-37).all()
