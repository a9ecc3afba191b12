"""The conv + scan prefill call (braid_gdn_conv_prefill_raw) against the two it
joins, conv1d_prefill then gdn_prefill_raw on dense copies of its q/k/v columns:
y (fp32, and bf16 where the scan rounds it), pad zeros, states and windows bit
for bit, over the pool types, ragged lengths around the stages' and conv
chunks' 16 tokens with an empty row and one past T, and each prefill layout."""
from __future__ import annotations

import pytest
import torch

from gpu_helpers import DEV, gen, raw_gates

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.int32) if t.dtype == torch.float32 else t.view(torch.int16)


@pytest.mark.parametrize("pool_dt", [torch.float16, torch.bfloat16, torch.float32],
                         ids=["f16-pool", "bf16-pool", "f32-pool"])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("layout", [None, 0, 1, 2, 4, 8])
def test_equals_conv_then_scan(kern, pool_dt, act, layout):
    H, G, T = 4, 2, 50
    lens = [50, 17, 0, 16, 33, 1, 99]
    B, C = len(lens), 2 * G * 128 + H * 128
    S = B + 2
    pool = (torch.randn(S, H, 128, 128, generator=gen(1), device=DEV) * 0.1).to(pool_dt)
    conv = torch.randn(S, C, 4, generator=gen(2), device=DEV)
    w = torch.randn(C, 4, generator=gen(3), device=DEV) * 0.3
    bias = torch.randn(C, generator=gen(4), device=DEV) * 0.1
    x = torch.randn(B, T, C, generator=gen(5), device=DEV).to(act)
    a, b, A, dtb = raw_gates((B, T, H), H, act, seed=6)
    slots = torch.randperm(S, generator=torch.Generator().manual_seed(7))[:B].to(torch.int32).to(DEV)
    for seq in (torch.tensor(lens, dtype=torch.int32, device=DEV), None):
        p1, c1, p2, c2 = pool.clone(), conv.clone(), pool.clone(), conv.clone()
        co = torch.empty(B, T, C, device=DEV)
        y1 = torch.empty(B, T, H, 128, device=DEV)
        y2 = torch.empty_like(y1)
        with kern.launch_override(prefill_layout=layout):
            kern.conv1d_prefill(c1, slots, x, w, bias, co, seq)
            q, k, v = torch.split(co, [G * 128, G * 128, H * 128], dim=-1)
            kern.gdn_prefill_raw(p1, slots, q.contiguous().view(B, T, G, 128),
                                 k.contiguous().view(B, T, G, 128),
                                 v.contiguous().view(B, T, H, 128), a, b, A, dtb, y1, seq)
            kern.gdn_conv_prefill_raw(p2, c2, slots, x, w, bias, a, b, A, dtb, y2, G, seq)
            assert torch.equal(_bits(y2), _bits(y1))
            assert torch.equal(_bits(p2), _bits(p1)) and torch.equal(c2, c1)
            y3 = torch.empty(B, T, H, 128, device=DEV, dtype=torch.bfloat16)
            if act == torch.bfloat16 and pool_dt != torch.float32:
                p3, c3 = pool.clone(), conv.clone()
                kern.gdn_conv_prefill_raw(p3, c3, slots, x, w, bias, a, b, A, dtb, y3, G, seq)
                assert torch.equal(_bits(y3), _bits(y1.to(torch.bfloat16)))
                assert torch.equal(_bits(p3), _bits(p1)) and torch.equal(c3, c1)
            else:
                with pytest.raises(RuntimeError, match="y is fp32"):
                    kern.gdn_conv_prefill_raw(p2, c2, slots, x, w, bias, a, b, A, dtb, y3, G, seq)
