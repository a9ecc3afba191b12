"""The fused conv + GDN decode + gated readout launch
(braid_gdn_conv_decode_readout) against the launches it fuses,
gdn_conv_decode_raw then gated_rmsnorm: core, FP8 codes, scale, states and conv
windows bit for bit, over the pool types, both activation types, one and two
heads per group, the smallest batch and one whose unit count (B * H) is no
multiple of four (the quantize pass reads the partials by fours)."""
from __future__ import annotations

import pytest
import torch

from gpu_helpers import DEV, gen, raw_gates

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pool_dt", [torch.float16, torch.bfloat16, torch.float32],
                         ids=["f16-pool", "bf16-pool", "f32-pool"])
@pytest.mark.parametrize("act", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
@pytest.mark.parametrize("B,H,G", [(1, 32, 16), (5, 3, 3), (64, 32, 16)])
def test_equals_the_separate_launches(kern, pool_dt, act, B, H, G):
    S, C = B + 3, 2 * G * 128 + H * 128
    pool = (torch.randn(S, H, 128, 128, generator=gen(1), device=DEV) * 0.1).to(pool_dt)
    conv = torch.randn(S, C, 4, generator=gen(2), device=DEV)
    w = torch.randn(C, 4, generator=gen(3), device=DEV) * 0.3
    bias = torch.randn(C, generator=gen(4), device=DEV) * 0.1
    x = torch.randn(B, C, generator=gen(5), device=DEV).to(act)
    z = torch.randn(B, 1, H * 128, generator=gen(6), device=DEV).to(act)
    gamma = torch.rand(128, generator=gen(7), device=DEV) + 0.5
    a, b, A, dtb = raw_gates((B, H), H, act, seed=8)
    slots = torch.randperm(S, generator=torch.Generator().manual_seed(9))[:B].to(torch.int32).to(DEV)
    p1, c1, p2, c2 = pool.clone(), conv.clone(), pool.clone(), conv.clone()
    for _ in range(2):
        y = torch.empty(B, H, 128, device=DEV)
        kern.gdn_conv_decode_raw(p1, c1, slots, x, w, bias, a, b, A, dtb, y, G)
        ref = kern.gated_rmsnorm(y, z, gamma, 1e-6)
        got = kern.gdn_conv_decode_readout(p2, c2, slots, x, w, bias, a, b, A, dtb, z, gamma,
                                           1e-6, G)
        for r, g, name in zip(ref, got, ("core", "codes", "scale")):
            assert r.shape == g.shape and r.dtype == g.dtype
            assert torch.equal(r.view(torch.uint8), g.view(torch.uint8)), name
    assert torch.equal(p1.view(torch.uint8), p2.view(torch.uint8)), "states differ"
    assert torch.equal(c1, c2), "conv windows differ"
    only = kern.gdn_conv_decode_readout(p2, c2, slots, x, w, bias, a, b, A, dtb, z, gamma, 1e-6, G,
                                        quantize=False)
    kern.gdn_conv_decode_raw(p1, c1, slots, x, w, bias, a, b, A, dtb, y, G)
    assert torch.equal(only, kern.gated_rmsnorm(y, z, gamma, 1e-6, quantize=False))
