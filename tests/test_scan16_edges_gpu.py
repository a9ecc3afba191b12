"""The matrix-core scan of 16-bit pools at its own edges, in every layout and
through the planner: lengths around its stages (16 tokens), its gate blocks (64)
and the tokens one store of y covers (4, 8, 16), an empty row, and rows at the
limits of the state's type. y, pad zeros and states equal the decode kernel
applied token by token, bit for bit; a sample is checked against 64 bits."""
from __future__ import annotations

import pytest
import torch

from gpu_helpers import DEV, gen, raw_gates

pytestmark = pytest.mark.gpu
H, G = 4, 2
LENS = [1, 3, 4, 5, 15, 16, 17, 31, 33, 63, 64, 65, 80, 0, 127, 129]


def _bits(t):
    return t.view(torch.int32) if t.dtype == torch.float32 else t.view(torch.int16)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("layout", [None, 0, 1, 2, 4, 8])
def test_equals_decode_at_the_edges(kern, dt, layout):
    B, T = len(LENS), max(LENS)
    pool = (torch.randn(B, H, 128, 128, generator=gen(1), device=DEV) * 0.1).to(dt)
    # One row of the smallest subnormals, one of large values.
    pool[4] = torch.where(pool[4] > 0, 1, -1).to(dt) * (2.0 ** -24 if dt == torch.float16 else 1e-39)
    pool[9] *= 1e4
    q = torch.randn(B, T, G, 128, generator=gen(2), device=DEV)
    k = torch.randn(B, T, G, 128, generator=gen(3), device=DEV)
    v = torch.randn(B, T, H, 128, generator=gen(4), device=DEV)
    q[2], k[2] = 0.0, 0.0          # zero vectors: the norms' epsilon
    k[6, :, :, 1:] *= 1e-6         # one dominant element: parts near subnormal
    a, b, A, dtb = raw_gates((B, T, H), H, torch.bfloat16, seed=5)
    slots = torch.arange(B, dtype=torch.int32, device=DEV)
    lens = torch.tensor(LENS, dtype=torch.int32, device=DEV)
    ps, ys = pool.clone(), torch.zeros(B, T, H, 128, device=DEV)
    for t in range(T):
        rows = [r for r, n in enumerate(LENS) if n > t]
        sel = torch.tensor(rows, device=DEV)
        y = torch.empty(len(rows), H, 128, device=DEV)
        kern.gdn_decode_raw(ps, slots[sel].contiguous(), q[sel, t].contiguous(),
                            k[sel, t].contiguous(), v[sel, t].contiguous(), a[sel, t].contiguous(),
                            b[sel, t].contiguous(), A, dtb, y)
        ys[sel, t] = y
    pc, yc = pool.clone(), torch.full((B, T, H, 128), 7.0, device=DEV)
    with kern.launch_override(prefill_layout=layout):
        kern.gdn_prefill_raw(pc, slots, q, k, v, a, b, A, dtb, yc, lens)
    assert torch.equal(_bits(yc), _bits(ys)), (yc - ys).abs().amax(dim=(1, 2, 3))
    assert torch.equal(_bits(pc), _bits(ps))


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
def test_one_token_against_64_bits(kern, dt):
    """Half an ulp of the state's type plus fp32 sums of 128 terms: the state
    within one unit, y within 1e-6 of the terms' magnitudes (the split of k_hat
    and q_hat leaves at most 2^-23 of an element, an fp32 sum 128 * 2^-24)."""
    B = 3
    pool = (torch.randn(B, H, 128, 128, generator=gen(6), device=DEV)).to(dt)
    q = torch.randn(B, G, 128, generator=gen(7), device=DEV)
    k = torch.randn(B, G, 128, generator=gen(8), device=DEV)
    v = torch.randn(B, H, 128, generator=gen(9), device=DEV)
    alpha = torch.rand(B, H, generator=gen(10), device=DEV)
    beta = torch.rand(B, H, generator=gen(11), device=DEV)
    S = pool.double()
    unit = lambda x: (x.double() * torch.rsqrt((x.double() ** 2).sum(-1, keepdim=True) + 1e-6)
                      ).repeat_interleave(H // G, dim=1)
    qh, kh = unit(q), unit(k)
    kv = (S * kh[..., None]).sum(-2)
    delta = (v.double() - alpha.double()[..., None] * kv) * beta.double()[..., None]
    S1 = alpha.double()[..., None, None] * S + kh[..., None] * delta[..., None, :]
    y64 = (S1 * qh[..., None]).sum(-2) * 128 ** -0.5
    mag = ((alpha.double()[..., None, None] * S).abs() * qh.abs()[..., None]).sum(-2) + delta.abs()
    y = torch.empty(B, H, 128, device=DEV)
    kern.gdn_decode(pool, torch.arange(B, dtype=torch.int32, device=DEV), q, k, v, alpha, beta, y)
    assert ((y.double() - y64).abs() <= 1e-6 * mag).all()
    eps = torch.finfo(dt).eps
    tiny = 2.0 ** -24 if dt == torch.float16 else 0.0
    assert ((pool.double() - S1).abs() <= eps * S1.abs() * 0.51 + 1e-6 * mag[:, :, None, :] + tiny).all()
