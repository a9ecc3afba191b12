"""quantize_act around the line between its one-workgroup launch (up to 16,384
elements, in eights, aligned) and its two launches: codes and scale equal torch's
spelling bit for bit, with NaN, infinite, zero and negative-zero elements at
either end, and through the no-alloc entry."""
from __future__ import annotations

import pytest
import torch

from gpu_helpers import DEV, gen

pytestmark = pytest.mark.gpu


def _torch(x):
    scale = (x.float().abs().amax() / 448).clamp(min=1e-12)
    q = (x.float() / scale).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q, scale


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [8, 12, 4096, 8184, 8192, 8200, 16376, 16384, 16385, 16392])
def test_matches_torch_at_the_line(kern, dt, n):
    x = torch.randn(n, generator=gen(n), device=DEV).to(dt)
    cases = [x, torch.zeros_like(x), -x.abs()]
    for bad in (float("nan"), float("inf"), -0.0):
        for at in (0, n - 1):
            y = x.clone()
            y[at] = bad
            cases.append(y)
    buf = torch.zeros(n + 8, device=DEV, dtype=dt)
    buf[1:n + 1] = x
    cases.append(buf[1:n + 1])  # not 16-byte aligned
    for c in cases:
        q, s = _torch(c)
        got_q, got_s = kern.quantize_act(c)
        assert torch.equal(got_q.view(torch.uint8), q.view(torch.uint8))
        assert torch.equal(got_s.view(-1).view(torch.int32), s.view(1).view(torch.int32)) or (
            s.isnan() and got_s.isnan())
        into, scale = torch.empty_like(got_q), torch.empty(1, device=DEV)
        kern.quantize_act_into(c, into, scale)
        assert torch.equal(into.view(torch.uint8), got_q.view(torch.uint8))
