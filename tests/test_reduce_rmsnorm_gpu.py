"""The split-K reduction fused with the residual add and RMSNorm, at the edges of how it requests
its partials (4 at once up to 4 splits, else 8: one more, a whole second batch, one past it) and of
its row loop (one, two and four pieces per thread, the last one partial): equal, bit for bit, to the
reduced product followed by the standalone norm, which rounds in the same order."""

from __future__ import annotations

import pytest
import torch

from turingserve_amd import hip_ops as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp16_scale,bias", [(False, False), (True, True)])
@pytest.mark.parametrize("Nn", [1536, 2056, 8192])
@pytest.mark.parametrize("splits", [2, 4, 5, 8, 9, 16, 17])
def test_reduce_rmsnorm_equals_the_separate_calls(splits, Nn, fp16_scale, bias):
    g = torch.Generator().manual_seed(splits * Nn)
    M, Kd = 3, 64 * 2 * splits
    x = torch.randn(M, Kd, generator=g).half().cuda()
    wq = torch.randint(-127, 128, (Nn, Kd), generator=g, dtype=torch.int32).to(torch.int8).cuda()
    scale = (torch.rand(Nn, generator=g) * 0.002 + 0.0005).cuda()
    scale = scale.half() if fp16_scale else scale
    b = torch.randn(Nn, generator=g).half().cuda() if bias else None
    res, nw = torch.randn(M, Nn, generator=g).half().cuda(), torch.rand(Nn, generator=g).half().cuda()
    cfg = (4, splits)                                         # 128 x 32 wide tiles, that many splits
    out, res_out = K.w8a16_add_rmsnorm(x, wq, scale, b, res, nw, 1e-6, cfg)
    want_out, want_res = K.rmsnorm_residual(K.w8a16_linear(x, wq, scale, b, cfg), res, nw, 1e-6)
    assert torch.equal(res_out, want_res) and torch.equal(out, want_out)
