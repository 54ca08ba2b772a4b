"""The products per head of few tokens, whose waves share K: edges of tokens, elements and K, with and without a gate.

The reference is float64.  A float32 sum of K products in runs of 32 is at most K / 16 roundings of 2^-24 of the sum of the magnitudes away (as many as
the runs and the four waves, twice over), the bfloat16 result one of 2^-9 of itself; the gate's own arithmetic is good to 2^-20."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 15, 16, 17, 40])
@pytest.mark.parametrize("H,K,N", [(1, 64, 1), (3, 72, 31), (4, 96, 33), (2, 136, 128), (16, 512, 128), (5, 520, 130), (16, 128, 512), (2, 1000, 64)])
@pytest.mark.parametrize("gated", [False, True])
def test_headwise(T, H, K, N, gated):
    from fms_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(T + K)
    xs, ys = K + 8, N + 3
    x = torch.randn(T, H * xs, generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn(H, N, K, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
    gate = torch.randn(T, H + 2, generator=g, device="cuda")[:, :H] if gated else None
    y = torch.full((T, H * ys), 7.0, device="cuda", dtype=torch.bfloat16)
    ops.headwise_linear(x, xs, w, y, ys, gate=gate)
    rows = x.view(T, H, xs)[:, :, :K].transpose(0, 1).double().contiguous()
    cols = w.double().transpose(1, 2).contiguous()
    factor = torch.sigmoid(gate.double())[:, :, None] if gated else 1.0
    want = torch.matmul(rows, cols).transpose(0, 1) * factor
    size = torch.matmul(rows.abs(), cols.abs()).transpose(0, 1)
    got = y.view(T, H, ys)
    allowed = size * (K / 16 + 8) * 2.0 ** -24 + want.abs() * (2.0 ** -8 + 2.0 ** -20)
    assert float(((got[:, :, :N].double() - want).abs() - allowed).max()) <= 0
    assert bool((got[:, :, N:] == 7).all())
