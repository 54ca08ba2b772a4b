"""The router's product and the choice as one kernel, and the choice on its own at the edges of what a lane keeps.

The logits' reference is float64; a float32 sum of K products by 64 lanes, K / 64 a lane in series, is at most K / 64 + 6 roundings of 2^-24 of
the sum of the magnitudes away.  The choice and its weights are those of `moe_route` for the same logits, bit by bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 8, 33, 128])
@pytest.mark.parametrize("K,outputs,experts,top", [(8, 1, 1, 1), (64, 5, 4, 4), (504, 33, 32, 4), (1024, 64, 64, 8), (1032, 66, 65, 3), (2048, 48, 47, 47), (200, 300, 299, 64)])
@pytest.mark.parametrize("score", ["softmax", "sigmoid", "sigmoid_normed"])
def test_router(T, K, outputs, experts, top, score):
    from fms_amd.kernels import ops

    g = torch.Generator(device="cuda").manual_seed(T * 1000 + K)
    wide = torch.randn(T, K + 8, generator=g, device="cuda").to(torch.bfloat16)
    x, w = wide[:, :K], (torch.randn(outputs, K, generator=g, device="cuda") * 0.1).to(torch.bfloat16)
    assert ops.moe_router_fits(x, w)
    ids, weights, logits = ops.moe_router(x, w, experts, top, score)
    want, size = x.double() @ w.double().T.contiguous(), x.double().abs() @ w.double().abs().T.contiguous()
    assert float(((logits.double() - want).abs() - size * (K / 64 + 7) * 2.0 ** -24).max()) <= 0
    same_ids, same_weights = ops.moe_route(logits, experts, top, score)
    assert torch.equal(ids, same_ids) and torch.equal(weights, same_weights)
    best = torch.topk(logits[:, :experts], top, dim=1)
    assert torch.equal(torch.gather(logits, 1, ids.long()), best.values)


@pytest.mark.parametrize("experts", [3, 64, 65, 256, 257, 1024])
def test_ties_go_to_the_lower_index(experts):
    from fms_amd.kernels import ops

    top = min(3, experts)
    logits = torch.zeros(5, experts, device="cuda")
    logits[1, experts - 1] = logits[1, experts // 2] = 1.0
    logits[2, :] = float("-inf")
    logits[3, 0] = float("nan")
    logits[4, :] = torch.arange(experts, device="cuda") % 3
    ids, _ = ops.moe_route(logits, experts, top)
    ids = ids.cpu().tolist()
    assert ids[0] == list(range(top))
    assert ids[1][:2] == sorted({experts // 2, experts - 1})[:2]
    assert all(0 <= i < experts for row in ids for i in row)
    assert ids[3] == [i for i in range(experts) if i != 0][:top] if experts > top else True
    twos = [e for e in range(experts) if e % 3 == 2]
    assert ids[4][: min(top, len(twos))] == twos[:top]
