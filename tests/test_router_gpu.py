"""The router's product and the choice as one kernel, and the choice on its own at the edges of what a lane keeps; the shared expert's unit.

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


@pytest.mark.parametrize("rows,width,hidden,kernels", [(16, 256, 128, 0), (17, 256, 128, 1), (32, 512, 512, 1), (33, 256, 128, 0), (32, 1024, 1024, 0)])
def test_the_shared_experts_unit_runs_where_it_is_faster(rows, width, hidden, kernels, monkeypatch):
    """Inside its product, or as a kernel behind it where 17 to 32 rows meet a small weight.  Against float64: gate and up are at most rounded to bfloat16
    (2^-9 each, the unit's slope is below 2), the hidden values and the result are rounded once more."""
    from fms_amd.kernels import ops
    from fms_amd.parts.experts import ExpertsFeedForward

    g = torch.Generator(device="cuda").manual_seed(rows + hidden)
    part = ExpertsFeedForward(width, 4, 2, 64, 7.0, shared_hidden_dim=hidden, shared_limit=1.5, shared_gate=False)
    for _, spec, owner, local in part.named_specs():
        owner.bind(local, (torch.randn(spec.shape, generator=g, device="cuda") * 0.05).to(torch.bfloat16))
    part.finalize(torch.device("cuda"), torch.bfloat16)
    part.w["experts.down"].zero_()  # the shared expert alone
    calls, unit = [], ops.clamped_gated_act
    monkeypatch.setattr(ops, "clamped_gated_act", lambda *a: calls.append(1) or unit(*a))
    x = torch.randn(rows, width, generator=g, device="cuda").to(torch.bfloat16)
    out = part.forward(x)
    assert len(calls) == kernels
    gate, up = (x.double() @ part.shared_gate_up.w["weight"].double().T.contiguous()).chunk(2, dim=1)
    z = gate.clamp(max=1.5)
    h = z * torch.sigmoid(1.702 * z) * (up.clamp(-1.5, 1.5) + 1.0)
    down = part.shared_down.w["weight"].double().T.contiguous()
    want = h @ down
    off = 2.0 ** -8 * ((gate.abs() * 2 * (up.abs() + 1) + up.abs() * z.abs() + h.abs()) @ down.abs()) + 2.0 ** -7 * want.abs()
    assert float(((out.double() - want).abs() - off).max()) <= 0
