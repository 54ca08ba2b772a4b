"""Rotation and cache write of few tokens against the kernel for many: the same tokens as part of a step that is too long for the first, bit by bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu

FEW = 384  # ROPE_FEW_TOKENS of rope.hip


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("heads,kvheads,dim,rot,pad", [(16, 4, 128, 128, 0), (3, 1, 8, 8, 0), (5, 5, 36, 20, 0), (4, 2, 64, 24, 4), (40, 8, 128, 0, 8)])
@pytest.mark.parametrize("tokens", [1, 7, FEW])
@pytest.mark.parametrize("cached", [True, False])
def test_few_tokens(dtype, heads, kvheads, dim, rot, pad, tokens, cached):
    from fms_amd.kernels import ops
    from fms_amd.kernels.library import check, load

    lib = load()
    g = torch.Generator(device="cuda").manual_seed(tokens + dim)
    width = (heads + 2 * kvheads) * dim
    base = torch.randn(tokens, width + pad, generator=g, device="cuda").to(dtype)
    angle = torch.rand(300, max(rot // 2, 1), generator=g, device="cuda")
    cos, sin = angle.cos().contiguous(), angle.sin().contiguous()
    positions = torch.randint(0, 300, (tokens,), generator=g, device="cuda", dtype=torch.int32)
    seqs = torch.arange(tokens, dtype=torch.int32, device="cuda")
    if tokens > 1:
        seqs[tokens // 2] = -1
    table = torch.arange(5 * tokens, dtype=torch.int32, device="cuda").view(tokens, 5)
    table[0, :] = -1  # a page that is not there
    results = []
    for rows in (tokens, FEW + 1 + tokens):  # alone, and with padding rows behind
        more = rows - tokens
        qkv = torch.cat([base, torch.zeros(more, width + pad, dtype=dtype, device="cuda")])
        keys = torch.zeros(5 * tokens, kvheads, 64, dim, dtype=dtype, device="cuda") if cached else None
        values = torch.zeros(5 * tokens, kvheads, dim, 64, dtype=dtype, device="cuda") if cached else None
        p = torch.cat([positions, torch.zeros(more, dtype=torch.int32, device="cuda")])
        s = torch.cat([seqs, torch.full((more,), -1, dtype=torch.int32, device="cuda")])
        check(lib.fmsamd_rope_kv_write(qkv.data_ptr(), ops._code(dtype), qkv.stride(0), p.data_ptr(), s.data_ptr(), table.data_ptr(), 5,
                                       cos.data_ptr() if rot else None, sin.data_ptr() if rot else None, rot, 300 if rot else 0,
                                       keys.data_ptr() if cached else None, values.data_ptr() if cached else None, rows, heads, kvheads, dim, dim,
                                       ops._stream()))
        results.append((qkv[:tokens], keys, values))
    for few, many in zip(*results):
        assert few is None or torch.equal(few, many)
    if cached and tokens > 2:
        assert bool(results[0][1].any()) and bool(results[0][2].any())
