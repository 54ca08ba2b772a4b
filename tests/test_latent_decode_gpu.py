"""Decode attention over a latent of 512 whose rows go straight into LDS: edges of tiles, parts, windows, head groups and padding rows.

The reference is float64 softmax over the same bfloat16 rows.  The kernel rounds the probabilities to bfloat16 (2^-9 of each, whatever their sum) and the
result once more: 2^-8 of the largest value that is averaged, here of the largest latent, bounds both."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rot", [0, 64])
@pytest.mark.parametrize("heads,sink", [(1, False), (16, True), (17, True), (40, False)])
@pytest.mark.parametrize("lengths,window", [([1], 0), ([1, 31, 32, 33, 63, 64, 65], 0), ([127, 128, 129, 0, 700, 2049], 0), ([5, 0, 400, 1300], 100), ([640, 641, 1025], 33),
                                            ([300] * 40, 0)])
def test_decode(rot, heads, sink, lengths, window):
    from fms_amd.kernels import ops

    T, width, scale = len(lengths), 512 + rot, 0.06
    g = torch.Generator(device="cuda").manual_seed(heads * 100 + T)
    pages = [max(1, -(-n // 64)) for n in lengths]
    cache = torch.randn(sum(pages) + 1, 1, 64, width, generator=g, device="cuda").to(torch.bfloat16)
    order = (torch.randperm(sum(pages), generator=g, device="cuda") + 1).int()
    table = torch.full((T, max(pages) + 1), -1, dtype=torch.int32, device="cuda")
    at = 0
    for i, p in enumerate(pages):
        table[i, :p] = order[at : at + p]
        at += p
    values = cache[:, :, :, :512].transpose(2, 3).contiguous()
    positions = torch.tensor([max(n - 1, 0) for n in lengths], dtype=torch.int32, device="cuda")
    seqs = torch.tensor([i if n else -1 for i, n in enumerate(lengths)], dtype=torch.int32, device="cuda")
    qa = (torch.randn(T, heads * width, generator=g, device="cuda") * 0.4).to(torch.bfloat16)
    sinks = torch.randn(heads, generator=g, device="cuda") if sink else None
    for bound in (max(lengths), 4096):
        out = ops.latent_attention(qa, positions, seqs, table, cache, sinks, heads, 512, rot, scale, window, decode=True, max_context=bound, vt_cache=values)
        for i, n in enumerate(lengths):
            got = out[i].view(heads, 512).double()
            if n == 0:
                assert not bool(got.any())
                continue
            rows = cache[table[i, : pages[i]].long()].reshape(-1, width)[:n].double()
            rows = rows[max(0, n - window) :] if window else rows
            s = qa[i].view(heads, width).double() @ rows.T.contiguous() * scale
            if sinks is not None:
                s = torch.cat([s, sinks.double()[:, None]], dim=1)
            want = torch.softmax(s, dim=1)[:, : rows.shape[0]].contiguous() @ rows[:, :512].contiguous()
            assert float((got - want).abs().max()) <= 2.0 ** -8 * float(rows.abs().max()), (n, bound)


@pytest.mark.parametrize("rot", [0, 64])
@pytest.mark.parametrize("decode", [True, False])
def test_a_cache_that_starts_between_16_byte_addresses(rot, decode):
    """Such a cache runs the kernel for any sizes: the same averages, both within the bound above of the float64 ones."""
    from fms_amd.kernels import ops

    heads, width, pages = 17, 512 + rot, 3
    g = torch.Generator(device="cuda").manual_seed(rot)
    cache = torch.randn(pages, 1, 64, width, generator=g, device="cuda").to(torch.bfloat16)
    flat = torch.zeros(cache.numel() + 4, dtype=torch.bfloat16, device="cuda")
    shifted = flat[4:].view(cache.shape)
    shifted.copy_(cache)
    assert shifted.data_ptr() % 16 == 8
    values = cache[:, :, :, :512].transpose(2, 3).contiguous()
    lengths = [130, 65, 191] if decode else list(range(60, 71))
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32, device="cuda")
    seqs = torch.arange(3, dtype=torch.int32, device="cuda") if decode else torch.zeros(len(lengths), dtype=torch.int32, device="cuda")
    table = torch.arange(pages, dtype=torch.int32, device="cuda").repeat(3, 1)
    qa = (torch.randn(len(lengths), heads * width, generator=g, device="cuda") * 0.4).to(torch.bfloat16)
    same, out = (ops.latent_attention(qa, positions, seqs, table, c, None, heads, 512, rot, 0.06, decode=decode, max_context=192, vt_cache=values)
                 for c in (cache, shifted))
    assert float((out.double() - same.double()).abs().max()) <= 2 * 2.0 ** -8 * float(cache.abs().max())
