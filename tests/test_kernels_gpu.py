"""Each kernel alone against a plain float32 torch formula, at sizes other than the engine's."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

import plain_llama as P  # noqa: E402

PAGE = 64


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from fms_amd.kernels import load, ops as _ops

    load()
    return _ops


def dev(t):
    return t.to("cuda")


def tol(dtype):
    return dict(atol=2e-5, rtol=2e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)


# --------------------------------------------------------------------------
def test_embed(ops):
    torch.manual_seed(0)
    for dtype in (torch.float32, torch.bfloat16):
        table = torch.randn(37, 24).to(dtype)
        ids = torch.tensor([0, 36, 5, 5, 17], dtype=torch.int32)
        out = ops.embed(dev(ids), dev(table)).cpu()
        assert out.dtype == torch.float32
        assert torch.equal(out, table.float()[ids.long()])


@pytest.mark.parametrize("width", [24, 100, 4096, 9000, 20000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_add_norm(ops, width, dtype):
    torch.manual_seed(1)
    T = 5
    resid = torch.randn(T, width) * 2
    branch = torch.randn(T, width).to(dtype)
    weight = (1 + 0.3 * torch.randn(width)).to(dtype)
    eps = 1e-3
    want_resid = resid + branch.float()
    want = P.rms_norm(want_resid, weight.float(), eps)
    r = dev(resid.clone())
    out = ops.add_norm(r, dev(branch), dev(weight), None, eps, dtype)
    torch.testing.assert_close(r.cpu(), want_resid)
    torch.testing.assert_close(out.cpu().float(), want, **tol(dtype))
    # no branch; selected rows only; the stream is left alone
    r2 = dev(resid.clone())
    rows = torch.tensor([3, 0], dtype=torch.int32)
    out2 = ops.add_norm(r2, dev(branch), dev(weight), None, eps, dtype, rows=dev(rows))
    torch.testing.assert_close(out2.cpu().float(), want[rows.long()], **tol(dtype))
    assert torch.equal(r2.cpu(), resid)
    out3 = ops.add_norm(dev(resid.clone()), None, dev(weight), None, eps, dtype)
    torch.testing.assert_close(out3.cpu().float(), P.rms_norm(resid, weight.float(), eps), **tol(dtype))


def test_kernels_run_on_the_current_stream(ops):
    """The number that the kernels are launched with is that of torch's current stream: by itself, inside stream contexts and while a
    graph is captured (whose replays then hold the kernel)."""
    here = lambda: ops._stream() == torch.cuda.current_stream().cuda_stream
    assert here()
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        assert here() and ops._stream() == a.cuda_stream
        with torch.cuda.stream(b):
            assert here() and ops._stream() == b.cuda_stream
        assert ops._stream() == a.cuda_stream
    x = dev(torch.ones(300))
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        assert here()
        ops.scale_(x, 2.0)
    for n in range(1, 4):
        graph.replay()
        assert bool((x == 2.0 ** n).all())
    assert here()


@pytest.mark.parametrize("heads, kvheads, dim, lens, contexts, window", [
    (4, 4, 16, [64], [64], 0), (2, 1, 128, [97], [97], 0), (6, 3, 112, [33], [200], 50), (32, 8, 64, [15, 1, 130, 31], [15, 300, 130, 95], 0),
    (32, 32, 48, [16, 40, 3], [16, 161, 257], 33)])
def test_float32_prompt_attention(ops, heads, kvheads, dim, lens, contexts, window):
    """The float32 prompt kernel beside 64 bits: rows of several sequences in a block, portions behind a cached context, windows,
    a context that ends inside a tile; behind the contexts the cache holds what is no number.  Then a value that is no number
    inside: only the queries that see it may show it."""
    gen = torch.Generator().manual_seed(dim)
    B, T, pages = len(lens), sum(lens), max(contexts) // 64 + 1
    k, v = torch.randn(B * pages, kvheads, 64, dim, generator=gen), torch.randn(B * pages, kvheads, dim, 64, generator=gen)
    table = torch.randperm(B * pages, generator=gen).to(torch.int32).view(B, pages)
    for b, n in enumerate(contexts):
        page = int(table[b, n // 64])
        k[page, :, n % 64 :], v[page, :, :, n % 64 :] = float("nan"), float("nan")
    q = torch.randn(T, (heads + 2 * kvheads) * dim, generator=gen)
    seq = torch.repeat_interleave(torch.arange(B), torch.tensor(lens)).to(torch.int32)
    pos = torch.cat([torch.arange(c - n, c) for n, c in zip(lens, contexts)]).to(torch.int32)

    def run(values):
        return ops.attention(dev(q), dev(pos), dev(seq), dev(table), dev(k), dev(values), heads, kvheads, dim, dim ** -0.5, window,
                             max_context=max(contexts)).cpu().view(T, heads, dim)

    got = run(v)
    for i in range(T):
        b, hi = int(seq[i]), int(pos[i]) + 1
        lo = max(0, hi - window) if window else 0
        keys = k[table[b].long()].permute(0, 2, 1, 3).reshape(-1, kvheads, dim)[lo:hi].double().repeat_interleave(heads // kvheads, dim=1)
        values = v[table[b].long()].permute(0, 3, 1, 2).reshape(-1, kvheads, dim)[lo:hi].double().repeat_interleave(heads // kvheads, dim=1)
        p = torch.softmax((keys * q[i, : heads * dim].view(heads, dim).double()).sum(-1) * dim ** -0.5, dim=0)
        # 24-bit sums of up to 300 terms of size one
        torch.testing.assert_close(got[i].double(), (p[:, :, None] * values).sum(0), atol=3e-6, rtol=1e-5)
    b = B - 1
    j = contexts[b] - lens[b] // 2 - 1  # a token of the last sequence's own
    broken = v.clone()
    broken[int(table[b, j // 64]), 0, 3, j % 64] = float("inf")
    got2 = run(broken)
    sees = (seq == b) & (pos >= j) & ((pos - j < window) if window else torch.ones(T, dtype=torch.bool))
    assert 0 < int(sees.sum()) < T
    shown = torch.zeros(T, heads, dim, dtype=torch.bool)
    shown[sees, : heads // kvheads, 3] = True
    assert not bool(torch.isfinite(got2[shown]).any()) and bool(torch.isfinite(got2[~shown]).all())
    torch.testing.assert_close(got2[~shown], got[~shown], atol=3e-6, rtol=1e-5)


@pytest.mark.parametrize("heads, kvheads, dim, window", [(4, 4, 16, 0), (6, 2, 128, 0), (3, 1, 48, 37)])
def test_float32_attention_has_the_same_bits_in_any_step(ops, heads, kvheads, dim, window):
    """A float32 row's attention alone, in its whole prompt, in portions, in decode steps (with padding rows, beside more sequences
    than a block has rows) and beside a long context: the same bits."""
    gen = torch.Generator().manual_seed(dim)
    contexts = [1, 7, 16, 17, 33, 70, 131] + [5 + 3 * i for i in range(12)] + [900]
    B, pages = len(contexts), 15
    k, v = dev(torch.randn(B * pages, kvheads, 64, dim, generator=gen)), dev(torch.randn(B * pages, kvheads, dim, 64, generator=gen))
    table = dev(torch.randperm(B * pages, generator=gen).to(torch.int32).view(B, pages))
    q = [dev(torch.randn(n, (heads + 2 * kvheads) * dim, generator=gen)) for n in contexts]

    def run(pieces, decode=False):  # [(sequence or -1, first position, tokens)] -> the rows' results
        ids = dev(torch.cat([torch.full((n,), b) for b, _, n in pieces]).to(torch.int32))
        pos = dev(torch.cat([torch.arange(at, at + n) for _, at, n in pieces]).to(torch.int32))
        rows = torch.cat([q[max(b, 0)][at : at + n] for b, at, n in pieces])
        return ops.attention(rows, pos, ids, table, k, v, heads, kvheads, dim, dim ** -0.5, window, decode=decode, max_context=max(contexts)).cpu()

    whole = [run([(b, 0, n)]) for b, n in enumerate(contexts)]
    together = run([(b, 0, n) for b, n in enumerate(contexts)]).split(contexts)
    for b, n in enumerate(contexts):
        assert torch.equal(together[b], whole[b])
        for cut in {1, n // 2, n - 1} - {0, n}:
            assert torch.equal(run([(b, 0, cut)]), whole[b][:cut]) and torch.equal(run([(b, cut, n - cut)]), whole[b][cut:])
    last = [(b, n - 1, 1) for b, n in enumerate(contexts)]
    single = run(last[:9] + [(-1, 0, 1)] + last[9:], decode=True)
    want = torch.cat([w[-1:] for w in whole])
    assert torch.equal(torch.cat([single[:9], single[10:]]), want) and not bool(single[9].any())
    mixed = run(last[7:] + [(5, 3, 60)])  # running sequences and a portion, in one step that is no decode step
    assert torch.equal(mixed, torch.cat([want[7:], whole[5][3:63]]))


@pytest.mark.parametrize("rows, width, act, weight_type", [(1, 4, torch.bfloat16, torch.bfloat16), (3, 260, torch.float32, torch.float32),
                                                           (257, 2048, torch.bfloat16, torch.float32), (2, 16384, torch.float32, torch.bfloat16),
                                                           (5, 4096, torch.bfloat16, None)])
def test_embed_norm_is_embed_and_add_norm(ops, rows, width, act, weight_type):
    """The same bits as the two kernels it stands for; sizes that it leaves to them; and a choice that advances positions."""
    gen = torch.Generator().manual_seed(width)
    table = dev(torch.randn(50, width, generator=gen).to(act))
    ids = dev(torch.randint(0, 50, (rows,), generator=gen, dtype=torch.int32))
    weight = None if weight_type is None else dev(torch.randn(width, generator=gen).to(weight_type))
    want = ops.embed(ids, table, 1.5)
    resid, normed = ops.embed_norm(ids, table, 1.5, weight, 1e-5)
    assert torch.equal(resid, want) and torch.equal(normed, ops.add_norm(want, None, weight, None, 1e-5, act))
    assert ops.embed_norm(ids, dev(torch.randn(50, width + 2, generator=gen)), 1.0, None, 1e-5) is None
    positions, seq = dev(torch.arange(rows, dtype=torch.int32)), dev((torch.arange(rows, dtype=torch.int32) % 3) - 1)
    logits = dev(torch.randn(rows, 50 * width, generator=gen)) if rows * width < 10000 else dev(torch.randn(rows, 60, generator=gen))
    assert torch.equal(ops.sample(logits, False, positions=positions, seq_of_token=seq), ops.sample(logits, False))
    assert torch.equal(positions, torch.arange(rows, device=seq.device, dtype=torch.int32) + (seq >= 0))


def test_add_norm_with_mean_and_shift(ops):
    torch.manual_seed(2)
    x = torch.randn(3, 48) + 1.5
    w, b = torch.randn(48), torch.randn(48)
    out = ops.add_norm(dev(x.clone()), None, dev(w), dev(b), 1e-5, torch.float32, use_mean=True)
    torch.testing.assert_close(out.cpu(), torch.nn.functional.layer_norm(x, (48,), w, b, 1e-5), atol=1e-5, rtol=1e-5)
    # a float32 weight with bfloat16 activations (a tensor the checkpoint keeps in 32-bit)
    out = ops.add_norm(dev(x.clone()), None, dev(w), None, 1e-5, torch.bfloat16)
    torch.testing.assert_close(out.cpu().float(), P.rms_norm(x, w, 1e-5), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gated_act(ops, dtype):
    torch.manual_seed(3)
    gu = torch.randn(7, 2 * 44).to(dtype)
    bias = torch.randn(2 * 44).to(dtype)
    out = ops.gated_act(dev(gu), dev(bias), "swish").cpu().float()
    g = gu.float() + bias.float()
    torch.testing.assert_close(out, P.silu(g[:, :44]) * g[:, 44:], **tol(dtype))
    out = ops.gated_act(dev(gu), None, "silu").cpu().float()
    torch.testing.assert_close(out, P.silu(gu.float()[:, :44]) * gu.float()[:, 44:], **tol(dtype))


def test_cast_and_bias(ops):
    x = torch.randn(1000)
    assert torch.equal(ops.cast(dev(x), torch.bfloat16).cpu(), x.to(torch.bfloat16))
    assert torch.equal(ops.cast(dev(x.to(torch.bfloat16)), torch.float32).cpu(), x.to(torch.bfloat16).float())
    m = torch.randn(4, 10)
    b = torch.randn(10)
    torch.testing.assert_close(ops.bias_add_(dev(m.clone()), dev(b)).cpu(), m + b)


def test_rope_table(ops):
    freqs = P.rope_frequencies(24, 500000.0)
    cos, sin = ops.rope_table(dev(freqs), 300)
    angles = torch.outer(torch.arange(300).float(), freqs)
    torch.testing.assert_close(cos.cpu(), torch.cos(angles), atol=2e-6, rtol=0)
    torch.testing.assert_close(sin.cpu(), torch.sin(angles), atol=2e-6, rtol=0)
    # large angles keep their accuracy (positions in the thousands times frequency one)
    cos, sin = ops.rope_table(dev(torch.tensor([1.0, 0.37])), 9000)
    a = torch.outer(torch.arange(9000).float(), torch.tensor([1.0, 0.37]))
    torch.testing.assert_close(cos.cpu(), torch.cos(a.double()).float(), atol=5e-7, rtol=0)


# --------------------------------------------------------------------------
# paged cache helpers
# --------------------------------------------------------------------------
def make_pages(lengths, K, D, dtype, seed=0, extra_pages=3):
    """Random page assignment: returns (block_table [B, P] int32, n_pages)."""
    g = torch.Generator().manual_seed(seed)
    per_seq = [-(-n // PAGE) for n in lengths]
    total = sum(per_seq) + extra_pages
    perm = torch.randperm(total, generator=g).tolist()
    width = max(per_seq)
    table = torch.full((len(lengths), width), -1, dtype=torch.int32)
    it = iter(perm)
    for b, n in enumerate(per_seq):
        for i in range(n):
            table[b, i] = next(it)
    return table, total


def fill_cache(table, ks, vs, n_pages, dtype):
    """ks[b]: [len, K, D] -> caches in the kernels' layout."""
    K, D = ks[0].shape[1:]
    kc = torch.zeros(n_pages, K, PAGE, D, dtype=dtype)
    vc = torch.zeros(n_pages, K, D, PAGE, dtype=dtype)
    for b, (k, v) in enumerate(zip(ks, vs)):
        for pos in range(k.shape[0]):
            page = int(table[b, pos // PAGE])
            kc[page, :, pos % PAGE, :] = k[pos].to(dtype)
            vc[page, :, :, pos % PAGE] = v[pos].to(dtype)
    return kc, vc


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,K,D,rot", [(4, 2, 16, 16), (3, 1, 24, 24), (2, 2, 32, 16), (2, 1, 6, 6), (8, 2, 128, 128), (3, 3, 256, 64)])
@pytest.mark.parametrize("starts,lens", [([0, 70, 5], [9, 3, 130]), ([0, 64, 8, 3], [200, 72, 56, 13])])
def test_rope_kv_write(ops, dtype, H, K, D, rot, starts, lens):
    """The second layout has runs of tokens that start at multiples of 8 places of their pages and cross page
    borders (whole 16-byte pieces of the transposed value pages), the first has none to speak of."""
    torch.manual_seed(4)
    total = [s + n for s, n in zip(starts, lens)]
    table, n_pages = make_pages(total, K, D, dtype, seed=1)
    T = sum(lens)
    qkv = torch.randn(T, (H + 2 * K) * D).to(dtype)
    positions = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lens)]).int()
    seq = torch.cat([torch.full((n,), b) for b, n in enumerate(lens)]).int()
    freqs = P.rope_frequencies(rot, 10000.0)
    cos, sin = ops.rope_table(dev(freqs), 256)
    kc = torch.zeros(n_pages, K, PAGE, D, dtype=dtype, device="cuda")
    vc = torch.zeros(n_pages, K, D, PAGE, dtype=dtype, device="cuda")
    q_dev = dev(qkv.clone())
    ops.rope_kv_write(q_dev, dev(positions), dev(seq), dev(table), cos, sin, rot, kc, vc, H, K, D)
    out = q_dev.cpu().float()
    x = qkv.float()
    q = x[:, : H * D].reshape(T, H, D)
    k = x[:, H * D : (H + K) * D].reshape(T, K, D)
    v = x[:, (H + K) * D :].reshape(T, K, D)

    def rotate(t):
        r = P.rope_rotate(t[..., :rot], positions, freqs)
        return torch.cat([r, t[..., rot:]], dim=-1)

    torch.testing.assert_close(out[:, : H * D].reshape(T, H, D), rotate(q), **tol(dtype))
    # v columns of qkv untouched
    assert torch.equal(out[:, (H + K) * D :], x[:, (H + K) * D :])
    kc, vc = kc.cpu().float(), vc.cpu().float()
    rk = rotate(k)
    for t in range(T):
        page = int(table[int(seq[t]), int(positions[t]) // PAGE])
        off = int(positions[t]) % PAGE
        torch.testing.assert_close(kc[page, :, off, :], rk[t], **tol(dtype))
        torch.testing.assert_close(vc[page, :, :, off], v[t].to(dtype).float(), **tol(dtype))
    # pages of no sequence stay zero: nothing was written elsewhere
    used = set(int(p) for p in table.flatten() if p >= 0)
    for p in range(n_pages):
        if p not in used:
            assert float(kc[p].abs().sum()) == 0 and float(vc[p].abs().sum()) == 0


@pytest.mark.parametrize("M", [1, 8, 20, 32, 40, 64, 81, 128, 129, 150, 161, 192])
@pytest.mark.parametrize("H,K,D,rot,E", [(4, 2, 16, 16, 64), (3, 1, 48, 48, 40), (8, 8, 32, 16, 256), (40, 4, 128, 128, 32), (30, 2, 136, 136, 32)])
def test_qkv_rope_write_equals_the_separate_kernels(ops, M, H, K, D, rot, E):
    """The decode-time fusion (projection + rotation + cache write) against linear followed by rope_kv_write."""
    torch.manual_seed(11)
    dtype = torch.bfloat16
    N = (H + 2 * K) * D
    x = torch.randn(M, E).to(dtype)
    w = (torch.randn(N, E) * 0.2).to(dtype)
    bias = torch.randn(N).to(dtype)
    positions = torch.randint(0, 200, (M,)).int()
    seq = torch.arange(M).int()
    if M > 2:
        seq[1] = -1  # a padding row: nothing of it may reach the cache
        seq[2:] -= 1
    n_seqs = int(seq.max()) + 1
    table, n_pages = make_pages([256] * n_seqs, K, D, dtype, seed=3)
    freqs = P.rope_frequencies(rot, 10000.0)
    cos, sin = ops.rope_table(dev(freqs), 256)
    for b in (None, bias):
        caches = []
        outs = []
        for fused in (False, True):
            kc = torch.zeros(n_pages, K, PAGE, D, dtype=dtype, device="cuda")
            vc = torch.zeros(n_pages, K, D, PAGE, dtype=dtype, device="cuda")
            args = (dev(positions), dev(seq), dev(table), cos, sin, rot, kc, vc, H, K, D)
            if fused:
                qkv = ops.qkv_rope_write(dev(x), dev(w), None if b is None else dev(b), *args)
            else:
                qkv = ops.linear(dev(x), dev(w), None if b is None else dev(b))
                ops.rope_kv_write(qkv, *args)
            outs.append(qkv[:, : H * D].cpu().float()[seq >= 0])  # a padding row's queries are never read
            caches.append((kc.cpu().float(), vc.cpu().float()))
        # The separate kernels round the projection to bfloat16 before they rotate it, the fused kernel rotates the
        # float32 sums: an element that the rotation makes small out of two large ones differs by up to the rounding
        # of those two, half a bfloat16 step (2^-9 of the largest value) each.
        step = 2.0 ** -8 * max(float(outs[0].abs().max()), float(caches[0][0].abs().max()))
        torch.testing.assert_close(outs[1], outs[0], atol=step, rtol=2e-2)
        torch.testing.assert_close(caches[1][0], caches[0][0], atol=step, rtol=2e-2)
        torch.testing.assert_close(caches[1][1], caches[0][1], atol=2e-2, rtol=2e-2)
        assert float(caches[0][0].abs().sum()) > 0


# --------------------------------------------------------------------------
def reference_attention(qs, ks, vs, starts, H, K, scale=None, window=0):
    """qs[b]: [n_b, H, D] queries at positions starts[b]..; ks/vs[b]: [len_b, K, D] all keys."""
    outs = []
    for q, k, v, s in zip(qs, ks, vs, starts):
        n = q.shape[0]
        full_q = torch.zeros(k.shape[0], H, q.shape[2])
        full_q[s : s + n] = q
        o = P.causal_attention(full_q, k.float(), v.float(), scale=scale, window=window)
        outs.append(o[s : s + n])
    return torch.cat(outs).reshape(sum(q.shape[0] for q in qs), -1)


def reference_attention_rows(qs, ks, vs, starts, H, K, scale=None, window=0):
    """The same attention for the query rows only (fms/modules/attention.py:215-294: head h reads kv head
    h // (H / K), key j is visible to the query at position p if j <= p, and p - j < window if there is one):
    for contexts so long that the whole square of scores of causal_attention would not fit."""
    outs = []
    for q, k, v, s in zip(qs, ks, vs, starts):
        n, _, D = q.shape
        sc = scale if scale is not None else 1 / math.sqrt(D)
        pos = torch.arange(s, s + n)[:, None]
        key = torch.arange(k.shape[0])[None, :]
        visible = key <= pos
        if window:
            visible &= pos - key < window
        o = torch.zeros(n, H, D)
        for h in range(H):
            kh = h // (H // K)
            scores = (q[:, h].double() @ k[:, kh].double().t()) * sc
            probs = torch.softmax(scores.masked_fill(~visible, float("-inf")), dim=-1)
            o[:, h] = (probs @ v[:, kh].double()).float()
        outs.append(o)
    return torch.cat(outs).reshape(sum(q.shape[0] for q in qs), -1)


def test_the_two_attention_references_agree():
    torch.manual_seed(3)
    ks, vs = [torch.randn(90, 2, 16)], [torch.randn(90, 2, 16)]
    qs = [torch.randn(7, 4, 16)]
    for window in (0, 20):
        torch.testing.assert_close(reference_attention_rows(qs, ks, vs, [83], 4, 2, window=window),
                                   reference_attention(qs, ks, vs, [83], 4, 2, window=window), atol=1e-5, rtol=1e-5)


def attention_case(ops, dtype, H, K, D, starts, lens, window=0, decode=False, scale=None, spike=False, **kw):
    torch.manual_seed(5)
    totals = [s + n for s, n in zip(starts, lens)]
    table, n_pages = make_pages(totals, K, D, dtype, seed=2)
    ks = [torch.randn(n, K, D).to(dtype).float() for n in totals]
    vs = [torch.randn(n, K, D).to(dtype).float() for n in totals]
    qs = [torch.randn(n, H, D).to(dtype).float() for n in lens]
    if spike:
        # one far key decides the result: a kernel that loses it (a split, a page, a mask edge) fails visibly
        for b in range(len(lens)):
            far = totals[b] // 3
            qs[b][-1, :, :] = 0
            qs[b][-1, :, 0] = 8.0
            ks[b][:, :, 0] = -1.0
            ks[b][far, :, 0] = 8.0
    kc, vc = fill_cache(table, ks, vs, n_pages, dtype)
    T = sum(lens)
    q_flat = torch.cat([q.reshape(q.shape[0], H * D) for q in qs]).to(dtype)
    # queries sit inside wider rows, as in the fused qkv buffer
    wide = torch.zeros(T, (H + 2 * K) * D, dtype=dtype)
    wide[:, : H * D] = q_flat
    positions = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lens)]).int()
    seq = torch.cat([torch.full((n,), b) for b, n in enumerate(lens)]).int()
    qblock = kw.pop("qblock", None) or ops.prefill_qblock(H, K, D, T)
    qb_start, qb_len, base = [], [], 0
    for n in lens:
        for off in range(0, n, qblock):
            qb_start.append(base + off)
            qb_len.append(min(qblock, n - off))
        base += n
    sc = scale if scale is not None else 1 / math.sqrt(D)
    out = ops.attention(
        dev(wide), dev(positions), dev(seq), dev(table), dev(kc), dev(vc), H, K, D, sc, window,
        decode=decode, max_context=max(totals),
        qblock_start=dev(torch.tensor(qb_start, dtype=torch.int32)), qblock_len=dev(torch.tensor(qb_len, dtype=torch.int32)), qblock_tokens=qblock, **kw,
    )
    rows_only = max(totals) > 3000  # the whole square of scores of a long context is too much for the plain function
    want = (reference_attention_rows if rows_only else reference_attention)(qs, ks, vs, starts, H, K, scale=sc, window=window)
    torch.testing.assert_close(out.cpu().float(), want, **(dict(atol=3e-5, rtol=3e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)))


@pytest.mark.parametrize("H,K,D", [(4, 2, 16), (4, 1, 24), (3, 3, 40), (2, 1, 8)])
def test_attention_generic_f32(ops, H, K, D):
    attention_case(ops, torch.float32, H, K, D, starts=[0, 0, 60], lens=[70, 1, 9])
    attention_case(ops, torch.float32, H, K, D, starts=[299, 64], lens=[1, 1], decode=True)


@pytest.mark.parametrize("H,K,D", [(4, 2, 16), (4, 1, 48), (6, 3, 128), (2, 2, 64), (32, 1, 32), (2, 1, 256), (5, 5, 80), (8, 2, 128), (12, 2, 64),
                                   (16, 2, 128), (4, 4, 128), (24, 1, 128)])
def test_attention_prefill_bf16(ops, H, K, D):
    attention_case(ops, torch.bfloat16, H, K, D, starts=[0, 0, 0], lens=[200, 1, 33])
    # a chunk that continues a cached prefix
    attention_case(ops, torch.bfloat16, H, K, D, starts=[100, 64, 0], lens=[70, 5, 129])
    attention_case(ops, torch.bfloat16, H, K, D, starts=[0, 30], lens=[300, 100])


@pytest.mark.parametrize("H,K,D", [(4, 2, 16), (4, 1, 48), (8, 2, 128), (2, 2, 64), (40, 2, 32), (2, 1, 256), (5, 5, 80),
                                   (16, 2, 128), (4, 4, 128), (24, 1, 128)])
def test_attention_decode_bf16(ops, H, K, D):
    attention_case(ops, torch.bfloat16, H, K, D, starts=[0, 63, 64, 700], lens=[1, 1, 1, 1], decode=True)
    attention_case(ops, torch.bfloat16, H, K, D, starts=[1500, 2], lens=[1, 1], decode=True, pages_per_block=2, waves=1)
    attention_case(ops, torch.bfloat16, H, K, D, starts=[1500, 2], lens=[1, 1], decode=True, pages_per_block=5, waves=3)
    attention_case(ops, torch.bfloat16, H, K, D, starts=[1500, 2], lens=[1, 1], decode=True, pages_per_block=24, waves=8)
    attention_case(ops, torch.bfloat16, H, K, D, starts=[1500, 2, 600], lens=[1, 1, 1], decode=True, pages_per_block=16, waves=4)
    # the order in which the blocks take the rows changes nothing; several pages a wave run as a pipeline
    attention_case(ops, torch.bfloat16, H, K, D, starts=[40, 1500, 2, 600], lens=[1, 1, 1, 1], decode=True, pages_per_block=24, waves=2,
                   row_order=dev(torch.tensor([1, 3, 0, 2], dtype=torch.int32)))
    if D == 128:
        # pages by way of LDS: blocks of up to 4 and of up to 8 waves, whole and partly filled pages, splits
        for pages, waves in ((64, 8), (64, 3), (5, 2), (2, 1), (16, 4)):
            attention_case(ops, torch.bfloat16, H, K, D, starts=[1500, 2, 600, 63, 64, 190], lens=[1, 1, 1, 1, 1, 1], decode=True,
                           pages_per_block=pages, waves=waves, staged=True)


@pytest.mark.parametrize("waves", [3, 8])
@pytest.mark.parametrize("longest", [1300, 1500])
def test_attention_decode_on_both_sides_of_what_the_caches_hold(ops, waves, longest):
    """Six sequences of 8 kv heads: up to 1302 tokens their pages are loaded as ones that stay in the caches, from there on not."""
    attention_case(ops, torch.bfloat16, 16, 8, 128, starts=[longest, 2, 600, 63, 64, 190], lens=[1] * 6, decode=True, pages_per_block=8, waves=waves)


@pytest.mark.parametrize("waves", [3, 8])
def test_attention_decode_of_pages_that_several_blocks_read(ops, waves):
    """More query heads a kv head than a tile holds, and more pages than the caches: every page is read by two blocks or three."""
    attention_case(ops, torch.bfloat16, 160, 8, 128, starts=[1500, 2, 600, 63, 64, 190], lens=[1] * 6, decode=True, pages_per_block=8, waves=waves)


# windows whose first key is the first, second, third and last of four, windows shorter than four keys and longer than a block's 256
@pytest.mark.parametrize("window", [1, 2, 3, 6, 65, 259, 300])
@pytest.mark.parametrize("H,K,D", [(4, 2, 40), (2, 1, 50), (3, 3, 128)])
def test_attention_generic_f32_window(ops, window, H, K, D):
    attention_case(ops, torch.float32, H, K, D, starts=[0, 301, 62], lens=[9, 6, 7], window=window)


@pytest.mark.parametrize("dtype,decode", [(torch.float32, False), (torch.bfloat16, False), (torch.bfloat16, True)])
def test_attention_far_key_and_window(ops, dtype, decode):
    lens = [1, 1] if decode else [40, 3]
    if decode:
        attention_case(ops, dtype, 8, 2, 128, starts=[900, 130], lens=lens, decode=True, spike=True, staged=True)
        attention_case(ops, dtype, 8, 2, 128, starts=[900, 130], lens=lens, decode=True, window=70, staged=True)
    attention_case(ops, dtype, 4, 2, 32, starts=[900, 130], lens=lens, decode=decode, spike=True)
    attention_case(ops, dtype, 4, 2, 32, starts=[900, 130], lens=lens, decode=decode, window=100)
    attention_case(ops, dtype, 4, 2, 32, starts=[900, 130], lens=lens, decode=decode, window=64, scale=0.3)
    attention_case(ops, dtype, 4, 2, 32, starts=[900, 130], lens=lens, decode=decode, window=1)


def test_attention_over_long_contexts(ops):
    """Contexts of 8200, 12000 and 20000 tokens beside short ones: the decode kernel with the split that the wrapper
    picks for such a bound and with others, pages through LDS and not, a far key that decides the result, a window
    whose edge lies thousands of tokens back; the prefill kernel for a chunk behind a cached prefix of 8000 tokens and for a prompt of 3200 tokens;
    the float32 kernel."""
    bf, f32 = torch.bfloat16, torch.float32
    attention_case(ops, bf, 8, 2, 128, starts=[8199, 19999, 2], lens=[1, 1, 1], decode=True, spike=True)
    attention_case(ops, bf, 8, 2, 128, starts=[8199, 19999, 2, 700], lens=[1, 1, 1, 1], decode=True, staged=True)
    attention_case(ops, bf, 8, 2, 128, starts=[8199, 19999, 2], lens=[1, 1, 1], decode=True, staged=True, window=5000)
    attention_case(ops, bf, 8, 2, 128, starts=[19999, 64], lens=[1, 1], decode=True, staged=True, pages_per_block=40, waves=8, spike=True)
    attention_case(ops, bf, 4, 1, 64, starts=[11999, 0], lens=[1, 1], decode=True, spike=True)
    attention_case(ops, bf, 6, 2, 80, starts=[9000], lens=[1], decode=True, window=4097)
    attention_case(ops, bf, 8, 2, 128, starts=[8000, 0], lens=[200, 70], spike=True)
    attention_case(ops, bf, 8, 2, 128, starts=[0, 0], lens=[3200, 33], spike=True)  # a long prompt whole: a hundred query blocks
    attention_case(ops, bf, 4, 4, 32, starts=[5000], lens=[100], window=3000)
    attention_case(ops, f32, 4, 2, 16, starts=[9000, 5], lens=[3, 2], spike=True)
    attention_case(ops, f32, 4, 2, 16, starts=[9000], lens=[1], decode=True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_score_terms(ops, dtype):
    """Further terms of the scores (fms/modules/positions.py:9-36, the reference's adjusted_mask; :78-105: a bias of
    -|key position - query position| * scale[head]): a slope per head times the distance, and a soft cap.  Against
    softmax(cap * tanh(q.k * scale / cap) - slope * distance) written out; the special cases: slope 0 and a cap far
    above the scores is plain attention, a steep slope leaves every query its own value."""
    torch.manual_seed(9)
    H, K, D = 6, 2, 16
    starts, lens = [0, 130, 5], [70, 2, 1]
    totals = [s + n for s, n in zip(starts, lens)]
    table, n_pages = make_pages(totals, K, D, dtype, seed=4)
    ks = [torch.randn(n, K, D).to(dtype).float() for n in totals]
    vs = [torch.randn(n, K, D).to(dtype).float() for n in totals]
    qs = [2 * torch.randn(n, H, D).to(dtype).float() for n in lens]
    kc, vc = fill_cache(table, ks, vs, n_pages, dtype)
    q_flat = torch.cat([q.reshape(q.shape[0], H * D) for q in qs]).to(dtype)
    positions = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lens)]).int()
    seq = torch.cat([torch.full((n,), b) for b, n in enumerate(lens)]).int()
    sc = 1 / math.sqrt(D)

    def run(slopes, cap):
        sl = dev(torch.tensor(slopes, dtype=torch.float32)) if slopes is not None else None
        return ops.attention(dev(q_flat), dev(positions), dev(seq), dev(table), dev(kc), dev(vc), H, K, D, sc, 0,
                             score_slopes=sl, soft_cap=cap, force_generic=True).cpu().float()

    def want(slopes, cap):
        outs = []
        for q, k, v, s in zip(qs, ks, vs, starts):
            n = q.shape[0]
            pos = torch.arange(s, s + n)[:, None]
            key = torch.arange(k.shape[0])[None, :]
            o = torch.zeros(n, H, D)
            for h in range(H):
                kh = h // (H // K)
                scores = (q[:, h].double() @ k[:, kh].double().t()) * sc
                if cap:
                    scores = cap * torch.tanh(scores / cap)
                if slopes is not None:
                    scores = scores - slopes[h] * (pos - key).abs()
                probs = torch.softmax(scores.masked_fill(key > pos, float("-inf")), dim=-1)
                o[:, h] = (probs @ v[:, kh].double()).float()
            outs.append(o.reshape(n, H * D))
        return torch.cat(outs)

    tolerance = dict(atol=3e-5, rtol=3e-5) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)
    slopes = [2.0 ** -(i + 1) for i in range(H)]
    plain = run(None, 0.0)
    torch.testing.assert_close(plain, want(None, 0.0), **tolerance)
    for sl, cap in ((slopes, 0.0), (None, 1.5), (slopes, 1.5)):
        got = run(sl, cap)
        torch.testing.assert_close(got, want(sl, cap), **tolerance)
        assert float((got - plain).abs().max()) > 0.05  # the term did something
    torch.testing.assert_close(run([0.0] * H, 1e4), plain, **tolerance)
    own = torch.cat([v[s : s + n].repeat_interleave(H // K, dim=1).reshape(n, H * D) for v, s, n in zip(vs, starts, lens)])
    torch.testing.assert_close(run([200.0] * H, 0.0), own, **tolerance)
    with pytest.raises(ValueError):
        run(slopes[:-1], 0.0)


def test_attention_generic_bf16_agrees(ops):
    attention_case(ops, torch.bfloat16, 4, 2, 16, starts=[0, 10], lens=[70, 3], force_generic=True)


# --------------------------------------------------------------------------
@pytest.mark.parametrize("M,N,K", [(1, 40, 24), (5, 100, 176), (64, 64, 64), (130, 257, 96), (70, 4096, 40)])
def test_gemm_f32(ops, M, N, K):
    torch.manual_seed(6)
    x, w, b = torch.randn(M, K), torch.randn(N, K), torch.randn(N)
    out = ops.linear(dev(x), dev(w), dev(b)).cpu()
    torch.testing.assert_close(out, (x.double() @ w.double().t() + b.double()).float(), atol=1e-4, rtol=1e-5)


# every tile shape with rows, columns and K past its last whole tile, in blocks of eight waves: 16x16 (9 by 300 of K = 2052, 17 by 300 of 516), 16x32 (9 by
# 4100 of 516), 16x48 (9 by 8200 of 516, 513 by 300 of 132), 16x64 (33 by 4100 of 132, 48 of 1028), 32x32 (17 by 8190 of 132, 513 by 300 of
# 516), the same with K one more (not 16-byte aligned); of four: 16x16 (1 by 300 of 261, 61 of 260), 16x32 (33 by 8200 of 129, 48 by 4100 of 260 and 261), 32x32
# (17 by 8190 of 84 and 261, 130 by 8200 of 261); through LDS: 32x64 (130 by 3000 of 132, 17 by 8200 of 132), 64x64 (301 by 8200 of 260, 33 of 1028), 64x128
# (513 by 16390 of 100, 130 by 8200 of 260).  Rows at an odd stride: those of eight and four waves.  K up to 80, odd K up to 128: sums in
# float64, waves of 16x16 (8 by 4096, 130 by 4100) and 32x32 (from 301 by 8200 on); K up to 4: a row of W a thread
@pytest.mark.parametrize("M,N,K", [(1, 17, 130), (8, 4096, 33), (17, 300, 516), (48, 4100, 260), (130, 3000, 132), (130, 4100, 65), (130, 4100, 68), (64, 8190, 100), (301, 8200, 36), (513, 16390, 20), (513, 16390, 7),
                                   (17, 300, 261), (48, 4100, 261), (130, 4100, 261), (130, 8200, 260), (301, 8200, 260), (513, 16390, 100),
                                   (301, 8200, 96), (301, 8200, 255), (17, 300, 255), (9, 12250, 260), (13, 12250, 261),
                                   (1, 300, 1), (17, 256, 2), (33, 255, 3), (16, 257, 4), (130, 1, 4),
                                   (9, 300, 2052), (9, 300, 2053), (9, 4100, 516), (9, 4100, 517), (9, 8200, 516), (513, 300, 132), (513, 300, 133),
                                   (33, 4100, 132), (33, 4100, 133), (48, 4100, 1028), (48, 4100, 1029), (17, 8190, 132), (17, 8190, 133), (513, 300, 516),
                                   (1, 300, 261), (61, 300, 260), (33, 8200, 129), (17, 8190, 84), (17, 8190, 261), (17, 8200, 132), (33, 8200, 1028),
                                   (130, 8200, 80), (301, 8200, 127), (17, 300, 81)])
@pytest.mark.parametrize("pad", [0, 1, 4])
def test_gemm_f32_tile_shapes(ops, M, N, K, pad):
    torch.manual_seed(61)
    wide, w, b = torch.randn(M, K + pad), torch.randn(N, K), torch.randn(N)
    x = wide[:, :K]
    out = ops.linear(dev(wide)[:, :K], dev(w), dev(b)).cpu().double()
    want = x.double() @ w.double().t() + b.double()
    # what a float32 sum of 16 products is off by at most (16 roundings of the sum of their sizes), and the float64 sum's one rounding at the
    # end.  The bfloat16 products are held to the same: the three that are left out are one rounding of a product (2^-24), the others are
    # exact, and a run of 32 is rounded in six instructions, five of them on sums of 2^-8 of its size
    bound = 2.0 ** -24 * (16.5 * (x.abs().double() @ w.abs().double().t()) + want.abs()) + 1e-30
    assert float(((out - want).abs() / bound).max()) <= 1.0


@pytest.mark.parametrize("K", [3, 7, 36, 80, 96, 100, 127, 129, 255, 257, 1000, 1028, 2049])
def test_gemm_f32_rows_keep_their_bits(ops, K):
    """A row has the same bits whatever else is in the product: blocks of 16x16 to 32x32 results whose four and eight waves share K, of 32x64, 64x64 and
    64x128 through LDS, and for rows that are not 16-byte aligned (an odd stride, an odd K) the former alone; short rows (K up to 80, odd ones up to
    128) in waves of 16x16 (up to 33 rows) and 32x32."""
    torch.manual_seed(62)
    N = 12790
    x, w, b = dev(torch.randn(301, K)), dev(torch.randn(N, K)), dev(torch.randn(N))
    odd = torch.zeros(301, K + 1, device="cuda")[:, :K].copy_(x)
    whole = ops.linear(x, w, b)
    for M in (1, 8, 17, 33, 61, 130):
        assert torch.equal(ops.linear(x[:M], w, b), whole[:M]), M
        assert torch.equal(ops.linear(odd[:M], w, b), whole[:M]), M
    assert torch.equal(ops.linear(odd, w, b), whole)
    assert torch.equal(ops.linear(x, w[:100], b[:100]), whole[:, :100])
    for N in (4096, 8200, 12200):  # 16x32, 16x48 of eight waves
        assert torch.equal(ops.linear(x[:9], w[:N], b[:N]), whole[:9, :N]), N


@pytest.mark.parametrize("M,N,K", [(8, 300, 64), (40, 4096, 132), (301, 4096, 256), (301, 4096, 131), (40, 300, 13)])
def test_gemm_f32_of_numbers_that_are_not_finite_or_nearly(ops, M, N, K):
    """Infinities and numbers that bfloat16 rounds to one show where 64 bits show them, and change no other result's bits; small numbers,
    whose third parts bfloat16 does not hold, count whole."""
    torch.manual_seed(65)
    x, w, b = torch.randn(M, K), torch.randn(N, K), torch.randn(N)
    clean = ops.linear(dev(x), dev(w), dev(b)).cpu()
    y, v = x.clone(), w.clone()
    y[1, 5], y[2, 6], y[3, 7], v[9, 8], v[10] = math.inf, math.nan, 3.4028e38, -math.inf, 0.0
    got = ops.linear(dev(y), dev(v), dev(b)).cpu()
    want = (y.double() @ v.double().t() + b.double()).float()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[got.isinf()])
    torch.testing.assert_close(got[3][want[3].isfinite()], want[3][want[3].isfinite()], rtol=2.0 ** -22, atol=1e-4)
    rows, cols = [0] + list(range(4, M)), [n for n in range(N) if n not in (9, 10)]
    assert torch.equal(got[rows][:, cols], clean[rows][:, cols])
    small = ops.linear(dev(x * 2.0 ** -120), dev(w), None).cpu().double()
    exact = (x * 2.0 ** -120).double() @ w.double().t()
    # the bound of the tile shapes' test
    bound = 2.0 ** -24 * (16.5 * exact.abs().new_tensor(2.0 ** -120) * (x.abs().double() @ w.abs().double().t()) + exact.abs())
    bound += 2.0 ** -148
    assert float(((small - exact).abs() / bound).max()) <= 1.0


@pytest.mark.parametrize("M,N,K", [(8, 300, 132), (301, 4096, 4096), (301, 8200, 256)])
@pytest.mark.parametrize("signs", [False, True])
def test_gemm_f32_of_the_largest_products_left_out(ops, M, N, K, signs):
    """Numbers whose second and third parts are as large as they get, 2^-8 and -2^-17 beside a first part of 1 to 2: the products of the two,
    which are not formed, are then 2^-24 each pair of factors, all of one sign where the factors are, and add up."""
    torch.manual_seed(69)
    rest = 2.0 ** -8 - 2.0 ** -17
    x, w = (1.0 + torch.randint(0, 128, shape).float() / 128 + rest for shape in ((M, K), (N, K)))
    if signs:
        x, w = x * (torch.randint(0, 2, x.shape) * 2 - 1), w * (torch.randint(0, 2, w.shape) * 2 - 1)
    got, exact, size = ops.linear(dev(x), dev(w), None).cpu().double(), x.double() @ w.double().t(), x.abs().double() @ w.abs().double().t()
    # what is left out is 2^-24 of a pair of ones at most; the runs' own roundings as in the tile shapes' test
    assert float(((got - exact).abs() / (2.0 ** -24 * (K + 15.5 * size + exact.abs()))).max()) <= 1.0
    # and the result as a whole no further off than half of float32's last bit, one rounding of every product
    assert float((got - exact).norm() / exact.norm()) < 2.0 ** -24 * (1.5 if signs else 1.0)


@pytest.mark.parametrize("M,N", [(8, 512), (130, 1024), (301, 4096)])
def test_gemm_f32_of_rows_with_runs_of_zeros(ops, M, N):
    """The matrix unit rounds down: what that adds up to cancels between the runs of 32 k-values, also where every other run is zero, or
    every other two or four.  The bound is what a product of float32 instructions was measured at (7.8e-8), less the noise of the norm."""
    torch.manual_seed(68)
    K = 11008
    w = torch.randn(N, K)
    for size in (1, 2, 4):
        for first in (0, 1):
            x = torch.randn(M, K)
            x.view(M, K // 32, 32)[:, (torch.arange(K // 32) // size) % 2 == first] = 0.0
            got, exact = ops.linear(dev(x), dev(w), None).cpu().double(), x.double() @ w.double().t()
            assert float((got - exact).norm() / exact.norm()) < 7.5e-8, (size, first)


@pytest.mark.parametrize("M,N,K", [(5, 300, 40), (8, 12288, 132), (16, 4100, 520), (40, 4096, 132), (130, 4100, 260), (301, 4096, 256), (40, 4096, 131)])
@pytest.mark.parametrize("down", [-105, -115, -125, -140])
def test_gemm_f32_of_small_numbers(ops, M, N, K, down):
    """Rows of x and of W with a small number, or all small, beside large factors: float32's 24 bits count, down to its subnormal numbers,
    and the rows beside them keep their bits."""
    torch.manual_seed(67)
    x, w = torch.randn(M, K), torch.randn(N, K) * 2.0 ** 60
    clean = ops.linear(dev(x), dev(w), None).cpu()
    y, v = x.clone(), w.clone()
    y[1] *= 2.0 ** down
    y[3, K - 1] *= 2.0 ** down
    v[7] *= 2.0 ** (down - 60)
    v[N - 1, 0] *= 2.0 ** (down - 60)
    got = ops.linear(dev(y), dev(v), None).cpu()
    exact = y.double() @ v.double().t()
    # the bound of the tile shapes' test, and half a step of the smallest numbers
    bound = 2.0 ** -24 * (16.5 * (y.abs().double() @ v.abs().double().t()) + exact.abs()) + 2.0 ** -149
    assert float(((got.double() - exact).abs() / bound).max()) <= 1.0
    rows, cols = [m for m in range(M) if m not in (1, 3)], [n for n in range(N) if n not in (7, N - 1)]
    assert torch.equal(got[rows][:, cols], clean[rows][:, cols])
    for few in (1, 2, 4):  # the same bits in the tiles of fewer rows
        assert torch.equal(ops.linear(dev(y[:few]), dev(v), None).cpu(), got[:few])


@pytest.mark.parametrize("M,N", [(301, 4096), (8, 4096)])
def test_gemm_f32_of_results_that_are_not_finite_costs_little(ops, M, N):
    """A product whose results all overflow, or are all infinite, takes a few times as long as another."""
    torch.manual_seed(66)
    K = 4096
    x, w = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda")

    def time(rows, weights):
        ops.linear(rows, weights, None)
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(3):
            ops.linear(rows, weights, None)
        end.record()
        end.synchronize()
        return start.elapsed_time(end)

    usual = time(x, w)
    endless, large = x.clone(), x.abs() * 1e30
    endless[:, 7] = math.inf
    assert time(endless, w.abs()) < 12 * usual
    assert bool(ops.linear(large, w.abs() * 1e30, None).isinf().all())
    assert time(large, w.abs() * 1e30) < 12 * usual


@pytest.mark.parametrize("M,N,K", [(130, 3000, 132), (301, 8200, 260), (513, 16390, 128), (130, 4100, 64)])
def test_gemm_f32_of_rows_far_apart(ops, M, N, K):
    """Rows of x so far apart that a tile's lie just within the 32 bits of bytes that the kernels through LDS count in (32x64, 64x64, 64x128: 2^22
    floats less four), just past them (2^22, to the registers' kernels), and on either side of 32 bits for one of 128 rows; short rows beside them."""
    if torch.cuda.mem_get_info()[0] < 40e9:
        pytest.skip("needs 40 GB of memory")
    torch.manual_seed(64)
    x, w = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda")
    want = ops.linear(x, w, None)
    for stride in ((1 << 22) - 4, 1 << 22, (1 << 23) + 4, (1 << 23) - 4):
        far = torch.empty(M * stride, device="cuda").as_strided((M, K), (stride, 1)).copy_(x)
        assert torch.equal(ops.linear(far, w, None), want)
        del far
    torch.cuda.empty_cache()


def test_gemm_f32_of_more_results_than_a_launch_has_threads(ops):
    """1.7e10 results (69 GB): the threads of one launch are counted in 32 bits."""
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 80e9:
        pytest.skip("needs 80 GB of memory")
    torch.manual_seed(63)
    x, w = torch.randn(131072, 1, device="cuda"), torch.randn(131136, 1, device="cuda")
    out = ops.linear(x, w, None)
    for at in list(range(0, 131072, 8192)) + [131071]:
        assert torch.equal(out[at : at + 40], x[at : at + 40] * w.t())
    del out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("M", [1, 3, 16, 17, 33, 48, 64, 65, 96, 100, 128, 129, 144, 160, 170, 192, 193, 300])
@pytest.mark.parametrize("N,K", [(40, 24), (100, 176), (257, 96), (384, 96), (4096 + 16, 512), (20000, 64)])
def test_gemm_bf16(ops, M, N, K):
    torch.manual_seed(7)
    x = torch.randn(M, K).to(torch.bfloat16)
    w = (torch.randn(N, K) * 0.1).to(torch.bfloat16)
    b = torch.randn(N).to(torch.bfloat16)
    want = x.double() @ w.double().t()
    for out_dtype in (torch.bfloat16, torch.float32):
        for allow_library in (True, False):
            out = ops.linear(dev(x), dev(w), None, out_dtype=out_dtype, allow_library=allow_library).cpu()
            assert out.dtype == out_dtype
            torch.testing.assert_close(out.double(), want, atol=3e-2 if out_dtype == torch.bfloat16 else 2e-3, rtol=1e-2)
    out = ops.linear(dev(x), dev(w), dev(b), out_dtype=torch.float32, allow_library=False).cpu()
    torch.testing.assert_close(out.double(), want + b.double(), atol=2e-3, rtol=1e-2)
    # a float32 bias with bfloat16 weights, and a float32 weight with bfloat16 activations
    out = ops.linear(dev(x), dev(w), dev(b.float()), out_dtype=torch.float32).cpu()
    torch.testing.assert_close(out.double(), want + b.double(), atol=2e-3, rtol=1e-2)
    out = ops.linear(dev(x), dev(w.float()), None).cpu()
    assert out.dtype == torch.bfloat16
    torch.testing.assert_close(out.double(), want, atol=3e-2, rtol=1e-2)


@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 97, 129, 161, 192])
@pytest.mark.parametrize("N,K,skip", [(33004, 72, 0), (512, 4104, 0), (16384, 520, 0), (3080, 776, 0), (7168, 2056, 0), (20, 8200, 0), (300, 1032, 3), (2056, 4104, 3), (16392, 200, 5)])
def test_gemm_bf16_cuts_of_the_wide_product(ops, M, N, K, skip):
    """Two rounds of blocks, slices of K with a short last step, blocks that own fewer rows than they have places for, rows
    that start at no 16-byte address.

    A product of two bfloat16 is exact in float32; a sum of K of them in any order is off by at most K 2^-24 sum |x w|."""
    torch.manual_seed(9)
    rows = torch.randn(M, K + 8).to(torch.bfloat16)
    x = rows[:, skip : skip + K]
    w = (torch.randn(N, K) * 0.1).to(torch.bfloat16)
    out = ops.linear(dev(rows)[:, skip : skip + K], dev(w), None, out_dtype=torch.float32, allow_library=False).cpu().double()
    want = (x.float() @ w.float().t()).double() if N * K > 4e6 else x.double() @ w.double().t()
    bound = 2 * K * 2.0**-24 * (x.float().abs() @ w.float().abs().t()).double()  # (twice: the reference may be float32 too)
    assert bool(((out - want).abs() <= bound).all())


@pytest.mark.parametrize("N,K", [(40, 24), (304, 136), (768, 512), (8200, 512), (16384, 256), (16400, 504), (33000, 264)])
def test_short_products_keep_their_bits(ops, N, K):
    """17 to 192 rows and a K of up to 512: a row has the same bits in every product, whatever the number of rows, the
    kernel that takes them (gemm.hip up to 32 rows and below 16384 weight rows, else gemm_wide.hip) and its cut.  (Not so the
    scale of a norm that was left to the product: the partial sums it comes from are of runs of other lengths.)"""
    torch.manual_seed(10)
    x, w, b = dev(torch.randn(192, K).to(torch.bfloat16)), dev((torch.randn(N, K) * 0.1).to(torch.bfloat16)), dev(torch.randn(N).to(torch.bfloat16))
    stream, nw = dev(torch.randn(192, N)), dev(torch.randn(N))

    def products(M):
        resid = stream[:M].clone()
        scaled, _ = ops.linear_into_stream(x[:M], w, b, resid, nw, 1e-5)
        return [ops.linear(x[:M], w, None), ops.linear(x[:M], w, b, out_dtype=torch.float32), resid, scaled, ops.gated_linear(x[:M], w, b, "swish")]

    whole = products(192)
    for M in (17, 31, 32, 33, 64, 65, 100, 130, 160, 191):
        assert all(torch.equal(got, want[:M]) for got, want in zip(products(M), whole))


@pytest.mark.parametrize("M", [1, 5, 17, 64, 70, 200])
@pytest.mark.parametrize("N,K", [(37, 12), (100, 44), (60, 50), (301, 1000 + 4)])
def test_gemm_bf16_of_widths_that_are_no_multiple_of_8(ops, M, N, K):
    """Rows of such widths are not 16-byte aligned, which the MFMA kernels need: an element-wise kernel takes
    them, so that no width a configuration allows is refused.  Also a view whose row stride is odd."""
    torch.manual_seed(17)
    x = torch.randn(M, K).to(torch.bfloat16)
    w = (torch.randn(N, K) * 0.1).to(torch.bfloat16)
    b = torch.randn(N).to(torch.bfloat16)
    want = x.double() @ w.double().t()
    for out_dtype in (torch.bfloat16, torch.float32):
        out = ops.linear(dev(x), dev(w), None, out_dtype=out_dtype).cpu()
        assert out.dtype == out_dtype
        torch.testing.assert_close(out.double(), want, atol=3e-2 if out_dtype == torch.bfloat16 else 2e-3, rtol=1e-2)
    for bias in (b, b.float()):
        out = ops.linear(dev(x), dev(w), dev(bias), out_dtype=torch.float32).cpu()
        torch.testing.assert_close(out.double(), want + b.double(), atol=2e-3, rtol=1e-2)
    wide = dev(torch.randn(M, K + 3).to(torch.bfloat16))
    out = ops.linear(wide[:, :K], dev(w), None, out_dtype=torch.float32).cpu()
    torch.testing.assert_close(out.double(), wide[:, :K].cpu().double() @ w.double().t(), atol=2e-3, rtol=1e-2)
    if N % 2 == 0:
        out = ops.gated_linear(dev(x), dev(w), dev(b), "swish").cpu().float()
        gu = x.float() @ w.float().t() + b.float()
        want = P.silu(gu[:, : N // 2]) * gu[:, N // 2 :]
        torch.testing.assert_close(out, want, atol=4e-2, rtol=2e-2)


@pytest.mark.parametrize("M", [1, 8, 20, 40, 64, 100, 128, 130, 150, 177, 192, 200])
@pytest.mark.parametrize("hidden,K", [(44, 24), (77, 40), (176, 64), (1000, 96)])
def test_gated_linear(ops, M, hidden, K):
    torch.manual_seed(8)
    for dtype in (torch.bfloat16, torch.float32):
        x = torch.randn(M, K).to(dtype)
        w = (torch.randn(2 * hidden, K) * 0.2).to(dtype)
        b = torch.randn(2 * hidden).to(dtype)
        for bias in (None, b):
            out = ops.gated_linear(dev(x), dev(w), None if bias is None else dev(bias), "swish").cpu().float()
            gu = x.float() @ w.float().t() + (0 if bias is None else bias.float())
            want = P.silu(gu[:, :hidden]) * gu[:, hidden:]
            torch.testing.assert_close(out, want, **(dict(atol=1e-4, rtol=1e-4) if dtype == torch.float32 else dict(atol=4e-2, rtol=2e-2)))


@pytest.mark.parametrize("M", [1, 7, 16, 17, 32, 33, 64, 90, 128, 140, 165, 192])
@pytest.mark.parametrize("N,K,eps", [(48, 24, 1e-5), (96, 176, 1e-6), (4096 + 40, 64, 1e-5), (100, 96, 1e-3), (6144, 32, 1e-5)])
def test_linear_into_stream_and_deferred_row_norm(ops, M, N, K, eps):
    """The last product of a branch adds to the float32 stream and leaves the next norm's input; the
    products that read it (plain, gated, qkv with rotation) finish the norm.  Against the plain formulas:
    stream' = stream + x W^T + b;  y = rms_norm(stream') V^T."""
    torch.manual_seed(12)
    x = torch.randn(M, K).to(torch.bfloat16)
    w = (torch.randn(N, K) * 0.2).to(torch.bfloat16)
    b = torch.randn(N).to(torch.bfloat16)
    resid = torch.randn(M, N) * 3
    resid[0] *= 40  # rows of very different size: a row scale applied to the wrong row shows
    for norm_w in (torch.randn(N).abs().to(torch.bfloat16), torch.randn(N).abs(), None):
        for bias in (None, b):
            stream = dev(resid.clone())
            scaled, row_norm = ops.linear_into_stream(dev(x), dev(w), None if bias is None else dev(bias), stream,
                                                      None if norm_w is None else dev(norm_w), eps)
            want_stream = resid.double() + x.double() @ w.double().t() + (0 if bias is None else bias.double())
            torch.testing.assert_close(stream.cpu().double(), want_stream, atol=2e-3, rtol=1e-4)
            got = stream.cpu()
            torch.testing.assert_close(row_norm.partials.cpu().sum(-1), got.pow(2).sum(-1), rtol=1e-5, atol=1e-5)
            nw = torch.ones(N) if norm_w is None else norm_w.float()
            torch.testing.assert_close(scaled.cpu().float(), (got * nw).to(torch.bfloat16).float(), atol=0, rtol=1e-2)
            if N % 8:
                continue
            # consumers: what they make of (scaled, row_norm) against the product of the normed stream
            normed = P.rms_norm(got, nw, eps)
            N2 = 80
            v = (torch.randn(N2, N) * 0.2).to(torch.bfloat16)
            vb = torch.randn(N2).to(torch.bfloat16)
            bound = dict(atol=0.02 * float((normed @ v.float().t()).abs().max()) + 1e-3, rtol=2e-2)
            out = ops.linear(scaled, dev(v), dev(vb), row_norm=row_norm).cpu().float()
            torch.testing.assert_close(out, normed @ v.float().t() + vb.float(), **bound)
            out = ops.linear(scaled, dev(v), None, out_dtype=torch.float32, row_norm=row_norm).cpu()
            torch.testing.assert_close(out, normed @ v.float().t(), **bound)
            out = ops.gated_linear(scaled, dev(v), dev(vb), "swish", row_norm=row_norm).cpu().float()
            gu = normed @ v.float().t() + vb.float()
            want = P.silu(gu[:, :N2 // 2]) * gu[:, N2 // 2:]  # a product of two rounded values: its own scale
            torch.testing.assert_close(out, want, atol=0.02 * float(want.abs().max()) + 1e-3, rtol=2e-2)
            # the chain: a second product into the stream that reads the first one's rows
            stream2 = dev(resid.clone())
            w2 = (torch.randn(N, N) * 0.1).to(torch.bfloat16)
            ops.linear_into_stream(scaled, dev(w2), None, stream2, None, eps, row_norm=row_norm)
            torch.testing.assert_close(stream2.cpu(), resid + normed @ w2.float().t(), **bound)


@pytest.mark.parametrize("E,F,H,K", [(5120, 13824, 40, 40), (8192, 28672, 64, 8), (2560, 10240, 32, 32)])
def test_decode_products_at_the_layer_sizes_of_other_variants(ops, E, F, H, K):
    """The four products of a layer as a decode step runs them, at the sizes of the 13B, 70B and granite 3B variants
    (the 8B and 7B sizes run through whole models in test_model_shapes_gpu.py): output projection into the stream,
    gate/up with the activation and the deferred norm, down projection into the stream, qkv with rotation and cache
    write and the deferred norm.  Row counts of the kernels for up to 16 rows, for 17 to 32, for 33 to 128 and for 129 to 192.
    References are float32 products of the same operands, on the GPU."""
    torch.manual_seed(31)
    D = E // H
    eps = 1e-5
    wo = (torch.randn(E, E, device="cuda") * 0.02).bfloat16()
    wgu = (torch.randn(2 * F, E, device="cuda") * 0.02).bfloat16()
    wd = (torch.randn(E, F, device="cuda") * 0.02).bfloat16()
    wqkv = (torch.randn((H + 2 * K) * D, E, device="cuda") * 0.02).bfloat16()
    nw = (1 + 0.1 * torch.randn(E, device="cuda")).bfloat16()
    cos, sin = ops.rope_table(dev(P.rope_frequencies(D, 10000.0)), 512)
    for M in (8, 24, 80, 150):
        attn = torch.randn(M, E, device="cuda").bfloat16()
        resid = torch.randn(M, E, device="cuda") * 2
        resid[0] *= 20
        stream = resid.clone()
        # output projection: stream += attn Wo^T, scaled = stream * norm weight, partial sums of squares
        scaled, row_norm = ops.linear_into_stream(attn, wo, None, stream, nw, eps)
        want_stream = resid + attn.float() @ wo.float().t()
        torch.testing.assert_close(stream, want_stream, atol=2e-3, rtol=1e-4)
        normed = want_stream * torch.rsqrt(want_stream.pow(2).mean(-1, keepdim=True) + eps) * nw.float()
        # gate/up with the deferred norm
        hidden = ops.gated_linear(scaled, wgu, None, "swish", row_norm=row_norm)
        gu = normed @ wgu.float().t()
        want_hidden = P.silu(gu[:, :F]) * gu[:, F:]
        torch.testing.assert_close(hidden.float(), want_hidden, atol=0.02 * float(want_hidden.abs().max()) + 1e-3, rtol=2e-2)
        # down projection into the stream
        stream2 = want_stream.clone()
        ops.linear_into_stream(hidden, wd, None, stream2, nw, eps)
        torch.testing.assert_close(stream2, want_stream + hidden.float() @ wd.float().t(), atol=3e-3, rtol=1e-4)
        # qkv with rotation and cache write, against the product followed by the separate rotation kernel
        positions = torch.randint(0, 300, (M,)).int()
        seq = torch.arange(M).int()
        table, n_pages = make_pages([320] * M, K, D, torch.bfloat16, seed=4)
        res = []
        for fused in (True, False):
            kc = torch.zeros(n_pages, K, PAGE, D, dtype=torch.bfloat16, device="cuda")
            vc = torch.zeros(n_pages, K, D, PAGE, dtype=torch.bfloat16, device="cuda")
            args = (dev(positions), dev(seq), dev(table), cos, sin, D, kc, vc, H, K, D)
            if fused:
                qkv = ops.qkv_rope_write(scaled, wqkv, None, *args, row_norm=row_norm)
            else:
                qkv = (normed @ wqkv.float().t()).bfloat16()
                ops.rope_kv_write(qkv, *args)
            res.append((qkv[:, : H * D].float(), kc.float(), vc.float()))
        step = 2.0 ** -7 * max(float(res[1][0].abs().max()), float(res[1][1].abs().max()))  # see test_qkv_rope_write
        for a, b in zip(res[0], res[1]):
            assert float(b.abs().max()) > 0
            torch.testing.assert_close(a, b, atol=step, rtol=2e-2)


def test_qkv_rope_write_takes_a_deferred_row_norm(ops):
    torch.manual_seed(13)
    M, H, K, D, E, eps = 5, 4, 2, 32, 96, 1e-5
    N = (H + 2 * K) * D
    resid = torch.randn(M, E) * 2
    resid[3] *= 30
    nw = torch.randn(E).abs().to(torch.bfloat16)
    x0 = torch.zeros(M, 8).to(torch.bfloat16)
    stream = dev(resid.clone())
    scaled, row_norm = ops.linear_into_stream(dev(x0), dev(torch.zeros(E, 8).to(torch.bfloat16)), None, stream, dev(nw), eps)
    normed = ops.add_norm(dev(resid.clone()), None, dev(nw), None, eps, torch.bfloat16)
    w = (torch.randn(N, E) * 0.2).to(torch.bfloat16)
    positions = torch.randint(0, 200, (M,)).int()
    seq = torch.arange(M).int()
    table, n_pages = make_pages([256] * M, K, D, torch.bfloat16, seed=3)
    cos, sin = ops.rope_table(dev(P.rope_frequencies(D, 10000.0)), 256)
    res = []
    for x, rn in ((normed, None), (scaled, row_norm)):
        kc = torch.zeros(n_pages, K, PAGE, D, dtype=torch.bfloat16, device="cuda")
        vc = torch.zeros(n_pages, K, D, PAGE, dtype=torch.bfloat16, device="cuda")
        qkv = ops.qkv_rope_write(x, dev(w), None, dev(positions), dev(seq), dev(table), cos, sin, D, kc, vc, H, K, D, row_norm=rn)
        res.append((qkv[:, : H * D].cpu().float(), kc.cpu().float(), vc.cpu().float()))
    for a, b in zip(*res):
        assert a.abs().max() > 0
        torch.testing.assert_close(a, b, atol=0.02 * float(a.abs().max()), rtol=2e-2)


@pytest.mark.parametrize("vocab,width", [(128256, 4096), (32000, 4096), (49152, 2560)])
def test_output_head_at_served_vocabularies(ops, vocab, width):
    """The last product of a step at the vocabularies and widths of the registered variants: float32 logits from
    bfloat16 rows, for the row counts of decode batches (the weight-streaming kernels, 1 to 192 rows, in blocks of
    thousands) and above (this package's MFMA kernel), against the float32 product of the same operands; and the
    token choice on those logits."""
    torch.manual_seed(21)
    w = (torch.randn(vocab, width, device="cuda") * 0.02).bfloat16()
    wf = w.float()
    for M in (1, 8, 17, 33, 64, 128, 130, 192, 200):
        x = torch.randn(M, width, device="cuda").bfloat16()
        got = ops.linear(x, w, None, out_dtype=torch.float32)
        want = x.float() @ wf.t()
        assert got.dtype == torch.float32 and tuple(got.shape) == (M, vocab)
        torch.testing.assert_close(got, want, atol=2e-3, rtol=2e-3)
        assert ops.sample(got, False).tolist() == got.argmax(-1).tolist()
    del wf


# --------------------------------------------------------------------------
def test_argmax(ops):
    torch.manual_seed(9)
    logits = torch.randn(6, 1000)
    logits[2, 17] = logits[2, 900] = 50.0  # equal maxima: the lowest index wins
    out = ops.sample(dev(logits), False).cpu()
    want = logits.argmax(-1)
    want[2] = 17
    assert out.tolist() == want.tolist()
    big = torch.randn(2, 128256)
    assert ops.sample(dev(big), False).cpu().tolist() == big.argmax(-1).tolist()


@pytest.mark.parametrize("vocab,top_k,temperature", [(50, 0, 1.0), (384, 10, 0.8), (5000, 3, 2.0), (128256, 50, 0.7), (300, 1000, 1.0),
                                                     (128256, 0, 0.8), (128256, 10, 1.0), (32000, 256, 1.3), (5000, 300, 1.0), (128256, 512, 1.0), (49152, 700, 0.9),
                                                     (1031, 1030, 0.9), (64, 5, 1.0), (65, 64, 1.0)])
def test_sampling(ops, vocab, top_k, temperature):
    torch.manual_seed(10)
    rows = 64
    logits = torch.randn(rows, vocab) * 3
    seeds = [1234 + 7 * r for r in range(rows)]
    counters = [r % 5 for r in range(rows)]
    rng = torch.tensor([[s, c] for s, c in zip(seeds, counters)], dtype=torch.int64)
    rng_dev = dev(rng)
    out = ops.sample(dev(logits), True, temperature, top_k, rng_dev).cpu().tolist()
    assert rng_dev.cpu()[:, 1].tolist() == [c + 1 for c in counters]
    for r in range(rows):
        p = P.sampling_distribution(logits[r], temperature, top_k).double()
        cdf = torch.cumsum(p, 0)
        u = P.draw_uniform(seeds[r], counters[r])  # the plain implementation's own statement of the generator
        tok = out[r]
        assert p[tok] > 0, "a token outside the kept set was drawn"
        lo = float(cdf[tok] - p[tok])
        hi = float(cdf[tok])
        assert lo - 1e-5 <= u <= hi + 1e-5, (r, tok, u, lo, hi)
    if top_k == 3:
        kept = [set(torch.topk(logits[r], 3).indices.tolist()) for r in range(rows)]
        assert all(out[r] in kept[r] for r in range(rows))


def test_sampling_ties_at_threshold_survive(ops):
    logits = torch.full((1, 100), -5.0)
    logits[0, [3, 50, 77]] = 2.0  # top_k=2 but three equal maxima: all three stay
    seen = set()
    for c in range(200):
        rng = dev(torch.tensor([[99, c]], dtype=torch.int64))
        seen.add(int(ops.sample(dev(logits), True, 1.0, 2, rng).cpu()[0]))
    assert seen == {3, 50, 77}


@pytest.mark.parametrize("vocab", [900, 6000])
def test_sampling_with_many_equal_values(ops, vocab):
    """top_k far below the number of equal maxima: every one of them stays, so the draw is uniform over them, in
    index order.  600 of them fit the kernel's short list of candidates (which it has to put in index order);
    4000 do not, and the threshold is found over the whole row."""
    logits = torch.full((1, vocab), 1.5)
    logits[0, ::3] = -4.0  # a third are low values, the others equal maxima
    kept = [i for i in range(vocab) if i % 3]
    for c in range(40):
        rng = dev(torch.tensor([[5, c]], dtype=torch.int64))
        tok = int(ops.sample(dev(logits), True, 0.5, 7, rng).cpu()[0])
        u = P.draw_uniform(5, c)
        assert tok % 3, "a low value was drawn"
        assert abs(kept.index(tok) - u * len(kept)) <= 1.5, (c, tok, u)


def test_sampling_finds_a_far_value(ops):
    """One value stands out at each of many places of a large row, the row's ends and the borders of the stretches
    that the kernel cuts it into among them: with top_k=1 it is drawn whatever the uniform number is."""
    vocab = 128256
    places = [0, 1, 63, 64, 8063, 8064, 8065, 16127, 64512, 120959, 120960, 128191, 128192, vocab - 2, vocab - 1]
    torch.manual_seed(12)
    logits = torch.randn(len(places), vocab)
    for r, at in enumerate(places):
        logits[r, at] = 9.0
    rng = dev(torch.tensor([[77, r] for r in range(len(places))], dtype=torch.int64))
    assert ops.sample(dev(logits), True, 0.9, 1, rng).cpu().tolist() == places
    # and without top_k, at a temperature that leaves the others no mass to speak of
    rng = dev(torch.tensor([[78, r] for r in range(len(places))], dtype=torch.int64))
    assert ops.sample(dev(logits * 20), True, 0.05, 0, rng).cpu().tolist() == places


def test_kernels_refuse_what_they_cannot_do(ops):
    from fms_amd.kernels import KernelError

    with pytest.raises((KernelError, ValueError)):  # a deferred row norm needs rows the MFMA kernels can load
        ops.linear(dev(torch.zeros(2, 12, dtype=torch.bfloat16)), dev(torch.zeros(8, 12, dtype=torch.bfloat16)),
                   row_norm=ops.RowNorm(dev(torch.zeros(2, 1)), 1e-5))
    with pytest.raises(RuntimeError):
        ops.embed(torch.zeros(2, dtype=torch.int32), torch.zeros(4, 4))  # CPU tensors: no CPU path
    with pytest.raises((KernelError, ValueError)):
        ops.sample(dev(torch.zeros(1, 8)), True, 0.0, 0, dev(torch.zeros(1, 2, dtype=torch.int64)))


def test_the_probes_measure_this_gpu(ops):
    """What the benchmark divides by: a kernel that only reads and one that only issues matrix instructions.  On an
    MI355X the first lies between a quarter of and the whole published 8 TB/s, the second between a fifth of and the
    whole published 2.5 PFLOP/s; a probe whose loop the compiler removed, or that counts its work wrongly, falls outside."""
    read, mfma = ops.measured_peaks(read_mib=256, repeats=3)
    assert 2.0e12 < read < 8.0e12, f"a pure read measured at {read / 1e12:.2f} TB/s"
    assert 0.5e15 < mfma < 2.5e15, f"matrix instructions measured at {mfma / 1e15:.2f} PFLOP/s"

