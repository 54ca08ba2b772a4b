"""The bfloat16 products of many rows: every kind of tiles, their edges, several tiles a block, strides and biases.

The reference is the product in float64 of the same bfloat16 numbers.  A float32 sum of K products is at most about K / 32 roundings
of 2^-24 of the sum of the magnitudes away from it (32 products an instruction, one rounding each), allowed are K / 16; a
bfloat16 result is rounded once more, by 2^-9 of itself."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# rows, columns, K, tiles (fmsamd_gemm_tall_plan): one row more than the other kernels take, edges of the tiles, one round and several
PLAIN = [
    (193, 128, 256, 2), (257, 136, 384, 2), (257, 9224, 256, 4), (769, 12296, 384, 0), (4097, 2056, 256, 3), (1537, 12296, 256, 1),
    (3000, 2504, 640, 4), (4689, 4096, 256, 2), (4689, 12296, 256, 0), (4097, 9224, 384, 1), (4689, 2056, 640, 3),
]
GATED = [(193, 136, 256, 2), (193, 9224, 384, 4), (511, 9224, 256, 3), (257, 12296, 384, 0), (1111, 9224, 256, 1), (4689, 2504, 384, 1),
         (4689, 12296, 256, 2), (4689, 6152, 640, 0), (2277, 1032, 640, 4), (4097, 1032, 384, 3)]


def library():
    from fms_amd.kernels.library import load

    return load()


def rows_of(M, K, extra, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(M, K + extra, generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16)[:, :K]


def sums(x, w, bias):
    """(the product in float64, the sums of the magnitudes)"""
    x, w = x.double(), w.double()
    b = torch.zeros(w.shape[0], dtype=torch.float64, device=x.device) if bias is None else bias.double()
    return x @ w.T.contiguous() + b, x.abs() @ w.abs().T.contiguous() + b.abs()


@pytest.mark.parametrize("M,N,K,tiles", PLAIN)
@pytest.mark.parametrize("bias_dtype", [None, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_plain(M, N, K, tiles, bias_dtype, out_dtype):
    from fms_amd.kernels import ops

    lib = library()
    assert lib.fmsamd_gemm_tall_plan(M, N, K, 0) == tiles
    x, w = rows_of(M, K, 8, 1), rows_of(N, K, 0, 2).contiguous()
    bias = None if bias_dtype is None else torch.randn(N, device="cuda").to(bias_dtype)
    wide = torch.full((M + 1, N + 16), 7.0, dtype=out_dtype, device="cuda")
    out = wide[:M, 8 : 8 + N]
    assert lib.fmsamd_gemm_tall_bf16(x.data_ptr(), x.stride(0), w.data_ptr(), bias.data_ptr() if bias is not None else None,
                                     ops._code(bias_dtype) if bias is not None else 0, out.data_ptr(), ops._code(out_dtype), out.stride(0), M, N,
                                     K, ops._stream()) == 0
    want, size = sums(x, w, bias)
    allowed = size * (K / 16) * 2.0 ** -24
    if out_dtype == torch.bfloat16:
        allowed = allowed + want.abs() * 2.0 ** -8
    worst = ((out.double() - want).abs() - allowed).max()
    assert float(worst) <= 0
    assert bool((wide[M] == 7).all()) and bool((wide[:M, :8] == 7).all()) and bool((wide[:M, 8 + N :] == 7).all())


@pytest.mark.parametrize("M,N,K,tiles", GATED)
@pytest.mark.parametrize("kind", ["silu", "bias", "gelu", "clamp"])
def test_gated(M, N, K, tiles, kind):
    from fms_amd.kernels import ops

    lib = library()
    assert lib.fmsamd_gemm_tall_plan(M, N, K, 1) == tiles
    x, w = rows_of(M, K, 8, 3), (rows_of(2 * N, K, 0, 4) * 0.1).contiguous()
    bias = torch.randn(2 * N, device="cuda") if kind == "bias" else None
    clamp = ops.GateClamp(1.5, 1.702, 1.0) if kind == "clamp" else None
    wide = torch.full((M + 1, N + 16), 7.0, dtype=torch.bfloat16, device="cuda")
    out = wide[:M, 8 : 8 + N]
    assert lib.fmsamd_gemm_tall_gated_bf16(x.data_ptr(), x.stride(0), w.data_ptr(), bias.data_ptr() if bias is not None else None, 0, out.data_ptr(),
                                           out.stride(0), M, N, K, ops.ACTIVATIONS["gelu" if kind == "gelu" else "silu"], ops._clamp(clamp),
                                           ops._stream()) == 0
    s, size = sums(x, w, bias)
    gate, up = s[:, :N], s[:, N:]
    if clamp is not None:
        g = gate.clamp(max=1.5)
        act, up = g * torch.sigmoid(1.702 * g), up.clamp(-1.5, 1.5) + 1.0
    else:
        act = torch.nn.functional.gelu(gate) if kind == "gelu" else gate * torch.sigmoid(gate)
    want = act * up
    # the activations' slopes are below 1.2 (2 with the clamp's alpha); their own arithmetic is good to some 2^-21
    loose = size * (K / 16) * 2.0 ** -24
    allowed = want.abs() * 2.0 ** -8 + 2 * loose[:, :N] * up.abs() + loose[:, N:] * act.abs() + 2.0 ** -20 * (gate.abs() + 1) * (up.abs() + 1)
    assert float(((out.double() - want).abs() - allowed).max()) <= 0
    assert bool((wide[M] == 7).all()) and bool((wide[:M, :8] == 7).all()) and bool((wide[:M, 8 + N :] == 7).all())


@pytest.mark.parametrize("M,N,K", [(641, 4368, 2048), (2049, 1360, 2048), (2561, 6176, 2048)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_one_row_and_no_column_for_the_last_quarter(M, N, K, out_dtype):
    from fms_amd.kernels import ops

    assert library().fmsamd_gemm_tall_pays(M, N, K, 0) == 1 and library().fmsamd_gemm_tall_plan(M, N, K, 0) == 2
    x, w = rows_of(M, K, 0, 11).contiguous(), rows_of(N, K, 0, 12).contiguous()
    want, size = sums(x, w, None)
    allowed = size * (K / 16) * 2.0 ** -24 + (want.abs() * 2.0 ** -8 if out_dtype == torch.bfloat16 else 0)
    assert float(((ops.linear(x, w, out_dtype=out_dtype).double() - want).abs() - allowed).max()) <= 0


def test_one_row_and_no_column_for_the_last_quarter_of_a_gated_product():
    from fms_amd.kernels import ops

    M, N, K = 3201, 136, 1024
    assert library().fmsamd_gemm_tall_pays(M, N, K, 1) == 1 and library().fmsamd_gemm_tall_plan(M, N, K, 1) == 2
    x, w = rows_of(M, K, 0, 13).contiguous(), (rows_of(2 * N, K, 0, 14) * 0.1).contiguous()
    s, size = sums(x, w, None)
    gate, up = s[:, :N], s[:, N:]
    act = gate * torch.sigmoid(gate)
    want, loose = act * up, size * (K / 16) * 2.0 ** -24  # allowed: as in test_gated
    allowed = want.abs() * 2.0 ** -8 + 2 * loose[:, :N] * up.abs() + loose[:, N:] * act.abs() + 2.0 ** -20 * (gate.abs() + 1) * (up.abs() + 1)
    assert float(((ops.gated_linear(x, w, None, "silu").double() - want).abs() - allowed).max()) <= 0


def test_rows_keep_their_own_infinities():
    """An infinity or NaN in a row of x or W stays in its row or column, also where a tile has rows that do not exist."""
    from fms_amd.kernels import ops

    M, N, K = 1111, 2048, 512
    x, w = rows_of(M, K, 0, 5).contiguous(), rows_of(N, K, 0, 6).contiguous()
    clean = ops.linear(x, w)
    x[M - 1, 3], w[5, 7] = float("nan"), float("inf")
    out = ops.linear(x, w)
    assert bool(out[M - 1].isnan().all()) and not bool(out[: M - 1, 5].isfinite().any())
    keep = [n for n in range(N) if n != 5]
    assert torch.equal(out[: M - 1, keep], clean[: M - 1, keep])


def test_entry_points_take_what_they_took():
    """Rows, widths and addresses that the kernel does not take still run, elsewhere; the two ways agree."""
    from fms_amd.kernels import ops

    M, N, K = 2048, 2048, 2048
    lib = library()
    assert lib.fmsamd_gemm_tall_pays(M, N, K, 0) == 1 and lib.fmsamd_gemm_tall_pays(M, N // 2, K, 1) == 1
    base = rows_of(M, K + 8, 0, 7).contiguous()
    w = (rows_of(N, K, 0, 8) * 0.05).contiguous()
    flat = torch.zeros(N * K + 8, dtype=torch.bfloat16, device="cuda")
    odd = flat[4 : 4 + N * K].view(N, K)
    odd.copy_(w)
    x, shifted = base[:, :K], torch.zeros_like(base)[:, 4 : 4 + K]
    shifted.copy_(x)
    want, size = sums(x, w, None)
    allowed = size * (K / 16) * 2.0 ** -24 + want.abs() * 2.0 ** -8
    for xs, ws in ((x, w), (x.contiguous(), w), (shifted, w), (x.contiguous(), odd)):
        assert float(((ops.linear(xs, ws).double() - want).abs() - allowed).max()) <= 0
    x = rows_of(M, K, 0, 7).contiguous()
    gated = ops.gated_linear(x, w, None, "silu")
    wide = torch.zeros(M, N // 2 + 4, dtype=torch.bfloat16, device="cuda")
    assert ops.gated_linear(x, w, None, "silu", out=wide[:, : N // 2]).data_ptr() == wide.data_ptr()
    assert float((wide[:, : N // 2].float() - gated.float()).norm() / gated.float().norm()) < 2.0 ** -7
    assert ops.linear(x, w[:120].contiguous()).shape == (M, 120) and ops.linear(x, w[:300].contiguous()).shape == (M, 300)


@pytest.mark.parametrize("step", [0, 8, 2040])
def test_rows_may_overlap(step):
    """Rows of x that are one row many times over, or a window that slides along."""
    from fms_amd.kernels import ops

    M, N, K = 2048, 2048, 2048
    flat = torch.randn(step * (M - 1) + K, generator=torch.Generator(device="cuda").manual_seed(15), device="cuda").to(torch.bfloat16)
    x, w = flat.as_strided((M, K), (step, 1)), (rows_of(N, K, 0, 16) * 0.05).contiguous()
    for out_dtype in (torch.bfloat16, torch.float32):
        want, size = sums(x, w, None)
        allowed = size * (K / 16) * 2.0 ** -24 + want.abs() * 2.0 ** -8
        assert float(((ops.linear(x, w, out_dtype=out_dtype).double() - want).abs() - allowed).max()) <= 0
    gated, same = ops.gated_linear(x, w, None, "silu"), ops.gated_linear(x.contiguous(), w, None, "silu")
    assert float((gated.float() - same.float()).norm() / same.float().norm()) < 2.0 ** -7


@pytest.mark.parametrize("shift", [0, 2048])
def test_results_may_take_the_place_of_the_rows(shift):
    """A gated product whose results go where its rows stand reads them all first, also where it has tiles for several rounds of blocks."""
    from fms_amd.kernels import ops

    M, N, K = 8192, 2048, 4096
    x, w = rows_of(M, K, 0, 17).contiguous(), (rows_of(2 * N, K, 0, 18) * 0.05).contiguous()
    assert library().fmsamd_gemm_tall_pays(M, N, K, 1) == 1
    gu = x.float() @ w.float().T.contiguous()
    want = torch.nn.functional.silu(gu[:, :N]) * gu[:, N:]
    out = x[:, shift : shift + N]
    assert ops.gated_linear(x, w, None, "silu", out=out).data_ptr() == out.data_ptr()
    assert float((x[:, shift : shift + N].float() - want).norm() / want.norm()) < 2.0 ** -7  # three roundings of 2^-9, gate and up among them


def test_a_captured_product_replays():
    from fms_amd.kernels import ops

    x, w = rows_of(700, 512, 0, 9).contiguous(), rows_of(2 * 2048, 512, 0, 10).contiguous()
    want = ops.gated_linear(x, w, None, "silu").clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        ops.gated_linear(x, w, None, "silu")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.gated_linear(x, w, None, "silu")
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
