"""What the kernels on the ring of ring_product.h rest on, as far as it shows without a GPU."""

import importlib
import os
import re
import subprocess

import pytest


def loads_with_places(lines):
    """How many loads to LDS the assembly has; fails unless each has its place put into m0 in front of it and m0 is used by nothing else,
    with no way in or out between the two.  The compiler does not look into the loads, so the waits that the hardware leaves to the
    program are looked for as well: one instruction between m0 and the load, five between a scalar register that the vector unit wrote and
    a load that reads it."""
    placed, loads, at, placed_at, by_vector_unit = False, 0, 0, 0, {}
    for line in lines:
        code = line.split(";")[0].strip()
        if re.match(r"[a-z]\w+( |$)", code):
            at += 1 + int(code.split()[1] if code.startswith("s_nop") else 0)
        written = re.match(r"v_(?:readfirstlane|readlane|cmp)\w* s(?:(\d+)|\[(\d+):(\d+)\])", code)
        if written:
            one, first, last = written.groups()
            by_vector_unit.update({r: at for r in range(int(one or first), int(one or last) + 1)})
        if re.fullmatch(r"s_mov_b32 m0, s\d+", code):
            assert not placed, "m0 is written twice in front of a load"
            placed, placed_at = True, at
        elif re.match(r"buffer_load\w* .*\blds\b", code):
            assert placed, f"a load to LDS without a place: {code}"
            assert at - placed_at > 1, f"a load right behind its place: {code}"
            for one, first, last in re.findall(r"\bs(?:(\d+)\b|\[(\d+):(\d+)\])", code):
                for r in range(int(one or first), int(one or last) + 1):
                    assert at - by_vector_unit.get(r, -99) > 5, f"s{r} is read too soon: {code}"
            placed, loads = False, loads + 1
        else:
            assert not re.search(r"\bm0\b", code), f"another use of m0: {code}"
            assert not placed or not re.match(r"s_c?branch|s_call|s_setpc|s_swappc|s_endpgm|\S+:$", code), f"a way in or out in front of a load: {code}"
    return loads


def test_nothing_comes_between_the_place_of_a_load_and_the_load(tmp_path):
    """A load to LDS takes its place from m0, which is set one matrix instruction earlier: no other instruction of the kernels
    may write m0 in between."""
    build = importlib.import_module("fms_amd.kernels.build")
    try:
        hipcc = build.hipcc_path()
    except RuntimeError:
        pytest.skip("no hipcc")
    sources = [s for s in build.sources() if "ring_product.h" in open(s).read()]
    assert sources
    for src in sources:
        out = tmp_path / (os.path.basename(src) + ".s")
        subprocess.run([hipcc, *build.HIPCC_FLAGS, "-I", build.CSRC, "-S", "--cuda-device-only", src, "-o", str(out)],
                       check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
        assert loads_with_places(out.read_text().splitlines()) > 100


@pytest.mark.parametrize("between", [
    "", "v_readfirstlane_b32 s9, v1", "v_cmp_lt_u32_e64 s[10:11], v1, v2", "v_readlane_b32 s12, v1, 0", "v_readfirstlane_b32 m0, v1",
    "v_readlane_b32 m0, v1, s2", "s_add_u32 m0, m0, s3", "s_mov_b32 m0, s4", "s_mov_b32 s4, m0", ".LBB0_3:", "s_cbranch_scc1 .LBB0_3",
    "s_mov_b64 s[2:3], s[4:5] ; m0", "v_add_u32_e32 v1, v2, v3",
])
def test_what_may_stand_between_them(between):
    lines = ["s_mov_b32 m0, s5", between, "buffer_load_dwordx4 v1, s[8:11], s12 offen lds"]
    if between.startswith(("v_add_u32_e32", "s_mov_b64")):
        assert loads_with_places(lines) == 1
    else:
        with pytest.raises(AssertionError):
            loads_with_places(lines)


@pytest.mark.parametrize("gated", [0, 1])
def test_a_product_that_pays_is_one_that_fits(gated):
    """What the kernel for many rows refuses is never sent to it."""
    from fms_amd.kernels.library import load

    lib = load()
    for M, N, K in ((192, 4096, 256), (4096, 4092, 4096), (4096, 4096, 4096 + 64), (4096, 4096, 128), (4096, 120, 4096),
                    (1 << 20, 1 << 20, 256), (4096, 4096, 1 << 22), (300, 4096, 14336)):
        assert lib.fmsamd_gemm_tall_pays(M, N, K, gated) == 0 or (M, N, K) == (300, 4096, 14336) and gated
    for M, N, K in ((2048, 4096, 4096), (2048, 6144, 4096), (4689, 14336, 4096)):
        assert lib.fmsamd_gemm_tall_pays(M, N, K, gated) == 1
        assert 0 <= lib.fmsamd_gemm_tall_plan(M, N, K, gated) <= 4


@pytest.mark.parametrize("tiles", range(5))
@pytest.mark.parametrize("gated", [0, 1])
@pytest.mark.parametrize("size", [2, 4])
def test_every_store_of_a_product_lies_inside_its_output(tiles, gated, size):
    """Every result is stored and nothing else, whatever rows and columns are left for the last tiles and their halves and quarters."""
    from fms_amd.kernels.library import load

    lib = load()
    for rows in (193, 255, 256, 257, 384, 385, 513, 640, 641, 642, 1921, 2049, 2561, 3201, 4097):
        for cols in (128, 136, 248, 256, 264, 384, 392, 1360, 2048, 4368, 6176):
            for ldo in (cols, cols + 8, 3 * cols):
                assert lib.fmsamd_gemm_tall_stores(rows, cols, ldo, size, gated, tiles) == rows * cols // 8, (rows, cols, ldo)
    # the longest rows that are taken
    longest = (1 << 22) // size - 8
    for rows, cols in ((193, longest), (257, 264), (641, 4368)):
        assert lib.fmsamd_gemm_tall_stores(rows, cols, longest, size, gated, tiles) == rows * cols // 8
