"""What the kernels on the ring of ring_product.h rest on, as far as it shows without a GPU."""

import importlib
import os
import re
import subprocess

import pytest


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
        placed, loads = False, 0
        for line in out.read_text().splitlines():
            code = line.split(";")[0].strip()
            if re.match(r"s_\w+ m0,", code):
                assert not placed, f"{os.path.basename(src)}: m0 is written twice in front of a load"
                placed = True
            elif " lds" in code and code.startswith("buffer_load"):
                assert placed, f"{os.path.basename(src)}: a load to LDS without a place"
                placed, loads = False, loads + 1
            elif "m0" in code.replace("m0,", ""):
                assert not re.search(r"\bm0\b", code), f"{os.path.basename(src)}: another use of m0: {code}"
        assert loads > 100


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
