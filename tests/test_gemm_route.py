"""Which kernel a plain GEMM runs on (uwc_plain_gemm_route, the rule uwc_noisy_gemm and its fused siblings
take), on the host without a GPU."""
import pytest

NONE, I32, BF16, F32 = 0, 1, 2, 3
LARGE, COLUMNS, SKINNY, STREAM, STAGED = 16, 17, 18, 19, 20
CUS = 256


def route(m, n, k, out=I32, second=0, cus=CUS):
    from uwc_amd import _lib
    return _lib.lib().uwc_plain_gemm_route(m, n, k, out, second, cus)


def test_header_names_the_routes():
    import os
    from conftest import ROOT
    src = open(os.path.join(ROOT, "include", "uwc.h")).read()
    for name, v in (("LARGE", LARGE), ("LARGE_COLUMNS", COLUMNS), ("SKINNY", SKINNY), ("SKINNY_STREAM", STREAM),
                    ("STAGED", STAGED)):
        assert f"#define UWC_ROUTE_{name} {v} " in src


@pytest.mark.parametrize("m,n,want", [(128, 128, 0), (2048, 2048, 0), (2048, 4096, 1), (2048, 12288, 1), (1024, 28672, 1)])
def test_product_without_output_keeps_the_dma_kernel(m, n, want):
    """Whole 128 x 128 tiles without an output: the 4-step ring while a CU has at most one tile, else the
    2-step one; ragged ones the staged kernel."""
    assert route(m, n, 2048, NONE) == want
    assert route(m + 1, n, 2048, NONE) == STAGED and route(m, n, 2048 + 64, NONE) == STAGED


@pytest.mark.parametrize("out,second", [(I32, 0), (BF16, 0), (F32, 0), (F32, 1), (I32, 2)])
def test_large_tiles(out, second):
    """256 x 256 tiles from one per CU on with the last round 90% full; the columns before the last
    multiple of 256 from one per CU on (not with a residual); never for m or k off their multiples."""
    r = lambda m, n, k=1024: route(m, n, k, out, second)
    assert r(4096, 4096) == LARGE and r(8192, 12288) == LARGE
    assert r(4096, 3840) < 9 and r(2048, 12288) < 9  # 240 tiles; 384: a half-empty round
    assert r(2304 * 2, 256 * 25) < 9 and r(2304 * 2, 256 * 26) == LARGE  # 450 and 468 tiles in two rounds
    assert r(4097, 4096) < 9 and r(4096 + 128, 4096) < 9
    assert r(4096, 4096, 1024 + 64) == STAGED
    assert r(4096, 4096 + 4) == (COLUMNS if second != 1 else r(4096, 4096 + 4)) and r(4096, 4096 + 2) == STAGED
    assert r(4096, 3840 + 128) < 9
    if second == 1:
        assert r(4096, 4096 + 4) < 9


def test_small_and_odd_products():
    assert route(5, 6, 128) == SKINNY and route(65, 6, 128) == STAGED
    assert route(40, 132, 192) == SKINNY and route(64, 300, 4160) == STREAM
    assert route(40, 4098, 14336) == STREAM and route(64, 300, 4160, NONE) == STAGED
    assert route(0, 4, 128) == -1 and route(4, 4, 100) == -1 and route(4, 4, 128, F32, 2) == -1


@pytest.mark.parametrize("m,n,k,out,second,want", [
    (17, 28672, 4096, F32, 0, 6), (20, 32000, 4096, F32, 0, 6), (384, 12288, 2048, F32, 0, 1), (1280, 4096, 2048, I32, 0, 1),
    (1536, 3072, 1024, F32, 0, 1), (4096, 1152, 1152, F32, 0, 1), (300, 151936, 2048, I32, 2, 1), (40, 28672, 4096, F32, 0, 4)])
def test_form_of_products_timed_apart(m, n, k, out, second, want):
    """Products whose forms differ by 20% and more: the fastest one (wide weights at few rows, a little
    more than one 128 x 128 tile per CU, a vocabulary's both outputs)."""
    assert route(m, n, k, out, second) == want


@pytest.mark.parametrize("m,n,k", [(1 << 28, 4, 128), ((1 << 28) + 5, 16, 1152), ((1 << 30) + 1, 4, 128), (1, 1 << 24, 4096),
                                   (4, 1 << 28, 128), (1 << 20, 1 << 16, 128), (1 << 24, 28672, 2048)])
@pytest.mark.parametrize("second", [0, 1])
def test_form_grids_hold_fewer_than_2_to_32_threads(m, n, k, second):
    """Very long or wide products take tiles whose grid one launch can hold."""
    tiles = [(128, 128), (128, 128), (64, 128), (64, 64), (64, 64), (64, 32), (32, 32), (16, 32), (16, 16)]
    f = route(m, n, k, F32, second)
    if f in (LARGE, COLUMNS):
        return
    bm, bn = tiles[f]
    assert -(-m // bm) * -(-n // bn) * 256 < 1 << 32
