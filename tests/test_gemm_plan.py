"""The GEMM's plan (vdn_fp8_gemm_plan; no GPU needed): which kernels run a shape."""
import ctypes
import random

import pytest

from conftest import gemm_plan

CUS = 256


def _shapes(n, seed):
    rng = random.Random(seed)
    lg = lambda a, b: int(a * (b / a) ** rng.random())
    return [(lg(1, 40000), max(4, lg(4, 40000) // 4 * 4), max(16, lg(16, 40000) // rng.choice([16, 256]) * 16))
            for _ in range(n)] + [(lg(1, 40000), lg(64, 10000) * 4, 256 * lg(1, 128)) for _ in range(n)]


@pytest.mark.parametrize("rows16,split", [(True, True), (True, False), (False, True), (False, False)])
def test_a_plan_covers_every_tile(rows16, split):
    """Whole tiles, split tiles and parts add up to the output, within what each kernel takes."""
    for M, N, K in _shapes(400, 1):
        rows, whole, slices, units, a, b = gemm_plan(M, N, K, rows16, split)
        case = (M, N, K, rows16, split, rows, whole, slices, units, a, b)
        if rows == 0:
            assert whole == units == 0 and a and b, case
            continue
        assert K % 256 == 0 and rows in ((224, 256) if rows16 else (256,)), case
        tiles = -(-M // rows) * -(-N // 256)
        if units:
            assert split and K >= 8192 and not a and slices >= 2 and K // 256 >= slices, case
            assert whole + units // slices == tiles and units % slices == 0 and units <= CUS, case
        elif a:
            parts = (tiles - whole) * (256 // a) * (256 // b)
            assert rows == 256 and a in (128, 256) and b in (64, 128) and 0 < parts <= CUS, case
        else:
            assert whole == tiles, case


def test_the_size_query_answers_for_every_epilogue():
    """The workspace is sized by M, N and K alone; a call whose rows take the general epilogue
    (binary16 or binary32 output, rows that are not 16-byte) needs no more than that."""
    shapes = [(M, N, K) for M in range(1, 5000, 37) for N in (512, 4100, 5376, 15360, 28672) for K in (8192, 14336)]
    apart = 0
    for M, N, K in shapes + [(2817, 28672, 8192), (2912, 28672, 8192), (3329, 28672, 8192)]:
        answer, need = gemm_plan(M, N, K, True, True)[3], gemm_plan(M, N, K, False, True)[3]
        assert need <= answer, (M, N, K, need, answer)
        apart += gemm_plan(M, N, K, True, True) != gemm_plan(M, N, K, False, True)
    assert apart


def test_large_shapes_run_whole_tiles():
    assert gemm_plan(32760, 15360, 5120)[:2] == (256, 7680)
    assert gemm_plan(32760, 15360, 5120, rows16=False)[:2] == (256, 7680)


@pytest.mark.parametrize("M,N,K,rows16,want", [
    (2074, 10400, 256, True, (224, 410, 0, 0, 0, 0)),       # 19.5 us; 26.3 on the tile kernel's 256 x 128
    (3891, 2704, 256, True, (224, 198, 0, 0, 0, 0)),        # 16.7 us; 19.7 as 128 x 192
    (10329, 2232, 1024, False, (256, 256, 0, 0, 256, 128)), # 40.3 us; 44.7 as 256 x 128 throughout
    (1304, 2272, 1024, True, (0, 0, 0, 0, 128, 96)),        # 9.9 us; 12.1 as 192 x 96
])
def test_short_rows_count_the_epilogue(M, N, K, rows16, want):
    """At a K of a few blocks most of a round is its epilogue (times: one MI355X)."""
    assert gemm_plan(M, N, K, rows16) == want


def test_query_refusals():
    import vdn_fp8._lib as L
    lib = L.load()
    plan = (ctypes.c_int32 * 6)()
    us = ctypes.c_double()
    assert lib.vdn_fp8_gemm_plan(1, 4, 16, 1, 0, CUS, None, None) == L.EINVAL
    assert lib.vdn_fp8_gemm_plan(0, 4, 16, 1, 0, CUS, plan, None) == L.EINVAL
    assert lib.vdn_fp8_gemm_plan(1, 4, 16, 1, 0, -1, plan, None) == L.EINVAL
    assert lib.vdn_fp8_gemm_plan(1 << 40, 1 << 20, 16, 1, 0, CUS, plan, None) == L.EINVAL
    assert lib.vdn_fp8_gemm_plan(1, 4, 16, 1, 0, CUS, plan, ctypes.byref(us)) == L.OK and us.value > 0
