"""CPU: the tile that a 16-bit product with an activation takes, for rows and columns of every size, and the splits of K that others take (no kernel runs)."""
import ctypes

import pytest


@pytest.mark.parametrize("N", [128, 5632, 28672, 57344, 131072, 262144])
def test_few_rows_take_low_tiles(N):
    """A tile of 32 mb rows is never twice as high as the rows need: 64 up to 64 rows, 128 up to 128, also where the columns alone are two rounds of workgroups."""
    from proxy_inference_engine_amd import _ffi
    tile = ctypes.CDLL(str(_ffi.lib_path().parent / "libpie_base.so"))["_Z9w16l_tileiiiPiS_"]   # w16l_tile(M, N, K, &mb, &sw)
    mb, sw = ctypes.c_int(), ctypes.c_int()
    for K in (64, 2048, 8192):
        for M in (33, 64, 65, 100, 128, 129, 256, 257, 1000, 4096):
            tile(M, N, K, ctypes.byref(mb), ctypes.byref(sw))
            assert mb.value in (2, 4, 8) and sw.value in (1, 2), (M, K)
            assert 32 * mb.value < 2 * max(M, 33), (M, K, mb.value)


@pytest.mark.parametrize("N,K,rows,splits", [(8448, 2048, (43, 50, 61), 3), (6144, 2048, (33, 48, 62), 3), (10752, 4096, (122, 128), 2), (4096, 14336, (33, 64), 6), (14336, 4096, (33, 64), 2)])
def test_splits_that_were_measured(N, K, rows, splits):
    """The fastest split of each, by 5 to 30 % over the whole product or one split more: the workgroups' share of the stream decides, and what hides the launch that sums the slabs."""
    from proxy_inference_engine_amd import _ffi
    lib = _ffi.load()
    for M in rows:
        assert int(lib.pie_linear_w16m_workspace(M, N, K)) == splits * M * N * 4, M
