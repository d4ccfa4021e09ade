"""The stencil kernels' k chunks (host rule, no GPU needed)."""
import ctypes as C

import pytest


class _Grid(C.Structure):
    _fields_ = [("nx", C.c_int), ("ny", C.c_int), ("nz", C.c_int)] + \
               [(n, C.c_double) for n in ("dx_inv", "dy_inv", "re_inv", "dt", "u_crf")] + \
               [(n, C.c_void_p) for n in ("dzf", "dzf_inv", "dzc_inv", "dzflzi")] + \
               [("rk_kc", C.c_int)]


def _tiling(nx, ny, nz, kc=0):
    from powerllel_channel_amd import lib
    rk = (C.c_int * 5)()
    lib().pll_rk_tiling(C.byref(_Grid(nx, ny, nz, 1, 1, 1, 1, 0, None, None, None, None, kc)), rk)
    return list(rk)


@pytest.mark.parametrize("nx,ny", [(4, 2), (64, 64), (240, 140), (256, 192), (384, 384),
                                   (768, 384), (784, 350), (1536, 1024)])
def test_chunks_are_even(nx, ny):
    """Workgroups are handed to the XCDs chunk after chunk, so a short last chunk
    leaves XCDs idle: all chunks of a grid hold the same planes but one."""
    for nz in range(2, 400):
        ntx, nty, nkc, kc, _ = _tiling(nx, ny, nz)
        assert (ntx, nty) == ((nx + 63) // 64, (ny + 3) // 4)
        assert (nkc - 1) * kc < nz <= nkc * kc
        assert nkc * kc - nz < nkc, (nz, nkc, kc)
        assert kc <= 64


def test_chunk_override():
    """PLL_RK_KC stays as given."""
    assert _tiling(768, 384, 39, 7)[2:4] == [6, 7]
