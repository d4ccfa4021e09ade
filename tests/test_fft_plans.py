"""Points per thread that the transform plans take (no GPU needed)."""
import ctypes as C

import pytest


@pytest.fixture(scope="module")
def lib():
    from powerllel_channel_amd import lib as L
    return L()


def _points(lib, axis, L, cells=10 ** 9):
    E, n, rad = C.c_int(), C.c_int(), (C.c_int * 12)()
    rc = lib.pll_fft_plan_info_grid(L, int(axis == "y"), C.c_longlong(cells), C.byref(E),
                                    C.byref(n), rad)
    return E.value if rc == 0 else 0


def _smooth(L, primes):
    for q in primes:
        while L % q == 0:
            L //= q
    return L == 1


def _limit(E):
    return 256 if E >= 12 else 512


ALL = (2, 3, 4, 5, 6, 7, 8, 12, 24)


@pytest.mark.parametrize("axis", ["x", "y"])
def test_plan_points_per_thread(lib, axis):
    """Of a length's usable points per thread E (E divides it, at most 512
    threads a row, 256 from E = 12 on): 24 only where nothing else is usable;
    y tiles of two columns and more where any E but 24 gives them (from 128
    on); with a factor 11 or 13, the first of 12, 8, 6 that leaves room for two
    rows in a workgroup, on grids of more than 2^20 cells.  Lengths 2^a 3^b have
    plans of their own."""
    for L in range(2, 4096 if axis == "x" else 5120, 1 if axis == "x" else 2):
        usable = [E for E in ALL if L % E == 0 and L // E <= _limit(E)]
        E = _points(lib, axis, L)
        assert (E in usable) == (_smooth(L, (2, 3, 5, 7, 11, 13)) and bool(usable)), L
        if not E or _smooth(L, (2, 3)):
            continue
        assert E != 24 or usable == [24], (L, E)
        two = [e for e in usable if e != 24 and 2 * (L // e) <= _limit(e)]
        if axis == "y" and L >= 128 and two:
            assert E in two, (L, E, two)
        if not _smooth(L, (2, 3, 5, 7)):
            first = [e for e in (12, 8, 6) if e in two]
            assert not first or E == first[0], (L, E, first)


@pytest.mark.parametrize("axis,L,E", [
    ("y", 640, 5), ("y", 800, 5), ("y", 960, 5), ("y", 1344, 12), ("y", 1400, 8),
    ("y", 1568, 8), ("y", 126, 6), ("y", 462, 6), ("y", 832, 8), ("y", 936, 12),
    ("x", 126, 6), ("x", 294, 6), ("x", 660, 12), ("x", 726, 6), ("x", 1500, 6),
    ("x", 1300, 4), ("x", 1584, 8), ("x", 3360, 8)])
def test_plan_measured(lib, axis, L, E):
    """Lengths on either side of the rule's lines, as they were measured."""
    assert _points(lib, axis, L) == E


@pytest.mark.parametrize("axis,L,few,many", [("x", 132, 4, 12), ("x", 176, 4, 8), ("x", 330, 5, 6),
                                             ("x", 294, 3, 6), ("y", 66, 3, 6), ("y", 132, 4, 12),
                                             ("y", 208, 4, 8), ("y", 882, 3, 6), ("y", 1400, 5, 8),
                                             ("y", 960, 5, 5), ("y", 120, 5, 5), ("x", 3360, 8, 8)])
def test_plan_by_grid_size(lib, axis, L, few, many):
    """Up to 2^20 cells more threads to a row, above wider tiles."""
    assert _points(lib, axis, L, 2 ** 20) == few
    assert _points(lib, axis, L, 2 ** 20 + 1) == many


def test_no_24_points_on_small_grids(lib):
    for axis, L in [(a, n) for a in "xy" for n in range(2, 4096, 2)]:
        if not _smooth(L, (2, 3)) and _points(lib, axis, L, 1) == 24:
            assert not [E for E in ALL[:-1] if L % E == 0 and L // E <= _limit(E)], L


@pytest.mark.parametrize("want,L,taken", [("8", 80, True), ("2", 130, True), ("10", 80, False),
                                          ("2", 2000, False), ("9", 2268, False),
                                          ("x", 80, False), ("12", 64, False)])
def test_plan_override(lib, monkeypatch, want, L, taken):
    """PLL_FFT_E is taken where a kernel of as many points divides the length
    within its thread limit; otherwise the plan is the one without it."""
    plain = _points(lib, "y", L)
    monkeypatch.setenv("PLL_FFT_E", want)
    assert _points(lib, "y", L) == (int(want) if taken else plain) != 0
