"""CPU: the kernel variants that a plan takes by precision, sides and cells (tuned_variants)."""
import ctypes

import pytest


def radix(table, v):
    from pywignercuda_amd import _lib

    r, lanes = ctypes.c_int(), ctypes.c_int()
    assert _lib.lib().wh_variant_info(table, v, ctypes.byref(r), ctypes.byref(lanes)) == 0
    return r.value


def choice(precision, X, P, cl=False, members=1):
    from pywignercuda_amd.wigner2d import tuned_variants

    cells = X * P * members
    batch = cells * (16 if precision == "fp64" else 8) >= 256 << 20
    return tuned_variants(precision, [X] * members, [P] * members, cl, batch)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_friction_form_by_cells(precision):
    """P >= 1024 in FP64 arithmetic: the two-wave form (2) from two blocks per CU on, else radix 16
    in one wave or, for complex64 states on few cells, radix 8."""
    for P, X, members in ((2048, 1024, 1), (1024, 2048, 1), (2048, 2048, 1), (1024, 1024, 2), (2048, 2048, 4)):
        assert choice(precision, X, P, True, members)[2] == 2, (P, X, members)
    for P, X in ((1024, 1024), (2048, 512)):
        assert choice(precision, X, P, True)[2] == 0, (P, X)


def test_small_sides_keep_their_radix_in_ensembles():
    """Radix 16 in x for 2^20 and 2^21 cells of complex128 is for sides of 512 and more."""
    for side, members in ((128, 64), (128, 128), (256, 16), (256, 32)):
        assert radix(0, choice("fp64", side, side, members=members)[0]) == 4, (side, members)
    for X, P, members in ((512, 2048, 1), (2048, 512, 1), (2048, 1024, 1), (512, 512, 4), (512, 512, 8), (1024, 1024, 2)):
        assert radix(0, choice("fp64", X, P, members=members)[0]) == 16, (X, P, members)
