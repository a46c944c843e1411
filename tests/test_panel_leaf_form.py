"""Which leaf kernel the LU panel takes (no GPU needed)."""
import ctypes as C
import os

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def _form(c128, n, m, beside_fp64):
    out = (C.c_int * 3)()
    C.CDLL(os.path.join(HERE, "native", "libqbt_linalg.so")).qbt_leaf_form(c128, n, m, beside_fp64, out)
    return tuple(out)


LONG = (0, 0, 0)


@pytest.mark.parametrize("m", [4097, 6000, 8192])
def test_long_columns_beside_fp64_updates(m):
    """4097 to 8192 rows in registers beside the residue updates alone."""
    assert _form(1, 8704, m, 0) == (512, 16, 2)
    assert _form(1, 8704, m, 1) == LONG


@pytest.mark.parametrize("beside_fp64", [0, 1])
@pytest.mark.parametrize("c128", [0, 1])
def test_every_row_has_a_place(c128, beside_fp64):
    """The rows fit the threads, and threads x rows x columns the registers."""
    for n in (100, 1000, 4095, 4096, 8192, 9000):
        for m in {1, 511, 512, 513, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, n}:
            if m > n:
                continue
            t, r, w = _form(c128, n, m, beside_fp64)
            if t:
                assert m <= t * r and r * w <= (32 if c128 else 64) and w <= 32
            else:
                assert m > 4096
