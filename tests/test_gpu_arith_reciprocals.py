"""GPU self-test of the divisions that the kernels' bit-exactness rests on, against the compiler's
correctly rounded one: by a known reciprocal rounded to double (div_c), by a reciprocal refined from
the double that the divisor was rounded from, by two doubles (div_c2, denormal quotients included),
and div_rn at the edges of the operands that it takes through double (2^-60 and 2^60): 2^28 hashed
pairs and every pair of special values."""
import ctypes as C

import numpy as np
import pytest

from eden_amd import _native as N

pytestmark = pytest.mark.gpu


def _special_values():
    vals = [0.0, 1.0, 3.0, 1.0 / 3.0, np.inf, np.nan, 3.4028235e38, 1.17549435e-38, 1.1754942e-38]
    vals += [k * 2.0 ** -149 for k in (1, 2, 3, 5, 2 ** 20 + 1, 2 ** 22 - 1)]
    for e in [-126, -125, -100, -62, -61, -60, -59, -24, -1, 0, 1, 5, 24, 59, 60, 61, 62, 100, 126, 127]:
        for m in (1.0, np.nextafter(np.float32(1), np.float32(2)), 1.25, 1.5, np.nextafter(np.float32(2), np.float32(0))):
            vals.append(float(m) * 2.0 ** e)
    vals = np.array(vals, np.float32)
    return np.concatenate([vals, -vals])


def test_divisions_by_known_reciprocals():
    lib, sp = N.load_library(), _special_values()
    bad = (C.c_int64 * 3)(-1, -1, -1)
    assert lib.edenhip_diag_reciprocals(20261205, 1 << 28, N.ptr(sp), len(sp), bad) == 0
    print(f"[arith] mismatches {list(bad)}", flush=True)
    assert list(bad) == [0, 0, 0]


def test_division_at_the_edges_of_its_range():
    lib, sp = N.load_library(), _special_values()
    bad = C.c_int64(-1)
    assert lib.edenhip_diag_divide(7, 1 << 24, N.ptr(sp), len(sp), C.byref(bad)) == 0
    assert bad.value == 0
