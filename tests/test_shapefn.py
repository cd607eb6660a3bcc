"""The limits of the stateless deposits, which are checked before any array is
touched (so that no GPU is needed here)."""
import ctypes as C

import pytest

from csrst_amd import _lib

INT_MAX = 2 ** 31 - 1
# contributions per particle (current: items per particle), by order
PER = {"charge": (4, 9, 16), "diff": (8, 18, 32), "scatter": (4, 9, 16), "current": (4, 4, 4), "noalloc": (8, 24, 48)}


@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("op", sorted(PER))
def test_too_many_contributions_are_refused(op, order):
    """Contributions are numbered in 32 bits.  The first count beyond that, and
    the counts whose product wraps to a few in 32 bits, return CSRST_EINVAL."""
    L, i = _lib.lib(), C.c_int
    here = (C.c_double * 2)(1.0, 1.0)
    p, two = C.c_void_p(C.addressof(here)), here          # never read
    per = PER[op][order]
    for n in (INT_MAX // per + 1, min(2 ** 32 // per + 1, INT_MAX), INT_MAX):
        if op == "charge":
            rc = L.csrst_sf_charge_density(i(order), p, i(0), i(0), i(8), i(8), two, two, p, p, i(n), None)
        elif op == "diff":
            rc = L.csrst_sf_charge_density_diff(i(order), p, i(0), i(0), i(8), i(8), two, two, p, p, p, i(n), None)
        elif op == "scatter":
            rc = L.csrst_sg_scatter(i(order), i(0), p, i(8), i(8), two, two, p, p, i(n), None)
        else:
            f = L.csrst_sf_current_density if op == "current" else L.csrst_sf_current_density_noalloc
            rc = f(i(order), i(0), p, i(0), i(0), i(8), i(8), two, two, C.c_double(1.0), p, p, p, i(n), None)
        assert rc == -1, (n, rc)
        with pytest.raises(_lib.CsrstError, match="contributions"):
            _lib.check(rc)
