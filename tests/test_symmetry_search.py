"""The search for symmetries of the operators (host code of coral_amd_create)
ends soon where there are many ways to exchange variables and none of them is a
symmetry."""
import time
from types import SimpleNamespace as NS

import pytest


def alike(n):
    """n equations with a mass and a dx dy term of every variable: any exchange of
    variables and of equations keeps all magnitudes, and neither y -> -y nor a
    quarter turn keeps the signs (dx dy changes sign, the mass does not)."""
    def pieces(iz, k):
        return [NS(dsca=1.0, kx=k, ky=k, iz=iz, mz=0, var=v, eqn=e) for e in range(n) for v in range(n)]
    s = NS(nvars=n, bc_codes=[20] * n, eqn_orders=[2] * n, nl=[], mass=pieces(2, 0), stif=pieces(2, 1))
    return NS(kxky_systems=[s], zero_systems=[], full_vars=[], quad_vars=[])


@pytest.mark.parametrize("n", [2, 8])
def test_many_exchanges(native_lib, n):
    from coral_amd.solver import assembled_operator
    t = time.perf_counter()
    M, _, _ = assembled_operator(alike(n), 16, 16, 17, 1.0, 1.0, 0, "mass", 1, 1)
    assert M.shape == (15 * n, 15 * n)
    assert time.perf_counter() - t < 2.0   # (764 x 764 exchanges at eight variables)
