"""A variable with an infinity or a NaN in its spectrum spoils the products it
enters and no others, at line lengths where two lines share one transform:
108 and 288 points (several lines and one line per wavefront), 486, and 648 (two
wavefronts per line)."""
import numpy as np
import pytest

from conftest import product_recipe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("grid", [(72, 16, 17), (192, 16, 17), (324, 16, 17), (432, 16, 17)],
                         ids=lambda g: "x".join(map(str, g)))
def test_products_without_the_variable_are_unchanged(native_lib, grid, bad):
    from coral_amd import solver
    NX, NY, NZ = grid
    print("grid", grid, bad, flush=True)
    r = product_recipe("coral.equations.rbc_ra1e5")
    s, full = r.kxky_systems[0], [f.name for f in r.full_vars]
    rng = np.random.default_rng(1)
    with solver.Solver(r, NX, NY, NZ, 2 * np.pi, 2 * np.pi) as g:
        shape = (NX // 2, 3 * NY // 2, g.totals[0])
        k = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
        k[0] = 0.0
        z = [rng.standard_normal(n) for n in g.zero_totals]
        g.set_state([k], z)
        want = g.products()
        for name in ("u", "v", "w", "t"):
            f = full.index(name + "Full")
            kb = k.copy()
            kb[3, 5, s.var_names.index(name)] = bad   # (the lowest degrees come first, variable by variable)
            g.set_state([kb], z)
            got = g.products()
            for q, a, b in zip(r.quad_vars, got, want):
                if f in (q.ivar1, q.ivar2):
                    assert not np.isfinite(a).all()
                else:
                    # another partner in the transform: a few eps, as the transforms' own tests
                    assert np.linalg.norm(a - b) <= 2e-14 * np.linalg.norm(b), (name, q.ivar1, q.ivar2)
