"""The closure's fused lift on x-lines in tiles of 32 points (96 and 288) gives
the corrected quadratic spectra of the separate packing, GEMM, bias and
unpacking kernels bit for bit."""
import numpy as np
import pytest

from conftest import product_recipe, seeded_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,hidden", [(32, 128), (64, 256)])
@pytest.mark.parametrize("NX,NY", [(64, 64), (64, 16), (192, 16)])
def test_fused_lift_in_tiles_of_32(native_lib, monkeypatch, NX, NY, width, hidden):
    from coral_amd import closure
    from coral_amd.solver import Solver
    r = product_recipe("coral.equations.rbc_ra1e5")
    NZ, M = 17, 3
    basis = closure.fourier_basis(3 * NX // 2, 3 * NY // 2, M)
    cin = closure.input_width(4)
    lay = closure.Layout(cin=cin, cout=9, width=width, hidden=hidden, layers=2, nb=basis.shape[1])
    rng = np.random.default_rng(5)
    model = closure.Model(lay, M, closure.init_params(lay, 12) * 3.0, rng.normal(size=cin) * 0.1,
                          1.0 + rng.random(cin), rng.normal(size=9) * 0.1, 0.5 + rng.random(9))
    k0, z0 = seeded_state(r, NX, NY, NZ, 4, 4, 9, amps=(("u", 1.0), ("v", 1.0), ("w", 1.0), ("t", 0.1)))
    out = {}
    for mode in ("fused", "unfused"):
        if mode == "unfused":
            monkeypatch.setenv("CORAL_AMD_CLOSURE_UNFUSED", "1")
        with Solver(r, NX, NY, NZ, 2 * np.pi, 2 * np.pi) as g:
            g.set_state(k0, z0)
            g.set_closure(model)
            out[mode] = g.products()
    assert np.array_equal(out["fused"], out["unfused"])
