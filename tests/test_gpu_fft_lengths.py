"""The horizontal transforms at every line length with a wavefront plan: the
quadratic spectra of a broadband state and the single transforms against the
oracle (numpy/scipy FFTs in float64)."""
import numpy as np
import pytest

from oracle import coral_oracle as O

from conftest import product_recipe

pytestmark = pytest.mark.gpu

# 3 N / 2 = 24, 27, 36, ... points, on shallow grids and (the short lengths) deep ones
GRIDS = [(16, 18, 17), (18, 16, 17), (24, 16, 20), (32, 24, 17), (36, 32, 17), (48, 36, 17), (54, 48, 17),
         (64, 54, 17), (72, 64, 17), (96, 72, 17), (108, 96, 17), (128, 108, 17), (144, 128, 17), (162, 144, 17),
         (192, 162, 17), (216, 192, 17), (16, 216, 65), (16, 72, 129), (18, 72, 129), (24, 96, 129), (32, 96, 97),
         (36, 96, 97), (48, 96, 97), (54, 96, 97), (72, 48, 97), (108, 16, 129), (162, 16, 129), (16, 288, 17),
         (288, 16, 17), (16, 324, 17), (324, 16, 17), (384, 16, 17), (16, 384, 17), (432, 16, 17), (16, 432, 17),
         (486, 16, 17), (16, 486, 17)]


@pytest.mark.parametrize("grid", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_products_and_transforms_match_oracle(native_lib, grid):
    from coral_amd import solver
    NX, NY, NZ = grid
    print("grid", grid, flush=True)
    r = product_recipe("coral.equations.rbc_ra1e5")
    geo = O.Geometry(NX, NY, NZ, 2 * np.pi, 2 * np.pi)
    ora = O.OracleSolver(r, geo, "ARS_222")
    rng = np.random.default_rng(NX * 1000 + NY)
    k0 = [rng.standard_normal(f.shape) + 1j * rng.standard_normal(f.shape) for f in ora.field]
    for f in k0:
        f[~ora.keep] = 0.0
        f[0, 0] = 0.0
        O.project_kx0_plane(f, geo)
    z0 = [rng.standard_normal(z.shape) for z in ora.zfield]
    ora.field, ora.zfield = [f.copy() for f in k0], [z.copy() for z in z0]
    q = ora.quad_spectra(ora.field, ora.zfield)
    with solver.Solver(r, NX, NY, NZ, 2 * np.pi, 2 * np.pi) as g:
        g.set_state(k0, z0)
        got = g.products()
        spec = np.where(ora.keep[:, :, None], q[0], 0.0)
        phys = g.bwd_transform(spec)
        back = g.fwd_transform(phys)
        fields = [g.physical(i) for i in range(len(r.full_vars))]
        g.factorize_operators(1e-6)
        g.march_forward(1e-6, 1)
        cfl = g.cfl_dt()
    ora.step(1e-6)
    # FP64 FFTs of a few thousand points: a few eps in the l2 norm
    tol = 2e-14

    def rel(a, b):
        return np.linalg.norm(a - b) / np.linalg.norm(b)
    for i, s in enumerate(q):
        assert rel(got[i], np.where(ora.keep[:, :, None], s, 0.0)) <= tol, i
    want = O.spec_to_phys(spec, geo)
    assert rel(phys, want) <= tol
    assert rel(back, np.where(ora.keep[:, :, None], O.phys_to_spec(want, geo), 0.0)) <= tol
    ora.field, ora.zfield = k0, z0
    for a, b in zip(fields, ora.physical_full_variables()):
        assert rel(a, b) <= tol
    assert abs(cfl - ora.cfl_dt) <= 1e-9 * abs(ora.cfl_dt)


# lengths that share a transform between two lines scaled apart: several lines
# per wavefront (27, 108, 216), one (288, 486), two wavefronts per line (648)
@pytest.mark.parametrize("small", ["t", "w"])
@pytest.mark.parametrize("grid", [(18, 16, 17), (72, 48, 17), (144, 16, 17), (192, 16, 17), (324, 16, 17), (432, 16, 17)],
                         ids=lambda g: "x".join(map(str, g)))
def test_small_lines_keep_their_digits(native_lib, grid, small):
    """A variable of 1e-8 of the others (and its products beside theirs) comes out
    as accurate as the others: the lines of a pair are scaled by powers of two of
    their own.  Without that its errors would be 1e-8 of its size."""
    from coral_amd import solver
    NX, NY, NZ = grid
    print("grid", grid, small, flush=True)
    r = product_recipe("coral.equations.rbc_ra1e5")
    geo = O.Geometry(NX, NY, NZ, 2 * np.pi, 2 * np.pi)
    ora = O.OracleSolver(r, geo, "ARS_222")
    rng = np.random.default_rng(NX)
    k = rng.standard_normal(ora.field[0].shape) + 1j * rng.standard_normal(ora.field[0].shape)
    ops, v = ora.kops[0], r.kxky_systems[0].var_names.index(small)
    k[..., ops.posP[ops.var_first[v]:ops.var_first[v] + ops.var_size[v]]] *= 1e-8
    k[~ora.keep] = 0.0
    k[0, 0] = 0.0
    O.project_kx0_plane(k, geo)
    ora.field, ora.zfield = [k.copy()], [0.0 * z for z in ora.zfield]
    q = ora.quad_spectra(ora.field, ora.zfield)
    with solver.Solver(r, NX, NY, NZ, 2 * np.pi, 2 * np.pi) as g:
        g.set_state([k], ora.zfield)
        got = g.products()
    for i, s in enumerate(q):
        want = np.where(ora.keep[:, :, None], s, 0.0)
        assert np.linalg.norm(got[i] - want) <= 2e-14 * np.linalg.norm(want), i   # the bar of the test above
