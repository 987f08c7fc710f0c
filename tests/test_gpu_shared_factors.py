"""Factors shared between wavenumbers that the operators' symmetries relate:
the solve of every system, the time step and the factor counts against runs
that factor every wavenumber (CORAL_AMD_NO_SHARED_FACTORS=1)."""
import numpy as np
import pytest

from conftest import product_recipe

pytestmark = pytest.mark.gpu

TP = "rrbc_julien.coral.equations.toroidalPoloidal"
# recipe, NX, NY, NZ, Lx, Ly, wavenumbers per factorization: reflection and
# rotation, the reflection alone (unequal box), the rotation alone, none; uneven
# grids (partners outside the kept modes); complex factors; from 96 x 96 on, two
# right-hand sides per wavefront
CASES = [
    ("coral.equations.rbc_ra1e5", 16, 16, 17, 2.0, 2.0, 4, False),
    ("coral.equations.rbc_ra1e5", 16, 24, 18, 2.0, 3.0, 2, False),
    ("coral.equations.rbc_ra1e5", 24, 16, 17, 2.0, 2.0, 4, True),
    ("coral.equations.rrbc_ra5e7_ek1e-4", 16, 16, 17, 2.0, 2.0, 2, False),
    ("coral.equations.rrbc_ra5e7_ek1e-4", 16, 32, 19, 2.0, 2.0, 2, False),
    ("coral.equations.rrbc_ra5e7_ek1e-4", 16, 16, 17, 2.0, 3.0, 1, False),
    (TP, 16, 18, 20, 2.0, 2.0, 4, False),
    ("coral.equations.rbc_ra1e5", 96, 96, 33, 2.0, 2.0, 4, False),
    ("coral.equations.rrbc_ra5e7_ek1e-4", 96, 96, 33, 2.0, 2.0, 2, False),
]


def recipe_of(name):
    if name == TP:
        from conftest import recipe
        return recipe(name)
    return product_recipe(name)


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0].split('.')[-1]}-{c[1]}x{c[2]}x{c[3]}-{c[6]}{'c' * c[7]}" for c in CASES])
def test_shared_factors_match_factoring_every_system(native_lib, monkeypatch, case):
    from coral_amd import solver
    name, NX, NY, NZ, Lx, Ly, nshare, cplx = case
    print("case", case, flush=True)
    if cplx:
        monkeypatch.setenv("CORAL_AMD_COMPLEX_FACTORS", "1")
    r = recipe_of(name)
    rng = np.random.default_rng(7)
    out = []
    for off in (False, True):
        if off:
            monkeypatch.setenv("CORAL_AMD_NO_SHARED_FACTORS", "1")
        with solver.Solver(r, NX, NY, NZ, Lx, Ly) as g:
            g.factorize_operators(1e-5)
            kept = g.system_info(0)[3]
            nfac, share = g.factored_systems(0)
            assert share == (1 if off else nshare)
            assert nfac == kept if share == 1 else nfac < kept
            if share == nshare > 1 and NX == NY:
                # the axes' sets are incomplete, every other one is full
                assert nfac <= kept / nshare + NX + NY
            if not out:
                shape = (NX // 2, 3 * NY // 2, g.totals[0])
                rhs = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
                state = 1e-3 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
                z = [1e-3 * rng.standard_normal(n) for n in g.zero_totals]
                kx, ky, dx, dy = g.wavenumbers()
                state[dx] = 0.0
                state[:, dy] = 0.0
                state[0] = 0.0
            x = g.solve_system(0, rhs)
            g.set_state([state], z)
            g.march_forward(1e-5, 2)
            out.append((x, g.get_state()[0][0]))
    (x, s), (x1, s1) = out
    # both are backward stable solves of the same systems; the bar is the
    # parity tests'
    assert np.array_equal(x[0, 0], x1[0, 0])
    assert np.linalg.norm(x - x1) <= 1e-10 * np.linalg.norm(x1)
    per = np.linalg.norm(x - x1, axis=-1) / np.maximum(np.linalg.norm(x1, axis=-1), 1e-300)
    assert per.max() <= 1e-8, np.unravel_index(per.argmax(), per.shape)
    assert np.linalg.norm(s - s1) <= 1e-10 * np.linalg.norm(s1)


# recipe, NX = NY, NZ, whole systems (16 subdiagonals), complex factors: every
# window size (2, 3, 4 registers) and both element types with two right-hand
# sides per wavefront, which takes 1024 of such wavefronts
TWO = [
    ("radiative_heating.coral.equations", 96, 14, False, False),
    ("radiative_heating.coral.equations", 96, 14, False, True),
    ("coral.equations.rbc_ra1e5", 96, 14, False, True),
    ("coral.equations.rbc_ra1e5", 144, 14, True, False),
    ("coral.equations.rbc_ra1e5", 144, 14, True, True),
    ("coral.equations.rrbc_ra5e7_ek1e-4", 144, 14, True, True),
]


@pytest.mark.parametrize("case", TWO, ids=[f"{c[0].split('.')[-1]}-{c[1]}x{c[2]}{'w' * c[3]}{'c' * c[4]}" for c in TWO])
def test_two_right_hand_sides_per_wavefront(native_lib, monkeypatch, case):
    from coral_amd import solver
    name, NX, NZ, whole, cplx = case
    print("case", case, flush=True)
    monkeypatch.setenv("CORAL_AMD_NO_BLOCK_SPLIT", "1" if whole else "0")
    monkeypatch.setenv("CORAL_AMD_COMPLEX_FACTORS", "1" if cplx else "0")
    from conftest import recipe
    r = product_recipe(name) if name.startswith("coral.") else recipe(name)
    rng = np.random.default_rng(11)
    out, rhs = [], None
    for off in ("0", "1"):
        monkeypatch.setenv("CORAL_AMD_NO_SHARED_FACTORS", off)
        with solver.Solver(r, NX, NX, NZ, 2.0, 2.0) as g:
            g.factorize_operators(1e-5)
            nfac, share = g.factored_systems(0)
            nblk, _, kl, _ = g.factor_blocks(0)[:4]
            if off == "0":
                assert share >= 2 and (nfac * nblk + 3) // 4 * (share // 2) >= 1024
                assert (kl == 16) == whole and g.factor_is_real(0) == (not cplx)
                shape = (NX // 2, 3 * NX // 2, g.totals[0])
                rhs = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
            else:
                assert share == 1
            out.append(g.solve_system(0, rhs))
    x, x1 = out
    # the bars of the test above
    assert np.array_equal(x[0, 0], x1[0, 0])
    assert np.linalg.norm(x - x1) <= 1e-10 * np.linalg.norm(x1)
    per = np.linalg.norm(x - x1, axis=-1) / np.maximum(np.linalg.norm(x1, axis=-1), 1e-300)
    assert per.max() <= 1e-8, np.unravel_index(per.argmax(), per.shape)
