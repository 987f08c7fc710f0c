"""Host copies of states, volumes and spectra: sizes below and above one chunk
(1 MiB) and one chunk per thread (8 MiB), with ragged last chunks."""
import numpy as np
import pytest

from conftest import product_recipe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(4, 6, 17), (16, 24, 33), (48, 36, 41), (64, 96, 65)],
                         ids=lambda g: "x".join(map(str, g)))
def test_states_and_volumes_round_trip(native_lib, grid):
    from coral_amd import solver
    NX, NY, NZ = grid
    print("grid", grid, flush=True)
    r = product_recipe("coral.equations.rbc_ra1e5")
    rng = np.random.default_rng(3)
    with solver.Solver(r, NX, NY, NZ, 2.0, 3.0) as g:
        kx, ky, dx, dy = g.wavenumbers()
        a = rng.standard_normal((NX // 2, 3 * NY // 2, g.totals[0])) + 1j * rng.standard_normal(
            (NX // 2, 3 * NY // 2, g.totals[0]))
        g.set_field("kxky", 0, a)
        b = g.get_field("kxky", 0)
        a[dx] = 0.0
        a[:, dy] = 0.0
        a[0, 0] = 0.0
        assert np.array_equal(a, b)      # copied, not computed
        # a variable written from its own volume keeps its coefficients (forward
        # and inverse transforms and a stencil solve: tens of eps of the largest)
        a[0] = 0.0                       # (the kx = 0 plane of a real field is Hermitian)
        g.set_field("kxky", 0, a)
        v = g.variable_physical("kxky", 0, 3)
        g.set_variable_physical("kxky", 0, 3, v)
        c = g.get_field("kxky", 0)
        assert np.linalg.norm(c - a) <= 1e-12 * np.linalg.norm(a)
        g.set_variable_physical("kxky", 0, 3, v)      # the tables of its first use again
        assert np.array_equal(g.get_field("kxky", 0), c)


def test_two_threads_read_one_run(native_lib):
    """Threads that read states of one run at the same time (the calls release
    the interpreter's lock) each get the whole state."""
    from concurrent.futures import ThreadPoolExecutor

    from coral_amd import solver
    r = product_recipe("coral.equations.rbc_ra1e5")
    rng = np.random.default_rng(4)
    with solver.Solver(r, 64, 96, 65, 2.0, 3.0) as g:
        shape = (32, 144, g.totals[0])
        g.set_field("kxky", 0, rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
        want = g.get_field("kxky", 0)
        with ThreadPoolExecutor(4) as ex:
            for got in ex.map(lambda _: g.get_field("kxky", 0), range(16)):
                assert np.array_equal(got, want)
