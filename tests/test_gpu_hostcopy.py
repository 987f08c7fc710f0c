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


def _free_bytes():
    import ctypes

    from coral_amd import devmem
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert devmem.hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_reading_keeps_no_device_memory(native_lib):
    """Products, fields, variables and transforms leave only the volume that the
    physical fields are formed in and the small tables of a variable."""
    from coral_amd import solver
    r = product_recipe("coral.equations.rbc_ra1e5")
    rng = np.random.default_rng(5)
    with solver.Solver(r, 96, 96, 65, 2.0, 2.0) as g:
        shape = (48, 144, g.totals[0])
        g.set_field("kxky", 0, rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
        g.factorize_operators(1e-5)
        g.march_forward(1e-5, 1)
        volume = 8 * 144 * 144 * 97
        start = _free_bytes()
        g.physical(0)
        q = g.products()
        g.bwd_transform(q[0])
        v = g.variable_physical("kxky", 0, 2)
        g.fwd_transform(v)
        g.set_variable_physical("kxky", 0, 2, v)
        # the allocator hands out memory in pieces of up to 4 MiB; the spectra of
        # the nine products in the host's layout are 42 MB
        assert start - _free_bytes() <= volume + (8 << 20)


def test_recipe_without_products(native_lib):
    """One full variable and no products: the spectra are too small for a volume
    in the host's layout, which then has an array of its own."""
    from coral_amd import solver

    from conftest import recipe
    rng = np.random.default_rng(6)
    out = []
    for few in (False, True):
        r = recipe("heat_equation.coral.equations")
        if few:
            r.full_vars, r.quad_vars = r.full_vars[:1], []
            for s in r.kxky_systems + r.zero_systems:
                s.nl = []
        with solver.Solver(r, 32, 24, 33, 2.0, 3.0) as g:
            if not out:
                shape = (16, 36, g.totals[0])
                a = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
                a[0] = 0.0
            g.set_field("kxky", 0, a)
            v = g.variable_physical("kxky", 0, 0)
            g.set_variable_physical("kxky", 0, 0, 2.0 * v)
            out.append((v, g.get_field("kxky", 0), g.bwd_transform(g.fwd_transform(v))))
    for x, y in zip(*out):
        assert np.array_equal(x, y) and np.abs(x).max() > 0
