"""Which wavenumbers share one factorization (host code): every kept wavenumber
is served once, and at each member the oracle's operators are those of the
factored wavenumber with rows and columns renumbered and some signs changed."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import coral_oracle as O

from conftest import ROOT, product_recipe, recipe

RBC, RRBC = "coral.equations.rbc_ra1e5", "coral.equations.rrbc_ra5e7_ek1e-4"
# recipe, NX, NY, Lx, Ly, members at most
CASES = [
    (RBC, 8, 8, 2.0, 2.0, 4),
    (RBC, 8, 12, 2.0, 2.0, 4),
    (RBC, 16, 6, 2.0, 2.0, 4),
    (RBC, 8, 8, 2.0, 3.0, 2),
    (RRBC, 8, 8, 2.0, 2.0, 2),
    (RRBC, 6, 12, 2.0, 2.0, 2),
    (RRBC, 8, 8, 2.0, 3.0, 1),
    ("rrbc_julien.coral.equations.toroidalPoloidal", 8, 8, 2.0, 2.0, 4),
    ("stratified_channel.coral.equations.velocityPressure", 8, 8, 2.0, 2.0, 4),
    ("baroclinic_turbulence.coral.equations", 8, 8, 2.0, 2.0, 2),
]


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("probe") / "probe.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", so,
                    os.path.join(ROOT, "tests", "native", "sharing_probe.cpp"),
                    os.path.join(ROOT, "coral_amd", "csrc", "assembly.cpp")], check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0].split('.')[-1]}-{c[1]}x{c[2]}-{c[5]}" for c in CASES])
def test_members_have_the_factored_system(native_lib, probe, case):
    from coral_amd import solver
    name, NX, NY, Lx, Ly, nshare = case
    r = product_recipe(name) if name in (RBC, RRBC) else recipe(name)
    NZ, nkx, nky = 10, NX // 2, NY - 1
    prob, keep = solver.build_problem(r, NX, NY, NZ, Lx, Ly)
    ops = O.SystemOps(r.kxky_systems[0], NZ, 0.5, 1.0)
    n, total = nkx * nky, ops.total
    rep, mem, nrep = np.zeros(n, np.int32), np.full(4 * n, -9, np.int32), ctypes.c_int()
    row, col = np.zeros((3, total), np.int32), np.zeros((3, total), np.int32)
    rneg, cneg = np.zeros((3, total), np.uint8), np.zeros((3, total), np.uint8)
    nslot = probe.sharing_probe(ctypes.byref(prob), 0, ctypes.byref(nrep),
                                *[a.ctypes.data_as(ctypes.c_void_p) for a in (rep, mem, row, col, rneg, cneg)])
    assert nslot == nshare
    if nshare == 1:
        return
    rep, mem = rep[:nrep.value], mem[:nrep.value * nslot].reshape(-1, nslot)
    assert np.array_equal(mem[:, 0], rep)
    assert sorted(mem[mem >= 0]) == list(range(n)) and mem.min() >= -1
    assert (mem[rep == 0][0, 1:] == -1).all()           # (0, 0) stands alone
    groups = [ops.grouped_pieces(p) for p in (ops.sys.mass, ops.sys.stif)]

    def operator(which, s):
        jy = s % nky
        px, py = 2j * np.pi / Lx * (s // nky), 2j * np.pi / Ly * (jy if jy < NY // 2 else jy - nky)
        return sum(px ** a * py ** b * m for (a, b), m in groups[which])

    for s, members in zip(rep, mem):
        if s == 0:
            continue
        for which in (0, 1):
            A = operator(which, s)
            for q, o in enumerate(members[1:]):
                if o >= 0:
                    B = operator(which, o)[np.ix_(row[q], col[q])]
                    sign = np.where(rneg[q], -1.0, 1.0)[:, None] * np.where(cneg[q], -1.0, 1.0)
                    # sums of a few monomials: rounding of their powers
                    assert np.abs(B - sign * A).max() <= 1e-14 * np.abs(A).max(), (s, o, which)
