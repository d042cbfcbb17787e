"""The generated straight-line kinetics (phd_amd/csrc/mech_gen.h) is what
the generator writes for the bundled mechanism, and the generator takes the
mechanisms that the table-driven kinetics take."""
import copy
import ctypes as C
import os
import shutil
import subprocess
from types import SimpleNamespace

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_generated_file_is_current():
    from phd_amd import chemdata as cd
    from phd_amd.codegen_mech import OUT, generate
    with open(OUT) as f:
        assert f.read() == generate(cd.read_mechanism())


def _mixed_mid_temperatures(m):
    m.tmid[2] = 1400.0   # O
    m.tmid[5] = 800.0    # H2O


def _centring_temperatures(m):
    # Troe factors with a vanishing T3 or an endless T1, T2 beside finite ones
    r = [r for r in m.reactions if r["fal"] >= 3]
    r[0]["fpar"][3:6] = [0.8, 1.0e-100, 900.0]
    r[1]["fal"] = 4
    r[1]["fpar"][3:6] = [0.5, 700.0, 1.0e30]
    r[1]["fpar"] = r[1]["fpar"][:6] + [1.0e100] + r[1]["fpar"][7:]


@pytest.mark.parametrize("change,T0,T1", [
    (None, 250.0, 3000.0), (_mixed_mid_temperatures, 300.0, 3000.0),
    (_centring_temperatures, 300.0, 3000.0)])
def test_straight_line_like_tables(tmp_path, mech, change, T0, T1):
    """The generated right-hand side against the table-driven one, both on
    the host, at 400 states between two temperatures: within 1e-10 of the
    species' and of the temperature's largest rate (rates agree to a few
    hundred ulp where forward and reverse cancel), and the temperature column
    of the Jacobian against central differences (1e-6 of the column)."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    from phd_amd.codegen_mech import generate
    from phd_amd.solver import mech_flat
    m = copy.deepcopy(mech)
    if change:
        change(m)
    (tmp_path / "mech_gen.h").write_text(generate(m))
    (tmp_path / "h.cpp").write_text(open(os.path.join(HERE, "host_bdf.cpp")).read() + """
extern "C" void host_jac_T(double rho, const double *z, double *J) {
  double kt[GEN_NKT], f[N_];
  gen_kT(z[0], kt);
  gen_rhs(rho, z, kt, f);
  gen_jac_T(rho, z, kt, f, (double (*)[N_])J);
}
""")
    so = tmp_path / "h.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", str(tmp_path),
                    "-I", os.path.join(HERE, "..", "phd_amd", "csrc"), "-o", str(so),
                    str(tmp_path / "h.cpp")], check=True)
    L = C.CDLL(str(so))
    L.host_setup.argtypes = [C.c_void_p, C.c_long]
    L.host_rhs.argtypes = [C.c_int, C.c_double, C.c_void_p, C.c_void_p]
    L.host_jac_T.argtypes = [C.c_double, C.c_void_p, C.c_void_p]
    mf = mech_flat(m)
    assert L.host_setup(mf.ctypes.data, mf.size) == 0

    def rhs(kin, rho, z):
        f = np.zeros(10)
        L.host_rhs(kin, rho, z.ctypes.data, f.ctypes.data)
        return f

    rng = np.random.default_rng(3)
    for _ in range(400):
        z = np.concatenate([[rng.uniform(T0, T1)], rng.random(9) ** 3])
        z[1:] /= z[1:].sum()
        rho = 10 ** rng.uniform(-6.0, -3.0)
        f, g = rhs(0, rho, z), rhs(1, rho, z)
        assert np.all(np.isfinite(g))
        assert np.max(np.abs(f[1:] - g[1:])) <= 1e-10 * np.max(np.abs(f[1:])), z[0]
        assert abs(f[0] - g[0]) <= 1e-10 * abs(f[0]) + 1e-300, z[0]
        # a fixed mid temperature or centring slope aside
        if change is _centring_temperatures or np.min(np.abs(z[0] / m.tmid - 1.0)) < 1e-3:
            continue
        J, h = np.zeros((10, 10)), 1e-4 * z[0]
        L.host_jac_T(rho, z.ctypes.data, J.ctypes.data)
        fd = sum(c * rhs(1, rho, z + s * h * np.eye(10)[0])
                 for s, c in ((-2, 1), (-1, -8), (1, 8), (2, -1))) / (12 * h)
        assert np.all(np.abs(J[:, 0] - fd) <= 1e-6 * (np.abs(fd) + np.abs(fd).max()))


def test_basis_of_any_composition():
    """Species as fractions of others (3/7 of one with seven atoms)."""
    from phd_amd.codegen_mech import _basis
    a = np.zeros((3, 2, 7))
    a[:, 0, 5] = [0.0, 1.0e4, 2.0e4]   # the first is the basis species
    basis, B = _basis(SimpleNamespace(kk=3, ncf=np.array([[7.0], [3.0], [11.0]]), a=a))
    assert basis == [0]
    assert np.array_equal(B[:, 0], [1.0, 3.0 / 7.0, 11.0 / 7.0])


def test_duplicates_without_a_rate(mech):
    """The slope of a sum of Arrhenius terms that underflows or cancels is not
    formed as 0 / 0."""
    from phd_amd.codegen_mech import generate
    m = copy.deepcopy(mech)
    for r in m.reactions:
        if r["dup"]:
            r["EoR"] = abs(r["EoR"]) + 1.0
    src = generate(m)
    assert src.count("!= 0.0 ?") == len({r["eq"] for r in m.reactions if r["dup"]})
    assert "!= 0.0 ?" not in generate(mech)
