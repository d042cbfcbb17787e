"""The face reconstruction of izem_flux_mode 1 (phd_amd/csrc/iz_weno.h, host
build) against the reference's form (wenopar, wenorec: module_weno.f90:
114-190, 286-527) in extended precision, over the range of fluxes that its
comment states."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "phd_amd", "csrc")
L = np.longdouble


@pytest.fixture(scope="module")
def wlib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("weno")
    (d / "w.cpp").write_text('#define IZ_HD static\n#include "iz_weno.h"\n'
                             'extern "C" double face(int js, const double *p, const double *m) '
                             '{ const double r = d_weno5_face_fused<false>(js, p, m); return fabs(r) < INFINITY '
                             '? r : d_weno5_face_fused<true>(js, p, m); }\n')
    so = d / "w.so"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas", "-shared", "-fPIC",
                    "-I", CSRC, "-o", str(so), str(d / "w.cpp")], check=True)
    lib = C.CDLL(str(so))
    lib.face.restype = C.c_double
    lib.face.argtypes = [C.c_int, C.c_void_p, C.c_void_p]
    return lib


def side(q):
    """WENO5 value right of q[2] for the five values q."""
    q = q.astype(L)
    z1, z2, eps = L(13) / 12, L(1) / 4, L(10) ** -10
    v = [(2 * q[2] + 5 * q[3] - q[4]) / 6, (-q[1] + 5 * q[2] + 2 * q[3]) / 6,
         (2 * q[0] - 7 * q[1] + 11 * q[2]) / 6]
    b = [z1 * (q[2] - 2 * q[3] + q[4]) ** 2 + z2 * (3 * q[2] - 4 * q[3] + q[4]) ** 2,
         z1 * (q[1] - 2 * q[2] + q[3]) ** 2 + z2 * (q[1] - q[3]) ** 2,
         z1 * (q[0] - 2 * q[1] + q[2]) ** 2 + z2 * (q[0] - 4 * q[1] + 3 * q[2]) ** 2]
    a = [c / (eps + x) ** 2 for c, x in zip((L(3) / 10, L(6) / 10, L(1) / 10), b)]
    return sum(x * y for x, y in zip(a, v)) / sum(a)


@pytest.mark.parametrize("kind", ["random", "smooth", "jump", "mixed"])
def test_fused_face_over_its_range(wlib, kind):
    """Fluxes of 1e-12 to 1e70 units: within 1e-13 of the largest one (the
    weighted mean of candidates whose coefficients sum to less than 4 in
    magnitude; a few hundred roundings)."""
    rng = np.random.default_rng(4)
    for s in 10.0 ** np.arange(-12, 71):
        for _ in range(20):
            x = np.arange(6)
            g = {"random": lambda: rng.uniform(-1, 1, (2, 6)),
                 "smooth": lambda: 1.0 + 1e-3 * np.sin(0.3 * x + rng.uniform(0, 6, (2, 1))),
                 "jump": lambda: np.where(x < rng.integers(0, 7), 1.0, 1e-3) * np.ones((2, 1)),
                 "mixed": lambda: rng.uniform(-1, 1, (2, 6)) * np.array([[1.0], [1e-6]])}[kind]()
            gp, gm = np.ascontiguousarray(2.0 * s * g[0]), np.ascontiguousarray(2.0 * s * g[1])
            got = wlib.face(1, gp.ctypes.data, gm.ctypes.data)
            ref = side(gp[:5] / 2) + side(gm[:0:-1] / 2)
            assert abs(L(got) - ref) <= 1e-13 * max(np.abs(gp).max(), np.abs(gm).max()), (s, g)
