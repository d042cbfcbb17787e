"""Which kinetics form runs (phd_amd/csrc/chem_setup.h, host build): each
straight-line form is judged by its own run of the setup check."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "phd_amd", "csrc")


@pytest.fixture(scope="module")
def flib(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("forms")
    (d / "f.cpp").write_text(
        '#include "chem_setup.h"\nextern "C" {\n'
        'int form(int ok, int waves, int k) { return iz_chem_form(ok, waves, k); }\n'
        'int agree(int n, const double *T0, const int *n0, const double *T, const int *n1) '
        '{ return iz_forms_agree(n, T0, n0, T, n1); }\n}\n')
    so = d / "f.so"
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-I", CSRC, "-o", str(so),
                    str(d / "f.cpp")], check=True)
    return C.CDLL(str(so))


def test_form_of_a_request(flib):
    # a closed-form Jacobian that disagrees leaves the finite-difference form
    # to be asked for and to be the default
    want = {  # ok: (kinetics -1, 0, 1, 2) at one wave
        0: (0, 0, -1, -1), 1: (1, 0, 1, -1), 2: (2, 0, -1, 2), 3: (2, 0, 1, 2)}
    for ok, forms in want.items():
        assert tuple(flib.form(ok, 1, k) for k in (-1, 0, 1, 2)) == forms
        for waves in (2, 4):
            assert tuple(flib.form(ok, waves, k) for k in (-1, 0, 1, 2)) == (0, 0, -1, -1)


def test_verdict(flib):
    T0, n0 = np.linspace(1000.0, 1630.0, 64), np.full(64, 100, np.int32)

    def agree(T, n):
        a = [np.ascontiguousarray(x) for x in (T0, n0, T, n)]
        return flib.agree(64, *(C.c_void_p(x.ctypes.data) for x in a))

    assert agree(T0 * (1 + 9e-7), n0 + 2)
    for bad in (T0 * (1 + 2e-6), np.where(T0 > 1600, np.nan, T0), T0 + (T0 == 1000.0)):
        assert not agree(bad, n0)
    assert not agree(T0, n0 + 4)
