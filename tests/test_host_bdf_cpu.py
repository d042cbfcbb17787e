"""The chemistry integrator's source (phd_amd/csrc/chem_device.h), built for
the host with g++, against the reference's own compiled DVODE (oracle/_ref;
without that build DVODE as scipy ships it, oracle.VodeChem): both kinetics forms, the C3 cell recipe, the reactor
substep of izem_psr_batch.  Bars as in the GPU test: |dT| <= 2e-4 T and
|dY_k| <= 2e-4 |Y_k| + 1e-8 per cell, every cell integrated (ok)."""
import numpy as np
import pytest

@pytest.mark.parametrize("kinetics", [0, 1])
def test_host_integrator_vs_reference_dvode(host_bdf, thd, kinetics):
    from oracle.oracle import refchem
    from phd_amd import ics
    rc = refchem()
    n = 48
    T, p, Y = ics.config3_cells(thd, n, seed=11)
    Wmix = 1.0 / (Y / (np.array(thd.W) * 1000.0)).sum(axis=1)
    rho = (p * 10.0) * Wmix / (8.314510e7 * T)
    dt, rtol, atol = 1e-6, 1e-6, 1e-12
    Th, Yh = T.copy(), np.ascontiguousarray(Y.copy())
    nst, ok = np.zeros(n, np.int32), np.zeros(n, np.int32)
    host_bdf.host_psr(kinetics, n, Th.ctypes.data, rho.ctypes.data, Yh.ctypes.data, dt, rtol,
                      atol, 50, nst.ctypes.data, ok.ctypes.data)
    assert ok.all()
    errT, errY, steps = 0.0, 0.0, []
    for c in range(n):
        Tr, Yr, ist, ns, nfe, nje = rc.psr(T[c], rho[c], Y[c], dt, rtol, atol)
        assert ist == 2
        steps.append(ns)
        errT = max(errT, abs(Th[c] - Tr) / Tr)
        errY = max(errY, np.max(np.abs(Yh[c] - Yr) / (2e-4 * np.abs(Yr) + 1e-8)))
    print(f"host BDF vs DVODE: max |dT|/T {errT:.2e}, Y err / bound {errY:.2f}, "
          f"steps {nst.mean():.1f} (DVODE {np.mean(steps):.1f})")
    assert errT <= 2e-4
    assert errY <= 1.0
    assert np.all(np.abs(Yh.sum(axis=1) - 1.0) <= 1e-12)


def test_host_integrator_global_error_like_dvode(host_bdf, thd):
    """At the same rtol/atol the integrator's global error is like DVODE's:
    both measured against DVODE run at rtol 1e-11, atol 1e-17, in DVODE's
    error norm (tests/chembars.py), on C3 cells at two substeps and on the
    cells of a 3-D decaying-HIT state over an igniting 2e-4 s substep."""
    from oracle.oracle import Oracle, refchem
    from phd_amd import chemdata as cd, ics
    from tests import chembars
    from tests.flowcase import OracleRun, small_state
    rc = refchem()
    cases = []
    for seed, n, dt in ((11, 64, 1e-6), (7, 48, 1e-7), (5, 48, 1e-5)):
        T, p, Y = ics.config3_cells(thd, n, seed=seed)
        Wmix = 1.0 / (Y / (np.array(thd.W) * 1000.0)).sum(axis=1)
        cases.append((T, (p * 10.0) * Wmix / (8.314510e7 * T), Y, dt))
    adi = cd.Adim()
    box, v, T = small_state(adi, thd, "3d", 10)
    run = OracleRun(Oracle(), adi, thd, box, v, T)
    run.prim_all()
    I = box.interior()
    rho = run.v[(0,) + I].ravel()
    cases.append((run.T[I].ravel() * adi.T_ref, rho * adi.rho_ref * 1e-3,
                  np.ascontiguousarray((run.v[(slice(5, 14),) + I] / run.v[(0,) + I]).reshape(9, -1).T),
                  2e-4))
    for T, rho, Y, dt in cases:
        n = len(T)
        Th, Yh = T.copy(), np.ascontiguousarray(Y.copy())
        nst, ok = np.zeros(n, np.int32), np.zeros(n, np.int32)
        host_bdf.host_psr(1, n, Th.ctypes.data, np.ascontiguousarray(rho).ctypes.data,
                          Yh.ctypes.data, dt, 1e-6, 1e-12, 50, nst.ctypes.data, ok.ctypes.data)
        assert ok.all()
        e = chembars.dvode_errors(rc, T, rho, Y, dt, Th, Yh)
        print(f"{n} cells, dt {dt:g}: {chembars.summary(e)}")
        chembars.assert_like_dvode(e)


def test_closed_form_jacobian_columns(host_bdf, thd):
    """The generated mass-fraction columns of the reactor Jacobian (gen_jac)
    against fourth-order central differences of the same right-hand side,
    on ignition-range cells with radicals present (every reaction, third
    body and falloff branch active): within 1e-5 of each column's scale (the
    difference quotients themselves are good to about 1e-6)."""
    from phd_amd import ics
    T, p, Y = ics.config3_cells(thd, 24, seed=21)
    Y = Y.copy()
    Y[:, [0, 2, 4, 6, 7]] += np.array([1e-4, 2e-4, 3e-3, 1e-5, 2e-6])
    Y /= Y.sum(axis=1, keepdims=True)
    Wmix = 1.0 / (Y / (np.array(thd.W) * 1000.0)).sum(axis=1)
    rho = (p * 10.0) * Wmix / (8.314510e7 * T)
    worst = 0.0
    for c in range(len(T)):
        z = np.concatenate([[T[c]], Y[c]])
        J = np.zeros((10, 10))
        host_bdf.host_jac(rho[c], z.ctypes.data, J.ctypes.data)
        for j in range(1, 10):
            h = 1e-4 * max(z[j], 1e-6)
            cols = []
            for s in (-2, -1, 1, 2):
                zz = z.copy()
                zz[j] += s * h
                f = np.zeros(10)
                host_bdf.host_rhs(1, rho[c], zz.ctypes.data, f.ctypes.data)
                cols.append(f)
            fd = (cols[0] - 8 * cols[1] + 8 * cols[2] - cols[3]) / (12 * h)
            scale = np.max(np.abs(fd)) + 1e-30
            worst = max(worst, np.max(np.abs(J[:, j] - fd)) / scale)
    print("closed-form vs central-difference columns, worst", worst)
    assert worst <= 1e-5


def test_closed_form_jacobian_integrator_like_dvode(host_bdf, thd):
    """The integrator with the closed-form mass-fraction columns keeps
    DVODE's accuracy (tests/chembars.py) on C3 cells at 1e-6 s."""
    from oracle.oracle import refchem
    from phd_amd import ics
    from tests import chembars
    rc = refchem()
    T, p, Y = ics.config3_cells(thd, 64, seed=11)
    Wmix = 1.0 / (Y / (np.array(thd.W) * 1000.0)).sum(axis=1)
    rho = (p * 10.0) * Wmix / (8.314510e7 * T)
    out = {}
    for kin in (1, 2):
        Th, Yh = T.copy(), np.ascontiguousarray(Y.copy())
        nst, ok = np.zeros(64, np.int32), np.zeros(64, np.int32)
        host_bdf.host_psr(kin, 64, Th.ctypes.data, rho.ctypes.data, Yh.ctypes.data, 1e-6, 1e-6,
                          1e-12, 50, nst.ctypes.data, ok.ctypes.data)
        assert ok.all()
        out[kin] = (Th, Yh, nst.mean())
    e = chembars.dvode_errors(rc, T, rho, Y, 1e-6, out[2][0], out[2][1])
    print("closed-form Jacobian:", chembars.summary(e), "steps", out[2][2], "(FD", out[1][2], ")")
    chembars.assert_like_dvode(e)
