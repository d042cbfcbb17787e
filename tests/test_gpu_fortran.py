"""A Fortran host drives the library: libizem_fortran.so (the
ISO_C_BINDING module izem_hip_mod.f90 and the host driver izem_fdriver.f90,
compiled with the image's Fortran compiler) is loaded into this process and
does the set-up and one iteration of the main loop (devel-izem/src/
izem.f90:242-282) itself:

* izem_f_create: the context from thd_type's arrays in Fortran order
  (species dimension 29) through izem_thd_image;
* izem_f_chem_init: the mechanism from CHEMKIN-II's work arrays after CKINIT
  and the /CKSTRT/ pointers of the reference's own CHEMKIN-II library
  (oracle/_ref) through izem_mech_image_ckwrk;
* izem_f_main_iteration: timestep -> reaction_selec(dt/2) -> rk3(dt) ->
  reaction_selec(dt/2) (rk3 alone when inert), dt on the device.

On the 16^2 hot-spot case the Fortran-driven iteration equals the same
iteration driven through the C ABI from Python bit for bit (state,
temperature, time state); the inert iteration equals the oracle to 1e-12
and the reacting one lies within DVODE's own distance of the tight oracle
solution."""
from __future__ import annotations

import ctypes as C
import os

import numpy as np
import pytest

from tests.flowcase import OracleRun, P, oracle_reaction_dvode, small_state
from tests.fortran_host import THD_ORDER, ckwrk_addresses, thd_arrays, thd_ref_quantities

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _flib():
    from phd_amd import _lib, build
    if not os.path.exists(build.FORTRAN_LIB):
        pytest.skip("libizem_fortran.so not built (no Fortran compiler)")
    _lib.load()   # the same libizem_hip.so the Fortran library links
    L = C.CDLL(build.FORTRAN_LIB)
    vp = C.c_void_p
    L.izem_f_create.argtypes = [C.POINTER(vp), C.POINTER(_lib.Grid), C.POINTER(_lib.Opts),
                                C.c_int, C.c_int] + [vp] * 11
    L.izem_f_chem_init.argtypes = [vp, vp, vp, vp, C.c_double, C.c_double]
    L.izem_f_main_iteration.argtypes = [vp] * 10 + [C.c_int, C.POINTER(C.c_double),
                                                    C.POINTER(C.c_double)]
    return L


def _upload(s, run):
    import torch
    for name in ("v", "T", "W_i", "cp", "ha", "sensor"):
        getattr(s, name).copy_(torch.from_numpy(getattr(run, name)))
    torch.cuda.synchronize()


def _fortran_solver(F, box, opts, adi, thd, run, refchem=None):
    """A Solver whose context the Fortran host created (and, reacting, whose
    mechanism it loaded); the Solver's device buffers hold the state."""
    import torch
    from phd_amd import _lib
    from phd_amd.solver import Solver
    s = Solver(box, opts, adi=adi, thd=thd, mech=None)
    _lib.check(s.lib.izem_destroy(s.ctx), "izem_destroy")
    s.ctx = None
    arrays = thd_arrays(thd)
    ref = np.array(thd_ref_quantities(thd))
    ctx = C.c_void_p()
    F.izem_f_create(C.byref(ctx), C.byref(s.grid_struct), C.byref(s.opts_struct), 9, 29,
                    *[arrays[k].ctypes.data for k in THD_ORDER], ref.ctypes.data)
    assert ctx.value
    s.ctx = ctx
    _lib.check(s.lib.izem_flux_mode(ctx, opts.flux_mode), "izem_flux_mode")
    _lib.check(s.lib.izem_set_stream(ctx, C.c_void_p(
        torch.cuda.current_stream(s.dev).cuda_stream)), "izem_set_stream")
    if refchem is not None:
        iw, rw, ck = ckwrk_addresses(refchem)
        F.izem_f_chem_init(ctx, iw, rw, ck, opts.rtol, opts.atol)
    _upload(s, run)
    s.set_time_state([1.0, 1.0, 1.0, 1.0, 1.0, 0.0])
    return s


def _fortran_iteration(F, s, reaction):
    dtmin, DTmax = C.c_double(), C.c_double()
    p = [C.c_void_p(x.data_ptr()) for x in (*s.d_i, s.T, s.W_i, s.cp, s.ha, s.sensor, s.v)]
    print(f"fortran iteration, reaction {reaction}", flush=True)
    F.izem_f_main_iteration(s.ctx, *p, reaction, C.byref(dtmin), C.byref(DTmax))
    s.sync()
    return dtmin.value, DTmax.value


def _abi_iteration(s, reaction):
    s.timestep()
    dt = s.lib.izem_time_state(s.ctx) + 4 * 8
    if reaction:
        s.reaction_selec(dt, 0.5)
        s.rk3(dt)
        s.reaction_selec(dt, 0.5)
    else:
        s.rk3(dt)
    s.sync()


def _same(a, b):
    for name in ("v", "T", "W_i", "cp", "ha", "sensor"):
        assert np.array_equal(getattr(a, name).cpu().numpy(), getattr(b, name).cpu().numpy()), name
    assert np.array_equal(a.time_state(), b.time_state())


def test_fortran_host_inert_iteration(oracle, adi, thd):
    from phd_amd.solver import Options, Solver
    F = _flib()
    box, v, T = small_state(adi, thd, "2d", 16)
    run = OracleRun(oracle, adi, thd, box, v, T)
    run.prim_all()
    opts = Options(reaction=0)
    sa = Solver(box, opts, adi=adi, thd=thd)
    _upload(sa, run)
    sa.set_time_state([1.0, 1.0, 1.0, 1.0, 1.0, 0.0])
    _abi_iteration(sa, 0)
    sf = _fortran_solver(F, box, opts, adi, thd, run)
    dtmin, DTmax = _fortran_iteration(F, sf, 0)
    assert sf.status() == 0 and DTmax == 0.0
    _same(sf, sa)
    # the oracle's iteration
    o = run.opts(vis=1)
    ts = np.zeros(4)
    d = C.c_double(1.0)
    run.o.lib.ora_timestep(C.byref(run.g), C.byref(run.t), C.byref(run.a), C.byref(o),
                           P(run.d_i[0]), P(run.d_i[1]), P(run.d_i[2]), P(run.cp), P(run.W_i),
                           P(run.T), P(run.v), C.c_double(0.0), P(ts), C.byref(d))
    assert abs(dtmin - d.value) <= TOL * d.value
    st = run.o.lib.ora_rk3(C.byref(run.g), C.byref(run.t), C.byref(run.a), C.byref(o),
                           C.c_double(d.value), P(run.d_i[0]), P(run.d_i[1]), P(run.d_i[2]),
                           P(run.T), P(run.W_i), P(run.cp), P(run.ha),
                           run.sensor.ctypes.data_as(C.POINTER(C.c_uint8)), P(run.v), None)
    assert st == 0
    I = (slice(None),) + box.interior()
    vf = sf.v.cpu().numpy()
    scale = np.max(np.abs(run.v[I]), axis=(1, 2, 3))
    err = np.max(np.abs(vf[I] - run.v[I]), axis=(1, 2, 3)) / np.where(scale > 0, scale, 1.0)
    print(f"fortran host, inert 16^2: max rel err vs oracle {err.max():.2e}")
    assert err.max() <= TOL
    sa.close()
    sf.close()


def test_fortran_host_reacting_iteration(oracle, adi, thd, mech):
    from oracle.oracle import RefChem
    from phd_amd import ics
    from phd_amd.solver import Options, Solver
    from tests import chembars
    F = _flib()
    try:
        rc = RefChem()  # its COMMON blocks are the mechanism the Fortran host hands over
    except FileNotFoundError as e:
        pytest.skip(str(e))
    box, v, T = ics.config1_state(adi, thd, n=16, seed=7, T_peak=1800.0)
    run0 = OracleRun(oracle, adi, thd, box, v, T)
    run0.prim_all()
    rtol, atol = 1e-6, 1e-12
    opts = Options(rtol=rtol, atol=atol, CPR=1.0)
    sa = Solver(box, opts, adi=adi, thd=thd, mech=mech)
    _upload(sa, run0)
    sa.set_time_state([1.0, 1.0, 1.0, 1.0, 1.0, 0.0])
    _abi_iteration(sa, 1)
    sf = _fortran_solver(F, box, opts, adi, thd, run0, refchem=rc)
    dtmin, DTmax = _fortran_iteration(F, sf, 1)
    assert sf.status() == 0 and DTmax > 0.0
    _same(sf, sa)
    # the oracle's iteration with the reference's DVODE, at the run's and at
    # a tight tolerance
    outs = {}
    for name, tol in (("exact", chembars.TIGHT), ("dvode", (rtol, atol))):
        r = OracleRun(oracle, adi, thd, box, run0.v, run0.T)
        r.W_i[:], r.cp[:], r.ha[:] = run0.W_i, run0.cp, run0.ha
        o = r.opts(vis=1, reaction=1, CPR=1.0)
        ts = np.zeros(4)
        d = C.c_double(1.0)
        r.o.lib.ora_timestep(C.byref(r.g), C.byref(r.t), C.byref(r.a), C.byref(o),
                             P(r.d_i[0]), P(r.d_i[1]), P(r.d_i[2]), P(r.cp), P(r.W_i),
                             P(r.T), P(r.v), C.c_double(0.0), P(ts), C.byref(d))
        oracle_reaction_dvode(r, rc, adi, 0.5 * d.value, *tol)
        st = r.o.lib.ora_rk3(C.byref(r.g), C.byref(r.t), C.byref(r.a), C.byref(o),
                             C.c_double(d.value), P(r.d_i[0]), P(r.d_i[1]), P(r.d_i[2]),
                             P(r.T), P(r.W_i), P(r.cp), P(r.ha),
                             r.sensor.ctypes.data_as(C.POINTER(C.c_uint8)), P(r.v), None)
        assert st == 0
        oracle_reaction_dvode(r, rc, adi, 0.5 * d.value, *tol)
        outs[name] = (r, d.value)
    (rt, dt_t), (rd, _) = outs["exact"], outs["dvode"]
    assert abs(dtmin - dt_t) <= TOL * dt_t
    I = box.interior()

    def z(vv, TT):
        return np.concatenate([TT[I].reshape(-1, 1) * adi.T_ref,
                               (vv[(slice(5, 14),) + I] / vv[(0,) + I]).reshape(9, -1).T], axis=1)

    e = chembars.compare(z(sf.v.cpu().numpy(), sf.T.cpu().numpy()), z(rd.v, rd.T),
                         z(rt.v, rt.T), rtol, atol)
    print(f"fortran host, reacting 16^2: {chembars.summary(e)}")
    chembars.assert_like_dvode(e, floor=1e-3)
    sa.close()
    sf.close()
