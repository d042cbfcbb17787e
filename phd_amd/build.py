"""Build the IZEM HIP library for gfx950 in-tree (phd_amd/libizem_hip.so).

The flow and chemistry kernels are compiled with -ffp-contract=off.  The
flow kernels that keep the reference's operation order (flow.hip says which)
so reproduce its rounding; the others turn contraction on by a pragma.  The
chemistry integrator and its straight-line kinetics turn contraction on
expression by expression (a pragma), which rounds every inlined copy alike;
left to the optimiser it was decided per copy, and one build took twice
DVODE's steps on the same cells.  The surrogate's BF16 matrix-core kernels (mlp.hip) have
no parity constraint and keep contraction.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libizem_hip.so")

ARCH = os.environ.get("IZEM_OFFLOAD_ARCH", "gfx950")
COMMON = ["-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}", "-Wall",
          "-Wno-unused-function", "-Wno-unused-variable",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
SOURCES = {
    "flow.hip": ["-ffp-contract=off"],
    # the kinetics' few hundred literals are rebuilt at each use: hoisted out
    # of the step loop they fill the scalar registers and spill (900 of them)
    "chem.hip": ["-ffp-contract=off", "-mllvm", "-disable-machine-licm"],
    "step.hip": ["-ffp-contract=off"],
    "mlp.hip": ["-ffp-contract=fast"],
    "images.hip": ["-ffp-contract=off"],
}


def hipcc() -> str:
    for cand in ("/opt/rocm/bin/hipcc", "hipcc"):
        if os.path.exists(cand) or cand == "hipcc":
            return cand
    raise RuntimeError("hipcc not found")


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    objs = []
    for src, extra in SOURCES.items():
        obj = os.path.join(BUILD, src.replace(".hip", ".o"))
        cmd = [hipcc(), "-c", os.path.join(CSRC, src), "-o", obj] + COMMON + extra
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError(f"hipcc failed on {src}")
        objs.append(obj)
    tmp = LIB + ".tmp"
    cmd = [hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("link failed")
    os.replace(tmp, LIB)
    for nrv, ng in FLOW_VARIANTS:
        build_flow_variant(nrv, ng, verbose)
    build_io(verbose)
    build_fortran(verbose)
    return LIB


# flow-only builds for other (species count, ghost depth) pairs: the flow
# kernels of flow.hip compiled with IZ_NRV / IZ_NG set, without the
# chemistry, the surrogate and the captured step.  (9, 4): WENO7 for the
# H2/air species; (2, 4): the reference's O2/N2 shock tube.
FLOW_VARIANTS = ((9, 4), (2, 4))


def flow_variant_path(nrv: int, ng: int) -> str:
    return os.path.join(HERE, f"libizem_flow_nrv{nrv}_ng{ng}.so")


def build_flow_variant(nrv: int, ng: int, verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    defs = [f"-DIZ_NRV={nrv}", f"-DIZ_NG={ng}"]
    objs = []
    for src in ("flow.hip", "flow_only.hip"):
        obj = os.path.join(BUILD, src.replace(".hip", f"_nrv{nrv}_ng{ng}.o"))
        cmd = [hipcc(), "-c", os.path.join(CSRC, src), "-o", obj] + COMMON + \
            ["-ffp-contract=off"] + defs
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError(f"hipcc failed on {src} ({' '.join(defs)})")
        objs.append(obj)
    out = flow_variant_path(nrv, ng)
    tmp = out + ".tmp"
    r = subprocess.run([hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objs,
                       capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("link failed")
    os.replace(tmp, out)
    return out


HDF5 = os.environ.get("IZEM_HDF5_PREFIX", "/opt/conda")
IO_LIB = os.path.join(HERE, "libizem_io.so")


def build_io(verbose: bool = False) -> str | None:
    """libizem_io.so (restart files, host code) with the host compiler
    against the HDF5 C library; skipped with a message when HDF5 is absent."""
    inc, lib = os.path.join(HDF5, "include"), os.path.join(HDF5, "lib")
    if not os.path.exists(os.path.join(inc, "hdf5.h")):
        print(f"[build] HDF5 not found under {HDF5}: restart files unavailable", flush=True)
        return None
    tmp = IO_LIB + ".tmp"
    cmd = ["gcc", "-O2", "-fPIC", "-shared", "-std=c11", "-Wall", "-I", inc, "-o", tmp,
           os.path.join(CSRC, "restart_io.c"), "-L", lib, "-lhdf5", f"-Wl,-rpath,{lib}"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("restart I/O library build failed")
    os.replace(tmp, IO_LIB)
    return IO_LIB


FORTRAN_LIB = os.path.join(HERE, "libizem_fortran.so")
FORTRAN_SOURCES = ("izem_hip_mod.f90", "izem_fdriver.f90")


def fortran_compiler() -> str | None:
    import shutil
    return shutil.which("amdflang") or shutil.which("flang")


def build_fortran(verbose: bool = False) -> str | None:
    """libizem_fortran.so: the ISO_C_BINDING module and the Fortran host
    driver (fortran/), linked against libizem_hip.so; skipped with a message
    when no Fortran compiler is installed."""
    fc = fortran_compiler()
    if fc is None:
        print("[build] no Fortran compiler: libizem_fortran.so not built", flush=True)
        return None
    mod_dir = os.path.join(BUILD, "fortran")
    os.makedirs(mod_dir, exist_ok=True)
    tmp = FORTRAN_LIB + ".tmp"
    cmd = [fc, "-O2", "-fPIC", "-shared", "-J", mod_dir, "-o", tmp]
    cmd += [os.path.join(HERE, "fortran", f) for f in FORTRAN_SOURCES]
    cmd += ["-L" + HERE, "-lizem_hip", "-Wl,-rpath,$ORIGIN"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True, cwd=mod_dir)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("Fortran host library build failed")
    os.replace(tmp, FORTRAN_LIB)
    return FORTRAN_LIB


if __name__ == "__main__":
    print(build(verbose=True))
