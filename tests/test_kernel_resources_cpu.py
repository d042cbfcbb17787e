"""Registers of the built gfx950 kernels, from the metadata of the code
objects in libizem_hip.so."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "phd_amd", "libizem_hip.so")
LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name: (VGPRs, SGPRs spilled, scratch bytes) of every kernel."""
    tools = [os.path.join(LLVM, t) for t in ("llvm-objcopy", "llvm-readelf")]
    if not os.path.exists(LIB) or not all(map(os.path.exists, tools)):
        pytest.skip("libizem_hip.so not built, or no LLVM tools")
    d = tmp_path_factory.mktemp("co")
    fat = d / "fat"
    subprocess.run([tools[0], f"--dump-section=.hip_fatbin={fat}", LIB, str(d / "x")], check=True)
    data = fat.read_bytes()
    out = {}
    for i, at in enumerate(m.start() for m in re.finditer(b"\x7fELF", data)):
        co = d / f"{i}.co"
        co.write_bytes(data[at:])
        t = subprocess.run([tools[1], "--notes", str(co)], capture_output=True, text=True).stdout
        for k in re.split(r"(?m)^ {2,4}- \.", t)[1:]:
            f = dict(re.findall(r"\.?(\w+): +(\S+)", k))
            if "sgpr_spill_count" in f:
                out[f["name"]] = (int(f["vgpr_count"]), int(f["sgpr_spill_count"]),
                                  int(f["private_segment_fixed_size"]))
    assert out
    return out


@pytest.mark.parametrize("name,vgprs,spills", [
    ("k_force_probe", 168, 100), ("k_newton_apply", 168, 0)])
def test_newton_keeps_its_tables_out_of_registers(kernels, name, vgprs, spills):
    """The species' tables are read in the Newton iteration, not held: with
    them in registers (250 VGPRs, 660 to 760 SGPRs spilled) a launch over a small
    domain took twice as long.  168 VGPRs are what three waves per SIMD leave."""
    (k,) = [v for n, v in kernels.items() if name in n]
    assert k[0] <= vgprs and k[1] <= spills and k[2] == 0, k


def test_euler_faces_spill_nothing(kernels):
    """Two waves per SIMD and no scratch, in either mode and with rank views."""
    faces = {n: v for n, v in kernels.items() if "k_euler_faces" in n}
    assert len(faces) == 12
    assert all(v[0] <= 256 and v[2] == 0 for v in faces.values()), faces
