"""Host-side state that a GPU run cannot reach safely: contexts on a device
without memory left, in small programs that link the library and stand in for
the HIP runtime's allocation calls (tests/native)."""
import os
import subprocess

import pytest

import sanepic_amd

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NATIVE = os.path.join(ROOT, "tests", "native")
LIBDIR = os.path.dirname(sanepic_amd.LIB_PATH)


@pytest.mark.parametrize("program", ["recal_state", "arena_state", "streams_memory"])
def test_native(program, tmp_path):
    exe = str(tmp_path / program)
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + sanepic_amd.CSRC, "-I" + os.path.join(ROOT, "include"),
                    os.path.join(NATIVE, program + ".cpp"), "-o", exe, sanepic_amd.LIB_PATH,
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + LIBDIR, "-Wl,-rpath,/opt/rocm/lib"], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
