"""CPU: device code of the register kernels run by an emulated workgroup
(tests/wave_emu): what they read at the edges of their operands, where a GPU
run would show nothing or a fault."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
EMU = os.path.join(ROOT, "tests", "wave_emu")
CSRC = os.path.join(ROOT, "magma_amd", "csrc")


def _run(tmp_path, name, *args):
    clang = shutil.which("clang++", path="/opt/rocm/llvm/bin" + os.pathsep + os.environ.get("PATH", ""))
    if clang is None:
        pytest.skip("no clang++")
    for f in os.listdir(CSRC):                 # the kernels' headers, but for the one of inline assembly
        if f.endswith(".h") and f != "dpp_fma.h":
            os.symlink(os.path.join(CSRC, f), tmp_path / f)
    os.symlink(os.path.join(EMU, "dpp_fma.h"), tmp_path / "dpp_fma.h")
    with open(os.path.join(CSRC, "lu_mfma.hip")) as f:
        kernel, launch = f.read().split("\n}  // namespace\n", 1)
    assert "getrf_mfma_kernel(MatSet s)" in kernel and "<<<" in launch
    (tmp_path / "lu_kernel.inc").write_text(kernel + "\n}\n}\n")
    exe = str(tmp_path / name)
    subprocess.run([clang, "-std=c++20", "-O1", "-march=native", "-ffp-contract=off", "-w", "-I" + str(tmp_path),
                    "-I" + EMU, "-I" + os.path.join(ROOT, "include"), os.path.join(EMU, name + ".cpp"), "-o", exe],
                   check=True)
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), (r.returncode, r.stdout[-2000:] + r.stderr[-2000:])


def test_lu_of_empty_matrices(tmp_path):
    _run(tmp_path, "lu")


def test_sweeps_load_inside_the_matrix(tmp_path):
    _run(tmp_path, "sweeps", "loads")


def test_sweeps_keep_out_what_is_not_read(tmp_path):
    _run(tmp_path, "sweeps", "values")
