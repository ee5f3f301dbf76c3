"""The widths of a batched launch's kernel, from its host-side plan (CPU only)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "sparse-voxel-octrees_amd")


def test_each_form_takes_the_width_of_its_own_kernel(svo, tmp_path):
    exe = str(tmp_path / "batch_plan_test")
    subprocess.run(["g++", "-O2", "-std=c++17", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I", os.path.join(ROOT, "include"), "-I", os.path.join(PKG, "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "batch_plan_test.cpp"), "-L", PKG, "-lsvo_hip", f"-Wl,-rpath,{PKG}",
                    "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
