"""The plan of the 64-token-block INT8 attention prefill, on the CPU: the header
that the kernels and the host share, run over every context up to 32768 and random
ragged batches (tests/cpp/attn_plan_check.cpp).  No plan may need more units than
the grid has workgroups or more partials than the workspace holds."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_attn_plan_fits_grid_and_workspace(tmp_path):
    exe = str(tmp_path / "attn_plan_check")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-Werror",
                           "-I", os.path.join(ROOT, "qwen3.5_0.8b_deploy_amd", "csrc"), "-o", exe,
                           os.path.join(ROOT, "tests", "cpp", "attn_plan_check.cpp")])
    run = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(run.stdout)
    assert run.returncode == 0 and run.stdout.startswith("ok"), run.stdout
