"""How decode attention launches split their rings, and the workspace size
that must serve every one of them: csrc/attention_plan.hpp, the same code the
kernel and the launches use, swept on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_chunks_and_workspace(tmp_path):
    exe = str(tmp_path / "attention_plan")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "ane-lm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "attention_plan.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout


def test_size_is_the_plan_s():
    """The exported size is the swept one: two figures of it."""
    import anelm

    n = anelm.lib().anelm_gqa_workspace_size(1, 32, 8, 128, 1024)
    assert n >= 32 * 16 * 130 * 4 * 64 // 63          # 16 chunks of every head, then the counters
    assert anelm.lib().anelm_gqa_workspace_size(1, 32, 8, 128, 64) == 0
