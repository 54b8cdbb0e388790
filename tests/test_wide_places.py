"""The decode of several sequences in one launch loads no operand that it has not waited for: the kernel's own index functions (csrc/wide_places.h), over every
shape it covers.  CPU only."""
import os
import subprocess

from conftest import ROOT


def test_every_loaded_piece_is_waited_for(tmp_path):
    exe = tmp_path / "wide_places"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(ROOT, "mini-llm-cuda_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "wide_places.cpp"), "-o", str(exe)], check=True)
    run = subprocess.run([str(exe)], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout


def test_the_kernel_loads_through_these_functions():
    """Every load of operand planes in the kernel names its chunk by them."""
    text = open(os.path.join(ROOT, "mini-llm-cuda_amd", "csrc", "kernels_wide.hip")).read()
    loads = [line.strip() for line in text.splitlines() if "operand(av[" in line]
    assert len(loads) == 3 and all("wd_chunk(wave, " in line or "wd_part(part2, i, k)" in line for line in loads), loads
