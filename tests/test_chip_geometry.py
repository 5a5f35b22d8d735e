"""The blocks of the on-chip solver (reef3d_amd/csrc/chip_geom.h), checked on the host before
any kernel uses them: every tile in one slot of one block, every neighbour of every cell
where the kernel looks for it, no index outside its buffer."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_neighbour_is_where_the_kernel_looks(tmp_path):
    exe = tmp_path / "chip_check"
    subprocess.run(["g++", "-std=c++17", "-O2", os.path.join(HERE, "cpp", "chip_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.rstrip().endswith("ok")
