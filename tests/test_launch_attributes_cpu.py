"""The dynamic-LDS limit of the decode kernels, with stand-ins for the runtime's calls: no device, nothing runs."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_the_lds_limit_is_raised_once_for_each_kernel(pkg, tmp_path):
    lib = pkg.lib_path()
    exe = str(tmp_path / "stand_in_runtime")
    subprocess.run(["gcc", "-O1", "-Wall", "-rdynamic", os.path.join(HERE, "stand_in_runtime.c"), lib, "-Wl,-rpath," + os.path.dirname(lib),
                    "-Wl,--unresolved-symbols=ignore-in-shared-libs", "-o", exe], check=True)
    words = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=120).stdout.split()
    count = {name: int(value) for name, value in zip(words[::2], words[1::2])}
    assert count["calls"] > 1000 and count["kernels"] > 60, count
    assert count["missing"] == 0 and count["again"] == 0 and count["raised"] >= count["kernels"], count
