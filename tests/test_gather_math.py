"""The gather's host-and-device arithmetic, called on the CPU in the kernels'
precision (the programs in tests/csrc say what they compare and why their
bounds are what they are)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def program(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "legitengine_amd", "csrc"),
                    "-o", exe, os.path.join(ROOT, "tests", "csrc", name + ".cpp")], check=True)
    return exe


def test_trilinear_taps(tmp_path):
    r = subprocess.run([program(tmp_path, "check_taps")], capture_output=True, text=True, timeout=300)
    assert r.stdout.startswith("ok "), r.stdout
    samples, at_infinite, differences, pairs = (int(v) for v in r.stdout.split()[1:])
    assert samples == 4000000 and at_infinite > 10000 and differences > 10000 and pairs > 10000


def test_march_limit(tmp_path):
    exe = program(tmp_path, "check_gather_limit")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.stdout.startswith("ok "), r.stdout
    assert int(r.stdout.split()[1]) > 10 ** 6
    for mistake in (1, 2, 3, 4):
        r = subprocess.run([exe, str(mistake)], capture_output=True, text=True, timeout=300)
        assert r.returncode == 1 and "footprint" in r.stdout, (mistake, r.stdout)
