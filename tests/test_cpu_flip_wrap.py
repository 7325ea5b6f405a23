"""Flips and wraps of a block of slices in one launch, in the CPU emulation build, against the flip kernel
slice by slice with dense wraps on the host: the same decisions, fields, tables and counters, G to 1e-11
and ratios and measurements to 1e-10 (some slices' rounding of matrices of order one); bounds under
AddressSanitizer, races between wavefronts under ThreadSanitizer."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CLANG = "/opt/rocm/llvm/bin/clang++"


def _build(tmp_path_factory, sanitizer):
    if not os.path.exists(CLANG):
        pytest.skip("host clang++ with sanitizers not available")
    out = str(tmp_path_factory.mktemp("emu") / f"flip_wrap_{sanitizer}")
    cmd = [CLANG, "-std=c++20", "-O1", "-g", f"-fsanitize={sanitizer}", "-fno-omit-frame-pointer",
           "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "cpu_emu", "flip_wrap_harness.cpp"),
           "-o", out, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return out


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    return _build(tmp_path_factory, "address")


@pytest.mark.parametrize("args", [
    "2 2 4 1 0 4 1",     # the smallest, a whole measured sweep
    "4 4 6 2 2 3 0", "3 9 3 1 1 2 1", "4 11 2 1 0 2 0", "8 8 3 2 0 3 1", "5 16 2 1 0 1 0",
    "12 8 2 1 0 2 1", "16 6 2 1 1 5 1",  # 96 sites: both spins' wraps in LDS; more slices than are left
    "7 14 2 1 0 2 0", "16 8 2 1 0 2 1",  # above: one spin after the other
    "3 4 5 3 2 3 1 7",   # three chains of 12, 8, 8 sites in the 128-site form, ending one after the other
])
def test_flip_with_wraps(harness, args):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
    r = subprocess.run([harness, *args.split()], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0 and "ok" in r.stdout, (r.stdout + r.stderr)[-3000:]


@pytest.mark.parametrize("args", ["3 5 2 1 0 2 1", "4 9 1 1 0 1 0 6"])
def test_flip_with_wraps_race_free(tmp_path_factory, args):
    exe = _build(tmp_path_factory, "thread")
    env = dict(os.environ, TSAN_OPTIONS="halt_on_error=0 report_signal_unsafe=0")
    r = subprocess.run([exe, *args.split()], capture_output=True, text=True, env=env, timeout=900)
    assert "ok" in r.stdout, (r.stdout + r.stderr)[-3000:]
    assert "WARNING: ThreadSanitizer" not in r.stderr, r.stderr[:4000]
