"""The QR of matrices above 256 in the CPU emulation build (its kernels take any smaller size too):
reconstruction and orthogonality to 1e-12 at one column, ragged row tiles, more row tiles than
wavefronts and a zero column, beside a one-column matrix in a launch sized for a larger one; bounds
under AddressSanitizer, races between its wavefronts under ThreadSanitizer."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CLANG = "/opt/rocm/llvm/bin/clang++"


def _build(tmp_path_factory, sanitizer):
    if not os.path.exists(CLANG):
        pytest.skip("host clang++ with sanitizers not available")
    out = str(tmp_path_factory.mktemp("emu") / f"qr_large_{sanitizer}")
    cmd = [CLANG, "-std=c++20", "-O1", "-g", f"-fsanitize={sanitizer}", "-fno-omit-frame-pointer",
           "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "cpu_emu", "qr_large_harness.cpp"),
           "-o", out, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return out


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    return _build(tmp_path_factory, "address")


@pytest.mark.parametrize("args", ["1 2 1", "33 20 2", "131 40 3", "20 10 4 zero"])
def test_large_qr(harness, args):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
    r = subprocess.run([harness, *args.split()], capture_output=True, text=True, env=env, timeout=900)
    assert r.returncode == 0 and "ok" in r.stdout, (r.stdout + r.stderr)[-3000:]


def test_large_qr_race_free(tmp_path_factory):
    exe = _build(tmp_path_factory, "thread")
    env = dict(os.environ, TSAN_OPTIONS="halt_on_error=0 report_signal_unsafe=0")
    r = subprocess.run([exe, "40", "20", "2"], capture_output=True, text=True, env=env, timeout=900)
    assert "ok" in r.stdout, (r.stdout + r.stderr)[-3000:]
    assert "WARNING: ThreadSanitizer" not in r.stderr, r.stderr[:4000]
