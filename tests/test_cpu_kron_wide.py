"""E_K products of lattices with a direction of 17 to 32 sites in the CPU emulation build: left and right
products against the dense product to 1e-13 relative (sums of at most 64 terms each way, so rounding
stays below 64 eps), two tasks per launch, every access in bounds, no race between wavefronts."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CLANG = "/opt/rocm/llvm/bin/clang++"


def _build(tmp_path_factory, sanitizer):
    if not os.path.exists(CLANG):
        pytest.skip("host clang++ with sanitizers not available")
    out = str(tmp_path_factory.mktemp("emu") / f"kron_wide_{sanitizer}")
    cmd = [CLANG, "-std=c++20", "-O1", "-g", f"-fsanitize={sanitizer}", "-fno-omit-frame-pointer",
           "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "cpu_emu", "kron_wide_harness.cpp"),
           "-o", out, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return out


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    return _build(tmp_path_factory, "address")


@pytest.mark.parametrize("args", ["17 2 2 17 1", "24 5 3 32 2", "19 18 18 5 3", "6 31 21 4 4"])
def test_wide_products(harness, args):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
    r = subprocess.run([harness, *args.split()], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0 and "ok:" in r.stdout, (r.stdout + r.stderr)[-3000:]


def test_wide_products_race_free(tmp_path_factory):
    exe = _build(tmp_path_factory, "thread")
    env = dict(os.environ, TSAN_OPTIONS="halt_on_error=0 report_signal_unsafe=0")
    r = subprocess.run([exe, "2", "17", "18", "3", "5"], capture_output=True, text=True, env=env, timeout=900)
    assert "ok" in r.stdout, (r.stdout + r.stderr)[-3000:]
    assert "WARNING: ThreadSanitizer" not in r.stderr, r.stderr[:4000]
