"""The register-tile flip in the CPU emulation build against the rank-1 kernel: the same decisions,
field, tables and counters, G and the measurement to rounding, at the edges of every form's range
(and small chains in the largest form, as mixed batches run them); bounds under AddressSanitizer,
races between its wavefronts under ThreadSanitizer."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CLANG = "/opt/rocm/llvm/bin/clang++"


def _build(tmp_path_factory, sanitizer):
    if not os.path.exists(CLANG):
        pytest.skip("host clang++ with sanitizers not available")
    out = str(tmp_path_factory.mktemp("emu") / f"flip_tile_{sanitizer}")
    cmd = [CLANG, "-std=c++20", "-O1", "-g", f"-fsanitize={sanitizer}", "-fno-omit-frame-pointer",
           "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "cpu_emu", "flip_tile_harness.cpp"),
           "-o", out, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    return out


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    return _build(tmp_path_factory, "address")


@pytest.mark.parametrize("args", [
    "1 3 1 0 0 1", "16 4 2 3 1 20", "17 4 2 1 0 30", "32 4 1 3 1 30", "33 3 1 0 0 40", "48 3 1 2 1 40",
    "64 3 2 1 0 40", "65 3 1 2 1 60", "96 2 1 0 0 60", "112 2 1 1 1 60", "128 2 1 0 0 80",
    "20 4 3 2 0 30 7",  # three chains of 20, 19, 18 sites in the 128-site form, one past its last slice
])
def test_tile_flip_matches_rank1(harness, args):
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1")
    r = subprocess.run([harness, *args.split()], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0 and "ok" in r.stdout, (r.stdout + r.stderr)[-3000:]


@pytest.mark.parametrize("args", ["30 3 1 2 1 30", "40 3 1 1 0 40"])
def test_tile_flip_race_free(tmp_path_factory, args):
    exe = _build(tmp_path_factory, "thread")
    env = dict(os.environ, TSAN_OPTIONS="halt_on_error=0 report_signal_unsafe=0")
    r = subprocess.run([exe, *args.split()], capture_output=True, text=True, env=env, timeout=900)
    assert "ok" in r.stdout, (r.stdout + r.stderr)[-3000:]
    assert "WARNING: ThreadSanitizer" not in r.stderr, r.stderr[:4000]
