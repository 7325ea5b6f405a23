"""The left E_K products of a block of slices in one launch, in the CPU emulation build: the same bits as
one launch per product; bounds under AddressSanitizer, races between wavefronts under ThreadSanitizer."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CLANG = "/opt/rocm/llvm/bin/clang++"


@pytest.mark.parametrize("sanitizer,args", [
    ("address", "2 2 3 9 1"), ("address", "5 13 4 16 3"), ("address", "8 8 16 7 4"), ("address", "16 16 16 16 2"),
    ("thread", "5 6 4 3 2"),
])
def test_chain_equals_single_products(tmp_path, sanitizer, args):
    if not os.path.exists(CLANG):
        pytest.skip("host clang++ with sanitizers not available")
    exe = str(tmp_path / "kron_chain")
    cmd = [CLANG, "-std=c++20", "-O1", "-g", f"-fsanitize={sanitizer}", "-fno-omit-frame-pointer",
           "-I", os.path.join(ROOT, "include"), os.path.join(HERE, "cpu_emu", "kron_chain_harness.cpp"),
           "-o", exe, "-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1", TSAN_OPTIONS="report_signal_unsafe=0")
    r = subprocess.run([exe, *args.split()], capture_output=True, text=True, env=env, timeout=600)
    assert "ok" in r.stdout, (r.stdout + r.stderr)[-3000:]
    assert "WARNING: ThreadSanitizer" not in r.stderr, r.stderr[:4000]
