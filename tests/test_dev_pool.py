"""The pool of device blocks that a context keeps between calls (csrc/dev_pool.h), with an
allocator of fixed capacity under AddressSanitizer and UndefinedBehaviorSanitizer
(tests/native/check_pool.cpp): a request that fits the device is served whatever the pool's
rounding and whatever it holds."""
import os
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_pool_under_asan_ubsan(tmp_path):
    exe = tmp_path / "check_pool"
    subprocess.run(["g++", "-O1", "-g", "-fno-omit-frame-pointer", "-std=c++17", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=all", "-pthread", "-o", str(exe),
                    str(ROOT / "tests" / "native" / "check_pool.cpp")], check=True, capture_output=True, timeout=300)
    # verify_asan_link_order=0: the process environment may preload other libraries
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0", UBSAN_OPTIONS="print_stacktrace=1")
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]
    assert "OK: 0 failures" in r.stdout
