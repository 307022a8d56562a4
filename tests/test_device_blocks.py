"""Device arrays that share one allocation (DevBlock, DevBuf): tests/near's
block_check runs them over an allocator of its own, under AddressSanitizer and
UBSan.  An ensemble that allocates array by array spends half of a short call
on freeing them."""
import os
import subprocess

NEAR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "near")


def test_arrays_of_a_block_share_one_allocation():
    rocm = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1", CPLUS_INCLUDE_PATH=rocm)
    exe = os.path.join(NEAR, "block_check")
    subprocess.run(["make", "-s", "-C", NEAR, exe], check=True, env=env)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300, env=env)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "0 scenario(s) failed" in r.stdout
