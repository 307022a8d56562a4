"""The near form of Bird::step (krabmaga_amd/csrc/kg_near.hpp) on the CPU:
tests/near stages tiles as the flock kernel does and compares every bird with
the general form bit for bit, under AddressSanitizer and UBSan."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_near_form_equals_the_general_form():
    near = os.path.join(HERE, "near")
    subprocess.run(["make", "-s", "-C", near], check=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")
    r = subprocess.run([os.path.join(near, "near_check")], capture_output=True, text=True,
                       timeout=600, env=env)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "0 scenario(s) failed" in r.stdout
