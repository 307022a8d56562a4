"""The near form of Bird::step (krabmaga_amd/csrc/kg_near.hpp) and the
resident step (kg_resident.hpp) on the CPU: tests/near runs their phases as
the kernels do and compares every bird with the general form bit for bit,
under AddressSanitizer and UBSan."""
import os
import subprocess

import pytest

NEAR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "near")


@pytest.mark.parametrize("check", ["near_check", "resident_check"])
def test_phases_equal_the_general_form(check):
    subprocess.run(["make", "-s", "-C", NEAR], check=True)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")
    r = subprocess.run([os.path.join(NEAR, check)], capture_output=True, text=True,
                       timeout=600, env=env)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    assert "0 scenario(s) failed" in r.stdout
