"""The short division of the transport (fd2_div_by) on every quotient of
24-bit significands near a rounding boundary (oracle/check_div.c)."""
import os
import subprocess


def test_division_rounds_every_hard_quotient():
    here = os.path.join(os.path.dirname(__file__), "..", "oracle")
    subprocess.run(["make", "-s", "-C", here, "check_div"], check=True)
    r = subprocess.run([os.path.join(here, "check_div")], capture_output=True, text=True,
                       timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and " 0 wrong" in r.stdout, r.stdout + r.stderr
