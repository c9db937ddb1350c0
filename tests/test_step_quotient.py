"""The quotients of the traversal step against IEEE division, over every size a step can
have and a reciprocal that is up to one ulp off (tests/step_quotient_check.c)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_step_quotients_match_ieee(tmp_path):
    exe = str(tmp_path / "step_quotient_check")
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", os.path.join(HERE, "step_quotient_check.c"), "-o", exe,
                    "-lm"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and "mismatches 0" in r.stdout, r.stdout + r.stderr
