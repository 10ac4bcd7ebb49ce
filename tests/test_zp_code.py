"""The zero-point code rule without a division gives the codes of the IEEE operations (tests/native/check_zp_code.c)."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_codes_with_a_zero_point_match_ieee(tmp_path):
    exe = tmp_path / "check_zp_code"
    subprocess.run(["gcc", "-O2", "-mfma", "-fopenmp", "-ffp-contract=off", f"-I{ROOT / 'hyc-lora-release_amd' / 'csrc'}",
                    str(ROOT / "tests" / "native" / "check_zp_code.c"), "-lm", "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0 and "mismatches=0" in res.stdout, res.stdout
    assert int(res.stdout.split("triples=")[1].split()[0]) > 2_000_000_000
