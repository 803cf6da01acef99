"""The weight quantisers' division-free quotient (csrc/q38m_layout.hip) rounds
like the division for every bf16 pair of four binades, for W4 and W8
(tests/weight_quotient_check.c)."""
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_weight_quotients_round_like_the_division(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "weight_quotient_check.c"), "-lm"], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=300).stdout
    counts = re.findall(r"pairs (\d+) mismatches (\d+)", out)
    assert len(counts) == 2
    for pairs, mismatches in counts:
        assert int(pairs) > 10_000_000 and int(mismatches) == 0
