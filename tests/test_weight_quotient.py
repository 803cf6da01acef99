"""The weight quantisers' division-free quotient (csrc/q38m_layout.hip) rounds
like the division for every bf16 pair of six binades of group maxima, for W4 and
W8: the lowest ones that take it, the middle, the largest
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


def test_every_binade_is_walked(tmp_path):
    exe = str(tmp_path / "check")
    subprocess.run(["gcc", "-O2", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "weight_quotient_check.c"), "-lm"], check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=300).stdout
    binades = re.findall(r"binade (0x\w+) qmax (\d+) checked (\d+) differ (\d+)", out)
    assert len(binades) == 12
    for first, qmax, checked, differ in binades:
        assert int(checked) > 0 and int(differ) == 0, (first, qmax)
    # the crossing binades are partly on the fast path, the next ones wholly
    whole = {(b[0], b[1]): int(b[2]) for b in binades}
    for qmax, crossing, above in (("7", "0x0480", "0x0500"), ("127", "0x0680", "0x0700")):
        assert 0 < whole[crossing, qmax] < whole[above, qmax]
        assert whole[above, qmax] == sum(2 * (a + 1) for a in range(int(above, 16), int(above, 16) + 128))
