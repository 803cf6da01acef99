"""The stream-mix sigmoid table (csrc/q38m_silu_gen.c sigmoid ->
_build/q38m_sigmoid_table.inc, read by hyper_mix_up_kernel): for every bf16
argument the clamped lookup equals bf16(1 / (1 + exp(-v))) by the oracle's exp
and an IEEE division, the arguments outside the table's magnitudes included."""
import os
import re
import subprocess

import numpy as np

from conftest import PACKAGE_DIR


def test_lookup_equals_oracle_for_every_bf16(orc):
    name = os.path.join("_build", "q38m_sigmoid_table.inc")
    subprocess.run(["make", "-C", PACKAGE_DIR, "-s", name], check=True)
    with open(os.path.join(PACKAGE_DIR, name)) as f:
        table = np.array([int(w, 16) for w in re.findall(r"0x([0-9a-f]{8})u", f.read())], np.uint32)
    assert len(table) == 4096
    words = np.arange(65536, dtype=np.uint32)
    magnitude = words & 0x7fff
    words, magnitude = words[magnitude <= 0x7f80], magnitude[magnitude <= 0x7f80]
    at = np.clip(magnitude, 0x3b00, 0x42ff) - 0x3b00 + ((words >> 4) & 0x800)
    v = (words << 16).view(np.float32)
    with np.errstate(all="ignore"):
        want = orc.f32_to_bf16(np.float32(1.0) / (np.float32(1.0) + orc.expf(-v)))
    assert np.array_equal(table[at] >> 16, want.astype(np.uint32))
