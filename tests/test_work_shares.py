"""How the items of a wavefront's lanes are shared out among wavefronts
(hpg-libs_amd/csrc/fmi_items.h), on the host: up to the most items that the
32-bit form is taken for, and past them with 64 bits, every wavefront steps to
its own items and ends.  CPU only."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "hpg-libs_amd", "csrc")


@pytest.mark.parametrize("bits", [32, 64])
def test_every_wavefront_ends(bits):
    r = subprocess.run(["make", "-C", CSRC, "check"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([os.path.join(CSRC, "_build", "host_check"), "items", str(bits)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
