"""Rules of launches, on the host: how the items of a wavefront's lanes are shared out among wavefronts
(hpg-libs_amd/csrc/fmi_items.h), on the host: up to the most items that the
32-bit form is taken for, and past them with 64 bits, every wavefront steps to
its own items and ends; and what decides the 1-error search's load mode.  CPU
only."""
import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "hpg-libs_amd", "csrc")


def host_check(*args):
    r = subprocess.run(["make", "-C", CSRC, "check"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([os.path.join(CSRC, "_build", "host_check"), *args], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("bits", [32, 64])
def test_every_wavefront_ends(bits):
    host_check("items", str(bits))


def test_load_mode_leaves_out_row_contexts():
    """The load mode of the 1-error search follows from the arrays it reads: row
    contexts kept beside them do not move an index over its limit."""
    host_check("spread", "5000")
