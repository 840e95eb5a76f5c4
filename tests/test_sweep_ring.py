"""The record ring of the LU-SGS sweeps (k_sweep_wg): a record has arrived in its slot before
its first read, and the copy into a slot starts after a barrier that follows the slot's last read.
A model on the CPU runs the copy waves' own loop and takes the readers' phases from the same
header as the kernel; it finds a wait left out, a wait for one load too few and a copy a phase
early."""
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).parent
STEPS = [15, 16, 22, 38, 214]        # IMAX + 14: one cell, two, a tile's worth, more


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    exe = tmp_path_factory.mktemp("ring") / "model"
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-Wall", str(HERE / "sweep_ring_model.cpp"), "-o", str(exe)])
    return lambda n, wait="0", early=0: subprocess.check_output([str(exe), str(n), str(wait), str(early)],
                                                                text=True).splitlines()


@pytest.mark.parametrize("n", STEPS)
def test_schedule(model, n):
    assert model(n) == ["ok"] * 4


@pytest.mark.parametrize("n", STEPS)
@pytest.mark.parametrize("mistake", [dict(wait="none"), dict(wait="1"), dict(early=1)],
                         ids=["no_wait", "one_load_too_few", "copy_a_phase_early"])
def test_mistakes_are_found(model, n, mistake):
    assert all(line != "ok" for line in model(n, **mistake))
