"""The record ring of the LU-SGS sweeps (k_sweep_wg): a copy into a slot starts after a barrier
that follows the slot's last read, and a record has arrived before its first read.  The order of
the kernel's phases is taken from its source, so that a change of one side alone is found."""
import re
from pathlib import Path

import pytest

SRC = (Path(__file__).parents[1] / "finflo_amd/csrc/ffhip.hip").read_text()


def schedule():
    """(phase in which a copy wave starts the copy of record s + RS, its step's distance from s),
    and the phases in which wave 0 reads its face of record s, counted from step s."""
    k = SRC[SRC.index("k_sweep_wg(Prm p"):SRC.index("constexpr int KI = 16, KJ = 4;")]
    loop = re.search(r"wg_step_sync\(\);\s*for \(int s = 0; s < nsteps; s\+\+\) \{\s*(.*?)\n        \}", k, re.S).group(1)
    m = re.search(r"copy\(s( - 1)? \+ RS\)", loop)
    assert m, "the copy of the ring's next record"
    phase = 1 + loop[:m.start()].count("wg_step_sync()")
    copy = (1 if m.group(1) else 0, phase)
    ahead = "read_face(ring[slot]" in k
    return copy, (-1, 2) if ahead else (0, 2)


@pytest.mark.parametrize("n", [2, 8, 24, 200])
@pytest.mark.parametrize("rs", [3, 5, 6, 8])
def test_no_copy_before_the_last_read(rs, n):
    copy, face = schedule()
    for s in range(rs, n):
        old = s - rs
        start = (old + copy[0], copy[1])
        # waves 1 and 2 read record s in the first phase of step s, wave 0 its increments'
        # fields a step ahead and its face where the source says
        last = max((old, 1), (old - 1, 2), (old + face[0], face[1]))
        assert start > last, f"ring of {rs}: the copy of record {s} starts in {start}, last read in {last}"
