"""The oracle's build takes the reference's own sources only where they are: a reference folder
that is absent or empty is no error."""
import subprocess

import pytest

from oracle import oracle_py


@pytest.mark.parametrize("ref", ["absent", "empty", "sources"])
def test_reference_library_is_optional(monkeypatch, tmp_path, ref):
    folder = tmp_path / "reference"
    if ref != "absent":
        folder.mkdir()
    if ref == "sources":
        (folder / "charac.f").write_text("")
    goals = []
    monkeypatch.setattr(oracle_py, "REFDIR", str(folder), raising=False)
    monkeypatch.setattr(subprocess, "check_call", lambda cmd: goals.append(cmd[-1]))
    oracle_py.build()
    assert goals == (["all", "ref"] if ref == "sources" else ["all"])
