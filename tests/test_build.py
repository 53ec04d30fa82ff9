"""The build of a machine without torch or its headers: the C library's part runs, the
torch extension is left out with a note."""
import sys

import pytest

from xrgpu_amd import build as B


@pytest.mark.parametrize("missing", ["torch", "headers"])
def test_front_needs_torch(monkeypatch, capsys, tmp_path, missing):
    ran = []
    monkeypatch.setattr(B, "_run", lambda cmd, verbose: ran.append(cmd))
    if missing == "torch":
        monkeypatch.setitem(sys.modules, "torch", None)  # import torch raises ImportError
    else:
        monkeypatch.setattr(B.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    B.build_front("g++", False)
    assert not ran and "not built" in capsys.readouterr().err
