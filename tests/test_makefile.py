"""Every object of the native engine is rebuilt when a header that its source includes changes:
the two fp8 encodes (append kernel and decode) come from one header and store the same bytes
only when both are built from the same version of it."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "persistentkv-attention_amd", "csrc")
SOURCES = {"pkv_decode.o": "pkv_decode.hip", "pkv_append.o": "pkv_append.hip",
           "pkv_schedule.o": "pkv_schedule.cpp"}


def _includes(name):
    with open(os.path.join(CSRC, name)) as f:
        return re.findall(r'^#include "([^"]+)"', f.read(), re.M)


@pytest.mark.parametrize("target", SOURCES)
def test_objects_follow_their_headers(tmp_path, target):
    csrc, include = tmp_path / "pkg" / "csrc", tmp_path / "include"
    csrc.mkdir(parents=True)
    include.mkdir()
    (csrc / "Makefile").write_text(open(os.path.join(CSRC, "Makefile")).read())
    headers = _includes(SOURCES[target])
    assert headers
    paths = {h: csrc / h if os.path.exists(os.path.join(CSRC, h)) else include / h for h in headers}
    for p in [csrc / SOURCES[target], *paths.values()]:
        p.write_text("")
        os.utime(p, (1, 1))
    (csrc / target).write_text("")

    def up_to_date(*newer):
        cmd = ["make", "-q", "PYTHON=true", target]
        for h in newer:
            cmd += ["-W", os.path.relpath(paths[h], csrc)]
        return subprocess.run(cmd, cwd=csrc, capture_output=True).returncode == 0

    assert up_to_date()
    for h in headers:
        assert not up_to_date(h), f"{target} does not depend on {h}"
