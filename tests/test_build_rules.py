"""The library's Makefile rebuilds what includes a changed header."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "venusaur_amd", "csrc")


def _includes(name):
    """The headers of this folder that a file includes, directly or not."""
    out, todo = set(), [name]
    while todo:
        with open(os.path.join(CSRC, todo.pop())) as f:
            for h in re.findall(r'#include "([^"/]+)"', f.read()):
                if h not in out:
                    out.add(h)
                    todo.append(h)
    return out


@pytest.mark.parametrize("header", sorted(f for f in os.listdir(CSRC) if f.endswith(".h")))
def test_a_changed_header_rebuilds_every_object_that_includes_it(tmp_path, header):
    if shutil.which("make") is None:
        pytest.skip("no make")
    sources = [f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp"))]
    for f in sources:  # objects newer than every source
        obj = tmp_path / (os.path.splitext(f)[0] + ".o")
        obj.write_text("")
    (tmp_path / "lib.so").write_text("")
    args = ["make", "-n", "-C", CSRC, f"BUILD={tmp_path}", f"OUT={tmp_path}/lib.so", f"{tmp_path}/lib.so"]
    assert "-c vz_" not in subprocess.run(args, check=True, capture_output=True, text=True).stdout
    told = subprocess.run(args + ["-W", header], check=True, capture_output=True, text=True).stdout
    users = [f for f in sources if header in _includes(f)]
    assert users
    assert [f for f in users if f"-c {f}" not in told] == []
