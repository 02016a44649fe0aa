"""The library's Makefile and sources: a changed header rebuilds what includes
it; indices that outgrow 32 bits are formed in 64."""
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


def test_node_box_indices_are_64_bit():
    """Six floats a node: from 715,827,883 nodes on (a scene may have 2^30
    spheres) node * 6 no longer fits 32 bits.  Every box is found through
    node_box, which multiplies in 64."""
    with open(os.path.join(CSRC, "vz_lbvh.hip")) as f:
        text = f.read()
    helper = re.search(r"node_box\(.*?\)\s*\{(.*?)\}", text, re.S).group(1)
    assert "(size_t)node * 6" in helper
    assert re.findall(r"boxes\s*(?:\[|\+)[^;\n]*\*\s*6", text.replace(helper, "")) == []
