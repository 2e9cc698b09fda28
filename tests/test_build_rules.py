"""The Makefile of the kernels: an object file depends on every header that its source includes, also through others."""
import re
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).parents[1] / "wgml_amd" / "csrc"


def included(path, seen):
    for name in re.findall(r'^\s*#include "([^"]+)"', path.read_text(), re.M):
        header = (path.parent / name).resolve()
        if header not in seen:
            seen.add(header)
            included(header, seen)
    return seen


@pytest.mark.parametrize("source", sorted(p.name for p in CSRC.iterdir() if p.suffix in (".hip", ".cpp")))
def test_objects_depend_on_their_headers(source):
    rules = subprocess.run(["make", "-npB", "-C", str(CSRC)], capture_output=True, text=True, check=True).stdout
    rule = re.search(r"^build/%s\.o: (.*)$" % re.escape(source.rsplit(".", 1)[0]), rules, re.M)
    prerequisites = {(CSRC / p).resolve() for p in rule.group(1).split()}
    assert included(CSRC / source, {(CSRC / source).resolve()}) <= prerequisites
