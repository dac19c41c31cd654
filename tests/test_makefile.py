"""Every object of the library depends on all the headers that its source includes, those included by headers
too, so that a plain make builds what a change reaches."""
import os
import re

from conftest import ROOT

CSRC = os.path.join(ROOT, "rustpde_amd", "csrc")


def _included(path, seen):
    with open(path) as f:
        for name in re.findall(r'^\s*#include "([^"]+)"', f.read(), re.M):
            p = os.path.normpath(os.path.join(os.path.dirname(path), name))
            if p not in seen:
                seen.add(p)
                _included(p, seen)
    return seen


def test_objects_depend_on_their_headers():
    with open(os.path.join(CSRC, "Makefile")) as f:
        text = f.read()
    rules = re.findall(r"^(build/\w+\.o): (.+)$", text, re.M)
    assert {o for o, _ in rules} == set(re.search(r"^OBJS := (.+)$", text, re.M).group(1).split())
    for obj, deps in rules:
        paths = [os.path.normpath(os.path.join(CSRC, d)) for d in deps.split()]
        missing = _included(paths[0], set()) - set(paths[1:])
        assert not missing, (obj, sorted(os.path.basename(p) for p in missing))
