"""Copies into memory that the caller names, read off the HIP sources: the
library's streams are non-blocking, and a plain hipMemcpy whose destination
turns out to be device memory neither waits nor is ordered against them, so the
data of the call may arrive after a later call has rewritten its source."""
import glob
import os
import re

import pytest

from conftest import ROOT

SOURCES = sorted(glob.glob(os.path.join(ROOT, "quantumvortices_amd", "csrc", "*.hip")))


def calls(name, text):
    """Argument text of every call of `name` (parentheses balanced)."""
    text = re.sub(r"//[^\n]*", "", text)
    for m in re.finditer(r"\b%s\(" % name, text):
        depth, i = 1, m.end()
        while depth:
            depth += {"(": 1, ")": -1}.get(text[i], 0)
            i += 1
        yield text[m.end():i - 1]


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_copies_to_callers_are_on_a_stream(path):
    bad = [a for a in calls("hipMemcpy", open(path).read()) if "hipMemcpyDefault" in a]
    assert not bad, bad
