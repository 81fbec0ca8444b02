"""Copies and clears of device memory, read off the HIP sources: the library's
streams are non-blocking, and a plain hipMemcpy between device buffers (or into
memory that the caller names, which may be one) or a plain hipMemset neither
waits nor is ordered against them, so its data may arrive after later kernels
have run."""
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


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_device_copies_are_on_a_stream(path):
    bad = [a for a in calls("hipMemcpy", open(path).read()) if "hipMemcpyDeviceToDevice" in a]
    assert not bad, bad


# where a device-wide wait or a blocking upload on the default stream follows
# before anything else can run
CREATES = {"vk_gpe_create", "vk_ens_create", "fno_alloc", "vk_pattern_bandwidth"}


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_clears_are_on_a_stream(path):
    inside, bad = "", []
    for line in open(path):
        m = re.match(r"^[a-z][\w:<>*& \"]*?\b(\w+)\(.*", line)
        if m and not line.rstrip().endswith(";"):
            inside = m.group(1)
        if re.search(r"\bhipMemset(D\d+)?\(", line.split("//")[0]) and inside not in CREATES:
            bad.append((inside, line.strip()))
    assert not bad, bad
