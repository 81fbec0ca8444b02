"""Which caller memory a psi read writes from its kernel and which it copies to:
the rule alone, compiled for the host.  A buffer of another device than the
handle's takes the copy, whichever device is current."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "vk_target.hpp"
int main(int, char** v)
{
    auto n = [&](int i) { return (size_t)std::strtoull(v[i], nullptr, 0); };
    const vk::Target t{n(3) != 0, (int)n(4), (uintptr_t)n(5), n(6)};
    std::printf("%d\n", (int)vk::kernel_writable((uintptr_t)n(1), n(2), t, (int)n(7)));
}
"""

TOP = 2 ** 64 - 4096
CASES = [  # p, bytes, device memory, its device, allocation, its size, the handle's device, direct
    (4096, 512, 1, 0, 4096, 512, 0, 1),          # the whole allocation
    (4096 + 16, 496, 1, 0, 4096, 512, 0, 1),     # up to its end
    (4096 + 16, 512, 1, 0, 4096, 512, 0, 0),     # 16 bytes past it
    (4096, 528, 1, 0, 4096, 512, 0, 0),
    (4096 + 8, 256, 1, 0, 4096, 512, 0, 0),      # 8-byte alignment
    (4096, 512, 0, 0, 4096, 512, 0, 0),          # not device memory
    (4096, 512, 1, 1, 4096, 512, 0, 0),          # another device's
    (4096, 512, 1, 0, 4096, 512, 1, 0),
    (4096, 512, 1, 3, 4096, 512, 3, 1),
    (TOP, 2 ** 64 - 16, 1, 0, TOP, 512, 0, 0),   # no wrap around
    (4096 - 16, 32, 1, 0, 4096, 512, 0, 0),      # before the allocation
]


@pytest.mark.skipif(not shutil.which("g++"), reason="no host compiler")
def test_kernel_writable(tmp_path):
    (tmp_path / "m.cpp").write_text(MAIN)
    inc = os.path.join(ROOT, "quantumvortices_amd", "csrc")
    subprocess.check_call(["g++", "-std=c++17", "-I", inc, "-o", str(tmp_path / "m"), str(tmp_path / "m.cpp")])
    for *a, want in CASES:
        got = subprocess.check_output([str(tmp_path / "m")] + [str(x) for x in a], text=True)
        assert int(got) == want, a
