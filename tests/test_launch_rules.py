"""The launch rules of csrc/launch_rules.hpp walked on the host: every index that a kernel derives from its grid lies
inside the caller's buffers, over the shapes that the entry points accept. (A value test cannot see a read past a
buffer's end whose result is not used.)"""

from __future__ import annotations

import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "qwen-3.5-cuda_amd" / "csrc"

SHIM = """
#include "launch_rules.hpp"
extern "C" void prep_grid(int chunks, int kh, int vh, int* out) {
    const qk::PrepGrid g = qk::prep_grid(chunks, kh, vh);
    out[0] = g.heads;
    out[1] = g.step;
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", "-o", str(d / "shim.so"), str(d / "shim.cpp")],
                   check=True)
    return ctypes.CDLL(str(d / "shim.so"))


@pytest.mark.parametrize("chunks", [1, 2, 5, 8, 9, 13, 64, 300])
def test_chunked_prep_heads_stay_in_range(rules, chunks):
    """Workgroup y of the chunked recurrence's prep reads the gates of heads y, y + step, ... below value_heads, the
    first of them before it tests the bound: it exists in every workgroup (value heads that key heads do not divide
    among them), every value head is taken once, from its own key head, and every key head's K and Q written once."""
    out = (ctypes.c_int * 2)()
    for kh in (1, 2, 3, 4, 7, 8, 15, 16, 17):
        for vh in (1, 2, 3, 4, 6, 7, 8, 12, 16, 24, 31, 32, 33, 48, 64):
            rules.prep_grid(chunks, kh, vh, out)
            heads, step = out
            taken, written = [], []
            for y in range(heads):
                assert y < vh, (kh, vh)   # the gates read at the workgroup's start
                taken += [(h, y % kh) for h in range(y, vh, step)]
                if y < kh:
                    written.append(y % kh)
            assert sorted(taken) == [(h, h % kh) for h in range(vh)], (kh, vh)
            assert written == list(range(min(kh, vh))), (kh, vh)
