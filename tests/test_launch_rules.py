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
extern "C" int offsets_fit(int q4, int block_bytes, int M, int K) {
    return qk::gemm_offsets_fit(q4 != 0, block_bytes, M, K);
}
extern "C" int overlap(uintptr_t a, size_t n, uintptr_t b, size_t m) {
    return qk::floats_overlap(reinterpret_cast<const float*>(a), n, reinterpret_cast<const float*>(b), m);
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


@pytest.mark.parametrize("q4,block", [(1, 144), (0, 210)])
def test_gemm_row_offsets_fit_32_bits(rules, q4, block):
    """A matrix takes the matrix-core kernels only while the largest byte offset that a lane forms fits 32 bits: Q4_K's
    from the matrix's first row, Q6_K's from a workgroup's (256 rows at most: K up to 20 million)."""
    for K in (256, 2048, 4096, 1 << 20, 20_000_000 // 256 * 256, 20_500_000 // 256 * 256, 1 << 25, (1 << 28), (1 << 31) - 256):
        for M in (1, 2, 15, 16, 100, 255, 256, 257, 4096, 248320, (1 << 31) - 1):
            rows = M if q4 else min(M, 256)
            last = ((rows - 1) * (K // 256) + K // 256) * block   # one past the last row's last byte
            assert bool(rules.offsets_fit(q4, block, M, K)) == (last < 1 << 32), (M, K)


def test_floats_overlap(rules):
    f = rules.overlap
    f.argtypes = [ctypes.c_size_t] * 4
    base, n, m = 1 << 20, 6, 4
    for shift in range(-4 * m - 8, 4 * n + 9, 2):
        bytes_a, bytes_b = set(range(4 * n)), set(range(shift, shift + 4 * m))
        assert bool(f(base, n, base + shift, m)) == bool(bytes_a & bytes_b) == bool(f(base + shift, m, base, n)), shift
