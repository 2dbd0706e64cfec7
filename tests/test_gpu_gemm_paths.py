"""matmul_rows over the token counts where its kernels and tile shapes change.

The rule (csrc/gemm.hip, gemm_path) takes a GEMV per token below 3 (4) tokens, then four
matrix-core forms and the wide tiles; the sliced forms choose a tile shape by the launch's
total. Each case sits at an edge of that rule, of a tile (16, 32, 48, 64, 128 tokens; 16 to 256
rows) or of a K split (blocks per row that 2, 4 or 8 slices do not divide), against the oracle's
GEMV at the fp32 bar and half of it against the outputs' rms, as the other GEMV tests.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import assert_bits_equal, assert_f32_close, rel_err
from qwen35_hip import ops, synth

pytestmark = pytest.mark.gpu

F32 = np.float32


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _weight(kind, rows, K, seed):
    t = synth.q4k_table(rows, K, seed_tensor=seed) if kind == "Q4_K" else synth.q6k_table(rows, K, seed_tensor=seed)
    return t


@pytest.mark.parametrize("kind", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("T,M,K", [
    (2, 48, 2048), (3, 17, 2048), (3, 300, 256), (4, 65, 4096), (15, 130, 2304),    # GEMV / fp32, partial rounds of K
    (3, 4097, 2048), (9, 4113, 256), (15, 8200, 1280), (14, 16400, 512), (3, 2048, 4096), (5, 4100, 4352),   # fp32: 16 or 32 rows, 1 or 2 slices
    (3, 49151, 256), (3, 49152, 256),                                               # fp32 / GEMV by the matrix
    (16, 4100, 2048), (17, 64, 2048), (33, 129, 1024), (47, 300, 2048), (49, 96, 512),
    (127, 200, 2048), (128, 33, 2048), (129, 257, 2048), (129, 100, 1280),          # four slices / two / none (odd)
    (160, 80, 4096), (161, 80, 4096), (191, 500, 4608), (700, 2048, 512),
    (320, 130, 2048), (321, 130, 2048), (640, 64, 2048), (641, 300, 2048),          # whole K: both tile sizes
    (960, 64, 2048), (961, 70, 2048), (1024, 64, 2048), (1025, 64, 2048), (1025, 65, 1280), (1100, 3850, 1280), (1183, 3600, 256), (2048, 20, 4096), (2049, 20, 4096),
])
def test_matmul_rows_edges(oracle, kind, T, M, K):
    r = np.random.default_rng(T * 131 + M + K)
    w = _weight(kind, M, K, 5)
    x = r.standard_normal((T, K)).astype(F32)
    out = torch.full((T + 1, M), 5.0, device="cuda")
    ops.matmul_rows(_dev(w), kind, M * K, _dev(x), M, K, out=out)
    got = out.cpu().numpy()
    rows = sorted({0, 1, T // 2, T - 2, T - 1} | {t for t in (15, 16, 31, 47, 63, 64, 127, 128) if t < T})
    for t in rows:
        ref = oracle.gemv(w, ops.GGML_TYPES[kind], x[t], M, K)
        assert_f32_close(got[t], ref, group=M, what=f"{kind} {T}x{M}x{K} token {t}")
        rms = np.sqrt(np.mean(ref.astype(np.float64) ** 2))
        assert np.abs(got[t].astype(np.float64) - ref).max() <= 5e-6 * rms
    assert np.all(got[T] == 5.0)


@pytest.mark.parametrize("T", [2, 3, 9, 15, 20, 100, 200, 400, 800, 1100])
def test_matmul_rows_multi_keeps_the_bits(T):
    """Tile shapes follow the launch's total, sums do not: each matrix of a call gives the bits of its own call
    (thin matrices and both types among them)."""
    r = np.random.default_rng(T)
    K = 2048
    x = _dev(r.standard_normal((T, K)).astype(F32))
    jobs = [(_dev(_weight(kind, M, K, 20 + i)), kind, M * K, M, 0, None)
            for i, (kind, M) in enumerate([("Q4_K", 8192), ("Q4_K", 32), ("Q6_K", 512), ("Q4_K", 2048), ("Q6_K", 48), ("Q6_K", 4096)])]
    for (w, kind, ne, M, off, _), got in zip(jobs, ops.matmul_rows_multi(jobs, x, K)):
        assert_bits_equal(got.cpu().numpy(), ops.matmul_rows(w, kind, ne, x, M, K).cpu().numpy(), what=f"{kind} {M}")


@pytest.mark.parametrize("kind", ["Q4_K", "Q6_K"])
def test_few_tokens_as_exact_as_the_gemv(kind):
    """Below 16 tokens the fp32 matrix-core form replaces one fp32 GEMV per token: its 2-norm error against float64 is no
    larger than the GEMV's (both sums have the same bound; the margin is the spread over inputs)."""
    r = np.random.default_rng(3)
    M, K, T = 1024, 2048, 12
    w = _dev(_weight(kind, M, K, 9))
    x = r.standard_normal((T, K)).astype(F32)
    dx = _dev(x)
    eye = ops.dequant_gather_rows(w, kind, M * K, torch.arange(M, dtype=torch.int32, device="cuda"), K)
    ref = x.astype(np.float64) @ eye.cpu().numpy().astype(np.float64).T
    few = ops.matmul_rows(w, kind, M * K, dx, M, K).cpu().numpy()
    one = np.stack([ops.matmul_dispatch(w, kind, M * K, dx[t], M, K).cpu().numpy() for t in range(T)])
    err = [np.linalg.norm(v - ref) / np.linalg.norm(ref) for v in (few, one)]
    assert err[0] <= 1.1 * err[1], err


@pytest.mark.parametrize("kind", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("T,M,K", [(12, 1024, 2048), (3, 4112, 1024), (15, 512, 4608), (7, 8208, 256)])
def test_few_tokens_keep_small_channels_beside_a_large_one(kind, T, M, K):
    """A channel far above the others whose weights are zero leaves the others' 24 bits, as in the GEMV that these
    counts stand in for, and so do rows of very small or large values: the same bar as above. (Each M is on another
    tile shape: 16 rows with a slice or two of K per wave, 32 rows.)"""
    r = np.random.default_rng(T)
    blocks = _weight(kind, M, K, 9).reshape(M, K // 256, -1).copy()
    if kind == "Q4_K":   # scale and minimum of elements 0..31 of each row
        blocks[:, 0, 4] &= 0xC0
        blocks[:, 0, 8] &= 0xC0
    else:                # scale of elements 0..15
        blocks[:, 0, 192] = 0
    w = _dev(blocks.reshape(-1))
    full = ops.dequant_gather_rows(w, kind, M * K, torch.arange(M, dtype=torch.int32, device="cuda"), K).double().cpu().numpy()
    assert not full[:, 5].any()
    for big, scale in [(1e5, 1), (1e7, 1), (1e12, 1), (1e30, 1), (1, 1e-30), (1, 1e30)]:
        x = (r.standard_normal((T, K)) * scale).astype(F32)
        x[:, 5] = big * scale
        dx = _dev(x)
        ref = x.astype(np.float64) @ full.T
        few = ops.matmul_rows(w, kind, M * K, dx, M, K).cpu().numpy()
        one = np.stack([ops.matmul_dispatch(w, kind, M * K, dx[t], M, K).cpu().numpy() for t in range(T)])
        err = [np.linalg.norm(v - ref) / np.linalg.norm(ref) for v in (few, one)]
        assert err[0] <= 1.1 * err[1], (big, scale, err)


@pytest.mark.parametrize("T", [3, 15])
def test_few_tokens_over_their_inputs(T):
    """Below 16 tokens a token's outputs may lie where the tokens before it were read: one GEMV per token then, with
    its bits, in a single call and in one of several matrices."""
    M = K = 512
    w, v = _dev(_weight("Q4_K", M, K, 5)), _dev(_weight("Q6_K", 48, K, 6))
    x = _dev(np.random.default_rng(T).standard_normal((T, K)).astype(F32))
    ref = torch.stack([ops.matmul_dispatch(w, "Q4_K", M * K, x[t], M, K) for t in range(T)]).cpu().numpy()
    buf = torch.cat([torch.zeros((1, K), device="cuda"), x])
    ops.matmul_rows(w, "Q4_K", M * K, buf[1:], M, K, out=buf[:-1])
    assert_bits_equal(buf[:-1].cpu().numpy(), ref)
    buf = torch.cat([torch.zeros((1, K), device="cuda"), x])
    other = ops.matmul_rows_multi([(v, "Q6_K", 48 * K, 48, 0, None), (w, "Q4_K", M * K, M, 0, buf[:-1])], buf[1:], K)[0]
    assert_bits_equal(buf[:-1].cpu().numpy(), ref)
    one = torch.stack([ops.matmul_dispatch(v, "Q6_K", 48 * K, x[t], 48, K) for t in range(T)])
    assert_bits_equal(other.cpu().numpy(), one.cpu().numpy())


@pytest.mark.parametrize("kind", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("T", [5, 40, 150, 800])
def test_nonfinite_rows_in_every_form(oracle, kind, T):
    """A token row with an infinity gives the reference's pattern, a NaN row NaN, a zero row +0; others are
    unaffected (two rounds of K for the form with one exponent a round)."""
    M, K = 96, 4096 if T == 150 else 2048
    w = _weight(kind, M, K, 7)
    x = np.random.default_rng(T).standard_normal((T, K)).astype(F32)
    x[1, K - 1] = np.inf
    x[2, 7] = np.nan
    x[3] = 0.0
    got = ops.matmul_rows(_dev(w), kind, M * K, _dev(x), M, K).cpu().numpy()
    ref = oracle.gemv(w, ops.GGML_TYPES[kind], x[1], M, K)
    assert np.array_equal(np.isnan(got[1]), np.isnan(ref)) and np.array_equal(got[1][np.isinf(ref)], ref[np.isinf(ref)])
    assert np.isnan(got[2]).all() and np.array_equal(got[3].view(np.uint32), np.zeros(M, np.uint32))
    for t in (0, 4, T - 1):
        ref = oracle.gemv(w, ops.GGML_TYPES[kind], x[t], M, K)
        assert rel_err(got[t], ref, group=M).max() <= 1e-5


@pytest.mark.parametrize("kind", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("T,M,K", [(1183, 3600, 256), (200, 96, 4096), (18, 40, 1280)])
def test_nonfinite_rows_in_the_other_tiles(oracle, kind, T, M, K):
    """The same in the 128 x 256 tiles (both token halves, the ragged last tile), two slices of K, and the form that
    converts x itself."""
    w = _weight(kind, M, K, 7)
    x = np.random.default_rng(T).standard_normal((T, K)).astype(F32)
    inf = sorted({0, 70 % T, T - 1})
    x[inf, K // 2] = [np.inf, -np.inf, np.inf][:len(inf)]
    x[[1, T - 2], 7] = np.nan
    x[5] = 0.0
    got = ops.matmul_rows(_dev(w), kind, M * K, _dev(x), M, K).cpu().numpy()
    for t in inf:
        ref = oracle.gemv(w, ops.GGML_TYPES[kind], x[t], M, K)
        assert np.array_equal(np.isnan(got[t]), np.isnan(ref))
        assert np.array_equal(got[t][np.isinf(ref)], ref[np.isinf(ref)])
    assert np.isnan(got[[1, T - 2]]).all() and np.array_equal(got[5].view(np.uint32), np.zeros(M, np.uint32))
    for t in (2, 6, T - 3):
        assert rel_err(got[t], oracle.gemv(w, ops.GGML_TYPES[kind], x[t], M, K), group=M).max() <= 1e-5


@pytest.mark.parametrize("T", [3, 15, 40])
def test_rows_off_16_byte_alignment_are_the_gemv(T):
    M, K = 96, 2048
    w = _dev(_weight("Q4_K", M, K, 7))
    x = torch.randn(T * K + 1, generator=torch.Generator().manual_seed(T)).cuda()[1:].view(T, K)
    one = torch.stack([ops.matmul_dispatch(w, "Q4_K", M * K, x[t], M, K) for t in range(T)])
    assert_bits_equal(ops.matmul_rows(w, "Q4_K", M * K, x, M, K).cpu().numpy(), one.cpu().numpy())


@pytest.mark.parametrize("kind", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("T,K", [(1024, 2048), (1360, 1280), (512, 4096)])
def test_prep_spread_over_workgroups_keeps_the_bits(kind, T, K):
    """The last token count whose prep takes a workgroup per 512 elements of K, against one tile more (all of K in
    one workgroup): the first T tokens get the same bits."""
    w = _dev(_weight(kind, 300, K, 9))
    x = torch.randn((T + 16, K), generator=torch.Generator().manual_seed(T)).cuda()
    assert_bits_equal(ops.matmul_rows(w, kind, 300 * K, x[:T], 300, K).cpu().numpy(),
                      ops.matmul_rows(w, kind, 300 * K, x, 300, K)[:T].cpu().numpy())
