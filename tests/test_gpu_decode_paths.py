"""Decode kernels at the edges of their shape rules: the attention combine's batches (128 splits
of 32 or 16 keys, more, many), the MoE down projection with the 512-wide shared expert, and the
residual norm's form for few rows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import assert_bits_equal
from qwen35_hip import ops, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,pos", [
    (16, 2, 0), (16, 2, 31), (16, 2, 4095), (16, 2, 4096), (16, 2, 16383), (16, 2, 16384), (16, 2, 20011),
    (32, 2, 2047), (32, 2, 2048), (16, 1, 9000),
])
def test_attn_decode_splits(heads, kv, pos):
    """Against float64 under the dot-product bar, |got - ref| <= 1e-5 max(|ref|, c) with c = sum_t p_t |v_t| (times the
    gate): the fp32 sum over keys and the scores' rounding err by ulps of its terms, and an average over many keys is
    far below them (20012 keys of N(0, 1): rms 0.01 of c)."""
    g = torch.Generator(device="cuda").manual_seed(pos + heads)
    q = torch.randn(heads * 256, generator=g, device="cuda")
    k = torch.randn((pos + 1) * kv * 256, generator=g, device="cuda")
    v = torch.randn((pos + 1) * kv * 256, generator=g, device="cuda")
    gate = torch.randn(heads * 256, generator=g, device="cuda")
    out = ops.attn_decode(q, k, v, heads, kv, 256, pos, gate=gate)
    kk = k.double().view(pos + 1, kv, 256).permute(1, 2, 0).contiguous()
    p = torch.softmax(torch.bmm(q.double().view(kv, heads // kv, 256), kk) / 16, -1)
    vv, sg = v.double().view(pos + 1, kv, 256).transpose(0, 1).contiguous(), torch.sigmoid(gate.double())
    ref, c = torch.bmm(p, vv).view(-1) * sg, torch.bmm(p, vv.abs()).view(-1) * sg
    assert bool(((out.double() - ref).abs() <= 1e-5 * torch.maximum(ref.abs(), c)).all())


@pytest.mark.parametrize("td,ts", [("Q4_K", "Q4_K"), ("Q4_K", "Q6_K"), ("Q6_K", "Q4_K"), ("Q6_K", "Q6_K")])
@pytest.mark.parametrize("k,dm", [(8, 2048), (5, 64), (4, 4), (1, 260)])
def test_down_combine_small_shared_expert(td, ts, k, dm):
    """shared_dim 512 in one launch: the bits of the separate calls (expert GEMVs, shared GEMV, weighted sum, gated
    add), an expert id out of range giving NaN rows as there."""
    E, inter, S = 7, 512, 512
    r = np.random.default_rng(k * 100 + dm)
    tab = {"Q4_K": synth.q4k_table, "Q6_K": synth.q6k_table}
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    wd, wsd = dev(tab[td](E * dm, inter, seed_tensor=3)), dev(tab[ts](dm, S, seed_tensor=11))
    ids = dev(r.permutation(E)[:k].astype(np.int32)) if k <= E else dev(r.integers(0, E, k).astype(np.int32))
    wts = dev(r.random(k).astype(np.float32))
    hid, shid = dev(r.standard_normal((k, inter)).astype(np.float32)), dev(r.standard_normal(S).astype(np.float32))
    logit = dev(r.standard_normal(1).astype(np.float32))

    def separate(idx):
        eo = ops.moe_expert_matmul(wd, td, E * dm * inter, dm * inter, E, idx, hid, inter, dm, inter)
        so = ops.matmul_dispatch(wsd, ts, dm * S, shid, dm, S)
        out = ops.moe_weighted_sum_rows(torch.zeros(1, dm, device="cuda"), eo.view(1, k, dm), wts.view(1, k))
        return ops.moe_shared_add_rows(out, so.view(1, dm), logit).view(-1)

    bad = ids.clone()
    bad[0] = E
    for idx in (ids, bad):
        got = ops.moe_down_combine(wd, td, E * dm * inter, dm * inter, E, idx, wts, hid, inter, wsd, ts, dm * S, shid,
                                   logit, dm)
        assert_bits_equal(got.cpu().numpy(), separate(idx).cpu().numpy(), what=f"{td} {ts} k={k} {dm}")


@pytest.mark.parametrize("S", [512, 2048])
def test_down_combine_into_its_inputs(S):
    """out in the place of the routed or the shared hidden rows: the bits of a call with an out of its own."""
    E, inter, k, dm = 5, 512, 4, 512
    r = np.random.default_rng(S)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    wd, wsd = dev(synth.q4k_table(E * dm, inter, seed_tensor=3)), dev(synth.q4k_table(dm, S, seed_tensor=11))
    ids, wts = dev(np.array([3, 0, 4, 1], np.int32)), dev(r.random(k).astype(np.float32))
    hid, shid = dev(r.standard_normal((k, inter)).astype(np.float32)), dev(r.standard_normal(S).astype(np.float32))
    logit = dev(r.standard_normal(1).astype(np.float32))

    def call(h, sh, out=None):
        return ops.moe_down_combine(wd, "Q4_K", E * dm * inter, dm * inter, E, ids, wts, h, inter, wsd, "Q4_K", dm * S,
                                    sh, logit, dm, out=out)

    ref = call(hid, shid).cpu().numpy()
    h, sh = hid.clone(), shid.clone()
    assert_bits_equal(call(h, shid, out=h[1]).cpu().numpy(), ref, what="into hidden")
    assert_bits_equal(call(hid, sh, out=sh[S - dm:]).cpu().numpy(), ref, what="into shared_hidden")


@pytest.mark.parametrize("n", [512, 516, 1024, 2048, 2052, 4096])
def test_residual_norm_of_few_rows_keeps_the_bits(n):
    """Up to 256 rows a row has a wave per chunk, above one wave: a row gives the same bits alone, among 256 and among
    257, also in place."""
    g = torch.Generator(device="cuda").manual_seed(n)
    x, b = torch.randn((2, 257, n), generator=g, device="cuda")
    w = torch.randn(n, generator=g, device="cuda")
    many = ops.residual_rmsnorm_rows(x, b, w)
    for rows in (1, 3, 256):
        for got, ref in zip(ops.residual_rmsnorm_rows(x[:rows].contiguous(), b[:rows].contiguous(), w), many):
            assert_bits_equal(got.cpu().numpy(), ref[:rows].cpu().numpy(), what=f"{rows} x {n}")
    y = x[:5].clone()
    resid, normed = ops.residual_rmsnorm_rows(y, b[:5].contiguous(), w, resid=y)
    assert_bits_equal(resid.cpu().numpy(), many[0][:5].cpu().numpy(), what="resid in place")
    assert_bits_equal(normed.cpu().numpy(), many[1][:5].cpu().numpy(), what="normed in place")
