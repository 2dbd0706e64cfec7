"""Decode kernels at the edges of their shape rules: the attention combine's batches (128 splits
of 32 or 16 keys, more, many), and the MoE down projection with the 512-wide shared expert."""

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
