"""Decode kernels at the edges of their shape rules: the MoE down projection with the 512-wide shared expert."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from conftest import assert_bits_equal
from qwen35_hip import ops, synth

pytestmark = pytest.mark.gpu


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
