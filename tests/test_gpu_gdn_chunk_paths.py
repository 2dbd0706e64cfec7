"""The chunked recurrence at the edges of its routes: the token loop up to 28 rows, prep workgroups per value head
while they have a CU each, one per key head above (and with one, two or three value heads per key head, or uneven
numbers of them)."""

from __future__ import annotations

import pytest
import torch

from conftest import assert_bits_equal
from qwen35_hip import ops
from qwen35_hip._lib import check

pytestmark = pytest.mark.gpu


def _inputs(rows, kh, vh):
    g = torch.Generator(device="cuda").manual_seed(rows * 7 + vh)
    n = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    qk = torch.nn.functional.normalize(n(rows, 2 * kh, 128), dim=-1)
    qk[:, :kh] /= 128 ** 0.5
    qkv = torch.cat([qk.reshape(rows, -1), n(rows, vh * 128)], 1).contiguous()
    beta, decay = torch.sigmoid(n(rows, vh)), torch.exp(-torch.rand((rows, vh), generator=g, device="cuda") * 2)
    return qk, qkv, beta, decay, 0.1 * n(vh, 128, 128)


def _check(got, got_s, qk, qkv, beta, decay, state, kh, vh):
    """Output and state against the recurrence in float64, under the bar of the other recurrence tests: 1e-5 of the
    larger of the value and its condition scale (here each head's largest terms, |q||S| of the readout)."""
    rows = qk.shape[0]
    idx = torch.arange(vh, device="cuda") % kh
    S, out, cond = state.double(), [], []
    for t in range(rows):
        q, k = qk[t, :kh][idx].double(), qk[t, kh:][idx].double()
        v = qkv[t, 2 * kh * 128:].view(vh, 128).double()
        S = S * decay[t].double()[:, None, None]
        delta = (v - torch.bmm(k[:, None], S)[:, 0]) * beta[t].double()[:, None]
        S = S + k[:, :, None] * delta[:, None, :]
        out.append(torch.bmm(q[:, None], S)[:, 0])
        cond.append(torch.bmm(q.abs()[:, None], S.abs())[:, 0])
    ref, c = torch.stack(out).view(rows, -1), torch.stack(cond).view(rows, -1)
    assert bool(((got.double() - ref).abs() <= 1e-5 * torch.maximum(ref.abs(), c)).all())
    rms = S.square().mean((1, 2), keepdim=True).sqrt()
    assert bool(((got_s.double() - S).abs() <= 1e-5 * torch.maximum(S.abs(), rms)).all())


@pytest.mark.parametrize("rows,kh,vh", [(1, 16, 32), (28, 16, 32), (29, 16, 32), (64, 4, 4), (65, 4, 12), (512, 16, 32),
                                        (513, 16, 32), (100, 8, 4), (64, 2, 3), (130, 16, 24), (700, 16, 24), (65, 3, 8)])
def test_chunked_routes(rows, kh, vh):
    qk, qkv, beta, decay, state = _inputs(rows, kh, vh)
    got_s = state.clone()
    got = ops.gdn_recurrent_chunked(got_s, qkv, beta, decay, kh, vh, 128, 128)
    _check(got, got_s, qk, qkv, beta, decay, state, kh, vh)


def test_up_to_28_rows_are_the_token_loop():
    g = torch.Generator(device="cuda").manual_seed(5)
    qkv = torch.randn((28, 8192), generator=g, device="cuda")
    beta, decay = torch.rand((2, 28, 32), generator=g, device="cuda")
    state = torch.randn((32, 128, 128), generator=g, device="cuda")
    a, b = state.clone(), state.clone()
    one = ops.gdn_recurrent_chunked(a, qkv, beta, decay, 16, 32, 128, 128)
    two = ops.gdn_recurrent_rows(b, qkv, beta, decay, 16, 32, 128, 128)
    assert_bits_equal(one.cpu().numpy(), two.cpu().numpy(), what="out")
    assert_bits_equal(a.cpu().numpy(), b.cpu().numpy(), what="state")


@pytest.mark.parametrize("rows", [1, 9, 28, 29])
@pytest.mark.parametrize("part", ["q", "k", "v"])
def test_outputs_over_their_inputs(rows, part):
    """Outputs over the q, k or v of their own rows (q and k are read by other workgroups, the v of a column only by the
    one that writes it)."""
    kh, vh, lib = 16, 16, ops.load()
    qk, qkv, beta, decay, state = _inputs(rows, kh, vh)
    buf, s, row = qkv.clone(), state.clone(), qkv.shape[1]
    q = buf.data_ptr()
    out = q + 4 * 2048 * "qkv".index(part)
    ws = torch.empty(lib.qwen_gdn_recurrent_chunked_workspace_bytes(rows, vh), dtype=torch.uint8, device="cuda")
    check(lib.qwen_gdn_recurrent_chunked(s.data_ptr(), q, q + 4 * 2048, q + 8 * 2048, beta.data_ptr(), decay.data_ptr(),
                                         out, rows, kh, vh, 128, 128, 0 if rows == 1 else row, 0 if rows == 1 else row,
                                         ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    first = 2048 * "qkv".index(part)
    _check(buf[:, first:first + 2048], s, qk, qkv, beta, decay, state, kh, vh)


def test_row_strides_past_the_walks_limit_are_the_token_loop():
    """29 rows, the first count of the chunked kernels, at a stride of 2^31 / 256 floats and more: the token loop's bits
    (a row of the 0.97 GB buffer holds the 2 key and 2 value heads; the rest is never read)."""
    rows, stride, kh, vh, dv = 29, 8_400_000, 2, 2, 32
    g = torch.Generator(device="cuda").manual_seed(8)
    wide = torch.zeros((rows, stride), device="cuda")
    wide[:, :2 * kh * 128 + vh * dv] = 0.1 * torch.randn((rows, 2 * kh * 128 + vh * dv), generator=g, device="cuda")
    beta, decay = torch.rand((2, rows, vh), generator=g, device="cuda")
    state = torch.randn((vh, 128, dv), generator=g, device="cuda")
    lib, p = ops.load(), wide.data_ptr()
    ws = torch.empty(lib.qwen_gdn_recurrent_chunked_workspace_bytes(rows, vh), dtype=torch.uint8, device="cuda")
    res = []
    for fn, extra in ((lib.qwen_gdn_recurrent_chunked, (ws.data_ptr(), ws.numel())), (lib.qwen_gdn_recurrent_rows, ())):
        s, out = state.clone(), torch.empty((rows, vh * dv), device="cuda")
        check(fn(s.data_ptr(), p, p + 4 * kh * 128, p + 8 * kh * 128, beta.data_ptr(), decay.data_ptr(), out.data_ptr(),
                 rows, kh, vh, 128, dv, stride, vh * dv, *extra, torch.cuda.current_stream().cuda_stream))
        res.append((out.cpu().numpy(), s.cpu().numpy()))
    assert_bits_equal(res[0][0], res[1][0], what="out")
    assert_bits_equal(res[0][1], res[1][1], what="state")


@pytest.mark.parametrize("rows,kh,dim,kernel,heads,skew", [(1, 16, 128, 4, 32, 0), (3, 2, 64, 4, 3, 0), (24, 16, 128, 4, 32, 0),
                                                           (25, 1, 256, 4, 1, 0), (777, 16, 128, 4, 33, 0),
                                                           (9, 4, 32, 4, 8, 0), (9, 2, 128, 3, 8, 0), (9, 2, 128, 4, 8, 1)])
def test_frontend_gates_is_the_two_calls(rows, kh, dim, kernel, heads, skew):
    """One launch (heads of 64, 128 or 256 and 16-byte aligned buffers) and the general path, bit for bit against the
    separate calls; the history in place as well."""
    g = torch.Generator(device="cuda").manual_seed(rows + heads)
    n = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    c = 4 * kh * dim
    x, w, hist = n(rows * c + skew)[skew:].view(rows, c), n(c, kernel), n(c, kernel - 1)
    b, al, a, dt = 9 * n(rows, heads), 9 * n(rows, heads), -torch.exp(n(heads)), n(heads)
    b.view(-1)[0], al.view(-1)[-1] = float("inf"), float("nan")
    y, h = ops.gdn_frontend_rows(x, w, hist, k_heads=kh, key_dim=dim)
    beta, decay = ops.gdn_gate_values_rows(b, al, a, dt)
    inplace = hist.clone()
    for got in (ops.gdn_frontend_gates_rows(x, w, hist, b, al, a, dt, k_heads=kh, key_dim=dim),
                ops.gdn_frontend_gates_rows(x, w, inplace, b, al, a, dt, hist_out=inplace, k_heads=kh, key_dim=dim)):
        for name, u, v in zip(("y", "history", "beta", "decay"), got, (y, h, beta, decay)):
            assert torch.equal(u.view(torch.int32), v.view(torch.int32)), name
