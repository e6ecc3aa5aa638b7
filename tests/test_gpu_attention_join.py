"""The frame-special block's fused pieces against the parts they stand for.

`attention_join` against the oracle's LSE merge of two fp32 attentions: query
counts around the 64-query wave and 256-query workgroup, frames that end inside
one, several batches and heads, one shared key, a half with no weight.  Its
output has one 16-bit rounding of the own half, one of P and one of the
result, so a row's relative error is at most 4 * 2^-9 (bf16) or 4 * 2^-12
(fp16) of unit-scale values.  `attention_rows` and `shared_set` do no new
arithmetic: equal bit for bit.
"""
import pytest
import torch

import gpa_aggregator as A
from merging import _native
from merging.fused_attention import (attention_join, attention_keybias, attention_rows,
                                     combine_by_lse)
from oracle.attention import attention_reference, lse_combine

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


def _randn(g, *shape, dtype=torch.bfloat16, scale=0.7):
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,H,P,N", [(1, 1, 2, 1, 1), (1, 3, 2, 21, 31), (2, 2, 3, 64, 33),
                                       (1, 5, 1, 51, 160), (1, 2, 4, 201, 96), (2, 7, 2, 100, 300)])
def test_join_matches_oracle(dev, dtype, B, S, H, P, N):
    g = torch.Generator().manual_seed(B * S * P + N)
    M = S * P
    q, k, v = (_randn(g, B, H, t, 64, dtype=dtype) for t in (M, N, N))
    bias = _randn(g, B, H, 1, N, dtype=dtype)
    ok, ov = (_randn(g, B * S, H, 40, 64, dtype=dtype) for _ in range(2))
    q_f = q.view(B, H, S, P, 64).permute(0, 2, 1, 3, 4).reshape(B * S, H, P, 64)
    own_o, own_lse = attention_reference(q_f, ok, ov, None, 0.125)
    ref_o, ref_lse = attention_reference(q, k, v, bias, 0.125)
    back = lambda t: t.view(B, S, *t.shape[1:]).transpose(1, 2).flatten(2, 3)  # noqa: E731
    ref = lse_combine(back(own_o), back(own_lse), ref_o, ref_lse)
    ref = torch.as_tensor(ref).view(B, H, M, 64).transpose(1, 2).reshape(B, M, H * 64)
    got = attention_join(q.to(dev), k.to(dev), v.to(dev), bias.to(dev), 0.125,
                         own_o.to(dev, dtype), own_lse.float().to(dev), S).float().cpu()
    assert got.shape == ref.shape
    rel = (got - ref).view(B, M, H, 64).norm(dim=-1) / ref.view(B, M, H, 64).norm(dim=-1)
    assert rel.max().item() <= 4 * ULP[dtype], rel.max().item()


def test_join_takes_a_half_without_weight(dev):
    """An own half whose LSE lies far below or above the shared one's."""
    g = torch.Generator().manual_seed(1)
    q, k, v = (_randn(g, 1, 2, t, 64).to(dev) for t in (90, 50, 50))
    own = _randn(g, 3, 2, 30, 64).to(dev)
    rows = attention_rows(q, k, v, None, 0.125)
    for lse, want in ((-500.0, rows), (float("-inf"), rows),
                      (500.0, own.view(1, 3, 2, 30, 64).transpose(2, 3).reshape(1, 90, 128))):
        got = attention_join(q, k, v, None, 0.125, own,
                             torch.full((3, 2, 30), lse, device=dev), 3)
        assert (got.float() - want.float()).abs().max().item() <= 2.0 ** -8 * want.abs().max().item()


def test_join_refuses_what_does_not_fit(dev):
    q = torch.zeros(1, 2, 90, 64, device=dev, dtype=torch.bfloat16)
    o, lse = torch.zeros(3, 2, 30, 64, device=dev, dtype=torch.bfloat16), torch.zeros(3, 2, 30, device=dev)
    for args in ((o, lse, 4), (o, lse, 2), (o[:, :1], lse, 3), (o, lse.double(), 3), (o, lse, 0)):
        with pytest.raises(ValueError):
            _native.attn_keybias_join(q, q, q, None, 0.125, *args)


@pytest.mark.parametrize("D", [16, 32, 64, 128, 256])
def test_rows_equal_the_transposed_output(dev, D):
    g = torch.Generator().manual_seed(D)
    q, k, v = (_randn(g, 2, 3, t, D).to(dev) for t in (259, 77, 77))
    bias = _randn(g, 1, 1, 1, 77).to(dev)
    want = attention_keybias(q, k, v, bias, D ** -0.5).transpose(1, 2).reshape(2, 259, 3 * D)
    assert torch.equal(attention_rows(q, k, v, bias, D ** -0.5), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,pts,gh,gw,kp", [(1, 5, 6, 6, 8), (3, 5, 14, 9, 4), (2, 0, 7, 5, 2),
                                            (4, 1, 16, 16, 2), (2, 5, 37, 37, 3)])
def test_shared_set_equals_its_parts(dev, dtype, S, pts, gh, gw, kp):
    """Specials, pooled summaries and the bias in one output, for each pooling
    kernel (up to 32, up to 64 and more seeds); no special tokens; v a view
    of a wider row."""
    g = torch.Generator().manual_seed(S * gh * gw)
    B, H, P = 2, 2, gh * gw + pts
    k = _randn(g, B, H, S * P, 64, dtype=dtype).to(dev)
    v = _randn(g, B, S * P, 3, H, 64, dtype=dtype).to(dev)[:, :, 2].transpose(1, 2)
    pk, pv, size, _ = torch.ops.gpa.pool_shared(k, v, S, pts, gh, gw, kp, False)
    sp = lambda t: t.reshape(B, H, S, P, 64)[:, :, :, :pts].reshape(B, H, S * pts, 64)  # noqa: E731
    bias = torch.zeros(B, H, 1, S * pts + pk.shape[2], device=dev)
    bias[:, :, 0, S * pts:] = size.log().reshape(B, H, -1)
    got = _native.shared_set(k, v, S, pts, gh, gw, kp)
    for a, b in zip(got, (torch.cat((sp(k), pk), 2), torch.cat((sp(v), pv), 2), bias.to(dtype), size)):
        assert torch.equal(a, b)


def test_opcheck(dev):
    g = torch.Generator().manual_seed(2)
    q, k = (_randn(g, 1, 2, t, 64).to(dev) for t in (3 * 41, 50))
    torch.library.opcheck(torch.ops.gpa.attn_keybias_rows, (q, k, k, None, 0.125))
    torch.library.opcheck(torch.ops.gpa.shared_set, (q, q, 3, 5, 6, 6, 2))
    torch.library.opcheck(torch.ops.gpa.attn_keybias_join, (
        q, k, k, None, 0.125, q.view(2, 3, 41, 64).transpose(0, 1).contiguous(),
        torch.zeros(3, 2, 41, device=dev), 3))
    assert A.pool_kernel_applies(q, 6, 6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("S,H,P,n_own,n", [(4, 4, 206, 201, 120), (16, 2, 1374, 1369, 480)])
def test_join_is_no_further_from_64_bits_than_its_parts(dev, dtype, S, H, P, n_own, n):
    """The join rounds the shared half once less than the two calls and
    `combine_by_lse`, so its output differs from theirs, repeats itself exactly
    and lies no further from the softmax over both key sets in 64 bits."""
    g = torch.Generator(device=dev).manual_seed(S)
    q, sk, sv = (torch.randn(1, H, t, 64, device=dev, generator=g).to(dtype)
                 for t in (S * P, n, n))
    ok, ov = (torch.randn(S, H, n_own, 64, device=dev, generator=g).to(dtype) for _ in "kv")
    bias = torch.randint(1, 60, (1, H, 1, n), device=dev, generator=g).float().log().to(dtype)
    q_f = q.view(H, S, P, 64).transpose(0, 1).contiguous()
    own, own_lse = attention_keybias(q_f, ok, ov, None, 0.125, return_lse=True)
    got = attention_join(q, sk, sv, bias, 0.125, own, own_lse, S)
    assert torch.equal(got, attention_join(q, sk, sv, bias, 0.125, own, own_lse, S))
    shared, shared_lse = attention_keybias(q, sk, sv, bias, 0.125, return_lse=True)
    parts = combine_by_lse(own, own_lse, shared, shared_lse, S)
    keys = torch.cat((ok, sk.expand(S, H, n, 64)), 2).double().transpose(-1, -2).contiguous()
    values = torch.cat((ov, sv.expand(S, H, n, 64)), 2).double()
    x = q_f.double() @ keys * 0.125
    x[..., n_own:] += bias.double()
    ref = (torch.softmax(x, -1) @ values).permute(0, 2, 1, 3).reshape(1, S * P, H * 64)
    err, err_parts = ((t.double() - ref).norm().item() for t in (got, parts))
    assert err <= err_parts
