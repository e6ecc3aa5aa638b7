"""Head dim 64 on both sides of the lines up to which the attention forms its row
bounds itself (8,192 keys, 1,024 workgroups): certified, tile-0 and lazily moved offsets (logit
scales from 0.3 to 30), an outlier key in the first and in the last tile.

Bar: a row's relative error within 16-bit P and output, 4 * 2^-9 (bf16) or
4 * 2^-12 (fp16) of unit-scale values."""
import pytest
import torch

from merging import _native
from merging.fused_attention import attention_join, attention_keybias
from oracle.attention import attention_reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [8160, 8192, 8193])
@pytest.mark.parametrize("dtype,ulp", [(torch.bfloat16, 2.0 ** -9), (torch.float16, 2.0 ** -12)])
@pytest.mark.parametrize("scale,outlier", [(0.3, None), (3.0, None), (0.5, 0), (0.5, -1)])
def test_bounds_formed_in_the_kernel(dev, N, dtype, ulp, scale, outlier):
    g = torch.Generator().manual_seed(N)
    q = (torch.randn(1, 2, 130, 64, generator=g) * scale).to(dtype)
    k = torch.randn(1, 2, N, 64, generator=g) * scale
    if outlier is not None:
        k[:, :, outlier] *= 12.0
    k, v = k.to(dtype), torch.randn(1, 2, N, 64, generator=g).to(dtype)
    bias = torch.randint(1, 9, (1, 1, 1, N), generator=g).float().log().expand(1, 2, 1, N).to(dtype)
    o = attention_keybias(q.to(dev), k.to(dev), v.to(dev), bias.to(dev), 0.125)
    ref, _ = attention_reference(q, k, v, bias, 0.125)
    rel = (o.float().cpu() - ref).norm(dim=-1) / ref.norm(dim=-1)
    assert rel.max().item() <= 4 * ulp, rel.max().item()


def test_certified_on_both_sides(dev):
    """The same keys, one more at -inf: the same bound, the same offset."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, 1, t, 64, generator=g).mul(0.5).bfloat16().to(dev)
               for t in (200, 8193, 8193))
    bias = torch.zeros(1, 1, 1, 8193, device=dev)
    bias[..., 8192] = float("-inf")
    _, _, few = _native.attn_keybias_offset_flags(q, k[:, :, :8192], v[:, :, :8192],
                                                  bias[..., :8192], 0.125)
    _, _, more = _native.attn_keybias_offset_flags(q, k, v, bias, 0.125)
    assert not few.any() and not more.any()


@pytest.mark.parametrize("N", [1, 2, 31, 32, 33, 47, 64, 95, 128, 129, 159, 160, 161])
@pytest.mark.parametrize("join", [False, True])
def test_last_tile_without_bias(dev, N, join):
    """The last tile's mask of a call without bias, alone and joined: k and v are
    views of longer buffers whose rows past N hold NaN."""
    g = torch.Generator().manual_seed(N)
    q, k, v = (torch.randn(1, 2, t, 64, generator=g).bfloat16() for t in (70, N, N))
    long = [torch.full((1, 2, N + 200, 64), float("nan"), dtype=q.dtype, device=dev) for _ in "kv"]
    for buf, t in zip(long, (k, v)):
        buf[:, :, :N] = t.to(dev)
    kd, vd = (buf[:, :, :N] for buf in long)
    ref, ref_lse = attention_reference(q, k, v, None, 0.125)
    if join:
        other = torch.zeros(2, 2, 35, 64, dtype=q.dtype, device=dev)
        o = attention_join(q.to(dev), kd, vd, None, 0.125, other,
                           torch.full((2, 2, 35), -1e4, device=dev), 2)
        o = o.view(1, 70, 2, 64).transpose(1, 2)
    else:
        o, lse = attention_keybias(q.to(dev), kd, vd, None, 0.125, return_lse=True)
        assert (lse.cpu() - ref_lse).abs().max().item() <= 2.0 ** -8 / 0.6931   # bf16 P in the sum
    rel = (o.float().cpu() - ref).norm(dim=-1) / ref.norm(dim=-1)
    assert rel.max().item() <= 4 * 2.0 ** -9, rel.max().item()


@pytest.mark.parametrize("dtype,ulp", [(torch.bfloat16, 2.0 ** -9), (torch.float16, 2.0 ** -12)])
@pytest.mark.parametrize("B,H", [(64, 16), (205, 5)])
@pytest.mark.parametrize("scale", [0.3, 3.0])
def test_both_sides_of_the_grid_line(dev, dtype, ulp, B, H, scale):
    """1,024 and 1,025 workgroups: bounds formed in the kernel, and by a launch."""
    g = torch.Generator(device=dev).manual_seed(B)
    q, k, v = (torch.randn(B, H, t, 64, device=dev, generator=g) for t in (100, 301, 301))
    q, k, v = (q * scale).to(dtype), (k * scale).to(dtype), v.to(dtype)
    bias = torch.randint(1, 9, (B, 1, 1, 301), device=dev, generator=g).float().log().to(dtype)
    o = attention_keybias(q, k, v, bias.expand(B, H, 1, 301), 0.125)
    x = q.double() @ k.double().transpose(-1, -2).contiguous() * 0.125 + bias.double()
    ref = torch.softmax(x, -1) @ v.double()
    rel = (o.double() - ref).norm(dim=-1) / ref.norm(dim=-1)
    assert rel.max().item() <= 4 * ulp, rel.max().item()
