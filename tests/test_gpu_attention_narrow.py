"""Head dims 16 and 32 at the edges of their kernel's tiles: one key, the last
key tile one short of full, full and one over, every phase of the four-slot
key ring, query counts around a wave's 64 and a workgroup's 256; k and v as
views of longer buffers whose rows past N hold NaN, so a read past N shows;
the row max rising in the last tile; a row whose biases are all -inf.

Bar: rms of a 16-bit output's error relative to its row is at most
half a unit in the last place each for P and the output, 2 * 2^-9 (bf16) or
2 * 2^-12 (fp16), and the max over rows stays within four times that; the LSE
is fp32 sums of fp32 terms, 1e-4 absolute in log2 units.
"""
import pytest
import torch

from merging.fused_attention import attention_keybias
from oracle.attention import attention_reference

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}


def _case(D, M, N, dtype, seed, top=0.0):
    g = torch.Generator().manual_seed(seed)
    s = 0.5 * (64.0 / D) ** 0.25
    q = torch.randn(1, 2, M, D, generator=g) * s
    k = torch.randn(1, 2, N, D, generator=g) * s
    v = torch.randn(1, 2, N, D, generator=g)
    if top:
        q = q + 2.0 * D ** -0.5
        k[:, :, -1] = top / 2.0                  # q.k / sqrt(D) ~ top
    bias = torch.randint(1, 9, (1, 1, 1, N), generator=g).float().log().expand(1, 2, 1, N)
    return q.to(dtype), k.to(dtype), v.to(dtype), bias.contiguous()


def _run(dev, q, k, v, bias):
    D, N = q.shape[-1], k.shape[2]
    long = [torch.full((1, 2, N + 200, D), float("nan"), dtype=q.dtype, device=dev) for _ in "kv"]
    for buf, t in zip(long, (k, v)):
        buf[:, :, :N] = t.to(dev)
    o, lse = attention_keybias(q.to(dev), long[0][:, :, :N], long[1][:, :, :N], bias.to(dev),
                               D ** -0.5, return_lse=True)
    ref, ref_lse = attention_reference(q, k, v, bias, D ** -0.5)
    rel = (o.float().cpu() - ref).norm(dim=-1) / ref.norm(dim=-1)
    assert rel.max().item() <= 8 * ULP[q.dtype], rel.max().item()
    assert (lse.cpu() - ref_lse).abs().max().item() <= 1e-4


@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("M,N", [(1, 1), (63, 31), (64, 32), (65, 33), (255, 96), (256, 97),
                                 (257, 128), (300, 129), (129, 160), (513, 191)])
def test_tile_edges(dev, D, M, N):
    _run(dev, *_case(D, M, N, torch.bfloat16, seed=M + N))


@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("top", [12.0, 60.0])
def test_row_max_rises_in_the_last_tile(dev, D, dtype, top):
    _run(dev, *_case(D, 200, 290, dtype, seed=int(top), top=top))


@pytest.mark.parametrize("D", [16, 32])
def test_masked_keys(dev, D):
    """Keys at -inf and at fp32's lowest value have no weight; a whole row of
    -inf has no defined softmax and gives NaN, not a finite value."""
    q, k, v, bias = _case(D, 100, 150, torch.bfloat16, seed=3)
    bias = bias.clone()
    bias[..., :40] = float("-inf")                  # the whole first tile
    bias[..., 90:100] = torch.finfo(torch.float32).min
    o = attention_keybias(q.to(dev), k.to(dev), v.to(dev), bias.to(dev), D ** -0.5)
    keep = torch.cat((torch.arange(40, 90), torch.arange(100, 150)))
    ref, _ = attention_reference(q, k[:, :, keep], v[:, :, keep], bias[..., keep], D ** -0.5)
    rel = (o.float().cpu() - ref).norm(dim=-1) / ref.norm(dim=-1)
    assert rel.max().item() <= 8 * ULP[q.dtype]
    o = attention_keybias(q.to(dev), k.to(dev), v.to(dev),
                          torch.full_like(bias, float("-inf")).to(dev), D ** -0.5)
    assert torch.isnan(o).all()
