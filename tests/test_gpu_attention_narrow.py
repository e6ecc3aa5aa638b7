"""Head dims 16 and 32 at the edges of their two kernels' tiles: one key, the last
key tile one short of full, full and one over, every phase of the four-slot
key ring, query counts around a wave's 64 and a workgroup's 256; k and v as
views of longer buffers whose rows past N hold NaN, so a read past N shows;
the row max rising in the last tile; a row whose biases are all -inf.

Bar: rms of a 16-bit output's error relative to its row is at most
half a unit in the last place each for P and the output, 2 * 2^-9 (bf16) or
2 * 2^-12 (fp16), and the max over rows stays within four times that; the LSE
is fp32 sums of fp32 terms, 1e-4 absolute in log2 units.
"""
import math

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


# Up to 192 keys, or up to 512 / 2,048 / 4,096 on small grids, a call runs a
# kernel of its own; the cases above are all its.  Those below run the other one,
# or sit on either side of a line.

def _against_fp64(dev, B, H, M, N, D, dtype, kind, seed):
    """Token-major q, k and v (strided rows), NaN rows behind the keys; bias one
    row for all heads with a stride between keys, or a row per head."""
    g = torch.Generator(device=dev).manual_seed(seed)
    s = 0.5 * (64.0 / D) ** 0.25

    def rows(T, scale, tail=0):
        t = torch.full((B, T + tail, H, D), float("nan"), device=dev)
        t[:, :T] = scale * torch.randn(B, T, H, D, device=dev, generator=g)
        return t.to(dtype)[:, :T].transpose(1, 2)

    q, k, v = rows(M, s), rows(N, s, 40), rows(N, 1.0, 40)
    bias = None
    if kind is not None:
        log = torch.randint(1, 9, (B, H, 1, N), device=dev, generator=g).float().log().to(kind)
        bias = log if seed % 2 else torch.stack((log, log), -1)[:1, :1, :, :, 0].expand(B, H, 1, N)
    o, lse = attention_keybias(q, k, v, bias, D ** -0.5, return_lse=True)
    x = q.double() @ k.double().transpose(-1, -2).contiguous() * D ** -0.5
    if bias is not None:
        x = x + bias.double()
    ref, ref_lse = torch.softmax(x, -1) @ v.double(), torch.logsumexp(x, -1) / math.log(2.0)
    rel = (o.double() - ref).norm(dim=-1) / ref.norm(dim=-1)
    assert rel.max().item() <= 8 * ULP[dtype], rel.max().item()
    assert (lse - ref_lse).abs().max().item() <= 1e-4


FORMS = [(torch.bfloat16, None), (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32),
         (torch.float16, torch.float16), (torch.float16, None), (torch.float16, torch.float32)]


@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("dtype,kind", FORMS)
@pytest.mark.parametrize("B,H,M,N", [(65, 16, 1, 193), (65, 16, 64, 224), (22, 16, 257, 225),
                                     (22, 16, 300, 256), (23, 16, 257, 257), (65, 16, 65, 300)])
def test_many_heads(dev, D, dtype, kind, B, H, M, N):
    """Every phase of the key ring, whole and broken last tiles, query counts
    around a wave's 64 and a workgroup's 256, in every form of the operands."""
    _against_fp64(dev, B, H, M, N, D, dtype, kind, seed=M + N)


@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("over", [0, 1])
@pytest.mark.parametrize("dtype,kind", FORMS[:4])
@pytest.mark.parametrize("B,H,M,line", [
    (1, 2, 100, 2048), (1, 2, 100, 4096), (1, 16, 1374, 2048), (3, 16, 1374, 512),
    (8, 16, 1374, 192), (9, 16, 100, 1024)])
def test_both_sides_of_the_lines(dev, D, over, dtype, kind, B, H, M, line):
    _against_fp64(dev, B, H, M, line + over, D, dtype, kind, seed=line + M)


@pytest.mark.parametrize("D", [16, 32])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N", [2049, 290])
def test_rows_that_rise_and_rows_that_are_masked_over_many_heads(dev, D, dtype, N):
    """The row max moving up in the last tile and keys masked by -inf or by the
    lowest fp32 value, beside rows without any weight (NaN), where the rescale
    is per block of a wave; at either of the two kernels (290 keys: 70 heads x
    4 batch elements; 2,049: two heads)."""
    B, H = (2, 1) if N > 2048 else (4, 70)
    M = 500
    g = torch.Generator(device=dev).manual_seed(N)
    q = 0.3 * torch.randn(B, H, M, D, device=dev, generator=g) + 2.0 * D ** -0.5
    k = 0.3 * torch.randn(B, H, N, D, device=dev, generator=g)
    k[:, :, -1] = 30.0                               # q.k / sqrt(D) ~ 60 at the last key
    q, k = q.to(dtype), k.to(dtype)
    v = torch.randn(B, H, N, D, device=dev, generator=g).to(dtype)
    bias = torch.zeros(B, H, 1, N, device=dev)
    bias[..., :40] = float("-inf")
    bias[..., 90:100] = torch.finfo(torch.float32).min
    bias[B - 1, H - 1] = float("-inf")
    o = attention_keybias(q, k, v, bias, D ** -0.5)
    x = q.double() @ k.double().transpose(-1, -2).contiguous() * D ** -0.5 + bias.double()
    ref = torch.softmax(x, -1) @ v.double()
    live = torch.ones(B, H, dtype=torch.bool, device=dev)
    live[B - 1, H - 1] = False
    assert torch.isnan(o[~live]).all()
    rel = (o.double() - ref)[live].norm(dim=-1) / ref[live].norm(dim=-1)
    assert rel.max().item() <= 8 * ULP[dtype], rel.max().item()
