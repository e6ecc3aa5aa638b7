"""Blocks run as a chain (the last residual pass also writes the next block's
LayerNorm) against the same blocks called one by one: bit for bit, and a block
with a forward hook, a replaced forward or another dtype is called as a
module, its hook seeing and able to change what passes (everything else that
takes a block out of the chain: test_block_chain.py, on the CPU).  The LayerNorm
parameters of the qk norm in each format against the stacked fp32 ones."""
import pytest
import torch

import gpa_aggregator as A
from merging import _native

pytestmark = pytest.mark.gpu


def _one_by_one(monkeypatch):
    monkeypatch.setattr(A, "_chainable", lambda blk: False)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_chain_equals_blocks_called_alone(dev, monkeypatch, dtype):
    cfg = A.GpaConfig(img_size=84, vit_depth=3, embed_dim=512, num_heads=8)
    vit = A.init_random_(A.DinoV2Reg(cfg).to(dev), 3).to(dtype).eval()
    img = torch.rand(3, 3, 84, 84, device=dev, generator=torch.Generator(dev).manual_seed(1))
    with torch.no_grad(), torch.autocast("cuda", dtype):
        chained = vit(img.to(dtype))
        _one_by_one(monkeypatch)
        alone = vit(img.to(dtype))
    assert torch.equal(chained, alone)


def test_hooks_and_replaced_forwards_still_run(dev):
    cfg = A.GpaConfig(img_size=84, vit_depth=3, embed_dim=512, num_heads=8)
    vit = A.init_random_(A.DinoV2Reg(cfg).to(dev), 3).bfloat16().eval()
    img = torch.rand(2, 3, 84, 84, device=dev).bfloat16()

    def run():
        with torch.no_grad(), torch.autocast("cuda", torch.bfloat16):
            return vit(img)

    base, seen = run(), []
    handle = vit.blocks[1].register_forward_hook(lambda m, a, out: seen.append(out.shape))
    assert torch.equal(run(), base) and len(seen) == 1
    handle.remove()
    handle = vit.blocks[0].register_forward_hook(lambda m, a, out: torch.zeros_like(out))
    zeroed = run()
    handle.remove()
    vit.blocks[0].forward = lambda x, rope=None, gm=None: torch.zeros_like(x)
    assert torch.equal(run(), zeroed) and not torch.equal(zeroed, base)
    del vit.blocks[0].forward
    assert torch.equal(run(), base)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("param", [torch.float32, torch.bfloat16, torch.float16])
def test_qk_norm_params(dev, dtype, param):
    """Separate parameters, aligned and not, of one format and mixed."""
    g = torch.Generator(dev).manual_seed(4)
    H, P = 3, 21
    qkv = torch.randn(2, 2 * P, 3 * H * 64, device=dev, generator=g).to(dtype)
    rope = A.Rope2D(100.0).table(A.frame_positions(4, 5, dev), 64)
    flat = torch.randn(4 * 64 + 3, device=dev, generator=g).to(param)
    for off in (0, 3):
        p = [flat[off + 64 * i:off + 64 * i + 64] for i in range(4)]
        want = torch.ops.gpa.qk_norm_rope(qkv, torch.stack(p[:2]), torch.stack(p[2:]), 1e-5,
                                          rope.pos, rope.cs, H, False, True)
        got = _native.qk_norm_rope_params(qkv, *p, 1e-5, rope.pos, rope.cs, H, False, True)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    mixed = [p[0].float(), *p[1:]]
    got = _native.qk_norm_rope_params(qkv, *mixed, 1e-5, rope.pos, rope.cs, H, False, True)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
