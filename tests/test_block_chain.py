"""What is attached to a block's call runs when the block is part of a chain
(CPU, on the differentiable path: torch's attention, unfused norms): hooks of
every kind, a compiled block, replaced forwards and calls, tracers that
record the block."""
import pytest
import torch

import gpa_aggregator as A

MODULE = torch.nn.modules.module


@pytest.fixture
def vit():
    cfg = A.GpaConfig(img_size=84, vit_depth=3, embed_dim=64, num_heads=2, frame_attn="sdpa",
                      fused_norms=False)
    return A.init_random_(A.DinoV2Reg(cfg), 3)


def _image():
    return torch.rand(1, 3, 84, 84, generator=torch.Generator().manual_seed(1))


HOOKS = {
    "forward": lambda b, f: b.register_forward_hook(lambda m, a, o: f()),
    "forward_pre": lambda b, f: b.register_forward_pre_hook(lambda m, a: f()),
    "backward": lambda b, f: b.register_full_backward_hook(lambda m, i, o: f()),
    "backward_pre": lambda b, f: b.register_full_backward_pre_hook(lambda m, o: f()),
    "all_forward": lambda b, f: MODULE.register_module_forward_hook(
        lambda m, a, o: f() if m is b else None),
    "all_forward_pre": lambda b, f: MODULE.register_module_forward_pre_hook(
        lambda m, a: f() if m is b else None),
    "all_backward": lambda b, f: MODULE.register_module_full_backward_hook(
        lambda m, i, o: f() if m is b else None),
    "all_backward_pre": lambda b, f: MODULE.register_module_full_backward_pre_hook(
        lambda m, o: f() if m is b else None),
}


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("kind", HOOKS)
def test_hooks_run(vit, kind, which):
    seen = []
    handle = HOOKS[kind](vit.blocks[which], lambda: seen.append(kind))
    try:
        vit(_image().requires_grad_()).sum().backward()
    finally:
        handle.remove()
    assert seen == [kind]


def test_a_backward_hook_changes_the_gradients(vit):
    def grads():
        vit.zero_grad()
        vit(_image()).square().sum().backward()
        return vit.blocks[0].norm1.weight.grad.clone()

    base = grads()
    handle = vit.blocks[1].register_full_backward_hook(lambda m, gi, go: tuple(
        None if g is None else 2 * g for g in gi))
    doubled = grads()
    handle.remove()
    assert torch.equal(doubled, 2 * base) and torch.equal(grads(), base)


def test_a_compiled_block_is_compiled(vit):
    base, graphs = vit(_image()), []

    def backend(gm, example):
        graphs.append(gm)
        return gm.forward

    vit.blocks[1].compile(backend=backend)
    assert torch.equal(vit(_image()), base) and len(graphs) == 1


@pytest.mark.parametrize("name", ["forward", "__call__"])
def test_a_method_replaced_on_the_class_is_called(vit, monkeypatch, name):
    base, seen, old = vit(_image()), [], getattr(A.Block, name)

    def replaced(self, *args, **kwargs):
        seen.append(self)
        return old(self, *args, **kwargs)

    monkeypatch.setattr(A.Block, name, replaced)
    assert torch.equal(vit(_image()), base) and seen == list(vit.blocks)


def test_tracers_record_the_blocks(vit):
    class Tracer(torch.fx.Tracer):
        def is_leaf_module(self, m, name):
            return isinstance(m, (A.Block, torch.nn.LayerNorm))

    called = [n.target for n in Tracer().trace(vit).nodes if n.op == "call_module"]
    assert called == ["blocks.0", "blocks.1", "blocks.2", "norm"]
    graph = str(torch.jit.trace(vit, _image(), check_trace=False).graph)
    assert graph.count("prim::CallMethod") == 4            # the same modules


def test_other_modules_in_a_block_s_place(vit):
    """They are called with what the loop passes, the image tokens alone."""
    img, args = _image(), []
    base = vit(img)
    handle = vit.blocks[1].register_forward_pre_hook(lambda m, a: args.append(len(a)))
    assert torch.equal(vit(img), base) and args == [1]
    handle.remove()
    vit.blocks[1] = torch.nn.Sequential(vit.blocks[1])
    assert torch.equal(vit(img), base)
    vit.blocks[1] = torch.nn.Identity()
    assert vit(img).shape == base.shape


def test_arguments_of_the_aggregator_s_blocks():
    cfg = A.GpaConfig(img_size=84, vit_depth=1, depth=2, embed_dim=64, num_heads=2)
    model, seen = A.GpaAggregator(cfg), []

    class Record(torch.nn.Module):
        def __init__(self, name):
            super().__init__()
            self.name = name

        def forward(self, x, *args):
            seen.append((self.name, len(args)))
            return x

    class Embed(torch.nn.Module):
        def forward(self, images):
            return torch.zeros(images.shape[0], 36, 64)

    model.patch_embed = Embed()
    for i in range(cfg.depth):
        model.frame_blocks[i], model.global_blocks[i] = Record("frame"), Record("global")
    with torch.no_grad():
        model(torch.zeros(1, 2, 3, 84, 84))
    assert seen == [("frame", 1), ("global", 2)] * cfg.depth
