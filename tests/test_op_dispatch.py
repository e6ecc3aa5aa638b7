"""How the package's ops are dispatched (CPU): the callable that skips the
autograd kernel and the registered op answer alike wherever a caller can tell
them apart, on a small op registered the same way."""
import subprocess
import sys
from typing import Tuple

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch._subclasses.fake_tensor import FakeTensorMode

from merging import _native


@_native._op
def dispatch_probe(x: torch.Tensor, s: float) -> Tuple[torch.Tensor, torch.Tensor]:
    return x * s, x.sum()


@_native._fake("dispatch_probe")
def _probe_fake(x, s):
    return x.new_empty(x.shape), x.new_empty(())


@pytest.mark.parametrize("fn", [dispatch_probe, torch.ops.gpa.dispatch_probe])
def test_callable_and_op_agree(fn):
    x = torch.arange(4.0)
    out, total = fn(x, 2.0)
    assert torch.equal(out, 2 * x) and total == 6 and not out.requires_grad
    # gradients: the output asks for one, the backward raises
    out = fn(x.clone().requires_grad_(), 2.0)[0]
    assert out.requires_grad
    with pytest.raises(RuntimeError, match="no autograd formula"):
        out.sum().backward()
    with torch.no_grad():
        assert not fn(x.clone().requires_grad_(), 2.0)[0].requires_grad
    with torch.inference_mode():
        assert fn(x, 2.0)[0].is_inference()
    # tracing and transforms see the op itself
    assert "gpa.dispatch_probe" in make_fx(lambda t: fn(t, 2.0)[0])(x).code
    assert torch.equal(torch.vmap(lambda t: fn(t, 2.0)[0])(x.expand(3, 4)), (2 * x).expand(3, 4))
    with FakeTensorMode():
        assert fn(torch.empty(5), 2.0)[0].shape == (5,)
    assert torch.equal(torch.compile(lambda t: fn(t, 2.0)[0] + 1, backend="aot_eager",
                                     fullgraph=True)(x), 2 * x + 1)


def test_cpu_tensors_are_refused():
    q = torch.zeros(1, 1, 4, 64, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="GPU tensors"):
        _native.attn_keybias(q, q, q, None, 0.125, False)


def test_keyword_arguments():
    x = torch.arange(4.0)
    for out in (dispatch_probe(x, s=2.0), dispatch_probe(s=2.0, x=x)):
        assert torch.equal(out[0], 2 * x) and not out[0].requires_grad
    out = dispatch_probe(s=2.0, x=x.clone().requires_grad_())[0]
    assert out.requires_grad
    with pytest.raises(RuntimeError, match="no autograd formula"):
        out.sum().backward()
    with FakeTensorMode():
        a = torch.empty(1, 4, 64, device="cuda", dtype=torch.bfloat16)
        assert _native.sim_argmax(a=a, b=a, max_in_input_dtype=True)[0].dtype == torch.bfloat16


_TWO_COPIES = """
import importlib, importlib.util, sys
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
sys.path.insert(0, {pkg!r})
from merging import _native
from merging.fused_similarity import fused_similarity_argmax
spec = importlib.util.spec_from_file_location("another_native", _native.__file__)
other = importlib.util.module_from_spec(spec)
spec.loader.exec_module(other)
for again in (False, True):
    if again:
        importlib.reload(_native)
    with FakeTensorMode():
        a = torch.empty(1, 4, 64, device="cuda", dtype=torch.bfloat16)
        for call in (_native.sim_argmax, other.sim_argmax, torch.ops.gpa.sim_argmax):
            assert call(a, a)[1].shape == (1, 4)
        assert fused_similarity_argmax(a, a)[0].dtype == torch.bfloat16
    try:
        other.sim_argmax(torch.zeros(1, 4, 64), torch.zeros(1, 4, 64))
    except ValueError as e:
        assert "GPU tensors" in str(e)
    else:
        raise AssertionError("a CPU tensor was taken")
"""


def test_two_copies_of_the_module_in_one_process():
    """Loaded under a second name, then loaded again."""
    script = _TWO_COPIES.format(pkg=str(_native.LIB_PATH.parents[2]))
    done = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True,
                          timeout=120)
    assert done.returncode == 0, done.stderr
