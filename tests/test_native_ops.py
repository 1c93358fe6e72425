"""The native ops (csrc/torch_ops.cpp) under the parts of torch that a call can pass through: autograd,
which they refuse, modes and transforms, which see them as they see any other op, streams, and the
argument errors, raised before any launch.
"""

import pytest
import torch

import flash_lab
from flash_lab import _hip

pytestmark = pytest.mark.gpu


@pytest.fixture
def qkv():
    q = torch.randn(1, 40, 8, 64, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(1, 50, 2, 64, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    return q, k, v


@pytest.fixture
def step():
    q = torch.randn(2, 8, 64, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(2, 90, 2, 64, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    return q, k, v, torch.tensor([90, 7], device="cuda", dtype=torch.int32)


def test_backward_is_refused_and_forward_is_not(qkv, step):
    q, k, v = qkv
    want = flash_lab.attention(q, k, v)
    out = flash_lab.attention(q.clone().requires_grad_(), k, v)
    assert out.requires_grad and torch.equal(out, want)
    with pytest.raises(RuntimeError, match="no autograd formula was registered"):
        out.sum().backward()
    with torch.no_grad():
        assert not flash_lab.attention(q.clone().requires_grad_(), k, v).requires_grad
    qd, kc, vc, lens = step
    out, lse = flash_lab.decode(qd.clone().requires_grad_(), kc, vc, lens, return_lse=True)
    assert out.requires_grad and lse.requires_grad
    with pytest.raises(RuntimeError, match="no autograd formula was registered"):
        lse.sum().backward()


def test_modes_and_transforms_see_the_op(qkv):
    from torch.utils._python_dispatch import TorchDispatchMode

    q, k, v = qkv
    seen = []

    class Record(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Record():
        want = flash_lab.attention(q, k, v, causal=True)
    assert "flash_lab.attention_mma_pipelined.default" in seen
    got = torch.vmap(lambda x: flash_lab.attention(x, k, v, causal=True))(q[None].expand(2, -1, -1, -1, -1))
    assert torch.equal(got[0], want) and torch.equal(got[1], want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = flash_lab.attention(q, k, v, causal=True)
    side.synchronize()
    assert torch.equal(other, want)


def test_opcheck(step):
    torch.library.opcheck(torch.ops.flash_lab.decode_splitkv.default, (*step, 0.1, 0))


@pytest.mark.parametrize("change,message", [
    (dict(k=lambda k: k.cpu()), "k must be a CUDA tensor"),
    (dict(k=lambda k: k.half()), "must have dtype torch.bfloat16"),
    (dict(q=lambda q: q[0]), r"must be \[B, S, H, D\]"),
    (dict(v=lambda v: v[:, :4]), "the same shape"),
    (dict(q=lambda q: q.transpose(2, 3).contiguous().transpose(2, 3)), "contiguous in its last dimension"),
    (dict(q=lambda q: q[:, :0]), "empty input"),
], ids=["device", "dtype", "rank", "shape", "stride", "empty"])
def test_bad_arguments(qkv, change, message):
    args = dict(zip("qkv", qkv))
    for name, f in change.items():
        args[name] = f(args[name])
    with pytest.raises(RuntimeError, match=message):
        torch.ops.flash_lab.attention_mma(args["q"], args["k"], args["v"], True, 0.1)


def test_bound_functions_are_the_librarys():
    assert _hip.TORCH_BOUND[-1] == "fl_last_error" and all(name in _hip.SIGNATURES for name in _hip.TORCH_BOUND)
