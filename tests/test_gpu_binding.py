"""The native call path against the ctypes one: same results, same refusals."""
import pytest
import torch

from myvllm_amd import _lib, recurrent_gated_delta_rule
from myvllm_amd.norm import gdn_gating
from myvllm_amd.workloads import decode_case


class Sub(torch.Tensor):
    """A subclass: not a plain tensor, so its calls go through ctypes."""


def test_plain_tensors_only():
    """Anything but a plain tensor is left to ctypes (None), as is a call without a device."""
    _lib.load()
    t = torch.zeros(2, 8, dtype=torch.bfloat16)
    f = _lib._fast
    assert f.same_device(t) == -1 and f.same_device(t.as_subclass(Sub)) == -1 and f.same_device() == -1
    assert f.vec16_ok(t) is True and f.vec16_ok(t[:, 1:]) is False and f.vec16_ok(t.as_subclass(Sub)) is None
    assert f.vec16_ok(t.t()) is False and f.vec16_ok(torch.zeros(())) is None and f.vec16_ok(3) is None
    assert f.gdn_gating(*[t] * 6) is None and f.gdn_gating(None, *[t] * 5) is None
    assert f.gdn_gating(*[torch.zeros(1, 1, 1, 1, 1)] * 6) is None
    with pytest.raises(TypeError):
        f.gdn_gating(t)
    with pytest.raises(TypeError):
        f.gdn_chunk_prefill_workspace_size(1.5, 1, 1, 1, 1, 1)
    with pytest.raises(ValueError):
        gdn_gating(t, t, t, t)


@pytest.mark.gpu
def test_both_paths_agree(dev):
    c = decode_case(5, seed=3, num_slots=7, Hk=2, Hv=4)
    d = [t.to(dev) for t in (c.q, c.k, c.v, c.g, c.beta)]
    outs = []
    for wrap in (lambda t: t, lambda t: t.as_subclass(Sub)):
        st = c.state.to(dev)
        o = recurrent_gated_delta_rule(*[wrap(t) for t in d], wrap(st), c.idx.to(dev))
        outs.append((o.as_subclass(torch.Tensor), st))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    with pytest.raises(_lib.GdnError, match="shape"):
        recurrent_gated_delta_rule(d[0][:3], *d[1:], c.state.to(dev), c.idx.to(dev))
    # on the current stream, in order: the inputs are written there behind some milliseconds of work
    late = [torch.zeros_like(t) for t in d]
    st = torch.zeros_like(c.state.to(dev))
    state, idx = c.state.to(dev), c.idx.to(dev)
    big = torch.randn(8192, 8192, device=dev)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        for _ in range(4):
            big = torch.tanh(big @ big)
        for t, src in zip(late, d):
            t.copy_(src)
        st.copy_(state)
        o = recurrent_gated_delta_rule(*late, st, idx)
    s.synchronize()
    assert torch.equal(o, outs[0][0]) and torch.equal(st, outs[0][1])
