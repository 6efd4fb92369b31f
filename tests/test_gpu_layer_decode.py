"""GPU: the layer's decode-only call as three launches (in_proj, the fused step
with the gated norm, out_proj)."""
import pytest
import torch

from myvllm_amd import _lib
from myvllm_amd.cache import LinearAttentionCache
from myvllm_amd.layer import GatedDeltaNet

pytestmark = pytest.mark.gpu

HID, HK, HV, D = 256, 2, 4, 128
PARAMS = ("in_proj", "conv1d_weight", "A_log", "dt_bias", "norm_weight", "out_proj")


def _layer(dev, slots=8, dtype=torch.bfloat16, seed=1):
    layer = GatedDeltaNet(HID, HK, HV, D, D, dtype=dtype, device=dev)
    layer.init_random(std=0.05, seed=seed)
    cache = LinearAttentionCache(1, slots, 4, D, D, HK, HV, dtype, dev, conv_dtype=torch.float32)
    g = torch.Generator().manual_seed(seed)
    cache.conv_cache[0].copy_(torch.randn(cache.conv_cache[0].shape, generator=g))
    cache.recurrent_cache[0].copy_(torch.randn(cache.recurrent_cache[0].shape, generator=g) * 0.1)
    layer.conv_state, layer.recurrent_state = cache.layer(0)
    return layer


@pytest.mark.parametrize("name", PARAMS)
def test_parameter_on_the_host_is_refused(dev, monkeypatch, name):
    """A parameter that was never moved raises before any kernel is given its
    address.  (Every launch is replaced by one that fails the test, but for the
    general path's own, which check their tensors first.)"""
    layer = _layer(dev)
    setattr(layer, name, torch.nn.Parameter(getattr(layer, name).detach().cpu()))
    launched = []

    def call(fn, *args):
        launched.append(fn)
        assert all(t.is_cuda for t in args if isinstance(t, torch.Tensor)), f"{fn} was given a host tensor"

    monkeypatch.setattr(_lib, "call", call)
    x = torch.randn(3, HID, device=dev).bfloat16()
    idx = torch.arange(3, dtype=torch.int32, device=dev)
    with torch.no_grad(), pytest.raises((ValueError, RuntimeError)):
        layer(x, None, idx, idx, False)
    assert "gdn_linear" not in launched and "gdn_decode_step_fused_norm" not in launched
