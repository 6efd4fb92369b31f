"""GPU: the layer's decode-only call as three launches (in_proj, the fused step
with the gated norm, out_proj) vs the fp64 layer oracle and the general path,
with the layer tests' bars; where it is not taken; and from a captured graph."""
import contextlib

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from conftest import assert_out_close, assert_state_close
from myvllm_amd import _lib
from myvllm_amd.cache import LinearAttentionCache
from myvllm_amd.layer import GatedDeltaNet
from oracle.layer import gdn_layer_ref

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


def _inputs(dev, T, slots=24, dtype=torch.bfloat16, seed=3):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, HID, generator=g).to(dtype)
    return x.to(dev), torch.randperm(slots, generator=g)[:T].to(torch.int32).to(dev)


def _call(layer, x, idx, caches, conv_idx=None):
    """One step from the given caches: the output and both caches after it."""
    layer.conv_state.copy_(caches[0])
    layer.recurrent_state.copy_(caches[1])
    out = layer(x, None, idx if conv_idx is None else conv_idx, idx, False)
    torch.cuda.synchronize()
    return out.detach(), layer.conv_state.clone(), layer.recurrent_state.clone()


def _spy(monkeypatch):
    calls, real = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda fn, *a: (calls.append(fn), real(fn, *a))[1])
    return calls


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 2, 16, 17, 24])
def test_native_decode(dev, monkeypatch, T, dtype):
    """Sizes on both sides of the linear kernel's 16 tokens: the route taken, the result against the
    oracle and the general path, and the same bits when it is run again."""
    layer = _layer(dev, 24, dtype)
    x, idx = _inputs(dev, T, dtype=dtype)
    caches = layer.conv_state.clone(), layer.recurrent_state.clone()
    print(f"native decode T={T} {dtype}", flush=True)
    calls = _spy(monkeypatch)
    with torch.no_grad():
        got = _call(layer, x, idx, caches)
        assert calls == (["gdn_linear", "gdn_decode_step_fused_norm", "gdn_linear"] if T <= 16 else
                         ["gdn_decode_step_fused_norm"])
        for a, b in zip(got, _call(layer, x, idx, caches)):
            assert torch.equal(a, b)
    calls.clear()
    general = _call(layer, x, idx, caches)  # (gradients on: torch's products, the norm by itself)
    assert calls == ["gdn_decode_step_fused", "gdn_rms_norm_gated"]
    cz = layer.conv_dim + layer.v_size
    w = layer.in_proj.detach().cpu()
    conv, rec = caches[0].cpu().clone(), caches[1].cpu().clone()
    ref = gdn_layer_ref(x.cpu(), w[:cz], w[cz:], *(getattr(layer, n).detach().cpu() for n in (
        "conv1d_weight", "A_log", "dt_bias", "norm_weight", "out_proj")), conv, idx.cpu(), rec, idx.cpu(),
        torch.zeros(1, dtype=torch.int32), HK, num_decode_tokens=T)
    for out, cs, rs in (got, general):
        assert_out_close(out, ref)
        assert_state_close(rs.cpu(), rec, rtol=3e-2, atol=1e-3)
        assert torch.allclose(cs.cpu(), conv.float(), rtol=1e-2, atol=1e-2)
        # o, its norm and the output are rounded once each, o not at all in the native step: half a unit in
        # the last place (2^-9, 2^-12) per rounding on either side
        err = (out.double().cpu() - ref.double()).norm() / ref.double().norm()
        assert err < 4 * (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12), err


def test_native_decode_padding_and_layouts(dev):
    """Slots outside the caches (zero rows, caches untouched), int64 indices, rows of x apart and a
    weight at an odd address: as the general path gives it."""
    layer = _layer(dev, 24)
    x, idx = _inputs(dev, 6)
    idx = idx.long()
    idx[2], idx[4] = -1, 24
    wide = torch.zeros(6, HID + 24, dtype=x.dtype, device=dev)
    wide[:, 8: 8 + HID] = x
    caches = layer.conv_state.clone(), layer.recurrent_state.clone()
    general = _call(layer, x, idx, caches)
    print("native decode, padding", flush=True)
    with torch.no_grad():
        got = _call(layer, wide[:, 8: 8 + HID], idx, caches)
        flat = torch.empty(layer.out_proj.numel() + 1, dtype=x.dtype, device=dev)
        odd = flat[1:].view(layer.out_proj.shape).copy_(layer.out_proj)
        layer.out_proj = torch.nn.Parameter(odd)
        assert layer.out_proj.data_ptr() % 16
        shifted = _call(layer, x, idx, caches)
    for out, cs, rs in (got, shifted):
        assert not out[2].any() and not out[4].any()
        assert_out_close(out, general[0])
        assert torch.equal(cs, got[1]) and torch.equal(rs, got[2])
        assert_state_close(rs, general[2], rtol=3e-2, atol=1e-3)
    unused = torch.ones(24, dtype=torch.bool)
    unused[idx.cpu()[[0, 1, 3, 5]]] = False
    assert torch.equal(got[1].cpu()[unused], caches[0].cpu()[unused])
    assert torch.equal(got[2].cpu()[unused], caches[1].cpu()[unused])


class _Seen(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Dispatched(TorchDispatchMode):
    products = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.products += func in (torch.ops.aten.mm.default, torch.ops.aten.addmm.default)
        return func(*args, **(kwargs or {}))


class _Weight(torch.nn.Parameter):
    pass


@pytest.mark.parametrize("why", ["grad", "autocast", "function mode", "default device", "dispatch mode", "forward AD",
                                 "subclass", "fp32"])
def test_general_path_where_something_looks_on(dev, monkeypatch, why):
    """The general path where the torch products are recorded, counted or changed, or the tensors are
    not plain 16-bit ones; its result is the native one's."""
    dtype = torch.float32 if why == "fp32" else torch.bfloat16
    layer = _layer(dev, 24, dtype)
    x, idx = _inputs(dev, 3, dtype=dtype)
    caches = layer.conv_state.clone(), layer.recurrent_state.clone()
    with torch.no_grad():
        native = _call(layer, x, idx, caches)
    stack = contextlib.ExitStack()
    if why != "grad":
        stack.enter_context(torch.no_grad())
    if why == "subclass":
        layer.in_proj = torch.nn.Parameter(layer.in_proj.detach())
        layer.in_proj.__class__ = _Weight
    mode = _Dispatched()
    enter = {"autocast": lambda: torch.autocast("cuda", torch.bfloat16), "function mode": _Seen,
             "default device": lambda: torch.device("cuda"), "dispatch mode": lambda: mode,
             "forward AD": torch.autograd.forward_ad.dual_level}
    calls = _spy(monkeypatch)
    print(f"general path: {why}", flush=True)
    with stack:
        if why in enter:
            stack.enter_context(enter[why]())
        got = _call(layer, x, idx, caches)
    assert calls == ["gdn_decode_step_fused", "gdn_rms_norm_gated"]
    assert mode.products == (2 if why == "dispatch mode" else 0)
    assert_out_close(got[0], native[0])
    assert_state_close(got[2], native[2], rtol=3e-2, atol=1e-3)


@pytest.mark.parametrize("T", [5, 20])
def test_native_decode_replays_from_a_graph(dev, T):
    """Captured and replayed with eager work between the replays: bit for bit the eager step."""
    layer = _layer(dev, 24)
    x, idx = _inputs(dev, T)
    caches = layer.conv_state.clone(), layer.recurrent_state.clone()
    with torch.no_grad():
        ref = _call(layer, x, idx, caches)
        side = torch.cuda.Stream(device=dev)  # warm-up off the capture stream, as torch asks
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            layer(x, None, idx, idx, False)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = layer(x, None, idx, idx, False)
        for rep in range(3):
            layer.conv_state.copy_(caches[0])
            layer.recurrent_state.copy_(caches[1])
            out.zero_()
            torch.cuda.synchronize()
            print(f"native decode T={T}, graph replay {rep}", flush=True)
            graph.replay()
            torch.cuda.synchronize()
            for a, b in zip((out, layer.conv_state, layer.recurrent_state), ref):
                assert torch.equal(a, b)
            a = torch.randn(256, 256, device=dev)
            (a @ a).sum().item()
