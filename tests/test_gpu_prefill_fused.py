"""GPU: the fused chunked prefill (gdn_chunk_prefill_ex: one workgroup walks an
item's chunks) on the inputs that stress its carried units and bounds.  The
same batches through chunk_gated_delta_rule run split, having few sequences."""
import pytest
import torch

from conftest import assert_out_close, assert_state_close
from myvllm_amd import _lib
from myvllm_amd.workloads import prefill_case
from test_gpu_prefill import _check, _run

pytestmark = pytest.mark.gpu


def _fused(case, dev):
    T, Hk, K = case.q.shape
    assert _lib.load().gdn_chunk_prefill_workspace_size(T, case.cu.numel() - 1, Hk, case.v.shape[1], K, K) > 0
    return _run(case, dev, items_per_wg=-1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_fused_prefill_long_no_decay(dev, dtype):
    """64 chunks with g = 0: the per-column units and bound are carried through all of them (the bound
    is exact every 16 chunks)."""
    case = prefill_case([4096], seed=15, num_slots=1, Hk=1, Hv=2, dtype=dtype)
    case.g.zero_()
    print(f"fused prefill, no decay, {dtype}", flush=True)
    _check(case, *_fused(case, dev))


@pytest.mark.parametrize("g_scale", [0.01, 0.05, 1.6, 4.0])
def test_fused_prefill_decay(dev, g_scale):
    """Weak decays, and strong ones past the factored range."""
    case = prefill_case([400, 1000, 200], seed=14, num_slots=3, Hk=2, Hv=4, g_scale=g_scale)
    print(f"fused prefill, g_scale {g_scale}", flush=True)
    _check(case, *_fused(case, dev))


def test_fused_prefill_zero_decay_beta_one(dev):
    case = prefill_case([256], seed=9, num_slots=1, Hk=1, Hv=2)
    case.g.zero_()
    case.beta.fill_(1.0)
    print("fused prefill, beta one", flush=True)
    _check(case, *_fused(case, dev))


@pytest.mark.parametrize("rho, spiky", [(1.0, False), (8.0, False), (64.0, False), (128.0, False), (8.0, True),
                                        (128.0, True)])
def test_fused_prefill_key_magnitudes(dev, rho, spiky):
    """Keys of norm rho, in random directions or with their mass in one coordinate, over many chunks;
    beta divided by |k|^2, outputs and states in units of 1 / |k| (as test_prefill_key_magnitudes)."""
    case = prefill_case([700, 300, 200], seed=21, num_slots=4, Hk=2, Hv=4, g_scale=0.05)
    gen = torch.Generator().manual_seed(22)
    k = torch.nn.functional.normalize(torch.randn(case.k.shape, generator=gen), dim=-1)
    if spiky:
        k = k * 0.05
        k.scatter_(-1, torch.randint(0, k.shape[-1], k.shape[:2], generator=gen)[..., None], 1.0)
        k = torch.nn.functional.normalize(k, dim=-1)
    case.k = (k * rho).to(torch.bfloat16)
    case.beta = case.beta / case.k.float().pow(2).sum(-1).amax().item()
    case.state.mul_(1.0 / rho)
    print(f"fused prefill, keys of norm {rho} spiky={spiky}", flush=True)
    o, st, o_ref, st_ref = _fused(case, dev)
    assert_out_close(o.double() * rho, o_ref.double() * rho)
    sel = case.idx.long()
    assert_state_close(st[sel].double() * rho, st_ref[sel].double() * rho)
