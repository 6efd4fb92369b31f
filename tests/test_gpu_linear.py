"""The linear kernel of a few tokens vs fp64 (one rounding of the output's type
after fp32 sums: relative error norm below 2^-8 / sqrt(3) for bf16, 2^-11 /
sqrt(3) for fp16, with room for the sums), its refusals, and the decode step's
fused gated norm vs the separate ops."""
import pytest
import torch

from conftest import assert_out_close, assert_state_close
from myvllm_amd import _lib, gated_delta_net_decode_step
from myvllm_amd.layer import _linear, _own_linear
from myvllm_amd.norm import rms_norm_gated


def test_own_linear_rule():
    assert _own_linear(1, 12352, 2048) and _own_linear(7, 12352, 2048) and not _own_linear(8, 12352, 2048)
    assert _own_linear(16, 2048, 4096) and not _own_linear(17, 64, 256) and not _own_linear(0, 64, 256)
    assert not _own_linear(1, 64, 128) and not _own_linear(1, 62, 256) and not _own_linear(1, 64, 0)


def test_misaligned_operands_are_not_copied(monkeypatch):
    """A weight the kernel cannot read goes to torch's product as it lies: the test of its alignment copies nothing."""
    x = torch.ones(1, 256, dtype=torch.bfloat16)
    w = torch.ones(64 * 256 + 1, dtype=torch.bfloat16)[1:].view(64, 256)
    assert w.data_ptr() % 16 and _own_linear(1, 64, 256)
    monkeypatch.setattr(torch.Tensor, "contiguous", lambda *a, **kw: pytest.fail("copied"))
    assert not _lib.vec16_ok(w) and not _lib.vec16_ok(x.t()) and _lib.vec16_ok(x)
    assert (_linear(x, w) == 256).all()


@pytest.mark.parametrize(
    "M, N, K, code",
    [(17, 64, 256, -11), (2, 64, 128, -3), (2, 64, 0, -3)],
)
def test_linear_refusals(M, N, K, code):
    D = _lib.describe
    x, w, o = (torch.zeros(a, b, dtype=torch.bfloat16) for a, b in ((M, K), (N, K), (M, N)))
    assert _lib.load().gdn_linear(D(x), D(w), D(o), None) == code
    if code == -11:
        x, o = x[:2], o[:2]
        f = _lib.load().gdn_linear
        assert f(D(x), D(w[:, :128]), D(o), None) == -3 and f(D(x.float()), D(w), D(o), None) == -4
        assert f(D(x), D(torch.zeros(K, N, dtype=torch.bfloat16).t()), D(o), None) == -5
        assert f(D(x), D(torch.zeros(N, K + 1, dtype=torch.bfloat16)[:, 1:]), D(o), None) == -9


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 2, 15, 16])
@pytest.mark.parametrize(
    "N, K, dtype",
    [(16, 256, torch.bfloat16), (100, 768, torch.float16), (12352, 2048, torch.bfloat16), (36, 4352, torch.bfloat16)],
)
def test_linear(dev, M, N, K, dtype):
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=gen).to(dtype).to(dev)[:, :K]  # (rows apart)
    w = torch.randn(N + 1, K, generator=gen).to(dtype).to(dev)[:N]
    out = torch.full((M + 1, N + 4), 3.0, dtype=dtype, device=dev)
    print(f"linear M={M} N={N} K={K} {dtype}", flush=True)
    _lib.call("gdn_linear", x, w, out[:M, :N])
    ref = x.double().cpu() @ w.double().cpu().t()
    err = (out[:M, :N].double().cpu() - ref).norm() / ref.norm()
    assert err < (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) / 1.73, err
    assert (out[M:] == 3.0).all() and (out[:, N:] == 3.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("Hk, Hv, dtype", [(2, 2, torch.bfloat16), (2, 4, torch.bfloat16), (1, 4, torch.float16)])
def test_decode_step_with_norm(dev, Hk, Hv, dtype):
    """Same states as the step without the norm, and its fp32 output normed (the separate
    ops round o to 16 bits in between: half a unit in the last place more)."""
    B, D = 5, (2 * Hk + Hv) * 128
    gen = torch.Generator().manual_seed(Hk + Hv)
    r = lambda *s: torch.randn(*s, generator=gen)  # noqa: E731
    proj = r(B, D + Hv * 128 + 2 * Hv).to(dtype).to(dev)
    conv_w, A, dt, nw = r(D, 4).to(dev), r(Hv).to(dev), r(Hv).to(dev), (1 + 0.1 * r(128)).to(dev)
    cs0, st0 = r(B + 2, 3, D).to(dtype), r(B + 2, Hv, 128, 128) * 0.1
    idx = torch.tensor([3, -1, 0, 6, 1], dtype=torch.int32, device=dev)
    z = proj[:, D: D + Hv * 128].view(B, Hv, 128)
    b, a = proj[:, -2 * Hv: -Hv], proj[:, -Hv:]
    cs, st = cs0.to(dev), st0.to(dev)
    o = gated_delta_net_decode_step(proj[:, :D], conv_w, cs, idx, a, b, A, dt, st, idx, Hk)
    want = rms_norm_gated(o, z, nw, 1e-6)
    cs2, st2, got = cs0.to(dev), st0.to(dev), torch.empty_like(o)
    print(f"decode step with norm Hk={Hk} Hv={Hv} {dtype}", flush=True)
    _lib.call("gdn_decode_step_fused_norm", proj[:, :D], conv_w, cs2, idx, a, b, A, dt, st2, idx, z, nw, got, Hk,
              128 ** -0.5, 1e-6)
    assert torch.equal(cs, cs2) and torch.equal(st, st2)
    assert (got[1] == 0).all()
    assert_out_close(got, want)
    assert_state_close(st2, st)
    err = (got.double() - want.double()).norm() / want.double().norm()
    assert err < (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11), err
