"""GPU: packed attention at head dims the kernels read as they lie (any
multiple of 8, no padded copies) vs the fp64 oracle, with the attention
tests' bars.  k and v are views of one interleaved buffer whose gaps hold NaN
and infinities, so that a piece read past a row's end would show."""
import pytest
import torch

from conftest import assert_out_close
from myvllm_amd import _lib, flash_attention_prefill
from myvllm_amd.full_attention import _direct_head_dim
from myvllm_amd.workloads import attn_varlen_case
from oracle.attention import flash_attention_prefill_ref


def test_direct_head_dim_rule():
    """Rows of a multiple of 8 elements inside their stride go as they lie, the rest is padded."""
    def rule(D, Dv=None, stride=None, T=10, max_seqlen=10):
        t = torch.empty(T, 2, D, dtype=torch.bfloat16)
        kv = t if stride is None else torch.empty(T * max(stride, 1) + 4 * D,
                                                  dtype=torch.bfloat16).as_strided((T, 2, D), (stride, D, 1))
        return _direct_head_dim(t, kv, kv, D, D if Dv is None else Dv, max_seqlen)

    assert rule(72) and rule(8) and rule(248) and rule(72, stride=72)
    assert not rule(72, Dv=64) and not rule(12) and not rule(264) and not rule(0)
    assert not rule(72, stride=64) and not rule(72, stride=0)  # overlapping rows
    assert not rule(72, max_seqlen=2**24)  # past 32-bit offsets


@pytest.mark.parametrize("stride", [64, 0])
def test_any_dim_refuses_overlapping_rows(stride):
    D = _lib.describe
    q = torch.zeros(8, 2, 72, dtype=torch.bfloat16)
    k = D(q)
    k.stride[0] = stride
    cu = torch.tensor([0, 8], dtype=torch.int32)
    rc = _lib.load().flash_attention_varlen_any_dim(D(q), k, D(q), D(cu), D(q), 8, 1.0, 1, None)
    assert rc == _lib.load().flash_attention_varlen_any_dim(D(q), D(q), k, D(cu), D(q), 8, 1.0, 1, None)
    assert "stride" in _lib.strerror(rc).lower()


@pytest.mark.gpu
@pytest.mark.parametrize("Dh", [8, 40, 64 + 8, 80, 88, 96, 104, 120, 136, 200, 248])
@pytest.mark.parametrize("Hq, Hkv, causal, dtype", [(4, 4, False, torch.bfloat16), (8, 2, True, torch.float16)])
def test_any_head_dim(dev, Dh, Hq, Hkv, causal, dtype):
    lengths = [1, 64, 31, 200, 65]
    case = attn_varlen_case(lengths, seed=Dh + Hq, Hq=Hq, Hkv=Hkv, D=Dh, dtype=dtype)
    T = sum(lengths)
    print(f"any head dim {Dh} Hq={Hq} Hkv={Hkv} causal={causal} {dtype}", flush=True)
    ref = flash_attention_prefill_ref(case.q, case.k, case.v, case.cu, case.scale, is_causal=causal)
    # rows of k and v heads apart by gaps of NaN and +-inf, more past the end
    gap = torch.tensor([float("nan"), float("inf"), -float("inf"), 65504.0], dtype=dtype).repeat(4)
    buf = gap.repeat((T + 4) * 2 * Hkv, 1 + Dh // 16 + 1)[:, : Dh + 16].reshape(T + 4, 2 * Hkv, Dh + 16).contiguous()
    buf[:T, :Hkv, :Dh] = case.k
    buf[:T, Hkv:, :Dh] = case.v
    buf = buf.to(dev)
    k, v = buf[:T, :Hkv, :Dh], buf[:T, Hkv:, :Dh]
    out = torch.full((T, Hq, Dh + 8), 7.0, dtype=dtype, device=dev)
    got = flash_attention_prefill(case.q.to(dev), k, v, case.cu.to(dev), case.scale, Hq, Hkv, Dh, Dh, causal,
                                  out=out[..., :Dh])
    assert got.data_ptr() == out.data_ptr() and (out[..., Dh:] == 7.0).all()
    assert_out_close(got, ref)
    err = (got.double().cpu() - ref.double()).norm() / ref.double().norm()
    assert err < 5e-3, f"relative error norm {err:.3e}"


def test_misaligned_contiguous_input_is_copied():
    t = torch.arange(2 * 3 * 8 + 1, dtype=torch.bfloat16)[1:].view(2, 3, 8)
    assert t.is_contiguous() and t.data_ptr() % 16
    c = _lib.vec16(t)
    assert c.data_ptr() % 16 == 0 and torch.equal(c, t)


@pytest.mark.gpu
@pytest.mark.parametrize("Dh", [72, 64])
def test_misaligned_contiguous_rows(dev, Dh):
    """q, k and v contiguous at odd addresses, as views of one flat buffer."""
    case = attn_varlen_case([40, 33], seed=Dh, Hq=4, Hkv=4, D=Dh)
    buf = torch.empty(3 * case.q.numel() + 1, dtype=case.q.dtype, device=dev)
    q, k, v = (buf[1 + i * case.q.numel():][: case.q.numel()].view(case.q.shape).copy_(t)
               for i, t in enumerate((case.q, case.k, case.v)))
    assert q.is_contiguous() and q.data_ptr() % 16
    print(f"misaligned contiguous rows D={Dh}", flush=True)
    got = flash_attention_prefill(q, k, v, case.cu.to(dev), case.scale, 4, 4, Dh, Dh, True)
    assert_out_close(got, flash_attention_prefill_ref(case.q, case.k, case.v, case.cu, case.scale))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["fp32", "host", "q", "k", "v", "shifted"])
def test_out_of_any_kind(dev, kind):
    """An out of another dtype or device, or in an input's memory, takes a copy of the result, as it
    does where the head dim is padded."""
    case = attn_varlen_case([200, 65], seed=9, Hq=4, Hkv=4, D=72)
    q, k, v = (t.to(dev) for t in (case.q, case.k, case.v))
    want = flash_attention_prefill(q, k, v, case.cu.to(dev), case.scale, 4, 4, 72, 72, True)
    buf = torch.empty(k.numel() + 8 * 72, dtype=k.dtype, device=dev)
    if kind == "shifted":
        k = buf[8 * 72:].view(k.shape).copy_(k)
    out = {"fp32": torch.empty_like(q, dtype=torch.float32), "host": torch.empty_like(case.q), "q": q, "k": k, "v": v,
           "shifted": buf[: k.numel()].view(k.shape)}[kind]
    print(f"attention out {kind}", flush=True)
    got = flash_attention_prefill(q, k, v, case.cu.to(dev), case.scale, 4, 4, 72, 72, True, out=out)
    assert got is out and torch.equal(got.to(want.device, want.dtype), want)


@pytest.mark.gpu
# (ranked by length up to 64 sequences, past eight of them a quarter per wave; in index order past 64)
@pytest.mark.parametrize("N", [1, 7, 8, 9, 10, 63, 64, 65])
@pytest.mark.parametrize("Dh", [64, 72, 128])
def test_sequence_order(dev, N, Dh):
    """Ragged batches with empty and equal sequences on both sides of the ranking's limit."""
    lengths = [(37 * n * n + 11) % 150 if n % 7 else 0 for n in range(N)] if N > 1 else [129]
    lengths[N // 2] = lengths[-1] = 33
    case = attn_varlen_case(lengths, seed=N + Dh, Hq=4, Hkv=1, D=Dh)
    print(f"sequence order N={N} D={Dh}", flush=True)
    got = flash_attention_prefill(case.q.to(dev), case.k.to(dev), case.v.to(dev), case.cu.to(dev), case.scale, 4, 1, Dh,
                                  Dh, True)
    assert_out_close(got, flash_attention_prefill_ref(case.q, case.k, case.v, case.cu, case.scale))


@pytest.mark.gpu
@pytest.mark.parametrize("Dh", [64, 40])
@pytest.mark.parametrize(
    "lengths, causal",
    [
        ([257], True), ([256], True),  # 64-key tiles from 257 tokens on
        ([639], True), ([640], True),  # 640 and 768 workgroups: 64 and 32 keys
        ([639], False), ([640], False),
        ([300, 65, 1], True), ([300, 127, 0, 33], False),
    ],
)
def test_key_tiles_of_few_workgroups(dev, Dh, lengths, causal):
    case = attn_varlen_case(lengths, seed=Dh, Hq=128, Hkv=128, D=Dh)
    print(f"few workgroups D={Dh} {lengths} causal={causal}", flush=True)
    got = flash_attention_prefill(case.q.to(dev), case.k.to(dev), case.v.to(dev), case.cu.to(dev), case.scale, 128, 128,
                                  Dh, Dh, causal)
    ref = flash_attention_prefill_ref(case.q, case.k, case.v, case.cu, case.scale, is_causal=causal)
    assert_out_close(got, ref)
    err = (got.double().cpu() - ref.double()).norm() / ref.double().norm()
    assert err < 5e-3, f"relative error norm {err:.3e}"


@pytest.mark.gpu
@pytest.mark.parametrize("Dh, N", [(256, 3), (72, 3), (128, 70), (64, 1)])
@pytest.mark.parametrize("first, tail", [(0, 1), (5, 0), (7, 900)])
def test_uncovered_rows_are_zero(dev, Dh, N, first, tail):
    """Rows before cu[0] and past cu[N], few and many, are zeroed by the workgroups past the last tile."""
    lengths = [33 + (7 * n) % 64 for n in range(N)]
    case = attn_varlen_case(lengths, seed=N + Dh, Hq=4, Hkv=2, D=Dh)
    T = sum(lengths)
    pad = lambda t: torch.cat([torch.full_like(t[:1], 9.0).expand(first, -1, -1), t,  # noqa: E731
                               torch.full_like(t[:1], 9.0).expand(tail, -1, -1)]).contiguous().to(dev)
    cu = (case.cu + first).to(dev)
    out = torch.full((first + T + tail, 4, Dh), 5.0, dtype=case.q.dtype, device=dev)
    print(f"uncovered rows D={Dh} N={N} first={first} tail={tail}", flush=True)
    flash_attention_prefill(pad(case.q), pad(case.k), pad(case.v), cu, case.scale, 4, 2, Dh, Dh, True, out=out)
    assert (out[:first] == 0).all() and (out[first + T:] == 0).all()
    assert_out_close(out[first: first + T], flash_attention_prefill_ref(case.q, case.k, case.v, case.cu, case.scale))
