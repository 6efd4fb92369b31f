"""The split chunked prefill (few sequences: all chunks prepared at once, then
each item walked by several workgroups) vs the fp64 oracle, with the fused
kernel's bars, and its dispatch rule."""
import pytest
import torch

from conftest import assert_out_close, assert_state_close
from myvllm_amd import _lib, chunk_gated_delta_rule
from myvllm_amd.gated_delta_rule import chunk_prefill_ex
from myvllm_amd.workloads import prefill_case
from oracle.gdn import chunk_gated_delta_rule_ref


def _floats(T, N, Hk, Hv, K=128, V=128):
    return _lib.load().gdn_chunk_prefill_workspace_size(T, N, Hk, Hv, K, V)


def test_split_rule():
    """Few items with many chunks each are split, within 1 GiB of records; the rest is not."""
    assert _floats(192, 1, 16, 32) > 0 and _floats(191, 1, 16, 32) == 0
    assert _floats(512, 2, 16, 32) > 0 and _floats(511, 2, 16, 32) == 0
    assert _floats(30000, 3, 16, 32) == 0 and _floats(40000, 64, 1, 1) > 0 and _floats(40000, 65, 1, 1) == 0
    for args in ((0, 1, 16, 32), (-5, 1, 16, 32), (400, 0, 16, 32), (400, -1, 16, 32), (400, 1, 0, 32), (400, 1, 3, 32),
                 (400, 1, 16, 32, 64, 128), (400, 1, 16, 32, 128, 64), (2**31, 1, 16, 32)):
        assert _floats(*args) == 0, args
    for T in (384, 4096, 16384, 65536, 2**31 - 1):
        assert _floats(T, 1, 16, 32) * 4 <= 2**30


def _case(lengths, Hk=2, Hv=4, **kw):
    return prefill_case(lengths, seed=sum(lengths) % 97, num_slots=len(lengths) + 3, Hk=Hk, Hv=Hv, **kw)


@pytest.mark.parametrize("bad, code", [("short", -3), ("bf16", -4), ("align", -9)])
def test_split_workspace_checks(bad, code):
    """A workspace that does not fit is refused before anything is launched (all pointers here are the host's)."""
    c = _case([400])
    n = _floats(400, 1, 2, 4)
    ws = {"short": lambda: torch.empty(n - 1), "bf16": lambda: torch.empty(n, dtype=torch.bfloat16),
          "align": lambda: torch.empty(n + 1)[1:]}[bad]()
    D = _lib.describe
    rc = _lib.load().gdn_chunk_prefill_split(D(c.q), D(c.k), D(c.v), D(c.g), D(c.beta), D(c.state), D(c.idx), D(c.cu),
                                             D(torch.empty_like(c.v)), D(ws), 1.0, 64, None)
    assert rc == code


@pytest.mark.gpu
@pytest.mark.parametrize(
    "lengths, Hk, Hv, dtype, g_scale",
    [
        ([192], 2, 4, torch.bfloat16, 1.0),  # whole chunks
        ([384], 2, 4, torch.float16, 1.0),  # an even number of them
        ([449], 1, 1, torch.bfloat16, 1.0),  # one token past a chunk, an odd number of chunks
        ([1100, 1, 64], 2, 4, torch.float16, 1.0),  # sequences of one chunk beside a long one
        ([600, 0, 900, 63, 1000], 2, 8, torch.bfloat16, 0.05),  # 40 items: two column groups per workgroup; weak decay
        ([1030] + [500] * 15, 1, 4, torch.float16, 20.0),  # 64 items; decays past the factored range
        ([700], 16, 32, torch.bfloat16, 0.0),  # no decay
    ],
)
def test_split_prefill(dev, lengths, Hk, Hv, dtype, g_scale):
    c = _case(lengths, Hk, Hv, dtype=dtype, g_scale=g_scale)
    T = sum(lengths)
    assert _floats(T, len(lengths), Hk, Hv) > 0
    print(f"split prefill {lengths} Hk={Hk} Hv={Hv} {dtype} g_scale={g_scale}", flush=True)
    st_ref = c.state.clone()
    o_ref = chunk_gated_delta_rule_ref(c.q, c.k, c.v, c.g, c.beta, st_ref, c.idx, c.cu)
    st = c.state.to(dev)
    d = [t.to(dev) for t in (c.q, c.k, c.v, c.g, c.beta)]
    o = chunk_gated_delta_rule(*d, st, c.idx.to(dev), c.cu.to(dev))
    assert_out_close(o, o_ref)
    sel = c.idx.long()
    assert_state_close(st.cpu()[sel], st_ref[sel])
    rest = torch.ones(len(st_ref), dtype=torch.bool)
    rest[sel] = False
    assert torch.equal(st.cpu()[rest], c.state[rest])
    # not further from the oracle than the fused kernel, beyond the noise of either's roundings
    st2, o2 = c.state.to(dev), torch.empty_like(o)
    chunk_prefill_ex(*d, st2, c.idx.to(dev), c.cu.to(dev), o2, 128 ** -0.5)
    err = lambda x: (x.cpu()[sel].double() - st_ref[sel].double()).norm() / st_ref[sel].double().norm()  # noqa: E731
    assert err(st) < 1.5 * err(st2) + 1e-8, (err(st), err(st2))


@pytest.mark.gpu
def test_split_prefill_padding_strides_and_graph(dev):
    """Padding slots, int64 indices, uncovered rows, strided views and a captured graph replayed on new inputs."""
    lengths = [500, 300, 700]
    c = _case(lengths)
    T = sum(lengths) + 9  # nine rows no sequence covers
    big = torch.zeros(T, 2 * 2 + 4, 128, dtype=torch.bfloat16)
    big[: T - 9, :2], big[: T - 9, 2:4], big[: T - 9, 4:] = c.q, c.k, c.v
    g, beta = torch.zeros(T, 4), torch.zeros(T, 4, dtype=torch.bfloat16)
    g[: T - 9], beta[: T - 9] = c.g, c.beta
    idx = c.idx.to(torch.int64)
    idx[1] = -1
    cu = c.cu.to(torch.int64)
    dbig, dg, dbeta, st, didx, dcu = (t.to(dev) for t in (big, g, beta, c.state, idx, cu))
    out = torch.full((T, 4, 128), 5.0, dtype=torch.bfloat16, device=dev)
    args = (dbig[:, :2], dbig[:, 2:4], dbig[:, 4:], dg, dbeta, st, didx, dcu)
    chunk_gated_delta_rule(*args, out=out)  # (warm: the library is loaded outside the capture)
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr):
        chunk_gated_delta_rule(*args, out=out)
    for rep in range(3):
        dbig.copy_(big.roll(rep, 0))
        st.copy_(c.state)
        out.fill_(5.0)
        print(f"split prefill replay {rep}", flush=True)
        gr.replay()
        torch.cuda.synchronize()
        b = big.roll(rep, 0)
        st_ref = c.state.clone()
        o_ref = chunk_gated_delta_rule_ref(b[:, :2], b[:, 2:4], b[:, 4:], g, beta.float(), st_ref, idx, cu)
        o_ref[500:800] = 0
        o_ref[T - 9:] = 0
        assert_out_close(out, o_ref)
        assert (out[500:800] == 0).all() and (out[T - 9:] == 0).all()
        assert_state_close(st, st_ref)


@pytest.mark.gpu
@pytest.mark.parametrize("lengths, Hk, Hv", [([200, 333], 2, 4), ([450, 700, 64], 4, 16)])
def test_split_prefill_fp32(dev, lengths, Hk, Hv):
    """fp32 q, k, v: both passes (v hi from the slot's state, v lo added from zero) run split, with
    a padding sequence and an uncovered row; against the fused kernel's passes on the same inputs."""
    c = _case(lengths, Hk, Hv, dtype=torch.float32)
    T = sum(lengths)
    assert _floats(T + 1, len(lengths), Hk, Hv) > 0
    pad = lambda t: torch.cat([t, t[:1]]).contiguous().to(dev)  # noqa: E731
    d = [pad(t) for t in (c.q, c.k, c.v, c.g, c.beta)]
    idx = c.idx.clone()
    idx[-1] = -1
    print(f"split prefill fp32 {lengths} Hk={Hk} Hv={Hv}", flush=True)
    st = c.state.to(dev)
    o = chunk_gated_delta_rule(*d, st, idx.to(dev), c.cu.to(dev), out=torch.full_like(d[2], 7.0))
    assert o.dtype == torch.float32 and (o[T:] == 0).all() and (o[T - lengths[-1]: T] == 0).all()
    st2, o2 = c.state.to(dev), torch.full_like(d[2], 7.0)
    qh, kh, vh = d[0].half(), d[1].half(), d[2].half()
    args = (d[3], d[4], st2, idx.to(dev), c.cu.to(dev), o2, 128 ** -0.5)
    chunk_prefill_ex(qh, kh, vh, *args)
    chunk_prefill_ex(qh, kh, (d[2] - vh.float()).half(), *args,
                     flags=_lib.PREFILL_ZERO_INIT | _lib.PREFILL_ACCUM_STATE | _lib.PREFILL_ACCUM_OUT)
    # (the splits of either keep 22 bits; P and the hi parts that feed o only keep 11)
    assert (st - st2).norm() < 3e-6 * st2.norm()
    assert (o - o2).norm() < 2e-3 * o2.norm()
    st_ref = c.state.clone()
    o_ref = chunk_gated_delta_rule_ref(c.q, c.k, c.v, c.g, c.beta, st_ref, idx, c.cu)
    assert_out_close(o[:T], o_ref, rtol=2e-3, atol=1e-3)


@pytest.mark.gpu
def test_split_prefill_fp32_largest_token_stride(dev):
    """fp32 rows 2^24 elements apart, the largest stride the entry takes (13 GB of rows): 64 of
    them are 2^32 bytes.  Bit for bit the result of contiguous rows."""
    c = _case([200], Hk=1, Hv=2, dtype=torch.float32)
    assert _floats(200, 1, 1, 2) > 0
    d = [t.to(dev) for t in (c.q, c.k, c.v, c.g, c.beta)]
    print("split prefill fp32, token stride 2^24", flush=True)
    outs = []
    for out in (None, torch.empty(199 * 2**24 + 256, device=dev).as_strided((200, 2, 128), (2**24, 128, 1))):
        st = c.state.to(dev)
        if out is not None:
            out.fill_(7.0)
        outs.append((chunk_gated_delta_rule(*d, st, c.idx.to(dev), c.cu.to(dev), out=out).clone(), st))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
