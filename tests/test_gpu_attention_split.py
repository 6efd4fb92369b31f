"""GPU: the split paged prefill (few new tokens over a long context: the key
range of a row runs as several workgroups) vs the fp64 oracle and vs the
unsplit entry.  Same bars as the attention tests; between the two entries the
outputs differ by the order of fp32 sums and by P rounded against another
base, so they also share the 5e-3 relative norm."""
import random

import pytest
import torch

from conftest import assert_out_close
from myvllm_amd import _lib, paged_flash_attention_prefill
from myvllm_amd.full_attention import _prefill_workspace
from myvllm_amd.workloads import paged_case
from oracle.attention import paged_attention_ref


def _splits(T, N, Hq, Hkv, D, cap):
    f = _lib.load().paged_attention_prefill_workspace_size(T, N, Hq, Hkv, D, cap)
    R = Hq // Hkv
    gh = 4 if R % 4 == 0 else (2 if R % 2 == 0 else 1)
    rows = (T // (32 * (4 // gh)) + N) * (Hq // gh)
    per = rows * 4 * (32 * D + 128)
    assert f % per == 0
    return max(1, f // per)


def test_split_rule():
    """Few rows over long tables are split; full batches, short tables and empty calls are not,
    and the partials stay within 512 MiB."""
    assert _splits(16, 1, 16, 2, 256, 8192) > 8
    assert 1 < _splits(4538, 4, 16, 2, 256, 16832) <= 8
    assert _splits(19041, 16, 16, 2, 256, 6144) == 1
    assert _splits(64, 2, 16, 2, 256, 256) == 1
    for T, N, Hq, Hkv, D, cap in ((0, 1, 16, 2, 256, 8192), (16, 0, 16, 2, 256, 8192), (16, -1, 16, 2, 256, 8192),
                                  (16, 1, 16, 2, 96, 8192), (16, 1, 16, 3, 256, 8192), (16, 1, 16, 2, 256, 0)):
        assert _lib.load().paged_attention_prefill_workspace_size(T, N, Hq, Hkv, D, cap) == 0
    for T in (1, 100, 2000, 30000):
        for cap in (1 << 12, 1 << 20, 1 << 30):
            assert _lib.load().paged_attention_prefill_workspace_size(T, 3, 16, 2, 256, cap) * 4 <= 1 << 29


def _on_host(page=16, block_stride=None):
    """Tensors of a call that is split at pages of 16 (never read)."""
    q = torch.empty(5, 4, 64, dtype=torch.bfloat16)
    kc = torch.empty(1, page, 1, 64, dtype=torch.bfloat16)
    if block_stride:
        kc = kc.as_strided(kc.shape, (block_stride, *kc.stride()[1:]))
    return q, kc, kc, torch.zeros(1, 4096 // page, dtype=torch.int32), torch.tensor([0, 5], dtype=torch.int32), page


def test_workspace_only_where_the_kernel_splits():
    """Pages that are no multiple of 16 and wide block strides take the per-row kernel: no workspace."""
    assert _prefill_workspace(*_on_host()) is not None and _prefill_workspace(*_on_host(page=32)) is not None
    assert _prefill_workspace(*_on_host(page=8)) is None and _prefill_workspace(*_on_host(page=24)) is None
    assert _prefill_workspace(*_on_host(block_stride=2**31)) is None
    assert _prefill_workspace(*_on_host(block_stride=2**31 - 8)) is not None


def test_wrong_ranks_are_left_to_the_entry():
    q, kc, vc, tab, cu, page = _on_host()
    for args in ((q[0], kc, vc, tab, cu), (q, kc[0], vc, tab, cu), (q, kc, vc[0], tab, cu), (q, kc, vc, tab[0], cu),
                 (q, kc, vc, tab, cu[0])):
        assert _prefill_workspace(*args, page) is None


@pytest.mark.gpu
@pytest.mark.parametrize("bad", ["q", "tables", "cu"])
def test_paged_prefill_wrong_rank(dev, bad):
    """Refused by the entry's own error, as a wrong rank is everywhere else."""
    case = paged_case([3000, 40], [5, 40], page=16, seed=3, Hq=16, Hkv=2, D=256)
    d = dict(q=case.q, k=case.k_cache, v=case.v_cache, tables=case.block_tables, ctx=case.context_lens, cu=case.cu)
    d[bad] = d[bad][0]
    d = [t.to(dev) for t in d.values()]
    with pytest.raises(_lib.GdnError, match="dimensions"):
        paged_flash_attention_prefill(*d, None, case.scale, 16, max_seqlen=40)


@pytest.mark.gpu
@pytest.mark.parametrize(
    "ctx, new, page, Hq, Hkv, Dh, dtype, tab64",
    [
        ([4096, 37, 1500], [3, 37, 40], 16, 16, 2, 256, torch.bfloat16, False),  # one row of many pieces, rows of one
        ([2048, 2049, 511], [1, 33, 1], 16, 8, 1, 256, torch.float16, True),  # ends on and past a piece's end
        ([3000, 0, 20], [70, 0, 50], 16, 16, 4, 128, torch.bfloat16, False),  # an empty sequence; queries without keys
        ([5000, 1], [129, 1], 48, 4, 4, 128, torch.bfloat16, True),  # one head per kv head: four query blocks
        ([2500, 700], [31, 90], 32, 8, 4, 64, torch.float16, False),  # two heads per kv head
    ],
)
def test_split_paged_prefill(dev, ctx, new, page, Hq, Hkv, Dh, dtype, tab64):
    case = paged_case(ctx, new, page=page, seed=len(ctx) + page, Hq=Hq, Hkv=Hkv, D=Dh, dtype=dtype)
    assert _splits(sum(new), len(new), Hq, Hkv, Dh, case.block_tables.shape[1] * page) > 1
    tab = case.block_tables.to(torch.int64) if tab64 else case.block_tables
    d = [t.to(dev) for t in (case.q, case.k_cache, case.v_cache, tab, case.context_lens, case.cu)]
    print(f"split paged prefill ctx={ctx} new={new} page={page} Hq={Hq} Hkv={Hkv} D={Dh}", flush=True)
    out = paged_flash_attention_prefill(*d, None, case.scale, page)
    ref = paged_attention_ref(case.q, case.k_cache, case.v_cache, case.block_tables, case.context_lens, case.cu,
                              case.scale).nan_to_num(0.0)  # (a query without keys: 0/0 there, a zero row here)
    assert torch.isfinite(out).all()
    plain = torch.empty_like(out)
    D = _lib.describe
    rc = _lib.load().paged_attention_prefill(*(D(t) for t in d), D(plain), max(new), float(case.scale),
                                             _lib.stream_handle(plain.device))
    _lib.check("paged_attention_prefill", rc)
    for got, want in ((out.cpu(), ref), (out.cpu(), plain.cpu())):
        assert_out_close(got, want)
        err = (got.double() - want.double()).norm() / want.double().norm().clamp_min(1e-12)
        assert err < 5e-3, f"relative error norm {err:.3e}"


@pytest.mark.gpu
@pytest.mark.parametrize("tail", [1, 300])
def test_split_paged_prefill_uncovered_rows(dev, tail):
    case = paged_case([3000, 40], [5, 40], page=16, seed=3, Hq=16, Hkv=2, D=256)
    assert _splits(45 + tail, 2, 16, 2, 256, case.block_tables.shape[1] * 16) > 1
    q = torch.cat([case.q, torch.full_like(case.q[:1], 9.0).expand(tail, -1, -1)]).contiguous()
    out = torch.full_like(q, 5.0).to(dev)
    print(f"split paged prefill, {tail} uncovered rows", flush=True)
    paged_flash_attention_prefill(q.to(dev), case.k_cache.to(dev), case.v_cache.to(dev), case.block_tables.to(dev),
                                  case.context_lens.to(dev), case.cu.to(dev), None, case.scale, 16, out=out)
    assert (out[45:] == 0).all()
    assert_out_close(out[:45], paged_attention_ref(case.q, case.k_cache, case.v_cache, case.block_tables,
                                                   case.context_lens, case.cu, case.scale))


@pytest.mark.gpu
def test_split_paged_prefill_decreasing_offsets(dev):
    """Offsets that decrease give more query tiles than the grid has rows: those past it have no
    place in the workspace, which ends where its size function says."""
    T, N, cap = 256, 5, 4096
    case = paged_case([cap] * N, [T] * N, page=16, seed=5, Hq=16, Hkv=2, D=256)
    n = _lib.load().paged_attention_prefill_workspace_size(T, N, 16, 2, 256, case.block_tables.shape[1] * 16)
    assert n > 0
    guard = 1 << 20
    buf = torch.full((n + guard,), 3.0, device=dev)
    cu = torch.tensor([0, T, 0, T, 0, T], dtype=torch.int32, device=dev)
    q = case.q[:T].to(dev)
    out = torch.empty_like(q)
    print("split paged prefill, decreasing offsets", flush=True)
    _lib.call("paged_attention_prefill_split", q, *(t.to(dev) for t in (case.k_cache, case.v_cache, case.block_tables,
                                                                        case.context_lens)), cu, out, buf[:n], T,
              float(case.scale))
    assert (buf[n:] == 3.0).all()
    assert torch.isfinite(out).all()


@pytest.mark.gpu
def test_paged_prefill_without_room_for_a_workspace(dev, monkeypatch):
    """Where the workspace is not to be had the call runs unsplit, as it needs none."""
    case = paged_case([3000, 40], [5, 40], page=16, seed=3, Hq=16, Hkv=2, D=256)
    d = [t.to(dev) for t in (case.q, case.k_cache, case.v_cache, case.block_tables, case.context_lens, case.cu)]
    plain = torch.empty_like(d[0])
    _lib.call("paged_attention_prefill", *d, plain, 40, float(case.scale))
    real, refused = torch.empty, []

    def empty(*a, **kw):
        if kw.get("dtype") is torch.float32:
            refused.append(a)
            raise torch.OutOfMemoryError("no room")
        return real(*a, **kw)

    monkeypatch.setattr(torch, "empty", empty)
    print("paged prefill, no workspace", flush=True)
    out = paged_flash_attention_prefill(*d, None, case.scale, 16, max_seqlen=40)
    assert refused and torch.equal(out, plain)


def _against_unsplit(d, max_len, scale):
    """The split entry over a marked workspace, and whether it wrote partials; the unsplit one."""
    q, kc, tab = d[0], d[1], d[3]
    n = _lib.load().paged_attention_prefill_workspace_size(q.shape[0], tab.shape[0], q.shape[1], kc.shape[2], q.shape[2],
                                                           tab.shape[1] * kc.shape[1])
    assert n > 0
    ws = torch.full((n + 4096,), 3.0, device=q.device)
    out, plain = torch.full_like(q, 9.0), torch.full_like(q, 9.0)
    _lib.call("paged_attention_prefill_split", *d, out, ws[:n], max_len, scale)
    _lib.call("paged_attention_prefill", *d, plain, max_len, scale)
    assert (ws[n:] == 3.0).all()
    return out, bool((ws[:n] != 3.0).any()), plain


def _close(out, plain):
    assert torch.isfinite(out).all()
    assert_out_close(out, plain)
    err = (out.double() - plain.double()).norm() / plain.double().norm().clamp_min(1e-12)
    assert err < 5e-3, f"relative error norm {err:.3e}"


@pytest.mark.gpu
@pytest.mark.parametrize("Hkv, Dh", [(2, 256), (4, 128), (4, 64)])
@pytest.mark.parametrize(
    "ctx, new, split",
    [
        ([4000, 130, 1500], [3, 40, 40], True),  # pieces of the contexts' lengths, not of the table's
        ([300, 90, 512], [30, 90, 64], False),  # nothing long enough: no partial is written
        ([0, 0, 6000], [0, 5, 1], True),
    ],
)
def test_split_paged_prefill_wide_table(dev, Hkv, Dh, ctx, new, split):
    """Tables 64 times as wide as the longest context (a server's, of its largest length)."""
    case = paged_case(ctx, new, page=16, seed=len(new), Hq=16, Hkv=Hkv, D=Dh)
    tab = torch.full((3, 64 * case.block_tables.shape[1]), -1, dtype=torch.int32)
    tab[:, : case.block_tables.shape[1]] = case.block_tables
    d = [t.to(dev) for t in (case.q, case.k_cache, case.v_cache, tab, case.context_lens, case.cu)]
    print(f"wide table D={Dh} ctx={ctx}", flush=True)
    out, wrote, plain = _against_unsplit(d, max(new), float(case.scale))
    assert wrote == split
    _close(out, plain)
    _close(out.cpu(), paged_attention_ref(case.q, case.k_cache, case.v_cache, case.block_tables, case.context_lens,
                                          case.cu, case.scale).nan_to_num(0.0))


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(16))
def test_split_paged_prefill_batches(dev, seed):
    """Batches of every kind against the unsplit entry: 1 to 150 sequences (more than a wave's lanes),
    empty ones, contexts shorter than their new tokens, tables tight and wide, either index type."""
    r = random.Random(seed)
    N = r.choice([1, 2, 5, 63, 64, 65, 150])
    Hq, Hkv, Dh = r.choice([(4, 1, 256), (4, 1, 128), (4, 1, 64)] if N > 5 else
                           [(16, 2, 256), (4, 1, 256), (16, 4, 128), (4, 4, 128), (8, 2, 64)])
    new = [r.choice([0, 1, 33, r.randint(1, 100)]) if N > 5 else r.randint(1, 300) for _ in range(N)]
    new[0] = max(new[0], 1)
    ctx = [max(0, n + r.choice([0, -5, r.randint(0, 300), r.randint(1500, 5000) if r.random() < 0.4 else 16]))
           for n in new]
    ctx[r.randrange(N)] = 6000
    case = paged_case([max(c, n) for c, n in zip(ctx, new)], new, page=r.choice([16, 48]), seed=seed, Hq=Hq, Hkv=Hkv,
                      D=Dh, dtype=r.choice([torch.bfloat16, torch.float16]))
    tab = torch.nn.functional.pad(case.block_tables, (0, r.choice([0, 200, 3000])), value=-1)
    wide = r.choice([torch.int32, torch.int64])
    d = [t.to(dev) for t in (case.q, case.k_cache, case.v_cache, tab.to(wide), torch.tensor(ctx, dtype=wide),
                             case.cu.to(r.choice([torch.int32, torch.int64])))]
    print(f"split batch {seed}: N={N} Hq={Hq} Hkv={Hkv} D={Dh} {int(case.cu[-1])} tokens", flush=True)
    out, _, plain = _against_unsplit(d, max(new), float(case.scale))
    _close(out, plain)
