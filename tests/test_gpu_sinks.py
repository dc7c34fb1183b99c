"""Sinks that weigh nothing (-inf, and the lowest value of the type, whose logarithm to base 2 is out of range) beside one that counts, where a
step of a kernel holds masked keys only: a window, chunks, portions behind cached keys, pages that are not there.  Against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
HEADS, KV = 4, 2
EPS = {torch.float32: 1e-5, torch.float16: 2**-10, torch.bfloat16: 2**-7}


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


def _sink(dtype):
    return torch.tensor([-float("inf"), torch.finfo(dtype).min, 0.5, -float("inf")], dtype=dtype)


def _attend(q, k, v, scale, seen, sink):
    """q [nq, H, D], k / v [nk, KV, D], seen [nq, nk] in fp64."""
    k, v = (t.double().repeat_interleave(q.shape[1] // k.shape[1], 1).transpose(0, 1).contiguous() for t in (k, v))
    s = (torch.matmul(q.double().transpose(0, 1), k.transpose(1, 2)) * scale).masked_fill(~seen, -float("inf"))
    s = torch.cat([s, sink.double()[:, None, None].expand(-1, s.shape[1], 1)], -1)
    return torch.matmul(s.softmax(-1).nan_to_num(0.0)[..., :-1], v).transpose(0, 1)


def _seen(nq, nk, window, chunk):
    pos, key = torch.arange(nq)[:, None] + nk - nq, torch.arange(nk)[None, :]
    first = pos // chunk * chunk if chunk else pos - window + 1 if window else 0 * pos
    return (key <= pos) & (key >= first)


def _close(got, want, dtype):
    # weights of 16 bits (half a unit each), a sum of them and a result of half a unit, at outputs of size one
    torch.testing.assert_close(got.double().cpu(), want, rtol=2 * EPS[dtype], atol=2 * EPS[dtype])


def _inputs(spans, dtype, d, kv=KV):
    g = torch.Generator().manual_seed(d)
    return ([torch.randn(n[i], h, d, generator=g).to(dtype) for n in spans] for i, h in ((0, HEADS), (1, kv), (1, kv)))


def _cu(ns):
    return torch.tensor([0, *torch.tensor(ns).cumsum(0).tolist()], dtype=torch.int32, device=DEV)


def _pages(ks, vs, block, lost=()):
    """Pages in no order; `lost`: places of the table without one."""
    width = max(-(-k.shape[0] // block) for k in ks)
    table = torch.randperm(len(ks) * width, generator=torch.Generator().manual_seed(1)).int().view(len(ks), width)
    kc, vc = (torch.zeros(len(ks) * width, block, *ks[0].shape[1:], dtype=ks[0].dtype) for _ in range(2))
    for s, (k, v) in enumerate(zip(ks, vs)):
        for i in range(-(-k.shape[0] // block)):
            part = slice(i * block, (i + 1) * block)
            kc[table[s, i], :k[part].shape[0]], vc[table[s, i], :k[part].shape[0]] = k[part], v[part]
    for i in lost:
        table[:, i] = -1
    return kc.to(DEV), vc.to(DEV), table.to(DEV)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("spans", [[(150, 150), (65, 65)], [(70, 77), (33, 40)]], ids=["whole", "behind 7 keys"])
@pytest.mark.parametrize("window, chunk", [(0, 0), (9, 0), (40, 0), (0, 32), (0, 50)])
def test_prompts(H, dtype, d, spans, window, chunk):
    qs, ks, vs = _inputs(spans, dtype, d)
    sink = _sink(dtype)
    want = torch.cat([_attend(q, k, v, d ** -0.5, _seen(q.shape[0], k.shape[0], window, chunk), sink) for q, k, v in zip(qs, ks, vs)])
    q, k, v = (torch.cat(t).to(DEV) for t in (qs, ks, vs))
    cq, ck, mq, mk = _cu([a for a, _ in spans]), _cu([b for _, b in spans]), max(a for a, _ in spans), max(b for _, b in spans)
    mask = H.AttnMask(window=window, sink=sink.to(DEV))
    kc, vc, table = _pages(ks, vs, 64)
    for flags in (0, H.MV_PREFILL_TILES):
        _close(H.prefill_varlen(q, k, v, cq, ck, mq, mk, d ** -0.5, flags=flags, chunk=chunk, mask=mask), want, dtype)
        _close(H.prefill_varlen(q, None, None, cq, ck, mq, mk, d ** -0.5, k_cache=kc, v_cache=vc, block_tables=table, flags=flags, chunk=chunk, mask=mask), want, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_the_vector_kernel_and_a_page_that_is_not_there(H, dtype, d):
    spans, lost = [(150, 150), (33, 97)], 0
    qs, ks, vs = _inputs(spans, dtype, d)
    sink, there = _sink(dtype), torch.arange(150) >= 16
    want = torch.cat([_attend(q, k, v, d ** -0.5, _seen(q.shape[0], k.shape[0], 0, 0) & there[:k.shape[0]], sink) for q, k, v in zip(qs, ks, vs)])
    kc, vc, table = _pages(ks, vs, 16, [lost])
    args = (torch.cat(qs).to(DEV), None, None, _cu([a for a, _ in spans]), _cu([b for _, b in spans]), 150, 150, d ** -0.5)
    for flags in (0, H.MV_PREFILL_TILES, H.MV_PREFILL_SIMPLE):
        _close(H.prefill_varlen(*args, k_cache=kc, v_cache=vc, block_tables=table, flags=flags, mask=H.AttnMask(sink=sink.to(DEV))), want, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kv, d", [(1, 64), (2, 64), (4, 64), (1, 128), (2, 128), (4, 128), (2, 256)])
@pytest.mark.parametrize("window, lost", [(0, ()), (5, ()), (90, ()), (0, (0,)), (200, (0, 2))])
def test_decode(H, dtype, kv, d, window, lost):
    lens = [1, 64, 65, 130, 200, 517, 1100]
    if lost:
        lens = lens[2:]
    qs, ks, vs = _inputs([(1, n) for n in lens], dtype, d, kv)
    sink, there = _sink(dtype), torch.ones(max(lens), dtype=torch.bool)
    for i in lost:
        there[i * 64:(i + 1) * 64] = False
    want = torch.cat([_attend(q, k, v, d ** -0.5, _seen(1, k.shape[0], window, 0) & there[:k.shape[0]], sink) for q, k, v in zip(qs, ks, vs)])
    kc, vc, table = _pages(ks, vs, 64, lost)
    q, at, mask = torch.cat(qs).to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV), H.AttnMask(window=window, sink=sink.to(DEV))
    for flags in [0] if dtype == torch.float32 else [0, H.MV_DECODE_VECTOR, H.MV_DECODE_MFMA, H.MV_DECODE_MFMA | H.MV_DECODE_KLDS_ON]:
        _close(H.paged_decode(q, kc, vc, table, at, d ** -0.5, flags=flags, mask=mask), want, dtype)
    for s in range(len(lens)):   # alone: the context in many parts
        _close(H.paged_decode(q[s:s + 1], kc, vc, table[s:s + 1], at[s:s + 1], d ** -0.5, mask=mask), want[s:s + 1], dtype)
