"""fp32 prefill attention on the matrix cores (csrc/prefill_f32.hip) against 64 bits and the vector kernel: edges of its tiles of 32 keys and
64 queries, every mask, pages with holes, values that are not finite."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def H():
    from minivllm_amd import hip_ops

    return hip_ops


@pytest.fixture(autouse=True)
def tiles(H, monkeypatch):
    monkeypatch.setattr(H, "PREFILL_FLAGS", H.MV_PREFILL_TILES)      # (also where the vector kernel is the quicker)


def _attend(q, k, v, scale, seen, cap=0.0, sink=None):
    """q [nq, H, D], k / v [nk, Hkv, D], seen [nq, nk] in fp64."""
    g = q.shape[1] // k.shape[1]
    s = torch.einsum("qhd,khd->hqk", q.double(), k.double().repeat_interleave(g, 1)) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    s = s.masked_fill(~seen, -float("inf"))
    if sink is not None:
        s = torch.cat([s, sink.double()[:, None, None].expand(-1, s.shape[1], 1)], -1)
    p = s.softmax(-1).nan_to_num(0.0)[..., :k.shape[0]]      # (no key at all: zeros)
    return torch.einsum("hqk,khd->qhd", p, v.double().repeat_interleave(g, 1))


def _mask(nq, nk, window=0, keep=0, chunk=0):
    pos, key = torch.arange(nq)[:, None] + nk - nq, torch.arange(nk)[None, :]
    first = pos.clamp(min=0) // chunk * chunk if chunk else (pos - window + 1 if window else torch.zeros_like(pos))
    return (key <= pos) & ((key >= first) | (key < (keep if window else 0)))


def _check(H, monkeypatch, spans, heads, kv, d, seed, window=0, keep=0, chunk=0, cap=0.0, sink=False, gate=False, block=0, holes=False):
    """spans: [(queries, keys)] of the sequences."""
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g)
    qs, ks, vs = ([rand(n, h, d) for n in ns] for ns, h in (([a for a, _ in spans], heads), ([b for _, b in spans], kv), ([b for _, b in spans], kv)))
    sinks, gates = rand(heads) if sink else None, rand(sum(a for a, _ in spans), heads * d) if gate else None
    cu = lambda ns: torch.tensor([0, *torch.tensor(ns).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    cq, ck, mq, mk = cu([a for a, _ in spans]), cu([b for _, b in spans]), max(a for a, _ in spans), max(b for _, b in spans)
    mask = H.AttnMask(window, keep, cap, 0.7 if gate else 1.0, None if sinks is None else sinks.to(DEV), None if gates is None else gates.to(DEV))
    kw, lost = {}, [torch.zeros(b, dtype=torch.bool) for _, b in spans]
    k, v = torch.cat(ks).to(DEV), torch.cat(vs).to(DEV)
    if block:
        pages = [-(-b // block) for _, b in spans]
        order, width = torch.randperm(sum(pages), generator=g).tolist(), max(pages)
        kc, vc = (torch.full((sum(pages) + 1, block, kv, d), float("nan"), device=DEV) for _ in range(2))
        table = torch.full((len(spans), width), -1, dtype=torch.int32)
        for i, (_, b) in enumerate(spans):
            for j in range(pages[i]):
                at, lo = order.pop(), j * block
                table[i, j] = at
                kc[at, :min(block, b - lo)], vc[at, :min(block, b - lo)] = ks[i][lo:lo + block].to(DEV), vs[i][lo:lo + block].to(DEV)
                if holes and j == 1:
                    table[i, j], lost[i][lo:lo + block] = -1, True
        kw, k, v = dict(k_cache=kc, v_cache=vc, block_tables=table.to(DEV)), None, None
    call = lambda: H.prefill_varlen(torch.cat(qs).to(DEV), k, v, cq, ck, mq, mk, d ** -0.5, chunk=chunk, mask=mask, **kw).cpu()
    got = call()
    with monkeypatch.context() as m:
        m.setattr(H, "PREFILL_FLAGS", H.MV_PREFILL_SIMPLE)
        other = call()
    want = torch.cat([_attend(a, b, c, d ** -0.5, _mask(a.shape[0], b.shape[0], window, keep, chunk) & ~l, cap, sinks)
                      for a, b, c, l in zip(qs, ks, vs, lost)])
    if gate:
        want = want * 0.7 * torch.sigmoid(gates.double()).unflatten(1, (heads, d))
    # sums of at most 300 products of 24 bits: a few 1e-6 of outputs of order one
    torch.testing.assert_close(got.double(), want, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(got, other, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("lens", [[1], [31, 32, 33], [63, 64, 65, 1], [128, 7, 200], [96, 97]], ids=str)
def test_whole_prompts_at_the_edges_of_tiles(H, monkeypatch, lens, d):
    _check(H, monkeypatch, [(n, n) for n in lens], 6, 2, d, sum(lens))


def test_many_prompts_at_the_edges_of_tiles(H, monkeypatch):
    """Enough of them for workgroups of 128 queries (those of 64: above)."""
    _check(H, monkeypatch, [(n, n) for n in [31, 32, 33, 63, 64, 65, 1, 95, 96, 97, 127, 128, 129, 255, 256, 257]], 32, 8, 64, 11)
    _check(H, monkeypatch, [(n, n) for n in [5, 128, 90] * 9], 32, 32, 64, 12, sink=True, gate=True)


@pytest.mark.parametrize("e", [47, 49, 55])
def test_large_scores(H, e):
    """Products of some +-2^96 .. 2^110: a row of one key is that key's value, whatever its score, down to the -1e30 of both kernels."""
    n = 130
    q, k, v = (torch.randn(n, 4, 64, generator=torch.Generator().manual_seed(i)).to(DEV) for i in range(3))
    q[0], k[0] = q[0].abs(), -k[0].abs()
    q, k = q * 2.0 ** e, k * 2.0 ** e
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    call = lambda flags: H.prefill_varlen(q, k, v, cu, cu, n, n, 0.0078125, flags=flags)
    got, want = call(H.MV_PREFILL_TILES), call(H.MV_PREFILL_SIMPLE)
    # (the largest score has all of the weight: values themselves, where two scores do not meet in their last bits)
    assert torch.equal(got[0], want[0]) and (e > 50 or torch.equal(got[0], v[0])) and ((got - want).abs().amax((1, 2)) < 1e-4).float().mean() > 0.95


@pytest.mark.parametrize("tokens, prompts, heads, d, tiles", [(8, 1, 12, 64, False), (40, 1, 12, 64, False), (65, 1, 12, 64, True), (80, 1, 12, 64, True), (65, 2, 32, 64, True),
                                                              (69, 4, 12, 64, True), (8, 64, 32, 64, False), (40, 1, 12, 128, False), (128, 1, 12, 128, True)])
def test_which_kernel_is_taken(H, tokens, prompts, heads, d, tiles):
    """The quicker one by the rule: few tokens key by key, a second tile of 64 keys by tiles."""
    q, k, v = (torch.randn(tokens * prompts, heads, d, generator=torch.Generator().manual_seed(i)).to(DEV) for i in range(3))
    cu = torch.arange(0, tokens * prompts + 1, tokens, dtype=torch.int32, device=DEV)
    call = lambda flags: H.prefill_varlen(q, k, v, cu, cu, tokens, tokens, d ** -0.5, flags=flags)
    by_tiles, by_keys = call(H.MV_PREFILL_TILES), call(H.MV_PREFILL_SIMPLE)
    assert not torch.equal(by_tiles, by_keys) and torch.equal(call(0), by_tiles if tiles else by_keys)


@pytest.mark.parametrize("kw", [dict(sink=True), dict(gate=True), dict(sink=True, gate=True)], ids=str)
def test_sinks_and_gates_of_whole_prompts(H, monkeypatch, kw):
    _check(H, monkeypatch, [(150, 150), (20, 20), (65, 65)], 4, 2, 64, 13, **kw)


@pytest.mark.parametrize("heads", [2, 400])      # workgroups of 64 queries, of 128
@pytest.mark.parametrize("what, at, value", [(0, 30, float("inf")), (0, 99, float("nan")), (1, 45, float("inf")), (1, 45, -float("inf")), (1, 0, float("nan")), (1, 64, 3.4e38),
                                             (0, 3, 3.4e38), (2, 70, 3.4e38), (2, 70, -float("inf"))], ids=str)
def test_numbers_that_have_no_parts(H, heads, what, at, value):
    """Infinities, NaN and numbers that bf16 rounds to infinity in q, k or v: as the vector kernel makes of them (its rows are what they go to)."""
    n = 200
    rows = [torch.randn(n, heads, 64, generator=torch.Generator().manual_seed(i)).to(DEV) for i in range(3)]
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    call = lambda flags: H.prefill_varlen(*rows, cu, cu, n, n, 0.125, flags=flags)
    before = call(H.MV_PREFILL_TILES)
    rows[what][at, 1, 5] = value
    got, want = call(H.MV_PREFILL_TILES), call(H.MV_PREFILL_SIMPLE)
    torch.testing.assert_close(got, want, rtol=1e-5, atol=1e-5, equal_nan=True)
    assert torch.equal(got[:, 0], before[:, 0])      # (the other heads' are not touched)


@pytest.mark.parametrize("heads", [2, 400])      # workgroups of 64 queries, of 128
@pytest.mark.parametrize("eq, ek, ev, gap", [(0, 0, -118, 0), (0, 0, -124, 0), (118, -121, 0, 0), (-121, 118, 0, 0), (90, -120, 0, 0), (100, -102, 0, 0), (-101, 99, 0, 0), (0, 0, 84, 0), (0, 0, -100, 110), (0, 0, 80, 122), (0, 0, 40, 122)], ids=str)
def test_small_numbers_keep_their_bits(H, heads, eq, ek, ev, gap):
    """q, k, v or probabilities below the numbers that three of bf16 add up to: as exact as ordinary ones.  ``gap``: key 0, whose values are zeros, is
    so many powers of two ahead of the others."""
    n = 200
    q, k, v = (torch.randn(n, heads, 64, generator=torch.Generator().manual_seed(i)) for i in range(3))
    if gap:
        q[..., 0], k[:, :, 0], k[0], v[0] = 8 * gap * 0.6931471805599453, 0.0, 0.0, 0.0
        k /= 8      # (no probability below 2^-126, which fp32's exponential has not)
        k[0, :, 0] = 1.0
    q, k, v = (x * 2.0 ** e for x, e in ((q, eq), (k, ek), (v, ev)))
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    got = H.prefill_varlen(*(x.to(DEV) for x in (q, k, v)), cu, cu, n, n, 0.125, flags=H.MV_PREFILL_TILES).cpu().double()
    some = slice(0, heads, max(1, heads // 4))
    want = _attend(q[:, some], k[:, some], v[:, some], 0.125, _mask(n, n))
    # sums of at most 200 products of 24 bits, by the size of a row's outputs; an exponent of `gap` has an error of some 2^-24 of it
    # (five roundings); numbers below 2^-126 are rounded at 2^-149
    bound = (1e-5 + gap * 5 * 2.0 ** -24) * want.abs().amax(-1, keepdim=True) + 2.0 ** -146
    assert ((got[:, some] - want).abs() <= bound).all()


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kw", [dict(window=1), dict(window=40, keep=3), dict(window=33, keep=70), dict(chunk=32), dict(chunk=50), dict(cap=2.0),
                                dict(sink=True), dict(gate=True), dict(window=64, keep=5, cap=3.0, sink=True, gate=True)], ids=str)
def test_masks(H, monkeypatch, kw, d):
    _check(H, monkeypatch, [(150, 150), (20, 20), (65, 65)], 4, 4, d, 3, **kw)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("block", [1, 16, 24, 64])
@pytest.mark.parametrize("kw", [{}, dict(window=30, keep=2), dict(chunk=40), dict(sink=True, holes=True)], ids=str)
def test_portions_over_pages(H, monkeypatch, block, kw, d):
    _check(H, monkeypatch, [(5, 130), (64, 64), (1, 33), (33, 97)], 4, 2, d, 5, block=block, **kw)


def test_more_queries_than_keys(H, monkeypatch):
    _check(H, monkeypatch, [(70, 40), (3, 3)], 2, 1, 64, 9)      # the first queries see no key: zeros


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("d", [64, 128])
def test_values_that_are_not_finite_reach_only_those_who_see_them(H, bad, d):
    n, at = 100, 45
    q, k, v = (torch.randn(n, 2, d, generator=torch.Generator().manual_seed(i)) for i in range(3))
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    want = H.prefill_varlen(q.to(DEV), k.to(DEV), v.to(DEV), cu, cu, n, n, d ** -0.5)
    v[at, 1, 3] = bad
    got = H.prefill_varlen(q.to(DEV), k.to(DEV), v.to(DEV), cu, cu, n, n, d ** -0.5)
    hit = torch.zeros(n, 2, d, dtype=torch.bool, device=DEV)
    hit[at:, 1, 3] = True
    assert not torch.isfinite(got[hit]).any()
    torch.testing.assert_close(got[~hit], want[~hit], rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("scale", [None, -0.05, 0.0])
@pytest.mark.parametrize("d", [64, 128])
def test_factors_of_scores_of_either_sign(H, d, scale):
    n, scale = 100, d ** -0.5 if scale is None else scale
    q, k, v = (torch.randn(n, 2, d, generator=torch.Generator().manual_seed(i)) for i in range(3))
    cu = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    got = H.prefill_varlen(q.to(DEV), k.to(DEV), v.to(DEV), cu, cu, n, n, scale)
    torch.testing.assert_close(got.double().cpu(), _attend(q, k, v, scale, _mask(n, n)), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("n, seqs", [(20, 200), (50, 80), (300, 12), (1000, 4)])
def test_no_further_from_64_bits_than_the_vector_kernel(H, n, seqs, d):
    """The error over all outputs (2-norm) of prompts of n tokens; half a million results and more, whose ratio of errors moves by a few thousandths from
    seed to seed."""
    g = torch.Generator(device=DEV).manual_seed(n)
    q, k, v = (torch.randn(seqs * n, 2, d, generator=g, device=DEV) for _ in range(3))
    cu = torch.arange(0, seqs * n + 1, n, dtype=torch.int32, device=DEV)
    lanes = lambda t: t.double().unflatten(0, (seqs, n)).transpose(1, 2).flatten(0, 1).contiguous()
    s = torch.matmul(lanes(q), lanes(k).transpose(1, 2).contiguous()) * d ** -0.5
    s.masked_fill_(torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1), -float("inf"))
    want = torch.matmul(s.softmax(-1), lanes(v))
    error = [(lanes(H.prefill_varlen(q, k, v, cu, cu, n, n, d ** -0.5, flags=f)) - want).norm() / want.norm() for f in (H.MV_PREFILL_TILES, H.MV_PREFILL_SIMPLE)]
    assert error[0] <= 1.01 * error[1], (error[0].item(), error[1].item())


# by what the vector kernel and the tiles take: few keys, single queries of paged keys; long prompts, many of a few tokens; a window, a chunk
@pytest.mark.parametrize("seqs, nq, nk, kw, vector", [(1, 8, 8, {}, True), (1, 40, 40, {}, True), (256, 1, 200, dict(paged=True), True), (1, 8, 400, dict(window=32), True),
                                                      (1, 300, 300, dict(chunk=16), True), (1, 100, 100, {}, False), (256, 16, 16, {}, False), (2, 500, 500, {}, False),
                                                      (1, 8, 400, dict(window=300), False)], ids=str)
@pytest.mark.parametrize("d", [64, 128])
def test_kernel_by_size(H, d, seqs, nq, nk, kw, vector):
    g = torch.Generator(device=DEV).manual_seed(nk)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    cu = lambda n: torch.arange(0, seqs * n + 1, n, dtype=torch.int32, device=DEV)
    q, k, v, cache = rand(seqs * nq, 8, d), rand(seqs * nk, 2, d), rand(seqs * nk, 2, d), {}
    if kw.get("paged"):
        kc, vc = (t.view(-1, 40, 2, d) for t in (k, v))
        k, v, cache = None, None, dict(k_cache=kc, v_cache=vc, block_tables=torch.arange(seqs * nk // 40, dtype=torch.int32, device=DEV).view(seqs, -1))
    call = lambda flags: H.prefill_varlen(q, k, v, cu(nq), cu(nk), nq, nk, d ** -0.5, flags=flags, chunk=kw.get("chunk", 0), mask=H.AttnMask(kw.get("window", 0)), **cache)
    by_size, one, other = call(0), call(H.MV_PREFILL_SIMPLE), call(H.MV_PREFILL_TILES)
    assert not torch.equal(one, other)
    assert torch.equal(by_size, one if vector else other)
    torch.testing.assert_close(one, other, rtol=1e-5, atol=1e-5)      # (as above)
