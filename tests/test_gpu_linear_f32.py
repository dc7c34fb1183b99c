"""fp32 projections from operands in parts of bf16 (csrc/linear_f32.hip), against 64 bits and the library."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _sum_of_parts(p):
    q = p.data.view(torch.bfloat16).view(-(-p.rows // 16), p.k // 32, 3, 4, 16, 8).double().sum(2)
    return q.permute(0, 3, 1, 2, 4).reshape(-1, p.k)[:p.rows]


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


@pytest.mark.parametrize("rows, k", [(1, 32), (15, 64), (16, 1024), (17, 1056), (33, 3072)])
def test_parts_add_up(rows, k):
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(rows)
    x = _randn(g, rows, k + 12)[:, 4:4 + k] * 10 ** (12 * _randn(g, rows, 1)).clamp(1e-30, 1e30)
    x[0, 0], x[0, 1] = torch.finfo(torch.float32).max, -torch.finfo(torch.float32).max      # (no bf16 is as large, rounded)
    w = _randn(g, 48, 64)
    a, b = H.split_f32(x, w)
    assert torch.equal(_sum_of_parts(a), x.double()) and torch.equal(_sum_of_parts(b), w.double())
    norm = torch.nn.LayerNorm(k, device=DEV).requires_grad_(False)
    norm.weight.copy_(1 + 0.1 * _randn(g, k)), norm.bias.copy_(0.1 * _randn(g, k))
    x = 1 + 3 * _randn(g, rows, k)
    a, b = H.split_f32(x, w, norm=norm)
    assert torch.equal(_sum_of_parts(b), w.double())
    want = F.layer_norm(x.double(), (k,), norm.weight.double(), norm.bias.double(), norm.eps)
    # mean, deviation and scale each within some units of 2^-24 of numbers of up to about 5; torch's own is as far off
    assert (_sum_of_parts(a) - want).abs().max() <= 2e-6


def _numbers(p):
    """What the parts stand for: their sum, or where the third is NaN the bits of the first and second."""
    q = p.data.view(torch.int16).view(-1, p.k // 32, 3, 4, 16, 8).permute(0, 4, 1, 3, 5, 2).reshape(-1, p.k, 3)[:p.rows].contiguous()
    bits = (q[..., 0].int() << 16) | (q[..., 1].int() & 0xffff)
    parts = q.view(torch.bfloat16)
    return torch.where(parts[..., 2].isnan(), bits.view(torch.float32).double(), parts.double().sum(-1))


def test_small_numbers_keep_their_bits():
    """Down to the smallest of fp32, also where bf16 has no number for the last of their bits."""
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(3)
    x = _randn(g, 48, 1056) * 2.0 ** torch.arange(-150, -102, device=DEV).double()[:, None]
    x = x.float()
    x[:, 7] = 1.0
    x[20, 8:40], x[21, 8:40] = 0.0, torch.finfo(torch.float32).tiny
    assert torch.equal(_numbers(H.split_f32(x)[0]), x.double())


def _chain_bound(x, w, y):
    # a chain of sums of four products, each rounded at its size; below 2^-126 each product and sum at 2^-149
    k = x.shape[1]
    return 2.0 ** -24 * ((x.double().abs() @ w.double().abs().T) * (k / 4 + 2) + 4 * y.abs()) + 2.0 ** -149 * (1.5 * k + 4)


@pytest.mark.parametrize("tile", [1, 2])
@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("e", [-108, -112, -118, -124, -130])
def test_products_of_small_numbers(e, which, tile):
    """Rows (weights) below the numbers that three of bf16 add up to, all of them or some beside larger ones that meet zeros."""
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(-e)
    a, b = _randn(g, 152, 160), _randn(g, 140, 160)
    a[:70] *= 2.0 ** e
    a[70:90, ::2] *= 2.0 ** e
    b[:, 1::2] *= torch.where(torch.arange(140, device=DEV) < 70, 0.0, 1.0)[:, None]
    x, w = (a, b) if which == 0 else (b, a)
    got, want = H.linear_f32(*H.split_f32(x, w), tile=tile), x.double() @ w.double().T
    assert ((got - want).abs() <= _chain_bound(x, w, want)).all()
    tiny, library = (got[:70], F.linear(x, w)[:70]) if which == 0 else (got[:, :70], F.linear(x, w)[:, :70])
    want = want[:70] if which == 0 else want[:, :70]
    off = lambda y: ((y.double() - want).norm() / want.norm()).item()
    assert off(tiny) <= off(library)
    # as they leave for another projection
    parts = H.linear_f32(*H.split_f32(x, w[:128].contiguous()), tile=tile, parts=True)
    assert torch.equal(_numbers(parts), H.linear_f32(*H.split_f32(x, w[:128].contiguous()), tile=tile).double())


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("rows, n, k", [(1, 4, 32), (16, 32, 64), (63, 60, 96), (64, 64, 160), (127, 128, 768), (129, 132, 768), (700, 1000, 256), (300, 96, 3072)])
def test_products(rows, n, k, tile):
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(rows + n)
    x, w, bias, residual = _randn(g, rows, k), _randn(g, n, k) * k ** -0.5, _randn(g, n), _randn(g, rows, n + 4)[:, :n]
    xs, ws = H.split_f32(x, w)
    want = x.double() @ w.double().T
    # 2^-24 of the sum of the products' sizes (sqrt(k) .. k of 1/sqrt(k)) for each of the k / 32 sums and what the parts leave out, and of the last additions
    bound = lambda y: 2.0 ** -24 * (x.double().abs() @ w.double().abs().T * (k / 32 + 2) + 4 * y.abs() + 4)
    assert ((H.linear_f32(xs, ws, tile=tile) - want).abs() <= bound(want)).all()
    got = H.linear_f32(xs, ws, bias, residual, relu=True, tile=tile)
    want = (want + bias).clamp(min=0) + residual
    assert got.shape == (rows, n) and ((got - want).abs() <= bound(want)).all()


def test_distance_from_64_bits():
    """No further off than the library's fp32."""
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(5)
    for k, scale in ((768, 1.0), (3072, 1.0), (768, 1e-30), (768, 1e15)):
        x, w = _randn(g, 1500, k).relu() * scale, _randn(g, 512, k) * 0.02
        x[:, 7] *= 1e4      # (a channel far above the others)
        want = x.double() @ w.double().T
        off = lambda y: ((y.double() - want).norm() / want.norm()).item()
        assert off(H.linear_f32(*H.split_f32(x, w))) <= off(F.linear(x, w))


@pytest.mark.parametrize("tile", [1, 2])
def test_not_finite(tile):
    """Infinities, NaN and sums that overflow come out as from the library; rows beside them are not touched."""
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(6)
    x, w = _randn(g, 200, 96), _randn(g, 160, 96)
    w[:80, :2], w[80:, :2] = 2.0, -0.25
    plain = H.linear_f32(*H.split_f32(x, w), tile=tile)
    x[3, 5], x[7, 9], x[13], x[13, :2] = float("inf"), float("nan"), 0.0, 3e38
    x[15, 3], x[15, 8] = float("inf"), -float("inf")
    xs, ws = H.split_f32(x, w)
    got, want = H.linear_f32(xs, ws, tile=tile), F.linear(x, w)
    for r in (3, 7, 13, 15):
        assert torch.equal(got[r].isnan(), want[r].isnan()) and torch.equal(got[r] == float("inf"), want[r] == float("inf"))
    assert got[13, :80].isinf().all() and torch.equal(got[13, 80:], torch.full((80,), -1.5e38, device=DEV))
    rest = [i for i in range(200) if i not in (3, 7, 13, 15)]
    assert torch.equal(got[rest], plain[rest])
    back = _sum_of_parts(H.linear_f32(xs, ws, relu=True, parts=True, tile=tile))
    assert torch.equal(back[3].isinf(), want[3] == float("inf")) and back[7].isnan().all()


@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("rows", [1, 16, 130])
def test_parts_out(rows, tile):
    """A projection's parts are those of its numbers."""
    from minivllm_amd import hip_ops as H

    g = torch.Generator(device=DEV).manual_seed(rows)
    x, w, bias, w2 = _randn(g, rows, 64), _randn(g, 160, 64), _randn(g, 160), _randn(g, 64, 160)
    xs, ws, w2s = H.split_f32(x, w, w2)
    plain, parts = H.linear_f32(xs, ws, bias, relu=True, tile=tile), H.linear_f32(xs, ws, bias, relu=True, parts=True, tile=tile)
    assert torch.equal(_sum_of_parts(parts), plain.double())
    assert torch.equal(H.linear_f32(parts, w2s, tile=tile), H.linear_f32(H.split_f32(plain)[0], w2s, tile=tile))


def test_who_goes_by_parts():
    """``linear``: plain fp32 numbers by parts; under autograd, autocast, vmap, forward mode, tracing, in other types and layouts what it was before."""
    from minivllm_amd import hip_ops as H
    from minivllm_amd.layers.linear import linear

    g = torch.Generator(device=DEV).manual_seed(8)
    x, w, bias = _randn(g, 1300, 96), _randn(g, 2048, 96) * 0.1, _randn(g, 2048)
    by_parts = H.linear_f32(*H.split_f32(x, w), bias)
    assert torch.equal(linear(x, w, bias), by_parts) and H.linear_f32_ok(x, w, bias)
    assert not torch.equal(by_parts, F.linear(x, w, bias))
    with torch.inference_mode():
        assert torch.equal(linear(x, w, bias), by_parts)
    wg = w.clone().requires_grad_()
    y = linear(x, wg, bias)
    assert y.requires_grad and torch.equal(y, F.linear(x, w, bias))
    with torch.no_grad():
        assert torch.equal(linear(x, wg, bias), by_parts)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert linear(x, w, bias).dtype == torch.bfloat16
    assert torch.equal(torch.func.vmap(lambda v: linear(v, w, bias))(x[None])[0], torch.func.vmap(lambda v: F.linear(v, w, bias))(x[None])[0])
    _, tangent = torch.func.jvp(lambda v: linear(v, w, bias), (x,), (x,))
    assert torch.allclose(tangent, F.linear(x, w), atol=1e-4)
    assert not H.linear_f32_ok(x[:, :40], w[:, :40], bias)              # inputs that are no multiple of 32
    assert not H.linear_f32_ok(x[:, 1:65], w[:, :64].contiguous(), bias)     # rows that are not aligned
    assert not H.linear_f32_ok(x, w.T.contiguous().T, bias)             # weights in another order
    odd = linear(x, w[:2046], bias[:2046])
    assert torch.equal(odd, F.linear(x, w[:2046], bias[:2046]))


def test_replays():
    """In a captured graph, with new numbers in the same buffers."""
    from minivllm_amd.layers.linear import linear

    g = torch.Generator(device=DEV).manual_seed(9)
    x, w = _randn(g, 1300, 96), _randn(g, 2048, 96)
    linear(x, w)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = linear(x, w)
    for _ in range(3):
        x.normal_(generator=g), w.normal_(generator=g)
        graph.replay()
        got = y.clone()
        assert torch.equal(got, linear(x, w))


def test_opt_layer():
    """An fp32 OPT layer as a whole against its modules one by one."""
    from types import SimpleNamespace

    from minivllm_amd.glue.opt import OPTDecoderLayer
    from minivllm_amd.utils.context import set_context

    with torch.device(DEV):
        layer = OPTDecoderLayer(SimpleNamespace(hidden_size=128, num_attention_heads=2, enable_bias=True, do_layer_norm_before=True, ffn_dim=512))
    layer.requires_grad_(False)
    g = torch.Generator(device=DEV).manual_seed(10)
    for p in layer.parameters():
        p.copy_(_randn(g, *p.shape) * (0.3 if p.dim() == 1 else p.shape[-1] ** -0.5))
    lengths = [4000, 4444, 17]
    cu = torch.tensor([0, 4000, 8444, 8461], dtype=torch.int32, device=DEV)
    x = _randn(g, sum(lengths), 128)
    set_context(True, max(lengths), max(lengths), cu, cu)
    assert layer._by_parts(x) and not layer._by_parts(x[:4000])
    with torch.inference_mode():
        got = layer(None, x)[0]
        a = layer.self_attn
        u = x + F.linear(a.attend(F.linear(F.layer_norm(x, (128,), layer.self_attn_layer_norm.weight, layer.self_attn_layer_norm.bias), a.qkv_proj.weight,
                                           a.qkv_proj.bias)), a.out_proj.weight, a.out_proj.bias)
        h = F.relu(F.linear(F.layer_norm(u, (128,), layer.final_layer_norm.weight, layer.final_layer_norm.bias), layer.fc1.weight, layer.fc1.bias))
        want = u + F.linear(h, layer.fc2.weight, layer.fc2.bias)
    # six roundings of 2^-24 each, of sums that cancel to a tenth, through four projections
    assert (got - want).norm() <= 3e-6 * want.norm()
    handle = layer.fc1.register_forward_hook(lambda m, i, o: None)
    assert not layer._by_parts(x)
    handle.remove()
