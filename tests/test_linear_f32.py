"""Who goes by parts of bf16 in fp32 (csrc/linear_f32.hip), and what its entry points refuse before they launch anything."""
import pytest
import torch

from minivllm_amd import hip_ops as H


def test_split_refuses():
    """The library is handed addresses: whatever they would be read wrongly from is refused on the host."""
    m, norm = torch.zeros(16, 64), torch.nn.LayerNorm(64)
    for bad in (m.bfloat16(), m.double(), m[:, ::2], m.T, m[0], m[None]):
        with pytest.raises(H.MvHipError, match="side by side"):
            H.split_f32(m, bad)
    for n in (0, H.MV_SPLIT_F32_MAX + 1):
        with pytest.raises(H.MvHipError, match="matrices"):
            H.split_f32(*[m] * n)
    for bad in (torch.nn.LayerNorm(32), torch.nn.LayerNorm(64).bfloat16(), torch.nn.LayerNorm((64, 64)), torch.nn.LayerNorm(64, elementwise_affine=False)):
        with pytest.raises(H.MvHipError, match="norm: 64"):
            H.split_f32(m, norm=bad)
    norm.bias = torch.nn.Parameter(torch.zeros(63))
    with pytest.raises(H.MvHipError, match="norm: 64"):
        H.split_f32(m, norm=norm)
    for call in (lambda: H.split_f32(m), lambda: H.split_f32(m, norm=torch.nn.LayerNorm(64))):
        with pytest.raises(H.MvHipError, match="device tensors"):
            call()


def test_linear_refuses():
    part = lambda rows, k, n=None: H.F32Parts(torch.zeros(n or -(-rows // 16) * k * 96, dtype=torch.uint8), rows, k)
    x, w = part(20, 64), part(48, 64)
    for a, b in ((part(20, 32), w), (part(20, 64, 100), w), (x, part(48, 64, 100)), (x._replace(data=x.data.view(torch.int16)), w), (x, w._replace(rows=49))):
        with pytest.raises(H.MvHipError, match="inputs of|parts of a matrix"):
            H.linear_f32(a, b)
    with pytest.raises(H.MvHipError, match="bias"):
        H.linear_f32(x, w, torch.zeros(47))
    with pytest.raises(H.MvHipError, match="residual"):
        H.linear_f32(x, w, residual=torch.zeros(20, 96)[:, ::2])
    with pytest.raises(H.MvHipError, match="device tensors"):
        H.linear_f32(x, w)


def _layer(monkeypatch, d=64, ffn=128):
    from types import SimpleNamespace

    from minivllm_amd.glue import opt

    monkeypatch.setattr(H, "linear_f32_ok", lambda *a: True)      # (which asks for a GPU)
    return opt.OPTDecoderLayer(SimpleNamespace(hidden_size=d, num_attention_heads=d // 64, enable_bias=True, do_layer_norm_before=True, ffn_dim=ffn)).requires_grad_(False)


@pytest.mark.parametrize("d, rows", [(128, 8385), (768, 1345), (1024, 1025), (2048, 1024), (4096, 1024), (9216, 1024)])
def test_rows_that_pay_for_a_layers_weights(monkeypatch, d, rows):
    """However wide a layer is, few rows do not pay for the parts of its weights."""
    with torch.device("meta"):
        layer, x = _layer(monkeypatch, d, 4 * d), torch.zeros(rows, d)
    assert layer._by_parts(x) and not layer._by_parts(x[:rows - 1])


def _other_modules(layer):
    from torch import nn

    from minivllm_amd.layers import ColumnParallelLinear

    class Scaled(ColumnParallelLinear):
        def forward(self, x):
            return 2 * super().forward(x)

    class Norm(nn.LayerNorm):
        pass

    att = type("Other", (type(layer.self_attn),), {})(64, 1)
    return [("fc1", nn.Sequential(layer.fc1)), ("fc1", nn.Linear(64, 128)), ("fc1", Scaled(64, 128, True)), ("fc2", nn.Linear(128, 64)), ("self_attn", att),
            ("self_attn_layer_norm", Norm(64)), ("final_layer_norm", nn.Identity()), ("final_layer_norm", nn.LayerNorm(64, elementwise_affine=False)),
            ("final_layer_norm", nn.LayerNorm((20000, 64)))]


@pytest.mark.parametrize("at", range(9))
def test_opt_layer_with_other_modules(monkeypatch, at):
    """An adapter or a norm in the place of a layer's own is called as a module."""
    layer, x = _layer(monkeypatch), torch.zeros(20000, 64)
    assert layer._by_parts(x)
    name, other = _other_modules(layer)[at]
    setattr(layer, name, other)
    assert not layer._by_parts(x)


def test_opt_layer_that_is_watched(monkeypatch):
    """So is one that has a hook, or a forward of its own."""
    from torch import nn

    layer, x = _layer(monkeypatch), torch.zeros(20000, 64)
    att = layer.self_attn
    for m in (att, att.qkv_proj, att.out_proj, layer.fc1, layer.fc2, layer.self_attn_layer_norm, layer.final_layer_norm):
        for hook in (m.register_forward_hook, m.register_forward_pre_hook):
            handle = hook(lambda *a: None)
            assert not layer._by_parts(x)
            handle.remove()
        m.forward = m.forward
        assert not layer._by_parts(x)
        del m.forward
    for hook in (nn.modules.module.register_module_forward_hook, nn.modules.module.register_module_forward_pre_hook):
        handle = hook(lambda *a: None)
        assert not layer._by_parts(x)
        handle.remove()
    assert layer._by_parts(x)


def test_forms_that_have_no_parts(monkeypatch):
    """Weights and biases in the other forms that ``F.linear`` takes go to it."""
    import torch.nn.functional as F

    from minivllm_amd.layers.linear import linear

    def refuse(*a):
        raise AssertionError("by parts")

    monkeypatch.setattr(H, "linear_f32_ok", lambda *a: True)
    monkeypatch.setattr(H, "split_f32", refuse)
    x, w = torch.randn(512, 4800), torch.randn(4800, 32)
    assert torch.equal(linear(x, w[:, 0].contiguous()), F.linear(x, w[:, 0].contiguous()))
    x = x[:, :32].contiguous()
    for bias in (torch.tensor(2.0), torch.randn(1), torch.randn(1, 4800), torch.randn(512, 4800)):
        assert torch.equal(linear(x, w, bias), F.linear(x, w, bias))
    for bias in (None, torch.randn(4800)):
        with pytest.raises(AssertionError, match="by parts"):
            linear(x, w, bias)


@pytest.mark.gpu
def test_who_is_asked_for():
    """A mode that sees functions sees the library's, a compiled program holds it whole; a default device changes nothing."""
    from torch.overrides import TorchFunctionMode

    from minivllm_amd.layers.linear import linear

    x, w = torch.randn(1300, 96, device="cuda:0"), torch.randn(2048, 96, device="cuda:0")
    by_parts, seen = H.linear_f32(*H.split_f32(x, w)), []

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Watch():
        y = linear(x, w)
    assert torch.nn.functional.linear in seen and torch.equal(y, torch.nn.functional.linear(x, w))
    with torch.device("cuda:0"):
        assert torch.equal(linear(x, w), by_parts)
    assert torch.equal(torch.compile(linear, backend="eager", fullgraph=True)(x, w), y)
    assert torch.equal(linear(torch._neg_view(x), w), torch.nn.functional.linear(-x, w))


@pytest.mark.gpu
def test_linear_refuses_vectors_elsewhere():
    x, w = H.split_f32(torch.zeros(20, 64, device="cuda:0"), torch.zeros(48, 64, device="cuda:0"))
    for kw in (dict(bias=torch.zeros(48)), dict(residual=torch.zeros(20, 48))):
        with pytest.raises(H.MvHipError, match="device tensors"):
            H.linear_f32(x, w, **kw)
