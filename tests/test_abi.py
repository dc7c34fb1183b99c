"""The C-ABI library loads (no GPU needed) and exports exactly what include/mvhip.h declares; the
product path refuses CPU tensors instead of falling back."""
import ctypes
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared():
    text = open(os.path.join(ROOT, "include", "mvhip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mv_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    from minivllm_amd import hip_ops

    names = _declared()
    assert len(names) >= 12
    lib = ctypes.CDLL(hip_ops.LIB_PATH)
    for n in names:
        assert hasattr(lib, n), f"{n} declared in mvhip.h but not exported"
    assert sorted(hip_ops.EXPORTED_SYMBOLS) == names      # the ctypes table covers the whole header
    assert hip_ops.version() == 1
    assert hip_ops.lib().mv_strerror(-5).decode().startswith("pointer or stride")
    assert b"ok" == hip_ops.lib().mv_strerror(0)


def test_workspace_size_queries_are_host_only():
    from minivllm_amd import hip_ops

    assert hip_ops.paged_decode_workspace_bytes(256, 16, 8, 128, 64, 64) == 256      # one split: no workspace
    small = hip_ops.paged_decode_workspace_bytes(1, 16, 8, 128, 64, 64)
    assert small > 256 and small % 256 == 0                                          # split-KV partials
    assert hip_ops.paged_decode_workspace_bytes(1, 16, 8, 96, 64, 64) == 256         # unsupported D: nothing


def test_when_state_space_prompts_are_cut():
    """Scratch memory is asked for where sequences are cut into segments: eight chunks of 64 tokens and more (six where a workgroup has one column tile), and
    few enough workgroups."""
    from minivllm_amd import hip_ops

    need = lambda seqs, rows, longest, heads=4, p=64, n=128, dtype=hip_ops.MV_BF16: hip_ops.lib().mv_ssm_prefill_workspace_bytes(
        seqs, rows, longest, heads, p, n, dtype)
    assert need(1, 448, 448) == 0 < need(1, 449, 449)
    assert need(1, 320, 320, p=80) == 0 < need(1, 321, 321, p=80)
    assert need(2, 2000, 1000, heads=64) > 0 == need(4, 4000, 1000, heads=64)            # half of the CUs have work, or all
    assert need(4, 5000, 4000, heads=64) > 0 == need(4, 16000, 4000, heads=64)           # one long sequence, or four
    assert need(2, 8000, 4000, heads=80) > 0 == need(2, 8000, 4000, heads=80, n=256)     # two workgroups to a CU, or one
    assert need(8, 8000, 8000, heads=64) == 0                                            # 512 workgroups
    assert need(1, 4000, 4000, dtype=hip_ops.MV_F32) == 0
    for rows in (0, -1, 999):          # fewer rows than the longest sequence: no bound that segments could be counted from
        assert need(1, rows, 1000) == 0


def test_struct_layouts_of_the_binding_match_the_library():
    """mv_decode_layers_persistent takes two structs by pointer: the ctypes declarations must have the library's layout."""
    from minivllm_amd import hip_ops

    assert hip_ops.lib().mv_persist_struct_bytes(1) == ctypes.sizeof(hip_ops.MvPersistArgs)
    assert hip_ops.lib().mv_persist_struct_bytes(0) == 8 * len(hip_ops.PERSIST_LAYER_FIELDS)   # a row of the int64 layer table
    assert hip_ops.lib().mv_decode_layers_persistent_workspace_bytes(1, 2048, 16, 8, 128, 6144, 64, 64) > 4096


def test_delta_prompts_with_convolution_need_its_state():
    """A pool of states without the kept inputs, or the other way round, is refused as mv_causal_conv refuses it, in the entry point and ahead of it."""
    from minivllm_amd import hip_ops as H

    at = torch.zeros(64, dtype=torch.uint8)
    p = (at.data_ptr() + 15) & ~15      # (nothing is read)
    s = H.DeltaShape(2, 2, 64, 64, 128, 256, 64, 0.125, False)

    def call(**kw):
        a = H.MvDeltaArgs(**dict(dict(x=p, beta=p, a=p, conv_w=p, dt_bias=p, a_log=p, state=p, state_slots=p, cu_q=p, cu_k=p, out=p, x_stride=s.channels, beta_stride=8,
                                      a_stride=8, out_stride=128, slots=3, n_seqs=1, max_q=70, total_q=70, channels=s.channels, taps=4, heads=2, groups=2, p=64,
                                      p_true=64, n=64, k_off=128, q_off=256), **kw))
        return H.lib().mv_delta_prefill_conv(ctypes.byref(a), p, H.MV_BF16, 0, None)

    assert call() == -1 and call(conv_state=p, state=None) == -1 and call(conv_state=p, taps=9) == -2 and call(conv_state=p + 8) == -5
    x, w, kept = (torch.zeros(*n, dtype=torch.bfloat16) for n in ((5, s.channels), (4, s.channels), (2, 3, 3, s.channels)))
    for slots, state in ((3, None), (3, kept[:, :, :2]), (3, kept.half()), (0, kept), (3, kept[:, :0])):
        with pytest.raises(H.MvHipError, match="convolution state"):
            H._delta_conv(H.MvDeltaArgs(slots=slots), s, x, w, state)
    for slots, state, weight in ((3, kept, w), (0, None, w), (0, kept[:, :0], w), (3, None, w[:1]), (3, kept[:, :, :0], w[:1])):
        g = H.MvDeltaArgs(slots=slots)
        H._delta_conv(g, s, x, weight, state)
        assert g.conv_state == (kept.data_ptr() if state is kept else None) and g.taps == weight.shape[0]


def test_no_cpu_fallback():
    from minivllm_amd import hip_ops

    x = torch.zeros(4, 128, dtype=torch.bfloat16)
    with pytest.raises(hip_ops.MvHipError, match="no CPU fallback"):
        hip_ops.rmsnorm(x, torch.ones(128, dtype=torch.bfloat16), 1e-6)
    with pytest.raises(hip_ops.MvHipError):
        hip_ops.silu_and_mul(x)


def test_product_never_imports_the_oracle():
    pkg = os.path.join(ROOT, "mini-vllm_amd")
    for d, _, files in os.walk(pkg):
        for f in files:
            if f.endswith(".py"):
                src = open(os.path.join(d, f)).read()
                assert not re.search(r"^\s*(from|import)\s+oracle\b", src, flags=re.M), f"{f} imports oracle"
