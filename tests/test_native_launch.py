"""The native launch path of the torch-facing wrappers (csrc/bind.cpp): what it declines without a GPU,
and on one that every form a wrapper accepts -- strides, given outputs, row-major and packed operands,
int32 and bf16 results, stored and missing workspaces -- is taken or declined as stated and gives bit for
bit what the wrapper's own code gives, and that what the wrapper refuses stays refused with the same error.
"""
import os
import subprocess
import sys

import pytest
import torch

import npu_kernels
from w8a8 import _lib, attention, build, fused, ops

DEV = "cuda"


def test_declines_what_it_does_not_take():
    n = _lib.launch_module()
    assert n is not None and ops._native is n, "the native launch path is not built"
    x, w, s = torch.zeros(1, 64, dtype=torch.bfloat16), torch.zeros(64, dtype=torch.int8), torch.zeros(16)
    assert n.gemv(x, w, 16, 64, s, None) is None          # host tensors
    assert n.gemv("x", w, 16, 64, s, None) is None        # not a tensor
    assert n.gemv(x, w, 16) is None                       # another number of arguments
    assert n.quant_packed(None) is None
    assert n.quant_packed(torch.nn.Parameter(x)) is None
    assert n.attention(x, x, x, 0, 0, 1.0, {}) is None
    assert n.wait_stream(x) is None


def test_a_module_that_does_not_fit_is_not_used(monkeypatch):
    n = _lib.launch_module()
    for name in ("torch_build", "sources"):
        with monkeypatch.context() as m:
            m.setattr(n, name, "another")
            assert _lib.launch_module() is None
        with monkeypatch.context() as m:
            m.delattr(n, name)
            assert _lib.launch_module() is None
    monkeypatch.setattr(_lib, "launch_sources", lambda: None)  # not shipped: nothing to compare
    assert _lib.launch_module() is n


def test_the_build_without_its_tools_leaves_it_out(monkeypatch, tmp_path):
    monkeypatch.setattr(build, "LAUNCH", str(tmp_path / "_launch.so"))
    with monkeypatch.context() as m:
        m.setattr(build.shutil, "which", lambda name: None)
        assert "g++" in build._build_launch()
    monkeypatch.setattr(torch.version, "hip", None)
    assert "ROCm" in build._build_launch()
    assert not list(tmp_path.iterdir())


def test_a_launch_that_fails_is_raised_and_not_run_again(monkeypatch):
    """Statuses decided before a launch decline; W8A8_EHIP, after which work may be queued, is raised as the
    wrappers raise it, and the wrapper does not make the call a second time."""
    n = _lib.launch_module()
    assert n.settle("w8a8_k_in", _lib.W8A8_OK) is True
    for status in (_lib.W8A8_EINVAL, _lib.W8A8_EALIGN, _lib.W8A8_ENOTSUP):
        assert n.settle("w8a8_k_in", status) is None
    with pytest.raises(_lib.W8A8Error, match="w8a8_k_in: EHIP") as e:
        n.settle("w8a8_k_in", _lib.W8A8_EHIP)
    assert e.value.status == _lib.W8A8_EHIP

    class Native:
        def __getattr__(self, name):
            return lambda *a: n.settle(f"w8a8_{name}", _lib.W8A8_EHIP)

    def call(*a):
        raise AssertionError("run again")
    for m in (ops, fused, attention):
        monkeypatch.setattr(m, "_native", Native())
        monkeypatch.setattr(m, "call", call)
    t, w = torch.zeros(2, 64), ops.PackedWeight(torch.zeros(1), 64, 64, sw=torch.zeros(64))
    for run in (lambda: ops.gemv_bf16(t, ops.GemvWeight(t, 64, 64), t), lambda: ops.linear_bf16(t, w),
                lambda: ops.gemm_bf16(t, t, w, epilogue="residual", residual=t, out=t), lambda: ops.gemm_i32(t, w),
                lambda: ops.quant_rows_packed(t), lambda: fused.k_in(t, t, 1e-6, packed=True),
                lambda: fused.k_qkv(t, t, t, t, t, t, t, 1e-6, 2, 1, 64, False), lambda: attention.attention(t, t, t),
                lambda: attention.attention_quant(t, t, t), lambda: attention.decode(t, t, t),
                lambda: npu_kernels.mm_i8(t, w, t)):
        with pytest.raises(_lib.W8A8Error, match="EHIP"):
            run()


def test_an_exception_inside_the_call_leaves_the_interpreter_whole():
    """A C++ exception while the GIL is released (a tensor without storage, ..) declines, with the GIL held
    again.  In a process of its own: without it the interpreter aborts."""
    code = ("import torch\nfrom w8a8 import _lib\nn = _lib.launch_module()\n"
            "assert [n.settle('w8a8_k_in', -1) for _ in range(100)] == [None] * 100\nprint('whole')")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100,
                       env={**os.environ, "PYTHONPATH": os.path.dirname(os.path.dirname(ops.__file__))})
    assert r.returncode == 0 and "whole" in r.stdout, r.stderr


class Recorded:
    """The native module; `taken` holds for each call made through it whether it was taken."""

    def __init__(self, module):
        self.module, self.taken = module, []

    def __getattr__(self, name):
        def run(*a):
            r = getattr(self.module, name)(*a)
            self.taken.append(r is not None)
            return r
        return run


def both(monkeypatch, call, native=None):
    """call() on the native path and on the wrappers' own code."""
    outs = []
    for native in (native or _lib.launch_module(), None):
        for m in (ops, fused, attention):
            monkeypatch.setattr(m, "_native", native)
        outs.append(call())
    return outs


def flat(r):
    if isinstance(r, ops.PackedActivation):
        return [torch.tensor([r.M, r.K]), r.data]
    if isinstance(r, (tuple, list)):
        return [t for x in r for t in flat(x)]
    return [r]


def bf(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(torch.bfloat16).to(DEV)


def forms():
    g = torch.Generator().manual_seed(3)
    w = torch.randint(-127, 128, (96, 128), generator=g, dtype=torch.int8).to(DEV)
    sw = (torch.rand(96, generator=g) * 0.01).to(DEV)
    pw, pg, gw = ops.pack_weight(w, "nk", sw=sw), ops.pack_weight(w[:64], "nk", 32, sw=sw[:64]), ops.pack_gemv_weight(w)
    wide = bf(33, 256, seed=1)
    x, xs = wide[:, :128].contiguous(), wide[:, 128:]  # xs: rows 256 apart
    ws = ops.workspace(x.device, ops.linear_workspace_bytes(33, 96, 128))
    res, one = bf(33, 96, seed=2), bf(1, 128, seed=4)
    q, sx = ops.quant_rows_packed(x)
    qr, _ = ops.quant_rows(x)
    acc = ops.gemm_i32(q, pw)
    y, n96, sc = ops.gemm_bf16(q, sx, pw), bf(96, seed=5), torch.ones(1, dtype=torch.bfloat16, device=DEV)
    cs, yq = bf(33, 128, seed=6), bf(33, 4 * 128, seed=7)
    qa, k, v = bf(2, 40, 128, seed=8), bf(1, 40, 128, seed=9), bf(1, 40, 128, seed=10)
    qt = bf(40, 2, 128, seed=11).transpose(0, 1)  # [H, T, D] with rows H * D apart
    # causal calls whose key ranges are split: their parts need a workspace
    qs, ks, vs = bf(8, 512, 256, seed=12), bf(1, 512, 256, seed=13), bf(1, 512, 256, seed=14)
    ql, kl, vl = bf(8, 2048, 256, seed=15), bf(1, 2048, 256, seed=16), bf(1, 2048, 256, seed=17)
    for T in (512, 2048):
        assert _lib.lib().w8a8_attention_workspace_bytes(8, 1, T, T, 256, 0, 0) > 0
    return {
        "gemv": lambda: ops.gemv_bf16(one, gw, sw), "gemv bf16 scales": lambda: ops.gemv_bf16(one, gw, sw.bfloat16()),
        "gemv strided out": lambda: ops.gemv_bf16(x[:3], gw, sw, torch.zeros(3, 128, dtype=torch.bfloat16, device=DEV)[:, :96]),
        "linear": lambda: ops.linear_bf16(x, pw), "linear strided": lambda: ops.linear_bf16(xs, pw),
        "linear empty": lambda: ops.linear_bf16(x[:0], pw),
        "linear given workspace": lambda: ops.linear_bf16(x, pw, ws_arg=ws),
        "linear gelu": lambda: ops.linear_bf16(x, pg, epilogue="gelu"),
        "linear residual": lambda: ops.linear_bf16(x, pw, epilogue="residual", residual=res),
        "linear residual_rms": lambda: ops.linear_bf16(x, pw, epilogue="residual_rms", residual=res, rms_w=n96),
        "linear unused residual": lambda: ops.linear_bf16(x, pw, residual=res),
        "gemm packed": lambda: ops.gemm_i32(q, pw), "gemm rows": lambda: ops.gemm_i32(qr, pw),
        "gemm given c": lambda: ops.gemm_i32(qr, pw, torch.zeros(33, 100, dtype=torch.int32, device=DEV)[:, :96]),
        "gemm_bf16": lambda: ops.gemm_bf16(qr, sx, pw, epilogue="residual", residual=res),
        "quant": lambda: ops.quant_rows_packed(xs), "k_in": lambda: fused.k_in(x, None, 1e-6, packed=True),
        "k_post_attn": lambda: fused.k_post_attn(y, None, None, res, n96, None, 1e-6, packed=True),
        "k_post_attn i32": lambda: fused.k_post_attn(acc, sx, sw, res, n96, n96, 1e-6, packed=True),
        "k_post_ff": lambda: fused.k_post_ff(acc, sx, sw, res, n96, 1e-6, packed=True),
        "k_ple_gate": lambda: fused.k_ple_gate(y, None, None, res, packed=True),
        "k_ple_out": lambda: fused.k_ple_out(y, None, None, res, n96, sc, 1e-6, n96, packed=True),
        "k_ple_out number": lambda: fused.k_ple_out(y, None, None, res, n96, 0.5, 1e-6, n96, packed=True),
        "k_qkv": lambda: fused.k_qkv(yq, None, None, cs, cs, None, None, 1e-6, 2, 1, 128, False),
        "k_qkv shared": lambda: fused.k_qkv(yq, None, None, cs, cs, None, None, 1e-6, 4, 0, 128, True),
        "attention": lambda: attention.attention(qa, k, v), "attention window": lambda: attention.attention(qa, k, v, 0, 16),
        "attention strided": lambda: attention.attention(qt, k, v, 0, 0, 0.5),
        "attention split": lambda: attention.attention(qs, ks, vs),
        "attention_quant": lambda: attention.attention_quant(qa, k, v),
        "attention_quant two steps": lambda: attention.attention_quant(qs, ks, vs),
        "attention_quant split": lambda: attention.attention_quant(ql, kl, vl),
        "decode": lambda: attention.decode(qa[:, -1], k, v, None, 8), "decode 3-D": lambda: attention.decode(qa[:, -1:], k, v),
    }


# What the native path leaves to the wrapper: all of a form's native calls, or, where the stream has no
# workspace stored yet, the first one alone.
DECLINED = {"linear unused residual", "k_ple_out number", "decode 3-D"}
NO_WORKSPACE_YET = {"attention split", "attention_quant split", "decode"}


@pytest.mark.gpu
def test_equals_the_wrappers_own_code(monkeypatch):
    for name, call in forms().items():
        print(f"native launch path: {name}", flush=True)
        monkeypatch.setattr(attention, "_WS", {})
        monkeypatch.setattr(attention, "_SPLIT_WS", {})
        for again in (False, True):
            native = Recorded(_lib.launch_module())
            got, want = (flat(r) for r in both(monkeypatch, call, native))
            if name == "attention_quant two steps":  # the fused call declined, attention and then no k_attn_out
                assert native.taken == [False, again]
            else:
                assert native.taken == [name not in DECLINED and (again or name not in NO_WORKSPACE_YET)], name
            assert len(got) == len(want), name
            for a, b in zip(got, want):
                assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride(), name
                if a.dtype == torch.int8 and a.dim() == 1:  # packed rows: the padding of the last block is zero in both
                    assert torch.equal(a, b), name
                else:
                    assert torch.equal(a.float().nan_to_num(), b.float().nan_to_num()), name


def short_operands(x, pw, gw, w, sw, res, rms_w):
    """Calls with a norm weight shorter than the row, or an output smaller than the result."""
    return [lambda: ops.linear_bf16(x, pw, epilogue="residual_rms", residual=res, rms_w=rms_w),
            lambda: ops.gemv_bf16(x, gw, sw, res[:1]), lambda: ops.gemv_bf16(x, gw, sw, res[:, :95]),
            lambda: ops.gemv_bf16(x, w, sw, res.view(1, -1))]


def test_short_operands_are_refused_before_the_call(monkeypatch):
    def call(*a):
        raise AssertionError("launched")
    monkeypatch.setattr(ops, "_native", None)
    monkeypatch.setattr(ops, "_check", lambda *a: None)  # the device
    monkeypatch.setattr(ops, "call", call)
    x, res = torch.zeros(2, 128, dtype=torch.bfloat16), torch.zeros(2, 96, dtype=torch.bfloat16)
    w, sw = torch.zeros(96, 128, dtype=torch.int8), torch.zeros(96)
    pw, gw = ops.PackedWeight(w, 96, 128, sw=sw), ops.GemvWeight(w, 96, 128)
    for run in short_operands(x, pw, gw, w, sw, res, res[0, :95]):
        with pytest.raises(ValueError):
            run()


@pytest.mark.gpu
def test_refusals_are_the_wrappers(monkeypatch):
    w = torch.ones(96, 128, dtype=torch.int8, device=DEV)
    sw = torch.ones(96, device=DEV)
    pw, gw, x = ops.pack_weight(w, "nk", sw=sw), ops.pack_gemv_weight(w), bf(2, 128)
    h = bf(4, 40, 128)
    small = torch.empty(8, dtype=torch.uint8, device=DEV)
    calls = [*short_operands(x, pw, gw, w, sw, bf(2, 96), bf(95)),
             lambda: ops.gemv_bf16(x.float(), gw, sw), lambda: ops.gemv_bf16(x[:, :64], gw, sw),
             lambda: ops.linear_bf16(x, pw, ws_arg=small),
             lambda: ops.gemv_bf16(bf(17, 128), gw, sw), lambda: ops.gemv_bf16(x.cpu(), gw, sw),
             lambda: ops.linear_bf16(bf(128, 2).t(), pw), lambda: ops.linear_bf16(x, pw, epilogue="residual"),
             lambda: ops.gemm_i32(torch.ones(2, 64, dtype=torch.int8, device=DEV), pw),
             lambda: fused.k_in(bf(2, 100), None, 1e-6, packed=True),
             lambda: attention.attention(h, h[:3], h[:3]), lambda: attention.attention(h, h[:1], h[:1], 10),
             lambda: attention.decode(h[:, 0], h[:1], h[:1], 40)]
    for i, call in enumerate(calls):
        def refused():
            with pytest.raises((TypeError, ValueError, RuntimeError)) as e:
                call()
            return e.type, str(e.value)
        a, b = both(monkeypatch, refused)
        assert a == b, i


@pytest.mark.gpu
def test_transformed_tensors_are_refused_as_by_the_wrappers(monkeypatch):
    """torch.func wraps tensors without a storage of their own: the error is the one of the wrapper's code."""
    gw, sw = ops.pack_gemv_weight(torch.ones(96, 128, dtype=torch.int8, device=DEV)), torch.ones(96, device=DEV)
    x = bf(3, 1, 128)

    def refused():
        with pytest.raises(RuntimeError) as e:
            torch.func.vmap(lambda r: ops.gemv_bf16(r, gw, sw))(x)
        return e.type, str(e.value)
    a, b = both(monkeypatch, refused)
    assert a == b
