"""The operator's native call (csrc/torch_call.cpp) against the Python autograd function that takes the unusual calls: the same
outputs, gradients, refusals and graph."""
import os
import shutil
import subprocess
import sys

import pytest
import torch

from acctransformer_amd import _capi
from acctransformer_amd.flash_attention.ops.flash_attention import flash_attention_impl as impl
from acctransformer_amd.flash_attention.ops.flash_attention.flash_attention_impl import get_flash_attention
from acctransformer_amd.infer.flash_attention.tik.flash_attention_tik import flash_attention_tik

DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_what_the_native_call_leaves_to_python():
    t = lambda *s: torch.zeros(*(s or (1, 2, 64, 64)), dtype=torch.float16)
    rest = (0, None, None, False, None, None, 0, 0, False, None, 65536, 65536, 0.1, 1.0, 0)
    assert _capi.native().forward(False, t(), t(), t(), *rest) is None                     # no device
    assert _capi.native().forward(False, t(64, 64), t(), t(), *rest) is None
    assert _capi.native().forward(False, None, t(), t(), *rest) is None
    with pytest.raises(TypeError):
        _capi.native().forward(False, t(), t(), t())


def test_the_native_call_uses_the_library_that_was_loaded(tmp_path):
    other = shutil.copy(_capi.lib_path(), tmp_path / "other.so")
    run = subprocess.run([sys.executable, "-c", f"""
from acctransformer_amd import _capi
_capi._LIB_PATH = {str(other)!r}
_capi.native()
maps = open('/proc/self/maps').read()
assert {str(other)!r} in maps and '_native.so' in maps and 'libacct_fa.so' not in maps
print('one library')
"""], capture_output=True, text=True, cwd=ROOT, timeout=300)
    assert run.stdout.strip() == "one library", run.stderr


def test_a_module_of_another_torch_does_not_load():
    run = subprocess.run([sys.executable, "-c", """
import torch
torch.__version__ = '0.0.0'
from acctransformer_amd import _capi
try:
    _capi.native()
except ImportError as e:
    print(e)
"""], capture_output=True, text=True, cwd=ROOT, timeout=300)
    assert "this is torch 0.0.0" in run.stdout and "make -C" in run.stdout, run.stderr


@pytest.mark.parametrize("torch_there", [True, False])
def test_the_c_abi_builds_without_torch(torch_there, tmp_path):
    python = sys.executable
    if not torch_there:
        python = str(tmp_path / "python")                   # an interpreter without installed packages
        (tmp_path / "python").write_text(f"#!/bin/sh\nexec {sys.executable} -S \"$@\"\n")
        os.chmod(python, 0o755)
    run = subprocess.run(["make", "-n", "-B", "-C", "acctransformer_amd/csrc", f"PYTHON={python}"], capture_output=True, text=True, cwd=ROOT,
                         timeout=300)
    assert run.returncode == 0 and "libacct_fa.so" in run.stdout and "libacct_fa_ms.so" in run.stdout, run.stderr
    assert ("torch_call.cpp" in run.stdout) == torch_there and ("no torch" in run.stdout) != torch_there


def _inputs(form):
    g = torch.Generator(device=DEV).manual_seed(5)
    B, N, Sq, Sk, D = 2, 3, 200, 264, 64
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).half()
    q, k, v, do = r(B, N, Sq, D), r(B, N, Sk, D), r(B, N, Sk, D), r(B, N, Sq, D)
    mask = drop = alibi = None
    if form == "bsnd":
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    if form == "columns":                                     # rows that are not contiguous are copied first
        q, k, v = (t.transpose(2, 3).contiguous().transpose(2, 3) for t in (q, k, v))
    if form == "mask u8":
        mask = (torch.rand(1, Sq, Sk, generator=g, device=DEV) < 0.3).to(torch.uint8)
    if form == "mask bool per batch":
        mask = torch.rand(B, Sq, Sk, generator=g, device=DEV) < 0.3
    if form == "mask f16":
        mask = (torch.rand(Sq, Sk, generator=g, device=DEV) < 0.3).half()
    if form == "tile":
        q = r(B, N, 264, D)
        do, mask = r(B, N, 264, D), torch.triu(torch.ones(1, 128, 128, device=DEV), 1).half()
    if form == "seed":
        drop = (1 << 40, 7)
    if form == "drop f16":
        drop = (torch.rand(B, N, Sq, Sk, generator=g, device=DEV) < 0.9).half() / 0.9
    if form == "bias":
        alibi = r(1, N, 1, Sk)
    if form == "bias f32":
        alibi = r(B, 1, Sq, Sk).float()
    if form == "other strides of dO":
        do = do.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "one gradient":
        k, v = k.detach(), v.detach()
    return q.requires_grad_(), k.requires_grad_(form != "one gradient"), v.requires_grad_(form != "one gradient"), do, mask, drop, alibi


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "bsnd", "columns", "mask u8", "mask bool per batch", "mask f16", "tile", "seed", "drop f16", "bias",
                                  "bias f32", "other strides of dO", "one gradient"])
def test_native_and_python_calls_agree(form, monkeypatch):
    q, k, v, do, *side = _inputs(form)
    op = get_flash_attention(scale=0.125, keep_prob=0.9)
    wanted = [t for t in (q, k, v) if t.requires_grad]
    res = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(impl, "_native_call", lambda *a: None)
        with torch.no_grad():
            plain = op(q, k, v, *side)
        with torch.autograd.graph.saved_tensors_hooks(lambda x: x.clone(), lambda x: x):        # other memory in the backward
            o, lse = op(q, k, v, *side)
        assert ("CppFunction" not in type(o.grad_fn).__name__) and o.grad_fn.name() == "_FlashAttentionFnBackward"
        assert o.requires_grad and not lse.requires_grad and not plain[0].requires_grad
        first = torch.autograd.grad(o, wanted, do, retain_graph=True)
        again = torch.autograd.grad(o, wanted, do)
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(o, wanted, do)
        assert all(torch.equal(a, b) for a, b in zip(first, again))
        res.append([o, lse, *plain, *first])
        bits = o.grad_fn.params
        res[-1] += [torch.tensor([bits.mask_kind, bits.mask_bits_filled, bits.drop_bits_filled, bits.drop_mask_kind, bits.drop_philox])]
    for a, b in zip(*res):
        assert torch.equal(a, b) and a.stride() == b.stride() and a.dtype == b.dtype


@pytest.mark.gpu
def test_native_call_refuses_as_before():
    q, k, v, do, *_ = _inputs("plain")
    op = get_flash_attention(scale=0.125, keep_prob=0.9)
    with pytest.raises(ValueError):
        op(q, k[:, :, :, :32], v)
    with pytest.raises(TypeError):
        op(q.float(), k.float(), v.float())
    with pytest.raises(ValueError):
        op(q, k, v, torch.zeros(3, 200, 264, dtype=torch.uint8, device=DEV))
    with pytest.raises(_capi.AcctError):                      # a bias row at an odd head dim
        op(*(torch.zeros(1, 1, 8, 40, device=DEV).half() for _ in range(3)), None, None, torch.zeros(1, 1, 1, 8, device=DEV).half())
    o, _ = op(q, k, v)
    odd = torch.zeros(o.numel() + 4, device=DEV).half()[4:].view(o.shape)      # 8 bytes off: refused in the backward
    with pytest.raises(_capi.AcctError, match="16-byte"):
        torch.autograd.grad(o, q, odd)
    with torch.no_grad():
        q.mul_(2)
    with pytest.raises(RuntimeError, match="inplace"):
        torch.autograd.grad(op(q, k, v)[0].sum() + o.sum(), q)


@pytest.mark.gpu
@pytest.mark.parametrize("record", [True, False])
@pytest.mark.parametrize("B, N, Sq, Sk", [(0, 2, 64, 64), (2, 0, 64, 64), (2, 2, 0, 64), (2, 2, 64, 0)])
def test_extents_of_zero_with_a_mask_are_refused_in_the_librarys_words(B, N, Sq, Sk, record):
    q, k, v = (torch.zeros(B, N, S, 64, dtype=torch.float16, device=DEV, requires_grad=record) for S in (Sq, Sk, Sk))
    with pytest.raises(_capi.AcctError, match="ACCT_E_SHAPE"):
        get_flash_attention(scale=0.125)(q, k, v, torch.zeros(1, Sq, Sk, dtype=torch.uint8, device=DEV))


@pytest.mark.gpu
def test_a_backward_gives_back_the_keep_bits():
    q, k, v, do, *_ = _inputs("plain")
    op = get_flash_attention(scale=0.125, keep_prob=0.9)
    o, _ = op(q, k, v, torch.zeros(1, 200, 264, dtype=torch.uint8, device=DEV), (3, 4))
    bits = o.grad_fn.drop_bits
    size, at = bits.numel(), bits.data_ptr()
    assert at == o.grad_fn.params.drop_bits and o.grad_fn.params.mask_bits
    del bits
    torch.autograd.grad(o, q, do, retain_graph=True)
    assert o.grad_fn.drop_bits.data_ptr() == at               # (a second backward may follow)
    before = torch.cuda.memory_allocated()
    dq, = torch.autograd.grad(o, q, do)
    assert torch.cuda.memory_allocated() <= before + dq.numel() * 2 - size
    p = o.grad_fn.params
    assert o.grad_fn.drop_bits is None and not p.drop_bits and not p.mask_bits and not p.q and p.Sq == 200 and p.drop_bits_filled


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("backend", ["eager", "aot_eager"])
@pytest.mark.parametrize("form", ["plain", "bsnd", "mask u8", "seed", "bias", "one gradient"])
def test_compiled_autograd(form, backend, native, monkeypatch):
    """The backward as a call in a compiled graph, twice (the second time with other tensors, and another dropout seed)."""
    from torch._dynamo import compiled_autograd
    if not native:
        monkeypatch.setattr(impl, "_native_call", lambda *a: None)
    q, k, v, do, mask, drop, alibi = _inputs(form)
    op = get_flash_attention(scale=0.125, keep_prob=0.9)
    wanted = [t for t in (q, k, v) if t.requires_grad]
    torch._dynamo.reset()
    for step in range(2):
        if drop is not None:
            drop = (drop[0], drop[1] + step)
        with torch.no_grad():
            q.mul_(1 + step)
        want = torch.autograd.grad(op(q * 1, k, v, mask, drop, alibi)[0], wanted, do)
        o, _ = op(q * 1, k, v, mask, drop, alibi)
        for t in wanted:
            t.grad = None
        with compiled_autograd._enable(torch.compile(backend=backend)):
            o.backward(do)
        assert all(torch.equal(a, t.grad) for a, t in zip(want, wanted))


@pytest.mark.gpu
@pytest.mark.parametrize("backend", ["eager", "aot_eager"])
def test_compiled_forward(backend):
    q, k, v, do, mask, _, alibi = _inputs("bias")
    op = get_flash_attention(scale=0.125)
    torch._dynamo.reset()
    want, got = ((o, *torch.autograd.grad(o, (q, k, v), do)) for o in (op(q * 1, k, v, mask, None, alibi)[0],
                                                                       torch.compile(lambda: op(q * 1, k, v, mask, None, alibi)[0], backend=backend)()))
    assert all(torch.equal(a, b) for a, b in zip(want, got))


@pytest.mark.gpu
def test_native_call_on_another_stream_and_in_the_inference_operator():
    q, k, v, do, *_ = _inputs("plain")
    op = get_flash_attention(scale=1.0)
    want, lse = op(q, k, v)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got, _ = op(q, k, v)
        dq, = torch.autograd.grad(got, q, do)
    s.synchronize()
    assert torch.equal(got, want) and torch.equal(dq, torch.autograd.grad(want, q, do)[0])
    y = flash_attention_tik(q, k[:, :, :200], v[:, :, :200])                     # never part of a graph
    assert not y.requires_grad and torch.equal(y, op(q, k[:, :, :200], v[:, :, :200])[0])
