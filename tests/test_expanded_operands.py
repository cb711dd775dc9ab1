"""Operands in unusual memory.  Heads or batches that share it (`k.expand(...)`): their gradients are those of materialised
copies.  Rows so far apart that 32-bit offsets within a tile do not reach: results are those of contiguous copies."""
import pytest
import torch

from acctransformer_amd import _capi
from acctransformer_amd.flash_attention.ops.flash_attention import flash_attention_impl as impl
from acctransformer_amd.flash_attention.ops.flash_attention.flash_attention_impl import get_flash_attention

DEV = "cuda:0"
B, N, SQ, SK, D = 2, 3, 130, 200, 64


def test_which_operands_are_copied():
    t = torch.zeros(B, N, 8, 16)
    for own in (t, t.transpose(1, 2), t[:, 1:2].expand(B, 1, 8, 16), t[:, :, ::2], torch.zeros(1, 1, 8, 16).expand(1, 1, 8, 16)):
        assert _capi._apart(own) is own
    for shared in (t[:, :1].expand(B, N, 8, 16), t[:1].expand(B, N, 8, 16), t.as_strided((B, N, 4, 16), (N * 8 * 16, 32, 16, 1))):
        copy = _capi._apart(shared)
        assert copy is not shared and copy.is_contiguous() and torch.equal(copy, shared)
    rows = t[:, :, :1].expand(B, N, 8, 16)                    # (refused by the library)
    assert _capi._apart(rows) is rows


def test_one_row_for_all_is_not_a_contiguous_tensor():
    t = torch.zeros(B, N, 8, 16, dtype=torch.float16)
    row = torch.zeros(16, dtype=torch.float16)
    for operands in ((row.expand(B, N, 8, 16), t, t), (t, row.expand(B, N, 8, 16), t), (t, t, row.expand(B, N, 8, 16))):
        with pytest.raises(_capi.AcctError, match="row stride"):
            _capi.make_params(*operands, scale=1.0)
    one = row.as_strided((B, N, 1, 16), (0, 0, 0, 1))         # (a single row per head is accepted)
    assert list(_capi.make_params(one, t, t, scale=1.0).q_stride) == [0, 0, 16]


@pytest.mark.gpu
def test_one_row_for_all_on_the_gpu():
    op = get_flash_attention(scale=0.125)
    q, row = _leaf((B, N, SQ, D), 1), _leaf((D,), 2)
    with pytest.raises(_capi.AcctError, match="row stride"):
        op(q, row.expand(B, N, SK, D), row.expand(B, N, SK, D))
    k = _leaf((B, N, SK, D), 3)
    with torch.no_grad():
        one = row.as_strided((B, N, 1, D), (0, 0, 0, 1))
        assert torch.equal(op(one, k, k)[0], op(one.contiguous(), k, k)[0])


def _leaf(shape, seed):
    return torch.randn(*shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).half().requires_grad_()


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("form", ["heads", "batches", "query", "windows"])
def test_gradients_of_expanded_operands(form, native, monkeypatch):
    if not native:
        monkeypatch.setattr(impl, "_native_call", lambda *a: None)
    op = get_flash_attention(scale=0.125)
    do = _leaf((B, N, SQ, D), 9).detach()
    kv = (B, 1, SK, D) if form == "heads" else (1, N, SK, D) if form == "batches" else (B, N, SK, D)
    leaves = [_leaf((B, 1, SQ, D) if form == "query" else (B, N, SQ, D), 1), _leaf(kv, 2), _leaf(kv, 3)]

    def operands(copied):
        q, k, v = leaves
        if form == "windows":                                 # heads are overlapping windows of one longer sequence
            k, v = (t.as_strided((B, N, 100, D), (N * SK * D, 50 * D, D, 1)) for t in (k, v))
        else:
            q, k, v = q.expand(B, N, SQ, D), k.expand(B, N, SK, D), v.expand(B, N, SK, D)
        return [t.contiguous() for t in (q, k, v)] if copied else [q, k, v]

    o, _ = op(*operands(False))
    got = torch.autograd.grad(o, leaves, do)
    ref, _ = op(*operands(True))
    want = torch.autograd.grad(ref, leaves, do)
    assert torch.equal(o, ref)
    for a, b in zip(got, want):                               # the same kernels on the same values, and autograd's own sums
        assert torch.equal(a, b)
    q, k, v = operands(False)
    o, lse = op(q, k, v)
    bprop = op.bprop(q, k, v, None, None, None, (o, lse), (do,))[:3]
    want = op.bprop(*operands(True), None, None, None, (o, lse), (do,))[:3]
    assert all(torch.equal(a, b) for a, b in zip(bprop, want))


@pytest.mark.gpu
@pytest.mark.parametrize("B, N, Sq, Sk, D", [(1, 2, 64, 300, 64), (1, 2, 64, 300, 128), (16, 16, 256, 260, 64), (16, 16, 256, 260, 128), (1, 2, 64, 200, 160), (2, 3, 1, 300, 64)])
@pytest.mark.parametrize("stride", [9 << 20, 16909312, 17 << 20, 35 << 20])
def test_forward_with_rows_far_apart(B, N, Sq, Sk, D, stride):
    g = torch.Generator(device=DEV).manual_seed(D)
    q, k, v = (torch.randn(B, N, S, D, generator=g, device=DEV).half() for S in (Sq, Sk, Sk))
    at = (2 * N * D, 2 * D, stride, 1)
    memory = torch.empty((Sk - 1) * stride + 2 * B * N * D, dtype=torch.float16, device=DEV)
    kw, vw = memory.as_strided(k.shape, at), memory.as_strided(v.shape, at, D)
    kw.copy_(k)
    vw.copy_(v)
    op = get_flash_attention(scale=0.125)
    for a, b in ((kw, v), (k, vw), (kw, vw)):
        for x, y in zip(op(q, a, b), op(q, k, v)):
            # (256-key tiles need half the stride: the same sums in other shares then)
            assert torch.equal(x, y) if stride >= _capi.FWD_ROW_STRIDE_END else torch.allclose(x, y, atol=2e-3 if x.dim() == 4 else 1e-4)
        # the library itself: the same, or refused where whole tiles are too long for their offsets
        try:
            o, lse = _capi.fa_fwd(_capi.make_params(q, a, b, scale=0.125), q)
        except _capi.AcctError as e:
            assert e.code == _capi.ACCT_E_SHAPE and Sq > 1 and stride >= (_capi._ROW_STRIDE_END if D > 128 else _capi.FWD_ROW_STRIDE_END)
        else:
            assert Sq == 1 or stride < (_capi._ROW_STRIDE_END if D > 128 else _capi.FWD_ROW_STRIDE_END)
            ref = _capi.fa_fwd(_capi.make_params(q, k, v, scale=0.125), q)
            assert torch.allclose(o, ref[0], atol=2e-3) and torch.allclose(lse, ref[1], atol=1e-4)


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("stride", [_capi._ROW_STRIDE_END - 8, _capi._ROW_STRIDE_END])
def test_gradients_with_rows_far_apart(stride, which, native, monkeypatch):
    if not native:
        monkeypatch.setattr(impl, "_native_call", lambda *a: None)
    op = get_flash_attention(scale=0.125)
    close = [_leaf((1, 2, 130, D), s) for s in (1, 2, 3)]
    wide = [t.detach() for t in close]
    memory = torch.empty(129 * stride + 2 * D, dtype=torch.float16, device=DEV)
    wide[which] = memory.as_strided((1, 2, 130, D), (2 * D, D, stride, 1)).copy_(wide[which])
    wide = [t.requires_grad_() for t in wide]
    do = _leaf((1, 2, 130, D), 4).detach()
    for a, b in zip(torch.autograd.grad(op(*wide)[0], wide, do), torch.autograd.grad(op(*close)[0], close, do)):
        assert torch.equal(a, b)
