"""The host path of a call: parameter blocks that are kept between calls, and the forward that runs without an autograd
function where nothing is recorded."""
import numpy as np
import pytest
import torch
from torch.autograd import forward_ad

from acctransformer_amd import _capi
from acctransformer_amd.flash_attention.ops.flash_attention.flash_attention_impl import get_flash_attention

DEV = "cuda:0"


def _block(*args, **kw):
    p = _capi.make_params(*args, **kw)
    return {n: (list(getattr(p, n)) if n.endswith("_stride") else getattr(p, n)) for n, _ in p._fields_}, p


def test_kept_parameter_blocks_equal_fresh_ones():
    B, N, S, D = 2, 2, 64, 64
    t = lambda: torch.randn(B, N, S, D).half()
    bsnd = lambda: torch.randn(B, S, N, D).half().transpose(1, 2)
    m, tile = torch.zeros(1, S, S, dtype=torch.uint8), torch.zeros(1, 128, 128, dtype=torch.uint8)
    variants = [
        ((t(), t(), t()), dict(scale=0.1)),
        ((bsnd(), t(), t()), dict(scale=0.1)),
        ((t(), t(), t()), dict(scale=0.2, next_block_num=0)),
        ((t(), t(), t()), dict(scale=0.1, mask_kind=_capi.MASK_DENSE_U8, attn_mask=m)),
        ((t(), t(), t()), dict(scale=0.1, mask_kind=_capi.MASK_DENSE_U8, attn_mask=m.expand(B, S, S).contiguous())),
        ((t(), t(), t()), dict(scale=0.1, mask_kind=_capi.MASK_DENSE_F16, attn_mask=m.half())),
        ((t(), t(), t()), dict(scale=0.1, mask_kind=_capi.MASK_TILE_U8, attn_mask=tile)),
        ((t(), t(), t()), dict(scale=0.1, keep_prob=0.9, drop_mask=torch.ones(B, N, S, S, dtype=torch.uint8))),
        ((t(), t(), t()), dict(scale=0.1, keep_prob=0.9, drop_seed=5 << 33, drop_offset=3)),
        ((t(), t(), t()), dict(scale=0.1, alibi=torch.zeros(1, N, 1, S).half())),
        ((t(), t(), t()), dict(scale=0.1, alibi=torch.zeros(B, N, S, S).half())),
    ]
    for args, kw in variants:
        _capi._blocks.clear()
        fresh, _ = _block(*args, **kw)
        others = [o for o in variants if o[0] is not args]
        for a, k in others:
            _block(*a, **k)
        kept, p = _block(*args, **kw)
        assert kept == fresh
        assert [x.data_ptr() for x in p._keepalive] == [fresh[n] for n in ("q", "k", "v", "attn_mask", "drop_mask", "alibi") if fresh[n]]
        # other addresses and another dropout stream on the kept block
        args2 = tuple(x.clone(memory_format=torch.preserve_format) for x in args)
        kw2 = dict(kw, drop_seed=9, drop_offset=1) if "drop_seed" in kw else kw
        again, _ = _block(*args2, **kw2)
        _capi._blocks.clear()
        assert again == _block(*args2, **kw2)[0]
    for i in range(2 * _capi._BLOCKS_MAX):
        _block(*variants[0][0], scale=1.0 + i)
    assert len(_capi._blocks) <= _capi._BLOCKS_MAX
    with pytest.raises(ValueError):                          # what is refused is refused every time
        _block(t(), t()[:, :, :8], t(), scale=0.1)
    with pytest.raises(ValueError):
        _block(t(), t()[:, :, :8], t(), scale=0.1)


@pytest.mark.parametrize("name, first, second", [("scale", 0.125, 0.25), ("keep_prob", 0.5, 0.75), ("prev_block_num", 3, 5),
                                                 ("next_block_num", 3, 5), ("row_block_prefix", 128, 256)])
def test_numbers_in_tensors_and_arrays(name, first, second):
    """A number may come as a 0-d tensor or array; one that is changed in place between two calls counts as it is."""
    q, k, v = (torch.randn(1, 1, 64, 64).half() for _ in range(3))
    for x in (torch.tensor(first), np.array(first)):
        kw = dict(dict(scale=0.1), **{name: x})
        assert _block(q, k, v, **kw)[0][name] == first
        x.fill_(second) if isinstance(x, torch.Tensor) else x.fill(second)
        assert _block(q, k, v, **kw)[0][name] == second
        assert _block(q, k, v, **dict(kw, **{name: first}))[0][name] == first


def test_blocks_of_tensors_without_memory():
    """A call on meta tensors has no addresses; a later one of the same shapes hands over its own."""
    shapes = [(1, 2, 64, 64)] * 3
    kw = dict(scale=0.1, mask_kind=_capi.MASK_DENSE_U8, keep_prob=0.5)
    _capi._blocks.clear()
    for device in ("meta", "cpu"):
        q, k, v = (torch.zeros(s, dtype=torch.float16, device=device) for s in shapes)
        mask = torch.zeros(1, 64, 64, dtype=torch.uint8, device=device)
        drop = torch.ones(1, 2, 64, 64, dtype=torch.uint8, device=device)
        alibi = torch.zeros(1, 2, 1, 64, dtype=torch.float16, device=device)
        got, p = _block(q, k, v, attn_mask=mask, drop_mask=drop, alibi=alibi, **kw)
    assert (got["q"], got["k"], got["v"]) == (q.data_ptr(), k.data_ptr(), v.data_ptr())
    assert (got["attn_mask"], got["drop_mask"], got["alibi"]) == (mask.data_ptr(), drop.data_ptr(), alibi.data_ptr())
    assert len(p._keepalive) == 6


@pytest.mark.parametrize("side", ["query", "attn_mask", "dropout_mask", "alibi_mask", None])
def test_a_side_input_that_asks_for_a_gradient_is_recorded(side, monkeypatch):
    """The output belongs to the graph as soon as any input asks for a gradient; masks and biases then get none."""
    monkeypatch.setattr(_capi, "fa_fwd", lambda p, q: (torch.zeros_like(q), torch.zeros(q.shape[:3])))
    monkeypatch.setattr(_capi, "fa_bwd", lambda p, q, k, v, o, do, lse: tuple(torch.zeros_like(t) for t in (q, k, v)))
    monkeypatch.setattr(_capi, "attach_drop_bits", lambda p, device: None)
    inputs = dict(query=torch.randn(1, 2, 64, 64).half(), key=torch.randn(1, 2, 64, 64).half(), value=torch.randn(1, 2, 64, 64).half(),
                  attn_mask=torch.zeros(1, 64, 64).half(), dropout_mask=torch.ones(1, 2, 64, 64).half(), alibi_mask=torch.zeros(1, 2, 1, 64).half())
    if side:
        inputs[side].requires_grad_(True)
    op = get_flash_attention(scale=0.125, keep_prob=0.9)
    o, lse = op(**inputs)
    assert o.requires_grad == (side is not None) and not lse.requires_grad
    if side:
        o.sum().backward()
        assert (inputs[side].grad is not None) == (side == "query")
    with torch.no_grad():
        assert not op(**inputs)[0].requires_grad
    assert op(**dict(inputs, dropout_mask=(3, 4), **({side: inputs[side].detach()} if side and side != "dropout_mask" else {})))[0].grad_fn is None


@pytest.mark.gpu
def test_forward_with_and_without_recording():
    q, k, v = (torch.randn(1, 2, 96, 64, device=DEV).half() for _ in range(3))
    op = get_flash_attention(scale=0.125)
    plain = op(q, k, v)
    assert plain[0].grad_fn is None
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda x: seen.append(x.shape) or x, lambda x: x):
        o, lse = op(q.requires_grad_(True), k, v)
    assert len(seen) == 5 and o.grad_fn is not None and not lse.requires_grad
    assert torch.equal(o, plain[0]) and torch.equal(lse, plain[1])
    with torch.no_grad():
        assert op(q, k, v)[0].grad_fn is None
    dq, = torch.autograd.grad(o.sum(), q, retain_graph=True)
    do = torch.ones_like(o)
    assert torch.equal(dq, torch.autograd.grad(o, q, do)[0]) and torch.isfinite(dq).all()
    q = q.detach()
    with forward_ad.dual_level(), pytest.raises(Exception):   # no forward-mode rule: refused, not ignored
        op(forward_ad.make_dual(q, torch.ones_like(q)), k, v)
    with pytest.raises(Exception):
        torch.func.vmap(lambda x: op(x, k, v)[0])(q[None])
