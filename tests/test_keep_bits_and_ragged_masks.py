"""GPU tests of the mask and dropout pre-passes where they leave work out or meet rows that are not 16-byte aligned:
keep bits of key blocks that the mask, the band, the causal compare or the row prefix hides, key counts that are no
multiple of 16 (or of 128), thresholds on both sides of 128 and at 256.  Forward and backward share one buffer of keep
bits where a gradient is asked for.  Gate: that of the parity tests (every element within 2e-3 + 1e-3 |oracle|)."""
import numpy as np
import pytest
import torch

from acctransformer_amd import _capi
from acctransformer_amd.flash_attention.ops.flash_attention.flash_attention_impl import get_flash_attention
from oracle import philox_dropout as phx
from oracle import unfused_attention as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _masks(kind, B, Sq, Sk):
    j, i = np.arange(Sk)[None, None, :], np.arange(Sq)[None, :, None]
    if kind == "causal":
        return (j > i).astype(np.uint8)
    if kind == "padded":                                  # key tails inside, at the edge of and behind a block
        lens = np.array([130, Sk])[:B, None, None]
        return np.broadcast_to(j >= lens, (B, Sq, Sk)).astype(np.uint8)
    if kind == "random":
        m = (np.random.default_rng(Sk).random((B, Sq, Sk)) < 0.3).astype(np.uint8)
        m[:, :, 0] = 0
        return m
    return None


@pytest.mark.parametrize("Sq, Sk, D, mask, nxt, drop, keep", [
    (300, 300, 64, "causal", 0, "seed", 0.9), (257, 257, 128, "causal", 65536, "seed", 0.3), (129, 513, 64, "padded", 65536, "seed", 1.0 - 1e-9),
    (200, 1000, 128, "padded", 65536, "seed", 0.5), (130, 300, 64, None, 0, "seed", 0.6), (300, 300, 128, "causal", 0, "u8", 0.7),
    (261, 261, 64, "causal", 0, "f16", 0.7), (140, 1155, 64, "padded", 65536, "u8", 0.7), (131, 1155, 64, "padded", 65536, "f16", 0.7),
    (270, 523, 64, "random", 65536, None, 1.0), (257, 259, 128, "padded", 65536, None, 1.0), (260, 260, 64, "causal", 0, None, 1.0)])
@pytest.mark.parametrize("wide", [False, True])
def test_pre_passes(Sq, Sk, D, mask, nxt, drop, keep, wide):
    B, N, g = 2, 1, torch.Generator().manual_seed(Sq + Sk)
    q, k, v = (torch.randn(B, N, S, D, generator=g).half() for S in (Sq, Sk, Sk))
    dO = torch.randn(B, N, Sq, D, generator=g).half()
    m = _masks(mask, B, Sq, Sk)
    okw = dict(scale=D ** -0.5, attn_mask=m, next_block_num=nxt)
    arg = None
    if drop == "seed":
        arg = (1234567891011, 7)
        okw.update(drop_mask=phx.dropout_keep_mask(B, N, Sq, Sk, *arg, keep), keep_prob=phx.keep_threshold(keep) / 256.0)
    elif drop is not None:
        d = (np.random.default_rng(Sq).random((B, N, Sq, Sk)) < keep).astype(np.uint8)
        okw.update(drop_mask=d, keep_prob=keep)
        arg = torch.from_numpy(d).to(DEV) if drop == "u8" else torch.from_numpy(d).to(DEV).half() / keep
    mt = None if m is None else torch.from_numpy(m).to(DEV)
    if mt is not None and wide:
        mt = mt.half()
    qd, kd, vd = (t.to(DEV).requires_grad_(True) for t in (q, k, v))
    op = get_flash_attention(next_block_num=nxt, scale=D ** -0.5, keep_prob=keep if drop else None)
    o, lse = op(qd, kd, vd, mt, arg)
    grads = torch.autograd.grad(o, (qd, kd, vd), dO.to(DEV))
    f = lambda t: t.detach().float().cpu().numpy()
    O, L = orc.unfused_fwd(f(q), f(k), f(v), **okw)
    refs = (O,) + orc.unfused_bwd(f(q), f(k), f(v), f(dO), **okw, O_saved=f(o))
    for name, ref, got in zip(("O", "dQ", "dK", "dV"), refs, (o,) + grads):
        ok, ratio, mx = orc.tolerance_gate(ref, f(got))
        assert ok, f"{name}: worst ratio {ratio:.3f}, max |d| {mx:.3e}"
    assert np.max(np.abs(L - f(lse))) < 1e-4 * max(1.0, np.abs(L).max() / 10)


def test_row_prefix_and_causal_kind_leave_out_the_same_blocks():
    """Without a shared buffer the blocks behind a row prefix or the causal compare are left out as well."""
    B, N, S, D, keep = 1, 2, 700, 64, 0.8
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(B, N, S, D, generator=g).half() for _ in range(3))
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    drop = phx.dropout_keep_mask(B, N, S, S, 99, 4, keep)
    for kw, m in ((dict(row_block_prefix=256), j >= (i // 256 + 1) * 256), (dict(mask_kind=_capi.MASK_CAUSAL), j > i)):
        qd = q.to(DEV)
        p = _capi.make_params(qd, k.to(DEV), v.to(DEV), scale=D ** -0.5, keep_prob=keep, drop_seed=99, drop_offset=4, **kw)
        o, _ = _capi.fa_fwd(p, qd)
        O, _ = orc.unfused_fwd(q.float().numpy(), k.float().numpy(), v.float().numpy(), scale=D ** -0.5, attn_mask=m[None].astype(np.uint8),
                               drop_mask=drop, keep_prob=phx.keep_threshold(keep) / 256.0)
        ok, ratio, mx = orc.tolerance_gate(O, o.float().cpu().numpy())
        assert ok, f"{kw}: worst ratio {ratio:.3f}, max |d| {mx:.3e}"


@pytest.mark.parametrize("source", ["seed", "u8"])
def test_shared_keep_bits_hold_for_another_band(source):
    """A lent buffer that a call with a narrow band filled serves a call on the same mask with a wider one."""
    B, N, S, D, keep = 1, 2, 400, 64, 0.7
    g = torch.Generator().manual_seed(11)
    q, k, v = (torch.randn(B, N, S, D, generator=g).half().to(DEV) for _ in range(3))
    kw = dict(scale=D ** -0.5, keep_prob=keep, mask_kind=_capi.MASK_DENSE_U8, attn_mask=torch.from_numpy(_masks("random", B, S, S)).to(DEV))
    kw.update(dict(drop_seed=77, drop_offset=2) if source == "seed" else
              dict(drop_mask=(torch.rand(B, N, S, S, generator=g) < keep).to(torch.uint8).to(DEV)))
    narrow, wide = _capi.make_params(q, k, v, prev_block_num=0, next_block_num=0, **kw), _capi.make_params(q, k, v, **kw)
    own = _capi.fa_fwd(wide, q)
    grads = _capi.fa_bwd(wide, q, k, v, own[0], q, own[1])
    bits = _capi.attach_drop_bits(narrow, DEV)
    bits.fill_(0xA5)
    _capi.fa_fwd(narrow, q)
    wide.drop_bits, wide.drop_bits_filled = narrow.drop_bits, 1
    shared = _capi.fa_fwd(wide, q)
    for a, b in zip(own + grads, shared + _capi.fa_bwd(wide, q, k, v, own[0], q, own[1])):
        assert torch.equal(a, b)
