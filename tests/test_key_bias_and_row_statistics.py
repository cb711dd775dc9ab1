"""GPU tests of the kernel variants for a bias that depends on the key only, and of the dK/dV kernel's accumulators that
start from the row statistics.  Key counts on the edges of the 64- and 128-key tiles, one to several query tiles (the
first one staged is ragged, the rest take the kept offsets), head dims with and without padding, grids that take one and
two key groups per wave; every kind of mask, so that both bodies of the variants run; rows that see nothing but masked keys,
whose LSE is near -10000; scales far below 1 / sqrt(D).  Reference: the operator in float32 with torch.  Gate: that of the parity tests (every element within
2e-3 + 1e-3 |reference| in fp16, 2e-2 + 1e-2 |reference| in bf16)."""
import pytest
import torch

from acctransformer_amd import _capi
from acctransformer_amd.flash_attention.ops.flash_attention.flash_attention_impl import get_flash_attention
from oracle import unfused_attention as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _mask(kind, B, Sq, Sk, g):
    i, j = torch.arange(Sq, device=DEV)[:, None], torch.arange(Sk, device=DEV)[None, :]
    if kind == "causal":
        return (j > i)[None].to(torch.uint8)
    if kind == "padded":
        lens = torch.randint(Sk // 3, Sk + 1, (B,), generator=g, device=DEV)
        return (j[None] >= lens[:, None, None]).expand(B, Sq, Sk).to(torch.uint8).contiguous()
    if kind in ("random", "blind rows"):
        m = (torch.rand(B, Sq, Sk, generator=g, device=DEV) < 0.3).to(torch.uint8)
        m[:, :, 0] = 0
        if kind == "blind rows":
            m[:, 3::7] = 1
        return m
    return None


def _check(B, N, Sq, Sk, D, dtype, mask, biased, scale=None, nxt=65536):
    g = torch.Generator(device=DEV).manual_seed(Sq * 7 + Sk + D)
    scale = D ** -0.5 if scale is None else scale
    q, k, v, dO = (torch.randn(B, N, S, D, generator=g, device=DEV).to(dtype) for S in (Sq, Sk, Sk, Sq))
    m = _mask(mask, B, Sq, Sk, g)
    al = torch.randn(1, N, 1, Sk, generator=g, device=DEV).to(dtype) if biased else None
    qf, kf, vf, df = (t.float() for t in (q, k, v, dO))
    s = qf @ kf.transpose(2, 3) * scale
    s = s + al.float() if biased else s
    s = s - 10000.0 * m[:, None].float() if m is not None else s
    if nxt == 0:
        b = torch.arange(Sk, device=DEV)[None, :] // 128 > torch.arange(Sq, device=DEV)[:, None] // 128
        s = s.masked_fill(b, float("-inf"))
    x = [t.clone().requires_grad_(True) for t in (q, k, v)]
    o, lse = get_flash_attention(scale=scale, next_block_num=nxt)(*x, m, None, al)
    got = (o,) + torch.autograd.grad(o, x, dO)
    P = torch.softmax(s, 3)
    # (D from the O that the backward is given, as it defines it)
    dS = P * (df @ vf.transpose(2, 3) - (df * o.detach().float()).sum(3, keepdim=True))
    want = (P @ vf, dS @ kf * scale, dS.transpose(2, 3) @ qf * scale, P.transpose(2, 3) @ df)
    wide = dtype == torch.bfloat16
    for name, a, b in zip(("O", "dQ", "dK", "dV"), want, got):
        ok, ratio, mx = orc.tolerance_gate(a.detach().cpu().numpy(), b.detach().float().cpu().numpy(), atol=2e-2 if wide else 2e-3, rtol=1e-2 if wide else 1e-3)
        assert ok, f"{name}: worst ratio {ratio:.3f}, max |d| {mx:.3e}"
    L = torch.logsumexp(s, 3)
    assert float((L - lse).abs().max()) < 1e-4 * max(1.0, float(L.abs().max()) / 10)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Sq, Sk, D, mask, nxt", [
    (64, 64, 64, None, 65536), (65, 72, 128, None, 65536), (200, 136, 80, "random", 65536), (264, 264, 128, "causal", 0),
    (257, 264, 64, "causal", 65536), (520, 520, 72, "causal", 0), (300, 640, 128, "padded", 65536), (385, 128, 96, "blind rows", 65536),
    (192, 1032, 128, None, 65536), (129, 131, 64, "random", 65536)])
def test_key_only_bias(Sq, Sk, D, mask, nxt, dtype):
    _check(2, 3, Sq, Sk, D, dtype, mask, True, nxt=nxt)


@pytest.mark.parametrize("D, mask, nxt, biased", [
    (128, "causal", 0, True), (128, "padded", 65536, True), (64, "random", 65536, True), (80, None, 65536, True),
    (128, "causal", 0, False), (128, "padded", 65536, False), (64, None, 65536, False), (80, "causal", 65536, False)])
def test_grids_of_two_key_groups(D, mask, nxt, biased):
    _check(2, 64, 584, 512, D, torch.float16, mask, biased, nxt=nxt)


@pytest.mark.parametrize("Sq, Sk, D, mask, scale", [
    (130, 140, 128, "blind rows", None), (300, 200, 64, "blind rows", None), (70, 256, 160, "blind rows", None), (257, 129, 40, "random", None),
    (200, 200, 64, None, 1e-3), (200, 200, 64, None, 1e-20), (200, 200, 128, None, 1e-35)])
def test_row_statistics_in_the_accumulators(Sq, Sk, D, mask, scale):
    _check(1, 4, Sq, Sk, D, torch.float16, mask, False, scale=scale)


def test_key_only_bias_without_a_mask_tensor():
    """ACCT_MASK_CAUSAL by index compare gives the bits of the same mask handed over as a tensor."""
    B, N, S, D = 1, 4, 328, 128
    g = torch.Generator(device=DEV).manual_seed(5)
    q, k, v, dO = (torch.randn(B, N, S, D, generator=g, device=DEV).half() for _ in range(4))
    al = torch.randn(1, N, 1, S, generator=g, device=DEV).half()
    m = _mask("causal", B, S, S, g)
    outs = []
    for kw in (dict(mask_kind=_capi.MASK_CAUSAL), dict(mask_kind=_capi.MASK_DENSE_U8, attn_mask=m)):
        p = _capi.make_params(q, k, v, scale=D ** -0.5, alibi=al, **kw)
        o, lse = _capi.fa_fwd(p, q)
        outs.append((o, lse) + _capi.fa_bwd(p, q, k, v, o, dO, lse))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
