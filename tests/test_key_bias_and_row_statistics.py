"""GPU tests of the kernel variants for a bias that depends on the key only, and of the row statistics in the dK/dV kernel.
Key counts on the edges of the 64- and 128-key tiles, one to several query tiles (the
first one staged is ragged, the rest take the kept offsets), head dims with and without padding, grids that take one and
two key groups per wave; every kind of mask, so that both bodies of the variants run; rows that see nothing but masked keys,
whose LSE is near -10000; scales far below 1 / sqrt(D).  Reference: the operator in float64 with torch.  Gate: that of the parity tests (every element within
2e-3 + 1e-3 |reference| in fp16, 2e-2 + 1e-2 |reference| in bf16).  Where scores, dP and D are exact in float32 the
kernel's own rounding is checked: P and dS are what one rounding of their difference to the row's statistic gives."""
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


def _check(B, N, Sq, Sk, D, dtype, mask, biased, scale=None, nxt=65536, prev=65536, prefix=0, per_batch=False, low=None, keep=1.0):
    g = torch.Generator(device=DEV).manual_seed(Sq * 7 + Sk + D)
    scale = D ** -0.5 if scale is None else scale
    q, k, v, dO = (torch.randn(B, N, S, D, generator=g, device=DEV).to(dtype) for S in (Sq, Sk, Sk, Sq))
    m = _mask(mask, B, Sq, Sk, g)
    al = torch.randn(B if per_batch else 1, N, 1, Sk, generator=g, device=DEV).to(dtype) if biased else None
    if low is not None:
        al[..., 1::3] = low if low != "lowest" else torch.finfo(dtype).min
    drop = (torch.rand(B, N, Sq, Sk, generator=g, device=DEV) < keep).to(torch.uint8) if keep < 1 else None
    qf, kf, vf, df = (t.double() for t in (q, k, v, dO))     # (beside a mask's 10000, float32 rounds a score to 5e-4)
    s = qf @ kf.transpose(2, 3) * scale
    s = s + al.double() if biased else s
    s = s - 10000.0 * m[:, None].double() if m is not None else s
    i, j = torch.arange(Sq, device=DEV)[:, None], torch.arange(Sk, device=DEV)[None, :]
    s = s.masked_fill((j // 128 > i // 128 + nxt) | (j // 128 < i // 128 - prev), float("-inf"))
    if prefix:
        s = s.masked_fill(j >= (i // prefix + 1) * prefix, float("-inf"))
    x = [t.clone().requires_grad_(True) for t in (q, k, v)]
    if prefix:                                           # (the C interface only)
        p = _capi.make_params(q, k, v, scale=scale, alibi=al, prev_block_num=prev, next_block_num=nxt, row_block_prefix=prefix, drop_mask=drop,
                              keep_prob=keep, mask_kind=_capi.MASK_DENSE_U8 if m is not None else _capi.MASK_NONE, attn_mask=m)
        o, lse = _capi.fa_fwd(p, q)
        got = (o,) + _capi.fa_bwd(p, q, k, v, o, dO, lse)
    else:
        o, lse = get_flash_attention(scale=scale, prev_block_num=prev, next_block_num=nxt, keep_prob=keep)(*x, m, drop, al)
        got = (o,) + torch.autograd.grad(o, x, dO)
    P = torch.softmax(s, 3)
    kept = drop.double() / keep if drop is not None else 1.0
    # (D from the O that the backward is given, as it defines it)
    dS = P * (df @ vf.transpose(2, 3) * kept - (df * o.detach().double()).sum(3, keepdim=True))
    want = ((P * kept) @ vf, dS @ kf * scale, dS.transpose(2, 3) @ qf * scale, (P * kept).transpose(2, 3) @ df)
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


# (B, N, Sq, Sk, D), mask, next_block_num, key-only bias, keep_prob: tests/test_index_math.py checks that the dK/dV plan gives
# each two key groups per wave.  (A causal launch of fewer rows has one.)
TWO_KEY_GROUPS = [
    ((2, 64, 768, 768, 128), "causal", 0, True, 1.0), ((2, 64, 584, 512, 128), "padded", 65536, True, 1.0), ((2, 64, 584, 512, 64), "random", 65536, True, 1.0),
    ((2, 64, 584, 512, 80), None, 65536, True, 1.0), ((2, 64, 768, 768, 128), "causal", 0, False, 1.0), ((2, 64, 584, 512, 128), "padded", 65536, False, 1.0),
    ((2, 64, 584, 512, 64), None, 65536, False, 1.0), ((2, 64, 584, 512, 80), "causal", 65536, False, 1.0), ((2, 64, 584, 512, 128), "random", 65536, False, 1.0),
    ((2, 64, 584, 456, 128), "padded", 65536, False, 0.8), ((2, 64, 768, 768, 128), "causal", 0, False, 0.8), ((2, 64, 584, 512, 64), "random", 65536, True, 0.8),
    ((2, 64, 584, 500, 128), None, 65536, True, 0.8)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape, mask, nxt, biased, keep", TWO_KEY_GROUPS)
def test_grids_of_two_key_groups(shape, mask, nxt, biased, keep, dtype):
    _check(*shape, dtype, mask, biased, nxt=nxt, keep=keep)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Sq, Sk, D, mask, prev, nxt, prefix, low", [
    (300, 392, 128, "random", 1, 1, 0, None), (520, 520, 64, "causal", 0, 0, 0, None), (640, 640, 80, None, 65536, 65536, 256, "lowest"),
    (400, 456, 128, "padded", 65536, 65536, 0, float("-inf")), (385, 264, 128, "blind rows", 2, 65536, 128, "lowest"), (700, 704, 128, "causal", 65536, 0, 0, float("-inf"))])
def test_key_only_bias_per_batch_entry(Sq, Sk, D, mask, prev, nxt, prefix, low, dtype):
    """One bias per batch entry and head, in bands, under row prefixes, and with keys that the bias hides."""
    _check(3, 2, Sq, Sk, D, dtype, mask, True, prev=prev, nxt=nxt, prefix=prefix, per_batch=True, low=low)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D, mask, keep", [(256, "random", 1.0), (256, None, 0.8), (256, "padded", 0.8), (160, "random", 1.0), (160, "random", 0.8)])
def test_wide_head_dims_over_several_query_tiles(D, mask, keep, dtype):
    _check(2, 3, 420, 390, D, dtype, mask, False, keep=keep)


@pytest.mark.parametrize("Sq, Sk, D, mask, scale", [
    (130, 140, 128, "blind rows", None), (300, 200, 64, "blind rows", None), (70, 256, 160, "blind rows", None), (257, 129, 40, "random", None),
    (200, 200, 64, None, 1e-3), (200, 200, 64, None, 1e-20), (200, 200, 128, None, 1e-35)])
def test_rows_of_masked_keys_and_small_scales(Sq, Sk, D, mask, scale):
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


@pytest.mark.parametrize("D", [64, 80, 128])
@pytest.mark.parametrize("heads", [2, 256])                    # one and two key groups per wave
@pytest.mark.parametrize("bias", ["none", "key", "full"])
def test_p_takes_one_rounding_of_score_minus_lse(D, heads, bias):
    """Scores (and bias / scale) are whole numbers near 16384, exact in float32 in any order, and LSE is close to them: P is
    exp2 of scale*log2e * S - LSE*log2e, rounded once, and dV with one-hot dO is P in fp16.  The difference of two numbers in
    the thousands taken in several roundings would move P by up to 1e-4, a quarter of an fp16 spacing, and 6 % of the entries with it;
    exp2's own last place moves 3e-5 of them.  Gate: 1 %."""
    g = torch.Generator(device=DEV).manual_seed(D + heads)
    Sk, scale = 256, 0.125
    const = 16 * 32 * 32
    def ints(S):
        x = torch.randint(-1, 2, (1, heads, S, D), generator=g, device=DEV).half()
        x[..., D - 16:] = 32
        return x
    q, k, v = ints(D), ints(Sk), torch.randn(1, heads, Sk, D, generator=g, device=DEV).half()
    dO = torch.eye(D, device=DEV).half().expand(1, heads, D, D).contiguous()
    al = None if bias == "none" else torch.randint(-8, 9, (1, heads, 1 if bias == "key" else D, Sk), generator=g, device=DEV).half() / 4
    S = q.double() @ k.double().transpose(2, 3) + (al.double() / scale if al is not None else 0)
    assert float((S - const).abs().max()) < 256
    lse = (scale * S.amax(3) + torch.rand(1, heads, D, generator=g, device=DEV, dtype=torch.float64)).float()
    log2e = torch.tensor(1.4426950408889634, dtype=torch.float32, device=DEV)
    mul, off = (torch.tensor(scale, dtype=torch.float32, device=DEV) * log2e).double(), (lse * log2e).double()
    want = torch.exp2((S * mul - off[..., None]).float().double()).half()
    p = _capi.make_params(q, k, v, scale=scale, alibi=al)
    dv = _capi.fa_bwd(p, q, k, v, torch.zeros_like(q), dO, lse)[2]
    differ = float((dv.transpose(2, 3) != want).double().mean())
    assert differ < 0.01, f"{100 * differ:.2f} % of P"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("heads", [2, 256])
def test_ds_takes_one_rounding_of_dp_minus_d(D, heads, dtype):
    """dP is a sum of whole numbers, exact in float32 although it passes 2^18 on the way, and D is a fraction: with P = 1
    (K = 0, LSE = 0) and one-hot Q, dK is dP - D in the element type, to the last bit."""
    g = torch.Generator(device=DEV).manual_seed(D + heads)
    Sk = 256
    eye = torch.eye(D, device=DEV).to(dtype).expand(1, heads, D, D).contiguous()
    dO = torch.ones(1, heads, D, D, device=DEV)
    v = torch.randint(-1, 2, (1, heads, Sk, D), generator=g, device=DEV).float()
    dO[..., :32], v[..., :16], v[..., 16:32] = 128, 128, -128
    o = torch.zeros(1, heads, D, D, device=DEV)
    o[..., D - 1] = torch.rand(1, heads, D, generator=g, device=DEV)
    dO, v, o = dO.to(dtype), v.to(dtype), o.to(dtype)
    k, lse = torch.zeros_like(v), torch.zeros(1, heads, D, device=DEV)
    p = _capi.make_params(eye, k, v, scale=1.0)
    dk = _capi.fa_bwd(p, eye, k, v, o, dO, lse)[1]
    want = (dO.double() @ v.double().transpose(2, 3) - o[..., D - 1:].double()).transpose(2, 3).to(dtype)
    assert torch.equal(dk, want), f"{int((dk != want).sum())} of {want.numel()} differ"
