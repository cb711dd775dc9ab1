"""GPU tests of the forward's pipelined tile loop (head dims up to 64, whole workgroups of 256 rows, rows that see 1024 keys and
more on average): an even and an odd number of tiles, a ragged last one, workgroups of one tile and two among the causal
ones, waves whose tiles start or end earlier than the workgroup's (causal, band, row prefix), with every step of the pipeline
in its fused form or not; and the plain loop that serves shorter walks, at the same edges.  Gate: that of the parity tests."""
import numpy as np
import pytest
import torch

from acctransformer_amd import _capi
from oracle import unfused_attention as orc
from test_key_group_merge import forward

pytestmark = pytest.mark.gpu


SHORT = [
    (256, 77, 64, "none"), (256, 129, 40, "none"), (230, 384, 64, "none"), (256, 500, 24, "none"), (256, 641, 64, "none"),
    (512, 512, 64, "causal"), (500, 700, 40, "causal"), (700, 300, 64, "causal"), (512, 512, 64, "causal tensor"),
    (768, 768, 64, "band"), (768, 769, 40, "late band"), (768, 768, 64, "prefix")]
LONG = [                                                       # (the pipelined loop's)
    (256, 1024, 64, "none"), (230, 1025, 40, "none"), (256, 1100, 64, "none"), (500, 1280, 24, "none"), (256, 1535, 40, "none"),
    (2048, 2048, 64, "causal"), (2200, 2100, 40, "causal"), (2050, 3000, 64, "causal"), (2048, 2048, 64, "causal tensor"),
    (4096, 4095, 40, "wide band"), (2048, 2050, 64, "wide late band"), (2048, 2048, 64, "prefix")]


def heads(Sq):
    return (16, 16) if Sq < 2048 else (2, 16) if Sq < 4096 else (1, 16)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Sq, Sk, D, side", SHORT + LONG)
def test_pipelined_forward(Sq, Sk, D, side, dtype):
    (B, N), g = heads(Sq), torch.Generator().manual_seed(Sq * 3 + Sk)
    q, k, v = (torch.randn(B, N, S, D, generator=g).to(dtype) for S in (Sq, Sk, Sk))
    kw, okw = dict(scale=D ** -0.5), dict(scale=D ** -0.5)
    triu = np.triu(np.ones((1, Sq, Sk), np.uint8), 1)
    if side == "causal":
        kw.update(mask_kind=_capi.MASK_CAUSAL)
        okw.update(attn_mask=triu)
    elif side == "causal tensor":
        kw.update(mask_kind=_capi.MASK_DENSE_U8, attn_mask=torch.from_numpy(triu).cuda())
        okw.update(attn_mask=triu)
    elif "band" in side:
        wide = 10 if "wide" in side else 2
        prev, nxt = (0, wide) if "late" in side else (wide, 0)
        kw.update(prev_block_num=prev, next_block_num=nxt)
        okw.update(prev_block_num=prev, next_block_num=nxt)
    elif side == "prefix":
        kw.update(row_block_prefix=384)
        okw.update(attn_mask=(np.arange(Sk)[None, None, :] >= ((np.arange(Sq) // 384 + 1) * 384)[None, :, None]).astype(np.uint8))
    o, lse = forward(q, k, v, kw)
    tol = dict(atol=2e-3, rtol=1e-3) if dtype == torch.float16 else dict(atol=2e-2, rtol=1e-2)
    for b in {0, B - 1}:                                 # (the heads of one batch entry at a time: the oracle is on the CPU)
        O, L = orc.unfused_fwd(*(t[b:b + 1].float().numpy() for t in (q, k, v)), **okw)
        ok, ratio, mx = orc.tolerance_gate(O, o[b:b + 1].float().cpu().numpy(), **tol)
        assert ok, f"batch {b}: worst ratio {ratio:.3f}, max |d| {mx:.3e}"
        assert np.max(np.abs(L - lse[b:b + 1].cpu().numpy())) < 1e-4 * max(1.0, np.abs(L).max() / 10), f"LSE, batch {b}"
