"""GPU tests of the launches that few query rows or few heads take: forward workgroups of key groups, and key ranges
cut into slices that a second kernel adds up.  Sizes sit on the edges of the 32-, 64- and 128-row units, with slices
in which some rows see no key at all.  Gate: that of the parity tests (every element within 2e-3 + 1e-3 |oracle|)."""
import ctypes

import numpy as np
import pytest
import torch

from acctransformer_amd import _capi
from oracle import unfused_attention as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _forward(p, q, workspace_bytes):
    lib = _capi.load()
    o, lse = torch.empty_like(q), torch.empty(q.shape[:3], dtype=torch.float32, device=DEV)
    p.o_stride = _capi._bhs_strides(o)
    ws = torch.empty(max(workspace_bytes, 256), dtype=torch.uint8, device=DEV)
    rc = lib.acct_fa_fwd(ctypes.byref(p), o.data_ptr(), lse.data_ptr(), ws.data_ptr(), workspace_bytes,
                         ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.acct_last_error().decode()
    return o, lse


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Sq, Sk, D, side, splits", [
    (64, 128, 64, "none", False), (65, 129, 128, "causal", False), (33, 31, 80, "none", False), (300, 520, 40, "mask", False),
    (257, 257, 128, "mask", False), (130, 500, 128, "drop", False), (200, 333, 64, "row_bias", False), (96, 264, 128, "bias", False),
    (128, 400, 160, "none", False), (1, 3000, 128, "none", True), (64, 8197, 40, "none", True), (200, 6000, 128, "mask", True),
    (40, 5000, 64, "drop", True), (72, 4104, 128, "row_bias", True), (70, 4104, 80, "bias", True), (31, 5000, 160, "none", True),
    (129, 4500, 256, "none", True), (1500, 4000, 128, "prefix", False), (2600, 4000, 128, "prefix", True), (300, 6000, 64, "band", True), (1500, 2000, 128, "narrow", False),
    (150, 17000, 64, "mask", True)])
def test_forward_of_small_grids(Sq, Sk, D, side, splits, dtype):
    B, N, g = 1, 2, torch.Generator().manual_seed(Sq * 7 + Sk)
    q, k, v = (torch.randn(B, N, S, D, generator=g).to(dtype) for S in (Sq, Sk, Sk))
    rng = np.random.default_rng(Sk)
    kw, okw = dict(scale=D ** -0.5), dict(scale=D ** -0.5)
    if side == "causal":
        kw.update(mask_kind=_capi.MASK_CAUSAL)
        okw.update(attn_mask=np.triu(np.ones((1, Sq, Sk), np.uint8), 1))
    if side == "mask":                                   # long runs of hidden keys: whole slices without a visible one
        m = (rng.random((B, Sq, Sk)) < 0.3).astype(np.uint8)
        m[:, : Sq // 2, 128:] = 1
        m[:, :, 0] = 0
        kw.update(mask_kind=_capi.MASK_DENSE_U8, attn_mask=torch.from_numpy(m).to(DEV))
        okw.update(attn_mask=m)
    if side == "prefix":
        prefix = 1280 if splits else 512                 # (the last group of rows sees 3840 or 1536 keys: the slices are cut from those)
        kw.update(row_block_prefix=prefix)
        okw.update(attn_mask=(np.arange(Sk)[None, None, :] >= ((np.arange(Sq) // prefix + 1) * prefix)[None, :, None]).astype(np.uint8))
    if side in ("band", "narrow"):                       # the slices are cut from what a row block sees: less than Sk, and not from 0
        prev, nxt = (1, 40) if side == "band" else (2, 1)
        kw.update(prev_block_num=prev, next_block_num=nxt)
        okw.update(prev_block_num=prev, next_block_num=nxt)
    if side == "drop":
        d = (rng.random((B, N, Sq, Sk)) < 0.8).astype(np.uint8)
        kw.update(drop_mask=torch.from_numpy(d).to(DEV), keep_prob=0.8)
        okw.update(drop_mask=d, keep_prob=0.8)
    if side in ("bias", "row_bias"):
        al = (0.3 * torch.randn(1, N, 1 if side == "row_bias" else Sq, Sk, generator=g)).to(dtype)
        kw.update(alibi=al.to(DEV))
        okw.update(alibi=al.float().numpy())
    qd = q.to(DEV)
    p = _capi.make_params(qd, k.to(DEV), v.to(DEV), **kw)
    lib = _capi.load()
    least, most = lib.acct_fa_fwd_workspace_bytes(ctypes.byref(p)), lib.acct_fa_fwd_split_workspace_bytes(ctypes.byref(p))
    assert (most > least) == splits, (least, most)
    O, L = orc.unfused_fwd(q.float().numpy(), k.float().numpy(), v.float().numpy(), **okw)
    tol = dict(atol=2e-3, rtol=1e-3) if dtype == torch.float16 else dict(atol=2e-2, rtol=1e-2)      # (the parity tests' gates)
    for size in {least, most}:
        o, lse = _forward(p, qd, size)
        ok, ratio, mx = orc.tolerance_gate(O, o.float().cpu().numpy(), **tol)
        assert ok, f"workspace {size}: worst ratio {ratio:.3f}, max |d| {mx:.3e}"
        assert np.max(np.abs(L - lse.cpu().numpy())) < 1e-4 * max(1.0, np.abs(L).max() / 10), f"LSE, workspace {size}"


@pytest.mark.parametrize("Sq, Sk, D", [(64, 8192, 40), (1, 3072, 128), (129, 4608, 256)])
def test_infinite_values_stay_infinite(Sq, Sk, D):
    """An infinity of V belongs to its output column only, whichever slice of the keys holds it.  (Whole key tiles: a tile
    that the keys end in repeats the last row of V with probability 0.)"""
    g = torch.Generator().manual_seed(Sk)
    q, k, v = (torch.randn(1, 2, S, D, generator=g).half() for S in (Sq, Sk, Sk))
    v[:, :, Sk - 1, 5], v[:, :, Sk // 2, 6], v[:, :, 0, 7] = float("inf"), float("-inf"), float("inf")
    qd = q.to(DEV)
    p = _capi.make_params(qd, k.to(DEV), v.to(DEV), scale=D ** -0.5)
    lib = _capi.load()
    for size in (lib.acct_fa_fwd_workspace_bytes(ctypes.byref(p)), lib.acct_fa_fwd_split_workspace_bytes(ctypes.byref(p))):
        o = _forward(p, qd, size)[0].cpu()
        assert (o[..., 5] == float("inf")).all() and (o[..., 6] == float("-inf")).all() and (o[..., 7] == float("inf")).all(), f"workspace {size}"
        finite = torch.ones(D, dtype=torch.bool)
        finite[5:8] = False
        assert torch.isfinite(o[..., finite]).all()
