"""GPU tests of the backward launches that grids below a full round take: dQ workgroups of two key groups, dK/dV
workgroups of 128 keys (one 32-key group per wave), query ranges cut into slices that a second kernel adds up.  Sizes
sit on the edges of the 32-, 64- and 128-row units; every launch runs with the workspace it asks for, and where
it cuts slices with one that is too small for all of them and one without room for any.  Gate: that of the parity tests (every element within 2e-3 + 1e-3 |oracle|)."""
import ctypes
import re

import numpy as np
import pytest
import torch

from acctransformer_amd import _capi
from oracle import unfused_attention as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _least_bwd_workspace(p):
    """The smallest workspace that acct_fa_bwd accepts, from the text with which it refuses none."""
    lib, buf = _capi.load(), (ctypes.c_char * 64)()
    addr = ctypes.addressof(buf) // 16 * 16 + 16
    assert lib.acct_fa_bwd(ctypes.byref(p), *([addr] * 6), None, 0, None) == -7
    return int(re.search(r"need (\d+) bytes", lib.acct_last_error().decode()).group(1))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Sq, Sk, D, side, sliced", [
    (64, 128, 64, "none", False), (65, 129, 128, "causal", False), (33, 31, 80, "none", False), (300, 520, 40, "mask", False),
    (257, 257, 128, "mask", False), (130, 500, 128, "drop", False), (200, 333, 64, "row_bias", False), (96, 264, 128, "bias", False),
    (161, 200, 80, "bias", False), (400, 77, 40, "none", True), (700, 77, 128, "drop", True), (650, 96, 64, "bias", True),
    (1100, 160, 160, "none", True), (513, 300, 256, "drop", True), (260, 390, 128, "tile", False)])
def test_backward_of_small_grids(Sq, Sk, D, side, sliced, dtype):
    B, N, g = 1, 2, torch.Generator().manual_seed(Sq * 5 + Sk)
    q, k, v = (torch.randn(B, N, S, D, generator=g).to(dtype) for S in (Sq, Sk, Sk))
    dO = torch.randn(B, N, Sq, D, generator=g).to(dtype)
    rng = np.random.default_rng(Sk)
    kw, okw = dict(scale=D ** -0.5), dict(scale=D ** -0.5)
    if side == "causal":
        kw.update(mask_kind=_capi.MASK_CAUSAL)
        okw.update(attn_mask=np.triu(np.ones((1, Sq, Sk), np.uint8), 1))
    if side == "tile":
        kw.update(mask_kind=_capi.MASK_TILE_U8, attn_mask=torch.triu(torch.ones(128, 128, dtype=torch.uint8), 1).to(DEV), next_block_num=0)
        okw.update(attn_mask=np.triu(np.ones((1, Sq, Sk), np.uint8), 1))
    if side == "mask":
        m = (rng.random((B, Sq, Sk)) < 0.3).astype(np.uint8)
        m[:, : Sq // 2, 128:] = 1
        m[:, :, 0] = 0
        kw.update(mask_kind=_capi.MASK_DENSE_U8, attn_mask=torch.from_numpy(m).to(DEV))
        okw.update(attn_mask=m)
    if side == "drop":
        d = (rng.random((B, N, Sq, Sk)) < 0.8).astype(np.uint8)
        kw.update(drop_mask=torch.from_numpy(d).to(DEV), keep_prob=0.8)
        okw.update(drop_mask=d, keep_prob=0.8)
    if side in ("bias", "row_bias"):
        al = (0.3 * torch.randn(1, N, 1 if side == "row_bias" else Sq, Sk, generator=g)).to(dtype)
        kw.update(alibi=al.to(DEV))
        okw.update(alibi=al.float().numpy())
    qd, kd, vd, dd = (t.to(DEV) for t in (q, k, v, dO))
    p = _capi.make_params(qd, kd, vd, **kw)
    o, lse = _capi.fa_fwd(p, qd)
    most = _capi.load().acct_fa_bwd_workspace_bytes(ctypes.byref(p))
    refs = orc.unfused_bwd(*(t.float().numpy() for t in (q, k, v, dO)), **okw, O_saved=o.float().cpu().numpy())
    first = None
    wide = dtype == torch.bfloat16
    least = _least_bwd_workspace(p)
    assert (most - (least + 255) // 256 * 256 > 0) == sliced
    for size in (most, most - 256, least) if sliced else (most,):      # all slices, fewer or none, none
        grads = _capi.fa_bwd(p, qd, kd, vd, o, dd, lse, workspace_bytes=size)
        for name, ref, got in zip(("dQ", "dK", "dV"), refs, grads):
            ok, ratio, mx = orc.tolerance_gate(ref, got.float().cpu().numpy(), atol=2e-2 if wide else 2e-3, rtol=1e-2 if wide else 1e-3)
            assert ok, f"{name}, workspace {size} of {most}: worst ratio {ratio:.3f}, max |d| {mx:.3e}"
        again = _capi.fa_bwd(p, qd, kd, vd, o, dd, lse, workspace_bytes=size)
        assert all(torch.equal(x, y) for x, y in zip(grads, again)), "not deterministic"
        first = first or grads
    assert torch.equal(first[0], grads[0])                   # dQ does not depend on the slices
