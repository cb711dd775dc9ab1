"""GPU tests of the forward's key groups: 256-key tiles at head dims up to 64 (tiles that span two blocks of a mask, ragged ends
in every 64-key share) and the merge that all groups of a workgroup take part in (2, 3, 4, 6, 8 and 10 column pieces per group).
Gate: that of the parity tests (every element within 2e-3 + 1e-3 |oracle|; bf16 2e-2 / 1e-2)."""
import ctypes

import numpy as np
import pytest
import torch

from acctransformer_amd import _capi
from oracle import unfused_attention as orc

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def forward(q, k, v, kw):
    qd = q.to(DEV)
    p = _capi.make_params(qd, k.to(DEV), v.to(DEV), **kw)
    lib = _capi.load()
    o, lse = torch.empty_like(qd), torch.empty(qd.shape[:3], dtype=torch.float32, device=DEV)
    p.o_stride = _capi._bhs_strides(o)
    size = lib.acct_fa_fwd_workspace_bytes(ctypes.byref(p))
    ws = torch.empty(max(size, 256), dtype=torch.uint8, device=DEV)
    rc = lib.acct_fa_fwd(ctypes.byref(p), o.data_ptr(), lse.data_ptr(), ws.data_ptr(), size, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.acct_last_error().decode()
    return o, lse


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B, N, Sq, Sk, D, side", [
    (1, 2, 64, 128, 64, "none"), (1, 2, 65, 129, 64, "none"), (1, 2, 1, 192, 40, "none"), (1, 2, 63, 193, 48, "causal"),
    (1, 2, 300, 256, 64, "causal"), (1, 2, 257, 257, 40, "causal"), (1, 3, 200, 320, 64, "padded"), (2, 2, 384, 384, 64, "padded"),
    (1, 2, 511, 513, 40, "padded"), (1, 2, 700, 700, 64, "mixed"), (1, 2, 640, 640, 64, "band"), (1, 2, 640, 641, 56, "late band"),
    (1, 2, 896, 896, 64, "prefix"), (1, 1, 130, 9000, 64, "mixed"),      # (more than 64 blocks: the class window moves)
    (2, 10, 1024, 300, 64, "causal"),                                   # 320 workgroups: 128-key tiles again
    # walks of as many 128-key tiles as 256-key ones do not pay for (above: 257 to 384 keys, bands of two blocks), and some that do
    (1, 2, 400, 450, 48, "causal"), (2, 2, 512, 512, 64, "causal"), (1, 3, 200, 450, 64, "padded"), (2, 2, 520, 512, 64, "padded"),
    (1, 2, 1100, 1100, 64, "wide band"), (1, 2, 1100, 1101, 56, "wide late band"), (1, 2, 900, 1290, 40, "wide band"),
    (20, 16, 77, 77, 64, "none"), (20, 16, 77, 150, 40, "padded"), (20, 16, 77, 200, 64, "mixed"), (1, 32, 1100, 1100, 64, "causal"),   # a merge alone
    (1, 2, 100, 300, 80, "none"), (1, 2, 100, 300, 128, "padded"),      # four groups, 3 and 4 pieces
    (4, 10, 500, 200, 64, "none"), (4, 10, 500, 200, 80, "none"), (4, 10, 500, 200, 128, "mixed"), (2, 10, 500, 200, 160, "none")])   # two groups
def test_forward_of_key_groups(B, N, Sq, Sk, D, side, dtype):
    g, rng = torch.Generator().manual_seed(Sq * 5 + Sk), np.random.default_rng(Sk + D)
    q, k, v = (torch.randn(B, N, S, D, generator=g).to(dtype) for S in (Sq, Sk, Sk))
    kw, okw, m = dict(scale=D ** -0.5), dict(scale=D ** -0.5), None
    if side == "causal":
        kw.update(mask_kind=_capi.MASK_CAUSAL)
        okw.update(attn_mask=np.triu(np.ones((1, Sq, Sk), np.uint8), 1))
    elif side == "padded":
        m = np.repeat((np.arange(Sk)[None, :] >= rng.integers(Sk // 4, Sk + 1, B)[:, None]).astype(np.uint8)[:, None], Sq, 1)
    elif side == "mixed":                                 # whole blocks hidden, clean and mixed ones, the first key of a row never hidden
        m = (rng.random((B, Sq, Sk)) < 0.3).astype(np.uint8)
        m[:, :, 128:256] = 1
        m[:, : Sq // 2, 256:384] = 0
        m[:, :, 0] = 0
    elif "band" in side:                                  # a first block in the upper half of a tile, and ends in the lower half
        width = 4 if "wide" in side else 1
        prev, nxt = (0, width) if "late" in side else (width, 0)
        kw.update(prev_block_num=prev, next_block_num=nxt)
        okw.update(prev_block_num=prev, next_block_num=nxt)
    elif side == "prefix":
        kw.update(row_block_prefix=384)
        okw.update(attn_mask=(np.arange(Sk)[None, None, :] >= ((np.arange(Sq) // 384 + 1) * 384)[None, :, None]).astype(np.uint8))
    if m is not None:
        kw.update(mask_kind=_capi.MASK_DENSE_U8, attn_mask=torch.from_numpy(m).to(DEV))
        okw.update(attn_mask=m)
    o, lse = forward(q, k, v, kw)
    O, L = orc.unfused_fwd(q.float().numpy(), k.float().numpy(), v.float().numpy(), **okw)
    tol = dict(atol=2e-3, rtol=1e-3) if dtype == torch.float16 else dict(atol=2e-2, rtol=1e-2)
    ok, ratio, mx = orc.tolerance_gate(O, o.float().cpu().numpy(), **tol)
    assert ok, f"worst ratio {ratio:.3f}, max |d| {mx:.3e}"
    assert np.max(np.abs(L - lse.cpu().numpy())) < 1e-4 * max(1.0, np.abs(L).max() / 10)


# a launch of more than one round and parts that fit into one: two key groups, whose merge the first one does alone there, or one
# group, whose first tile comes behind the Q fragments there
LONE_MERGES = [(20, 16, 77, 77, 64, 2), (20, 16, 77, 200, 40, 2), (33, 8, 130, 129, 64, 3), (22, 6, 300, 65, 56, 2)]
LATE_TILES = [(32, 16, 200, 77, 64, 2), (32, 16, 200, 100, 80, 2), (32, 16, 200, 128, 128, 2)]


@pytest.mark.parametrize("side", ["none", "mask", "dropout", "key bias", "bias"])
@pytest.mark.parametrize("B, N, Sq, Sk, D, parts", LONE_MERGES + LATE_TILES)
def test_launches_of_several_rounds_give_the_bits_of_their_parts(B, N, Sq, Sk, D, parts, side):
    if D == 40 and "bias" in side:
        pytest.skip("not built")
    g = torch.Generator(device=DEV).manual_seed(Sq + Sk)
    q, k, v = (torch.randn(B, N, S, D, generator=g, device=DEV).half() for S in (Sq, Sk, Sk))
    mask = (torch.rand(1, Sq, Sk, generator=g, device=DEV) < 0.4).to(torch.uint8)
    keep = (torch.rand(B, N, Sq, Sk, generator=g, device=DEV) < 0.8).to(torch.uint8)
    bias = torch.randn(B, N, 1 if side == "key bias" else Sq, Sk + Sk % 8, generator=g, device=DEV).half()[..., :Sk]

    def run(lo, hi):
        kw = dict(scale=D ** -0.5)
        if side == "mask":
            kw.update(mask_kind=_capi.MASK_DENSE_U8, attn_mask=mask)
        elif side == "dropout":
            kw.update(drop_mask=keep[lo:hi].contiguous(), keep_prob=0.8)
        elif "bias" in side:
            kw.update(alibi=bias[lo:hi])
        return _capi.fa_fwd(_capi.make_params(q[lo:hi], k[lo:hi], v[lo:hi], **kw), q[lo:hi])

    o, lse = run(0, B)
    for lo in range(0, B, B // parts):
        part, part_lse = run(lo, lo + B // parts)
        assert torch.equal(part, o[lo:lo + B // parts]) and torch.equal(part_lse, lse[lo:lo + B // parts])
