"""An infinity in the last rows of V stays one in O: the keys that pad the last tile of the forward have no probability, and
nothing of V may be multiplied by it."""
import pytest
import torch

from acctransformer_amd import _capi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("side", ["none", "mask", "dropout", "key bias", "bias"])
@pytest.mark.parametrize("B, N, Sq, D", [(1, 2, 64, 64), (1, 2, 64, 128), (4, 10, 500, 64), (4, 16, 512, 128), (16, 16, 256, 64), (16, 16, 256, 128),
                                         (1, 2, 70, 160), (1, 2, 70, 256), (2, 2, 200, 40)])
def test_infinities_of_v(B, N, Sq, D, side, dtype):
    if (D == 40 or D > 128) and "bias" in side:
        pytest.skip("not built")
    g = torch.Generator(device=DEV).manual_seed(D)
    for Sk in (1, 31, 33, 65, 100, 127, 129, 200, 257, 289, 300, 321, 500):
        q, k, v = (torch.randn(B, N, S, D, generator=g, device=DEV).to(dtype) for S in (Sq, Sk, Sk))
        v[:, :, Sk - 1, 5], v[:, :, Sk - 1, 6] = float("inf"), float("-inf")
        kw = dict(scale=0.25 * D ** -0.5)
        if side == "mask":
            m = (torch.rand(1, Sq, Sk, generator=g, device=DEV) < 0.5).to(torch.uint8)
            m[:, :, Sk - 1] = 0
            kw.update(mask_kind=_capi.MASK_DENSE_U8, attn_mask=m)
        elif side == "dropout":
            keep = (torch.rand(B, N, Sq, Sk, generator=g, device=DEV) < 0.8).to(torch.uint8)
            keep[..., Sk - 1] = 1
            kw.update(drop_mask=keep, keep_prob=0.8)
        elif "bias" in side:
            bias = torch.randn(1, N, 1 if side == "key bias" else Sq, Sk + Sk % 2, generator=g, device=DEV).to(dtype)
            kw.update(alibi=bias[..., :Sk])
        o, lse = _capi.fa_fwd(_capi.make_params(q, k, v, **kw), q)
        assert (o[..., 5] == float("inf")).all() and (o[..., 6] == float("-inf")).all(), Sk
        o[..., 5:7] = 0
        assert torch.isfinite(o).all() and torch.isfinite(lse).all(), Sk


@pytest.mark.parametrize("Sq, Sk, D", [(64, 20001, 64), (64, 20001, 128), (200, 9000, 80)])
def test_infinities_of_v_in_key_slices(Sq, Sk, D):
    g = torch.Generator(device=DEV).manual_seed(D)
    q, k, v = (torch.randn(1, 1, S, D, generator=g, device=DEV).half() for S in (Sq, Sk, Sk))
    v[:, :, Sk - 1, 5] = float("inf")
    o, _ = _capi.fa_fwd(_capi.make_params(q, k, v, scale=0.25 * D ** -0.5), q)
    assert (o[..., 5] == float("inf")).all() and torch.isfinite(o[..., :5]).all()
