"""The forward with one query row per head (csrc/fa_fwd_row.hip): batch edges, head dims, strides, parts of the key range, bands."""
import ctypes

import pytest
import torch

from acctransformer_amd import _capi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _call(q, k, v, room=None, **kw):
    lib = _capi.load()
    p = _capi.make_params(q, k, v, scale=q.shape[-1] ** -0.5, **kw)
    o, lse = torch.empty_like(q), torch.empty(q.shape[:3], dtype=torch.float32, device=DEV)
    p.o_stride = _capi._bhs_strides(o)
    need = lib.acct_fa_fwd_split_workspace_bytes(ctypes.byref(p))
    ws = torch.empty(max(need, 256), dtype=torch.uint8, device=DEV)
    rc = lib.acct_fa_fwd(ctypes.byref(p), o.data_ptr(), lse.data_ptr(), ws.data_ptr(), need if room is None else room,
                         ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.acct_last_error().decode()
    return o, lse, need


def _exact(q, k, v):
    s = (q.double() * q.shape[-1] ** -0.5) @ k.double().transpose(2, 3)
    return torch.softmax(s, -1) @ v.double(), torch.logsumexp(s, -1)


def _check(o, lse, q, k, v):
    # the sums are in float32, so what is left is the rounding of O to the element type (half a unit: 2^-11, bf16 2^-8) and, near
    # zero, the float32 sums of terms up to max |v|
    O, L = _exact(q, k, v)
    unit = 2.0 ** (-11 if o.dtype == torch.float16 else -8)
    assert ((o.double() - O).abs() <= 1.01 * unit * O.abs() + 2e-6 * v.double().abs().amax()).all()
    assert ((lse.double() - L).abs() <= 2e-6 * L.abs().clamp(min=1)).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B, N, Sk, D, parts", [
    (1, 3, 1, 64, False), (1, 1, 3, 8, False), (2, 3, 255, 40, False), (2, 3, 257, 64, False), (1, 300, 127, 72, False), (1, 2, 129, 128, False), (3, 2, 63, 136, False),
    (1, 2, 65, 256, False), (4, 16, 1000, 64, False), (1, 8, 4097, 128, True), (1, 1, 70000, 64, True), (2, 2, 5000, 160, True), (1, 320, 8192, 64, True), (1, 5, 9000, 80, True)])
def test_one_row_against_64_bits(B, N, Sk, D, parts, dtype):
    g = torch.Generator(device=DEV).manual_seed(Sk + D)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    q, k, v = r(B, N, 1, D), r(B, N, Sk, D), r(B, N, Sk, D)
    o, lse, need = _call(q, k, v)
    assert (need > 0) == parts
    _check(o, lse, q, k, v)
    if parts:                                                 # no room for the parts' sums: one part per head
        _check(*_call(q, k, v, room=0)[:2], q, k, v)
    # a view of a longer cache, rows of several heads beside each other
    k2, v2 = r(B, Sk + 5, N, D).transpose(1, 2)[:, :, :Sk], r(B, N, Sk + 9, D)[:, :, 3:3 + Sk]
    q2 = r(B, 1, N, D).transpose(1, 2)
    _check(*_call(q2, k2, v2)[:2], q2, k2, v2)


@pytest.mark.parametrize("Sk, D", [(127, 64), (1000, 40), (3001, 128), (700, 256)])
def test_one_row_of_shared_keys(Sk, D):
    """Keys and values that heads or batches share, and heads beside each other in a row: the same bits as from copies."""
    g = torch.Generator(device=DEV).manual_seed(Sk)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)
    B, N, q = 3, 4, r(3, 4, 1, D)
    for k, v in ((r(B, 1, Sk, D).expand(B, N, Sk, D), r(B, 1, Sk, D).expand(B, N, Sk, D)), (r(1, N, Sk, D).expand(B, N, Sk, D), r(B, N, Sk, D)),
                 (r(B, N, Sk, D), r(1, 1, Sk, D).expand(B, N, Sk, D)), (r(B, Sk, N, D).transpose(1, 2), r(B, Sk, N, D).transpose(1, 2))):
        o, lse, _ = _call(q, k, v)
        _check(o, lse, q, k, v)
        want, want_lse, _ = _call(q, k.contiguous(), v.contiguous())
        assert torch.equal(o, want) and torch.equal(lse, want_lse)


@pytest.mark.parametrize("seen, band", [(128, dict(next_block_num=0)), (384, dict(next_block_num=2)), (256, dict(row_block_prefix=256)), (500, dict(prev_block_num=0))])
def test_one_row_sees_its_band(seen, band):
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(2, 2, S, 64, generator=g, device=DEV).half() for S in (1, 500, 500))
    v[:, :, seen:] = float("nan")                             # not read
    o, lse, _ = _call(q, k, v, **band)
    _check(o, lse, q, k[:, :, :seen], v[:, :, :seen])


@pytest.mark.parametrize("Sk, D", [(300, 64), (3001, 128), (9001, 40)])
def test_one_row_with_infinities(Sk, D):
    g = torch.Generator(device=DEV).manual_seed(4)
    q, k, v = (torch.randn(1, 2, S, D, generator=g, device=DEV).half() for S in (1, Sk, Sk))
    v[:, :, Sk - 1, 5], v[:, :, Sk // 2, 6], v[:, :, 0, 7] = float("inf"), float("-inf"), float("inf")
    o = _call(q, k, v)[0]
    assert (o[..., 5] == float("inf")).all() and (o[..., 6] == float("-inf")).all() and (o[..., 7] == float("inf")).all()
    assert torch.isfinite(o[..., 8:]).all() and torch.isfinite(o[..., :5]).all()
    q[:], k[:] = 1.0, float("-inf")                           # no key has a probability: O = 0 and LSE = -inf, as for the other shapes
    o, lse, _ = _call(q, k, torch.ones_like(v))
    assert (o == 0).all() and (lse == float("-inf")).all()
    k[:, :, 1] = 0.5
    o, lse, _ = _call(q, k, torch.ones_like(v))
    assert torch.allclose(o.float(), torch.ones_like(o).float(), atol=1e-3) and torch.isfinite(lse).all()
    k[0, 0, 2] = float("nan")
    o = _call(q, k, torch.ones_like(v))[0]
    assert torch.isnan(o[0, 0]).all() and torch.isfinite(o[0, 1]).all()
