"""Performance cases of the attention operators and layers.

Every case is work that a program of this framework's user has it do, through the public entry points: the layers
`FlashAttention` and `TriangleAttention`, the operator `get_flash_attention` and the inference operator
`flash_attention_tik`.  `listed()` names one case of each kind; `draw(rng)` gives another size of one of the kinds.

The kinds (`"kind"` of a case) and what they stand for:

  layer_infer   forward of the layer in eval mode, from the smallest calls on: B1 N4 S512 D64 is the reference's own
                CPU-sized configuration.  Launches and host work count here.
  train_tile    small training step of the layer with the compact (1,128,128) causal tile: (4,8,128,80) is in the
                reference's shape grid.
  decode        one new token per sequence against a key / value cache that is longer than its present contents.
  long_keys     a block of queries against a very long key sequence: 256 x 131072 is in the reference's tests.
  infer_self    the inference operator on the self attention of an image model: head dims 40, 64, 80, 160.
  train_cross   training step of a cross attention onto 77 text tokens (the wukong shapes), head dims 40 to 160.
  train_causal  the benchmark: causal training step with the mask handed over as a uint8 tensor, B4 N16 S2048 D128.
  train_bsnd    training step in bf16 on projections laid out [B,S,N,D], odd sequence lengths, no mask.
  train_padded  training step on a padded batch with dropout drawn by the library, B16 N16 S1024 D128.
  train_alibi   causal training step with the per-head key bias of ALiBi, B2 N32 S4096 D128.
  train_masks   training step with the reference's own fp16 masks (causal mask and dropout mask as tensors): the
                shape of the reference's performance test, B4 N8 S4096 D128.
  triangle      forward of the triangle layer, four row blocks, B8 N32 S4096 D128.
"""
import math

import torch

from acctransformer_amd.flash_attention.nn.layer.flash_attention import FlashAttention
from acctransformer_amd.flash_attention.ops.flash_attention.flash_attention_impl import get_flash_attention
from acctransformer_amd.infer.flash_attention.tik.flash_attention_tik import flash_attention_tik
from acctransformer_amd.triangle_attention.triangle_attention import TriangleAttention

DEVICE = "cuda"
_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
_TRAINING = ("train_tile", "train_cross", "train_causal", "train_bsnd", "train_padded", "train_alibi", "train_masks")
_MOST_FLOPS = 1.1e12           # no drawn case computes more than the largest listed one


def _case(kind, dtype, B, N, Sq, Sk, D, **more):
    return dict(kind=kind, dtype=dtype, B=B, N=N, Sq=Sq, Sk=Sk, D=D, **more)


def listed():
    cases = [
        # one short sequence through the layer, no gradient: what a single call costs
        _case("layer_infer", "fp16", 1, 4, 512, 512, 64, causal=False),
        # the smallest training step: one 128-row block per head
        _case("train_tile", "fp16", 4, 8, 128, 128, 80),
        # one token per sequence, eight sequences, the cache three quarters full
        _case("decode", "bf16", 8, 32, 1, 3000, 128),
        # one head's 256 queries against 128K keys
        _case("long_keys", "fp16", 1, 1, 256, 131072, 128),
        # image self attention at 64 x 64 latents, head dim 40
        _case("infer_self", "fp16", 2, 8, 4096, 4096, 40),
        # its cross attention one level further down, training
        _case("train_cross", "fp16", 4, 8, 1024, 77, 80),
        # the headline benchmark
        _case("train_causal", "fp16", 4, 16, 2048, 2048, 128),
        # encoder training on unpadded sequences of an odd length
        _case("train_bsnd", "bf16", 8, 12, 1000, 1000, 64),
        # padded batch, dropout 0.1
        _case("train_padded", "fp16", 16, 16, 1024, 1024, 128),
        # decoder training with ALiBi
        _case("train_alibi", "fp16", 2, 32, 4096, 4096, 128),
        # the reference's performance test: every mask a tensor
        _case("train_masks", "fp16", 4, 8, 4096, 4096, 128),
        # large forward that leaves the upper triangle out
        _case("triangle", "fp16", 8, 32, 4096, 4096, 128, block=1024),
    ]
    for c in cases:
        c["name"] = c["kind"]
    return cases


def _log(rng, lo, hi):
    """A whole number between lo and hi, its logarithm uniform."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_once(rng):
    kind = rng.choice(("layer_infer", "train_tile", "decode", "long_keys", "infer_self", "train_cross", "train_causal",
                       "train_bsnd", "train_padded", "train_alibi", "train_masks", "triangle"))
    both = lambda: rng.choice(("fp16", "bf16"))
    if kind == "layer_infer":
        S = _log(rng, 32, 2048)
        return _case(kind, both(), rng.randint(1, 4), rng.choice((4, 8, 12, 16)), S, S, rng.choice((64, 80, 128)),
                     causal=rng.random() < 0.5)
    if kind == "train_tile":
        S = _log(rng, 64, 1024)
        return _case(kind, both(), rng.randint(1, 4), rng.randint(1, 8), S, S, rng.choice((64, 80, 128)))
    if kind == "decode":
        return _case(kind, both(), _log(rng, 1, 32), rng.choice((8, 16, 32)), 1, _log(rng, 64, 8192), rng.choice((64, 128)))
    if kind == "long_keys":
        return _case(kind, both(), 1, rng.randint(1, 8), _log(rng, 64, 512), _log(rng, 8192, 131072), rng.choice((64, 128)))
    if kind == "infer_self":
        S = _log(rng, 64, 4096)
        return _case(kind, "fp16", rng.randint(1, 4), 8, S, S, rng.choice((40, 64, 80, 160)))
    if kind == "train_cross":
        return _case(kind, both(), rng.randint(1, 8), 8, _log(rng, 64, 4096), 77, rng.choice((40, 64, 80, 160)))
    if kind == "train_causal":
        S = _log(rng, 512, 4096)
        return _case(kind, both(), rng.randint(1, 8), rng.choice((8, 12, 16, 32)), S, S, rng.choice((64, 128)))
    if kind == "train_bsnd":
        S = _log(rng, 128, 2048)
        return _case(kind, "bf16", rng.randint(1, 16), rng.choice((8, 12, 16)), S, S, rng.choice((64, 128)))
    if kind == "train_padded":
        S = _log(rng, 256, 1024)
        return _case(kind, both(), rng.randint(2, 16), rng.choice((8, 12, 16)), S, S, rng.choice((64, 128)))
    if kind == "train_alibi":
        S = 8 * _log(rng, 64, 512)
        return _case(kind, both(), rng.randint(1, 4), rng.choice((8, 16, 32)), S, S, rng.choice((64, 128)))
    if kind == "train_masks":
        S = _log(rng, 512, 4096)
        return _case(kind, "fp16", rng.randint(1, 4), 8, S, S, rng.choice((64, 128)))
    S = 512 * rng.randint(2, 8)
    return _case(kind, both(), rng.randint(1, 8), rng.choice((8, 16, 32)), S, S, rng.choice((64, 128)), block=S // 4)


def draw(rng):
    while True:
        case = _draw_once(rng)
        if work(case)["flops"] <= _MOST_FLOPS:
            return case


class _State:
    pass


def _triu(S, dtype):
    return torch.triu(torch.ones(1, S, S, dtype=dtype, device=DEVICE), 1)


def prepare(case, seed):
    kind, dtype = case["kind"], _DTYPES[case["dtype"]]
    B, N, Sq, Sk, D = (case[x] for x in ("B", "N", "Sq", "Sk", "D"))
    g = torch.Generator(device=DEVICE).manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, generator=g, device=DEVICE).to(dtype)

    s = _State()
    s.kind, s.args, s.dout = kind, (), None
    if kind == "decode":
        # the cache is a buffer for a power of two of positions; the present contents are a view of it
        cap = 1 << (Sk - 1).bit_length()
        s.q, s.k, s.v = randn(B, N, 1, D), randn(B, N, cap, D)[:, :, :Sk], randn(B, N, cap, D)[:, :, :Sk]
    elif kind == "train_bsnd":
        s.q, s.k, s.v = (randn(B, S, N, D).transpose(1, 2) for S in (Sq, Sk, Sk))
        s.dout = randn(B, Sq, N * D)
    else:
        s.q, s.k, s.v = randn(B, N, Sq, D), randn(B, N, Sk, D), randn(B, N, Sk, D)
        if kind in _TRAINING:
            s.dout = randn(B, N, Sq, D)
    if kind in _TRAINING:
        for t in (s.q, s.k, s.v):
            t.requires_grad_(True)
    scale = D ** -0.5

    if kind == "layer_infer":
        s.fn = FlashAttention(D, next_block_num=0 if case["causal"] else 65536).eval()
        s.args = (_triu(Sq, torch.uint8),) if case["causal"] else ()
    elif kind == "train_tile":
        s.fn = FlashAttention(D, next_block_num=0).train()
        s.args = (_triu(128, dtype),)
    elif kind in ("decode", "long_keys", "train_bsnd"):
        s.fn = get_flash_attention(scale=scale)
    elif kind == "infer_self":
        s.q = (s.q * 0.3).to(dtype)                      # the operator does not scale q k^T
        s.fn = flash_attention_tik
    elif kind == "train_cross":
        s.fn = get_flash_attention(tiling_stgy_name="wukong", scale=scale)
    elif kind == "train_causal":
        s.fn = FlashAttention(D, next_block_num=0).train()
        s.args = (_triu(Sq, torch.uint8),)
    elif kind == "train_padded":
        s.fn = FlashAttention(D, dropout_rate=0.1).train()
        lens = torch.randint(Sk // 4, Sk + 1, (B,), generator=g, device=DEVICE)
        mask = (torch.arange(Sk, device=DEVICE)[None, None, :] >= lens[:, None, None]).to(torch.uint8)
        s.args = (mask.expand(B, Sq, Sk).contiguous(), None, (seed, 1))     # the pair fixes the dropout stream
    elif kind == "train_alibi":
        s.fn = get_flash_attention(next_block_num=0, scale=scale)
        slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / N) for h in range(N)], device=DEVICE)
        # slope_h * (j - (S - 1)): the constant of a row cancels in the softmax
        pos = torch.arange(Sk, device=DEVICE, dtype=torch.float32) - (Sk - 1)
        s.args = (_triu(Sq, torch.uint8), None, (slopes[None, :, None, None] * pos).to(dtype))
    elif kind == "train_masks":
        s.fn = get_flash_attention(next_block_num=0, scale=scale, keep_prob=0.9)
        drop = torch.rand(B, N, Sq, Sk, generator=g, device=DEVICE, dtype=torch.float16) < 0.9
        s.args = (_triu(Sq, dtype), drop.to(dtype).div_(0.9))
    elif kind == "triangle":
        s.fn = TriangleAttention(block_size=case["block"]).eval()
        s.q = (s.q * scale).to(dtype)                    # the layer does not scale q k^T
        s.args = (_triu(Sq, torch.uint8).expand(B, Sq, Sk).contiguous(),)
    else:
        raise ValueError(kind)
    return s


def run(state):
    s = state
    if s.dout is None:
        with torch.no_grad():
            return s.fn(s.q, s.k, s.v, *s.args)
    out = s.fn(s.q, s.k, s.v, *s.args)
    o = out[0] if isinstance(out, tuple) else out
    y = o.transpose(1, 2).flatten(2) if s.kind == "train_bsnd" else o
    grads = torch.autograd.grad(y, (s.q, s.k, s.v), s.dout)
    return (out,) + grads


def _visible_pairs(case):
    """(query row, key) pairs of one head and batch entry that the operator has to compute."""
    Sq, Sk, kind = case["Sq"], case["Sk"], case["kind"]
    if kind == "layer_infer":
        return Sq * (Sq + 1) / 2 if case["causal"] else Sq * Sk
    if kind in ("train_tile", "train_causal", "train_alibi", "train_masks", "triangle"):
        return Sq * (Sq + 1) / 2
    if kind == "train_padded":
        return Sq * Sk * 0.625                           # lengths uniform between a quarter and the whole
    return Sq * Sk


def work(case):
    kind = case["kind"]
    B, N, Sq, Sk, D = (case[x] for x in ("B", "N", "Sq", "Sk", "D"))
    training = kind in _TRAINING
    q, k = B * N * Sq * D * 2, B * N * Sk * D * 2
    # q, k, v in and o out; in training dO in and dq, dk, dv out as well
    io = 2 * q + 2 * k + (2 * q + 2 * k if training else 0)
    if kind in ("decode", "long_keys", "train_cross", "train_bsnd", "train_alibi", "train_masks"):
        io += B * N * Sq * 4                             # the operator hands the row statistics out
    if kind in ("train_causal", "train_alibi") or (kind == "layer_infer" and case["causal"]):
        io += Sq * Sk
    elif kind in ("train_padded", "triangle"):
        io += B * Sq * Sk
    elif kind == "train_masks":
        io += 2 * Sq * Sk + 2 * B * N * Sq * Sk
    return {"bytes": io, "flops": (14 if training else 4) * B * N * _visible_pairs(case) * D}


def tolerance(case):
    # Measured against the same operator in 64-bit arithmetic on the same inputs: relative error of O and of the
    # gradients up to 5e-4 in fp16 and 3.1e-3 in bf16, largest single difference 0.011 and 0.072 of the root mean
    # square (the probabilities and dS are rounded to the element type before their products, and so are the
    # results); four times that.
    fp16 = case["dtype"] == "fp16"
    return {"rel": 2e-3 if fp16 else 1.2e-2, "max": 0.045 if fp16 else 0.3}
