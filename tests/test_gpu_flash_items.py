"""GPU tests that a flash workgroup's items do not reach into each other: one workgroup runs
several items (4 query blocks of one head) one after another, and what an item leaves behind,
above all the reference max of its softmax, must not be taken over by the next.

Heads differ in their logits by far more than the exponential's range (about 87), in orders that
put each kind before and after each other kind.  Reference: float64 softmax attention of the
bf16 inputs; the probabilities and the output are rounded to bf16 (2^-9 each, relative) and the
sums are f32, so a row stays within 2^-7 of the largest value.  Where no item is split, a head's
rows are the same bits as in a call with that head alone.
"""
import math

import pytest
import torch

from icsa_hip.editing_sparse_attention import _editing_sparse_attention_hip
from icsa_hip.hip_host import flash_attn_func

pytestmark = pytest.mark.gpu


def _ref(q, k, v):
    q, k, v = (x.double().cpu().permute(0, 2, 1, 3) for x in (q, k, v))
    p = torch.softmax(q @ k.transpose(-1, -2) / math.sqrt(q.shape[-1]), dim=-1)
    return (p @ v).permute(0, 2, 1, 3)


def _inputs(B, H, Sq, Sk, seed, dev):
    """q of each head scaled by 0, 1 or 40: largest logits 0, about 4 and about 160."""
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, S, H, 128, generator=g) for S in (Sq, Sk, Sk))
    scale = torch.tensor([0.0, 1.0, 40.0])[torch.randint(3, (B, 1, H, 1), generator=g)]
    scale[:, :, :4] = torch.tensor([40.0, 0.0, 0.0, 40.0]).view(1, 1, 4, 1)[:, :, :H]
    return [x.to(torch.bfloat16).to(dev) for x in (q * scale, k, v)]


SHAPES = [
    (1, 257, 64, 77),       # bundles of two 2-tile items
    (2, 130, 100, 700),     # bundles over a batch boundary, 11 tiles, a partial last one
    (1, 100, 64, 1500),     # split: 256 chunks of 9 or 10 of an item's 24 tiles, two items in many
    (1, 90, 250, 2113),     # split: 256 chunks of 11 or 12 of 34 tiles
]


@pytest.mark.parametrize("B,H,Sq,Sk", SHAPES)
def test_items_of_different_score_levels(gpu, B, H, Sq, Sk):
    q, k, v = _inputs(B, H, Sq, Sk, 7 * Sk + Sq, gpu)
    x = flash_attn_func(q, k, v, out_dtype=torch.float32)
    ref = _ref(q, k, v)
    err = (x.double().cpu() - ref).abs().amax(dim=(1, 3))          # [B, H]
    assert (err <= 2.0 ** -7 * ref.abs().amax(dim=(1, 3))).all(), err


@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,Sq,Sk", SHAPES[:2] + [
    (1, 300, 48, 64),       # rows 32 .. 47: a wave with 16 of its 32 rows
    (1, 260, 33, 130),      # and with one
    (1, 130, 290, 200),     # the same in each head's second item
])
def test_whole_items_as_alone(gpu, B, H, Sq, Sk, out):
    q, k, v = _inputs(B, H, Sq, Sk, 11 * Sk + Sq, gpu)
    x = flash_attn_func(q, k, v, out_dtype=out)
    for b, h in [(b, h) for b in range(B) for h in range(0, H, 5)] + [(B - 1, h) for h in range(4)]:
        y = flash_attn_func(q[b:b + 1, :, h:h + 1], k[b:b + 1, :, h:h + 1], v[b:b + 1, :, h:h + 1], out_dtype=out)
        assert torch.equal(x[b, :, h], y[0, :, 0]), (b, h)


@pytest.mark.parametrize("B,H,Sq,Sk", SHAPES)
def test_infinite_scores_stay_in_their_head(gpu, B, H, Sq, Sk):
    q, k, v = _inputs(B, H, Sq, Sk, 13 * Sk + Sq, gpu)
    x = flash_attn_func(q, k, v)
    bad = k.clone()
    bad[:, 1, ::3, 5] = math.inf                     # every third head has one such key
    q2 = q.clone()
    q2[:, :, ::3, 5] = 1.0                           # of score +inf
    y = flash_attn_func(q2, bad, v)
    keep = torch.arange(H, device=gpu) % 3 != 0
    assert torch.equal(x[:, :, keep], y[:, :, keep])


@pytest.mark.parametrize("S,t", [
    (1024, 512),            # 9 key tiles, two whole items a head
    (649, 320),             # 5 key tiles; items of 4 and of 1 block, a last block of 9 rows that may
                            # come anywhere among a head's 5 peaked ones
])
def test_layer_heads_as_alone(gpu, S, t):
    """The layer's peaked blocks, two items a workgroup."""
    H = 140
    g = torch.Generator().manual_seed(S)
    q, k, v = (torch.randn(1, S, H, 128, generator=g) for _ in range(3))
    level = torch.tensor([40.0, 0.0, 1.0])[torch.randint(3, (1, (S + 63) // 64, H, 1), generator=g)]
    q = q * level.repeat_interleave(64, dim=1)[:, :S]
    q, k, v = (x.to(torch.bfloat16).to(gpu) for x in (q, k, v))
    x, _ = _editing_sparse_attention_hip(q, k, v, t)
    assert x.isfinite().all()
    for h in range(0, H, 7):
        y, _ = _editing_sparse_attention_hip(*(a[:, :, h:h + 1] for a in (q, k, v)), t)
        assert torch.equal(x[:, :, h], y[:, :, 0]), h


def test_small_call_allocates_little(gpu):
    """64 queries, 1,000 keys, one head: V^T (256 KB), no partials; 64 queries, 1,500 keys: 6 chunks of
    one item, 7 partials of 135 KB at most."""
    for Sk, most in ((1000, 2 ** 19), (1500, 2 ** 21)):
        q, k, v = _inputs(1, 1, 64, Sk, Sk, gpu)
        flash_attn_func(q, k, v)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        flash_attn_func(q, k, v)
        assert torch.cuda.max_memory_allocated() - before <= most
