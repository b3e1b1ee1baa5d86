"""GPU tests of how the flash kernel deals out its work: whole items in bundles, and the last
round's items cut into tile ranges whose partials are summed.

The items (4 query blocks of one head) number ceil(Sq / 256) B H; 256 of them run at a time.
Reference: float64 softmax attention of the bf16 inputs.  Bound: the probabilities and the
output are rounded to bf16 (2^-9 each, relative), the sums are f32; a random-sign sum of
rounded terms stays within 2^-7 of the row's largest |v|-weighted value here.
"""
import ctypes
import math

import pytest
import torch

from icsa_hip import _lib
from icsa_hip.editing_sparse_attention import _editing_sparse_attention_hip
from icsa_hip.hip_host import flash_attn_func

pytestmark = pytest.mark.gpu


def _ref(q, k, v):
    q, k, v = (x.double().cpu().permute(0, 2, 1, 3) for x in (q, k, v))
    p = torch.softmax(q @ k.transpose(-1, -2) / math.sqrt(q.shape[-1]), dim=-1)
    return (p @ v).permute(0, 2, 1, 3)


def _inputs(B, H, Sq, Sk, seed, dev):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, S, H, 128, generator=g).to(torch.bfloat16).to(dev) for S in (Sq, Sk, Sk)]


@pytest.mark.parametrize("B,H,Sq,Sk", [
    (1, 1, 64, 1024),       # one item, 16 tiles: run whole
    (1, 1, 65, 833),        # 14 tiles, a partial last one; a second block of one row
    (2, 1, 300, 2000),      # split: 4 items, 2 of them of one block, 8 chunks each
    (1, 3, 1000, 1500),     # split: 12 items, 6 chunks each
    (1, 40, 1800, 1000),    # one full round of items and 64 more, 16 tiles: run whole
    (1, 1, 64, 832),        # 13 tiles
    (1, 1, 64, 768),        # 12 tiles: no size of call is split
    (1, 257, 64, 77),       # one item past a round, 2 tiles each: two items a workgroup
    (1, 130, 700, 64),      # one-tile items, two a workgroup, queries ending inside a block
    (1, 1, 64, 1088),       # 17 tiles: run whole
    (1, 1, 64, 1152),       # 18 tiles: the shortest item that is split, 4 chunks
    (1, 2, 500, 2900),      # 4 items of 46 tiles in 46 chunks: one in four ends an item and starts the next
    (1, 40, 1800, 1200),    # one full round of items and 64 split ones, 256 chunks of 4 or 5 tiles
])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_flash_work_split(gpu, B, H, Sq, Sk, out):
    q, k, v = _inputs(B, H, Sq, Sk, 1000 * Sk + Sq, gpu)
    x = flash_attn_func(q, k, v, out_dtype=out)
    y = flash_attn_func(q, k, v, out_dtype=out)
    torch.cuda.synchronize()
    assert torch.equal(x, y), "not the same twice"
    ref = _ref(q, k, v)
    err = (x.double().cpu() - ref).abs().max().item()
    assert err <= 2.0 ** -7 * ref.abs().max().item(), err


def test_flash_workspace_without_partials(gpu):
    """A workspace that ends after V^T runs the same call unsplit; the two differ by the
    order of f32 sums and the reference max of the bf16 probabilities only."""
    q, k, v = _inputs(1, 2, 500, 3000, 7, gpu)
    x = flash_attn_func(q, k, v, out_dtype=torch.float32)
    L = _lib.lib()
    vt_bytes = 2 * 128 * 47 * 64 * 2
    assert L.icsa_flash_attn_workspace_size(1, 3000, 2, 128) > vt_bytes
    ws = torch.empty(vt_bytes, dtype=torch.uint8, device=gpu)
    y = torch.empty_like(x)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = lambda t: [t.stride(0), t.stride(1), t.stride(2)]
    rc = L.icsa_flash_attn(p(q), *st(q), p(k), *st(k), p(v), *st(v), 1, 500, 3000, 2, 128, p(y), _lib.F32,
                           *st(y), p(ws), vt_bytes, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    torch.cuda.synchronize()
    assert (x - y).abs().max().item() <= 2.0 ** -8 * x.abs().max().item()


def test_flash_split_with_masked_range(gpu):
    """Keys of score -inf over more than a chunk carry no weight (a chunk whose scores are
    all -inf adds nothing)."""
    q, k, v = _inputs(1, 1, 64, 2048, 3, gpu)
    q = q.abs() + 0.25
    k[:, 1024:] = -math.inf
    x = flash_attn_func(q, k, v, out_dtype=torch.float32)
    ref = _ref(q, k[:, :1024], v[:, :1024])
    assert (x.double().cpu() - ref).abs().max().item() <= 2.0 ** -7 * ref.abs().max().item()


def test_split_residual_per_dim(gpu):
    """The residual weight of split items as a full [S, H, D] tensor: x(alpha) - x(0) is
    alpha times the compressed output, in f32."""
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(1, 2200, 2, 128, generator=g).to(gpu) for _ in range(3))
    al = torch.randn(1, 2200, 2, 128, generator=g).to(gpu)
    x0, w = _editing_sparse_attention_hip(q, k, v, 1100, 0.0, keep_workspace=True)
    xa, _ = _editing_sparse_attention_hip(q, k, v, 1100, al)
    oc = w["out_c"].repeat_interleave(64, dim=2)[:, :, :2200].permute(0, 2, 1, 3)
    assert (xa - torch.addcmul(x0, al, oc)).abs().max().item() <= 1e-6 * xa.abs().max().item()
