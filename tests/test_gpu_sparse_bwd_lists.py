"""GPU tests of the backward's work lists where they can go wrong: query-block counts around the
64-bit words of the bitmap by key block, key blocks that no query block selects, entries out of
range, and interval range counts from one to one per query block.  Oracle and bar as in
test_gpu_sparse_bwd (its docstring derives the bound)."""
import pytest
import torch

from oracle.sparse_bwd import sparse_piecewise_attn_bwd
from icsa_hip import sparse_piecewise_attn_1st_intervals_bwd_hip, sparse_piecewise_attn_1st_intervals_fwd_hip
from test_gpu_sparse_bwd import _case, _check_grad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,TQ,TKV,sparsity", [
    (1, 1, 63 * 64, 512, 0.25),        # 63, 64, 65 query blocks: one word, full, two words
    (1, 2, 64 * 64, 500, 0.25),
    (1, 1, 64 * 64 + 1, 1000, 0.125),  # the last query block is one row
    (1, 1, 129 * 64 - 7, 300, 0.5),    # three words, a ragged end on both sides
    (1, 1, 64, 64 * 70, 0.05),         # one query block: most key blocks unselected, two chunks
    (2, 40, 128, 130, 0.5),            # more (head, chunk) pairs than ranges are worth
])
def test_backward_lists(gpu, B, H, TQ, TKV, sparsity):
    print(f"[case] bwd lists B={B} H={H} TQ={TQ} TKV={TKV} sparsity={sparsity}", flush=True)
    q, k, v, do, out, lse, idx = _case(gpu, B, H, TQ, TKV, sparsity, seed=50)
    got = sparse_piecewise_attn_1st_intervals_bwd_hip(do.to(gpu), q.to(gpu), k.to(gpu), v.to(gpu), out, lse, idx,
                                                      grad_dtype=torch.float32)
    ref = sparse_piecewise_attn_bwd(do, q, k, v, out.cpu(), lse.cpu(), idx.long().cpu())
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        _check_grad(name, g, r)


def test_backward_skips_out_of_range_entries(gpu):
    """Entries outside [0, NKV) take no part: the same gradients as without them (their blocks
    count as unselected in both)."""
    q, k, v, do, out, lse, idx = _case(gpu, 1, 2, 300, 1000, 0.25, seed=60)
    args = [x.to(gpu) for x in (do, q, k, v)]
    short = idx[..., :2].contiguous()
    bad = torch.full((1, 2, 5, 1), -1, dtype=torch.int32, device=gpu)
    padded = torch.cat([bad, short[..., :1], bad + 17, short[..., 1:]], dim=-1)     # -1 and NKV = 16
    a = sparse_piecewise_attn_1st_intervals_bwd_hip(*args, out, lse, short, check_indices=False)
    b = sparse_piecewise_attn_1st_intervals_bwd_hip(*args, out, lse, padded, check_indices=False)
    assert all(torch.equal(x, y) for x, y in zip(a, b))
