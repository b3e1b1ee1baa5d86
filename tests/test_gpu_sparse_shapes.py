"""GPU tests of the sparse host entry where its one pooling pass covers unequal lengths: far more
query than key blocks and the reverse, key-block counts around the 64 rows its bf16 sums are
padded to.  Reference and bar: the oracle on the same block lists, as test_gpu_kernels."""
import pytest
import torch

import oracle as O
from icsa_hip import _lib
from icsa_hip import sparse_piecewise_attn_1st_intervals_fwd_hip, sparse_piecewise_attn_1st_intervals_hip
from parity import compare_out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,TQ,TKV", [(1, 2, 64 * 130, 64), (2, 1, 64, 64 * 65), (1, 1, 128, 64 * 64),
                                        (1, 3, 64 * 63, 64 * 63)])
def test_sparse_host_unequal_lengths(gpu, B, H, TQ, TKV):
    g = torch.Generator().manual_seed(TQ + TKV)
    q, k, v = (torch.randn(B, H, T, 128, generator=g).to(torch.bfloat16) for T in (TQ, TKV, TKV))
    out, idx = sparse_piecewise_attn_1st_intervals_hip(q.to(gpu), k.to(gpu), v.to(gpu), 0.1, return_indices=True)
    ref = O.sparse_piecewise_attn(q, k, v, 0.1, indices=idx.long().cpu())
    compare_out(out, ref[0] if isinstance(ref, tuple) else ref)
    # the training forward returns the same lists and output for whole blocks
    out2, _, idx2 = sparse_piecewise_attn_1st_intervals_fwd_hip(q.to(gpu), k.to(gpu), v.to(gpu), 0.1)
    assert torch.equal(idx, idx2) and torch.equal(out, out2)


def test_lists_in_and_out_in_one_buffer(gpu):
    """The C entry with inject_idx == idx_out: the lists stay as given, the output is theirs."""
    B, H, T = 1, 2, 64 * 20
    g = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn(B, H, T, 128, generator=g).to(torch.bfloat16).to(gpu) for _ in range(3))
    lists = torch.stack([torch.randperm(20, generator=g)[:2].sort().values for _ in range(B * H * 20)])
    lists = lists.view(B, H, 20, 2).int().to(gpu)
    want = sparse_piecewise_attn_1st_intervals_hip(q, k, v, 0.1, indices=lists)
    L = _lib.lib()
    n = L.icsa_sparse_piecewise_workspace_size(B, H, T, T, 128, 0.1)
    ws, out, io = torch.empty(n, dtype=torch.uint8, device=gpu), torch.empty_like(q), lists.clone()
    st = list(q.stride()[:3])
    rc = L.icsa_sparse_piecewise_attn(q.data_ptr(), *st, k.data_ptr(), *st, v.data_ptr(), *st, B, H, T, T, 128, 0.1,
                                      io.data_ptr(), io.data_ptr(), out.data_ptr(), *st, ws.data_ptr(), n,
                                      torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    assert torch.equal(io, lists) and torch.equal(out, want)
