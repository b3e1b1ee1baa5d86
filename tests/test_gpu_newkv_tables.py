"""GPU tests of the layer at the edges of its merged table launches: one to three blocks in all,
odd and even counts of straddling blocks (two share a workgroup), new-KV lengths on both sides
of the 32 blocks a workgroup copies, block counts around the 64 columns of a value-mean tile,
and so few heads that the logits take one column tile a range.  Reference and bars: the oracle,
as every pipeline case."""
import ctypes

import pytest
import torch

from icsa_hip import _lib
from icsa_hip.editing_sparse_attention import _editing_sparse_attention_hip
from icsa_hip.synthetic import make_inputs
from test_gpu_pipeline import _run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,real,pad,srr", [(1, 64, 0, 0.5), (1, 65, 0, 0.5), (2, 1024, 0, 0.5), (1, 2048, 0, 0.03),
                                            (1, 2049, 0, 0.1), (3, 2030, 40, 0.13), (1, 4160, 8, 0.06)])
def test_layer_table_edges(gpu, H, real, pad, srr):
    q, k, v, t = make_inputs(H=H, real=real, pad=pad, B=1, kind="random", seed=real)
    _run_case(gpu, q, k, v, t, srr=srr)
    _run_case(gpu, q.float(), k.float(), v.float(), t, srr=srr)


def test_workspace_without_its_optional_slot(gpu, monkeypatch):
    """A workspace that ends before the last slot: no interval bound, so the sparse kernel takes its
    max pass; with every block diffuse the output keeps its bits."""
    L = _lib.lib()
    layout, n = L.icsa_editing_workspace_layout, len(_lib.WS_SLOTS)
    q, k, v, t = make_inputs(H=2, real=1024, pad=0, B=1, kind="random", seed=3)
    args = (q.to(gpu), k.to(gpu), v.to(gpu), t, 0.5, 0.0625, 0.125, 0.0)
    full, _ = _editing_sparse_attention_hip(*args)

    def short(*a):
        size = layout(*a)
        end = ctypes.cast(a[-1], ctypes.POINTER(ctypes.c_int64))[n - 1]
        assert end < size
        return end

    monkeypatch.setattr(L, "icsa_editing_workspace_layout", short)
    x, _ = _editing_sparse_attention_hip(*args)
    assert torch.equal(x, full)
