"""GPU test of the rankings behind the layer's selection: the source list and the query order must
be the exact descending order of the scores the library stored, ties to the smaller index, for
list lengths around the 64 elements a workgroup ranks, and equal scores throughout (constant
keys).  Reference: a stable sort of the stored scores, so the comparison is exact."""
import pytest
import torch

from icsa_hip.editing_sparse_attention import _editing_sparse_attention_hip
from icsa_hip.synthetic import make_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,blocks,flat", [(1, 1, False), (2, 3, False), (1, 63, False), (1, 64, True), (3, 65, False),
                                           (1, 129, True), (1, 300, False)])
def test_rankings_are_exact(gpu, H, blocks, flat):
    q, k, v, t = make_inputs(H=H, real=64 * blocks, pad=0, kind="random", seed=blocks)
    if flat:
        k = torch.ones_like(k)
    x, w = _editing_sparse_attention_hip(q.to(gpu), k.to(gpu), v.to(gpu), t, 0.5, 0.0625, 1.0, 0.5,
                                         keep_workspace=True)
    z = w["sizes"]
    order = torch.sort(w["sharpness"].cpu(), dim=-1, descending=True, stable=True).indices
    assert torch.equal(w["order"].cpu().long(), order)
    if z["topK"] > 0:
        score = w["src_score"].cpu()[..., :z["n_s"]]
        sel = torch.sort(score, dim=-1, descending=True, stable=True).indices[..., :z["topK"]]
        assert torch.equal(w["sel"].cpu().long(), sel)
        kvmap = w["kvmap"].cpu().long()
        assert torch.equal(kvmap[..., :z["n_t"]], torch.arange(z["n_t"]).expand_as(kvmap[..., :z["n_t"]]))
        n = min(z["topK"], z["NKV"] - z["n_t"])
        assert torch.equal(kvmap[..., z["n_t"]:z["n_t"] + n], z["n_t"] + sel[..., :n])
        assert (kvmap[..., z["n_t"] + n:] == -1).all()
