"""GPU tests of the layer at the edges of its merged table launches: one to three blocks in all,
odd and even counts of straddling blocks (two share a workgroup), new-KV lengths on both sides
of the 32 blocks a workgroup copies, block counts around the 64 columns of a value-mean tile,
and so few heads that the logits take one column tile a range.  Reference and bars: the oracle,
as every pipeline case."""
import pytest

from icsa_hip.synthetic import make_inputs
from test_gpu_pipeline import _run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,real,pad,srr", [(1, 64, 0, 0.5), (1, 65, 0, 0.5), (2, 1024, 0, 0.5), (1, 2048, 0, 0.03),
                                            (1, 2049, 0, 0.1), (3, 2030, 40, 0.13), (1, 4160, 8, 0.06)])
def test_layer_table_edges(gpu, H, real, pad, srr):
    q, k, v, t = make_inputs(H=H, real=real, pad=pad, B=1, kind="random", seed=real)
    _run_case(gpu, q, k, v, t, srr=srr)
    _run_case(gpu, q.float(), k.float(), v.float(), t, srr=srr)
