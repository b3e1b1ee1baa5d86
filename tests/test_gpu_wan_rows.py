"""GPU test of the q / k producer's one-pass kernel against its two-pass kernels: a batch of eight
takes the one-pass kernel where the rule of csrc/wan_qk_rule.h gives it the call, each of its
sequences alone the two-pass kernels.  The sums run in the same order in both, so the comparison
is exact.  Head counts at the edges of the row chunks (4 heads each) and of the
instantiations, whole and ragged last blocks, one input or two, with and without block sums and
gate."""
import pytest
import torch

from icsa_hip.wan import wan_freqs, wan_qk_prologue

pytestmark = pytest.mark.gpu


# 64-token blocks of one head from which a batch of eight takes the one-pass kernel (below: 12,000)
SERVED = {6: 12000, 13: 12000, 21: 19400, 24: 19400, 40: 14000}


@pytest.mark.parametrize("H,extra,two,sums", [(6, 5, True, True), (13, 63, True, True), (21, 40, True, False),
                                              (24, 1, False, True), (40, 17, True, True)])
def test_one_pass_equals_two_passes_where_it_serves(gpu, H, extra, two, sums):
    test_one_pass_equals_two_passes(gpu, H, extra, two, sums, SERVED[H])


@pytest.mark.parametrize("H,extra,two,sums", [(1, 1, True, True), (3, 0, True, True), (12, 0, True, True),
                                              (13, 63, True, True), (20, 0, False, True), (21, 40, True, False),
                                              (40, 17, True, True)])
def test_one_pass_equals_two_passes(gpu, H, extra, two, sums, blocks=12000):
    B, D = 8, 128
    S = 64 * -(-blocks // (B * H * (2 if two else 1))) + extra
    g = torch.Generator().manual_seed(S + H)
    yq = torch.randn(B, S, H * D, generator=g).to(torch.bfloat16).to(gpu)
    yk = (torch.randn(B, S, H * D, generator=g) * 3).to(torch.bfloat16).to(gpu) if two else None
    wq, wk = (torch.rand(H * D, generator=g).to(gpu) + 0.5 for _ in range(2))
    a = torch.randn(B, S, 1, generator=g).to(torch.bfloat16).to(gpu) if two else None
    grids = [[2, 7 + b, 40] for b in range(B)]
    src = [[1, 9, 30 + b] for b in range(B)]
    freqs = wan_freqs()

    def run(sl):
        return wan_qk_prologue(yq[sl], None if yk is None else yk[sl], wq, wk if two else None, grids[sl], src[sl], 1,
                               freqs, H, None if a is None else a[sl], want_sums=sums)

    whole = run(slice(0, B))
    for b in range(B):
        part = run(slice(b, b + 1))
        for name, x, y in zip(("q", "k", "qsum", "ksum", "gate"), whole, part):
            assert (x is None) == (y is None)
            if x is not None:
                assert torch.equal(x[b:b + 1], y), f"{name} of batch {b}"
