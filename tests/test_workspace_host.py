"""CPU tests of the workspace size queries: arguments at which there is nothing to deal out."""
import os
import subprocess
import sys

import pytest

from icsa_hip import _lib

pytestmark = pytest.mark.cpu


@pytest.mark.parametrize("B,H,S,t,srr", [
    (1, 40, 65536, 0, 0.0),          # no target, no source blocks retained: no key tiles
    (2, 200, 256, 0, 0.125),         # no target, a source too short for one retained block
    (1, 40, 65536, 128, -2 / 1022),  # a negative share that takes the target's blocks away
])
def test_size_of_a_layer_without_keys(B, H, S, t, srr):
    """A size, not an abort (in a process of its own: a division by zero would end it)."""
    code = ("from icsa_hip import _lib\n"
            f"print(_lib.lib().icsa_editing_workspace_size({B}, {S}, {H}, 128, {t}, 0.0625, {srr!r}, 0.5, 0, 0, 0))")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, PYTHONPATH=os.path.dirname(os.path.dirname(_lib.__file__))))
    assert r.returncode == 0, r.returncode
    assert int(r.stdout) > 0


def test_dense_size_follows_the_queries():
    L = _lib.lib()
    for B, H, Sq, Sk in ((1, 1, 64, 1000), (1, 1, 64, 65536), (1, 3, 1000, 1500), (1, 40, 65520, 512),
                         (2, 12, 9373, 9373), (1, 5, 32768, 32768), (1, 257, 64, 77)):
        vt = -(-B * H * 128 * -(-Sk // 64) * 64 * 2 // 256) * 256
        size = L.icsa_flash_attn_workspace_size_for(B, Sq, Sk, H, 128)
        assert vt <= size <= L.icsa_flash_attn_workspace_size(B, Sk, H, 128)
        items = B * H * -(-Sq // 256)
        # a partial (8 waves of O, max and sum in f32: 135 KB) a chunk and split item, 4 tiles a chunk
        part = 8 * (64 * 64 + 2 * 64) * 4
        assert size - vt <= part * items * (-(-Sk // 256) + 1), (B, H, Sq, Sk)
    assert L.icsa_flash_attn_workspace_size_for(1, 64, 1000, 1, 128) == 128 * 1024 * 2      # not split
    assert L.icsa_flash_attn_workspace_size_for(1, 64, 128, 1, 96) < 0
