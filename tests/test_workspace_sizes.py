"""The workspace size queries on the host: they answer for any shape, served or not (a caller may ask before
it knows whether the layer is), and never end the process."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# T, N, K, rank: no output or reduction column, fewer than a tile's 128, and widths past any buffer
UNSERVED = [(1, 0, 128, 0), (1, 64, 128, 8), (7, 128, 0, 0), (128, 127, 4096, 16), (128, 4096, 127, 16),
            (1, 0, 0, 64), (0, 128, 128, 8), (1, 2 ** 62, 128, 0)]


def test_unserved_shapes_are_answered():
    """In a process of its own, so that an arithmetic fault is a failed test. Shapes below a tile get the
    sizes that the path for more tokens states."""
    code = f"""
import sys
sys.path.insert(0, {ROOT!r})
from r9700training_amd import R97Q_DECODE_AUTO, R97Q_DECODE_FUSED, lib
L = lib()
for s in {UNSERVED!r}:
    got = []
    for mode in (R97Q_DECODE_AUTO, R97Q_DECODE_FUSED):
        L.r97q_set_decode_once(mode)
        got.append((L.r97q_fwd_workspace_bytes(*s), L.r97q_bwd_workspace_bytes(*s)))
    print(s, got, flush=True)
    assert got[0] == got[1], s
"""
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, (p.returncode, p.stdout, p.stderr[-2000:])
