"""GPU parity of the wave-per-edge kernels (edgewise_wave.hip) against the float64 oracle, at the
edges of their tiles: channel counts around multiples of 16, one to four 16-slot blocks, layouts
whose widest groups share blocks, repeated, missing and unmixed degrees, and edge counts from one
up.  The launch log shows that they ran.  Tolerance: every stage accumulates in float32, as the
shape-generic kernels do, and is held to the same 1e-5 of the largest entry."""
import pytest

from flash_eq import _native as NAT
from test_gpu_edgewise import _run_parity, _select

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lin,lout,cin,cout,E", [
    # one slot, one channel (a single output can be a sum of four ranks that cancels, whose relative
    # error float32 does not bound: 17 edges bound it by the largest of 17)
    ([0], [0], 1, 1, 17),
    ([0, 1, 2], [0, 1, 2], 16, 16, 1),                      # one edge
    ([0, 1], [0, 1, 2], 32, 64, 3),
    ([0, 1, 2, 3], [0, 1, 2, 3], 17, 15, 66),               # one full block, ragged channels
    ([0, 1, 2, 3], [0, 1, 2, 3], 64, 48, 65),
    ([0, 1, 2, 3, 4], [0, 1, 2, 3, 4], 33, 31, 130),        # two blocks
    ([0, 1, 2, 3, 4, 5], [0, 1, 2, 3, 4, 5], 16, 24, 129),  # three blocks
    ([0, 1, 2, 3, 4, 5, 6], [0, 1, 2, 3, 4, 5, 6], 32, 32, 1031),   # four, the last with two slots
    ([0, 1, 2, 3, 4, 5, 6], [0, 1], 20, 48, 33),            # inputs no weight mixes
    ([0], [0, 1, 2, 3, 4, 5, 6], 5, 7, 18),                 # outputs no weight mixes
    ([3, 1, 1], [2, 2, 0, 4], 12, 9, 257),                  # repeated and missing degrees, any order
])
def test_wave_parity(dev, monkeypatch, lin, lout, cin, cout, E):
    _select(monkeypatch, "split")
    NAT.profile_summary()
    NAT.profile_enable(True)
    try:
        _run_parity(dev, lin, lout, cin, cout, E, seed=E, rmin=0.2)
    finally:
        NAT.profile_enable(False)
    launched = NAT.profile_summary()
    assert "k_ewg_bwd_x" in launched and "k_ewg_bwd_c" in launched, launched
    assert "k_ew_fwd" not in launched and "k_ew_bwd" not in launched, launched


def test_wave_parity_log_bins(dev, monkeypatch):
    _select(monkeypatch, "split")
    _run_parity(dev, [0, 1, 2, 3], [0, 1, 2, 3], 32, 32, 515, seed=4, log=True, rmin=0.2)
