"""Homogeneous batches too small for one point per lane: long, middle and short
series in one launch with 64 / 32 / 16, 16 and 4 lanes per point, against the same points
one per lane (GM_TUNE_MIE_LANES = 1).

Both forms are checked against the oracle elsewhere (1e-9); here against each other at
that bound: efficiencies 1e-9 relative, |a_n|, |b_n| <= 1 within 1e-9.
"""
import numpy as np
import pytest

from test_gpu_mie_long import _run

pytestmark = pytest.mark.gpu


# lanes 64 (n_max > 1200; the middle part from 8192 points on), 32 and 16; sizes on both
# sides of the parts' bounds (n_max 48 and 208), a part without points, one point
@pytest.mark.parametrize("n, lo, hi", [
    (1, 2000.0, 2000.0), (700, 0.01, 2000.0), (9000, 0.01, 2000.0), (30001, 1.0, 1500.0),
    (9000, 250.0, 1500.0), (9000, 20.0, 900.0), (3000, 0.01, 200.0), (20000, 30.0, 50.0)])
def test_parts_match_serial(gpu, n, lo, hi):
    x = np.exp(np.linspace(np.log(lo), np.log(hi), n))
    np.random.default_rng(n).shuffle(x)
    got, ref = _run(x, 0), _run(x, 1)
    for a, b in zip(got[:2], ref[:2]):
        assert float((a - b).abs().max()) <= 1e-9
    for q in (0, 1, 4):
        d = (got[2][q] - ref[2][q]).abs() / ref[2][q].abs()
        assert float(d.max()) <= 1e-9, q
