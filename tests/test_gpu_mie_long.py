"""Long series of a lane-per-point homogeneous batch run a wavefront each: the
same points with the split off (GM_TUNE_MIE_LANES = 1, every point serial).

Both forms are checked against the oracle elsewhere (1e-9); here against each
other at that bound: efficiencies 1e-9 relative, |a_n|, |b_n| <= 1 within 1e-9.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 64 * 256 * 16 + 77     # one point per lane from 262144 points on


def _run(x, lanes):
    import torch
    from geosmie_amd import _lib
    from geosmie_amd._lib import check, ptr
    from geosmie_amd.autotune import set_knob
    h = _lib.private_ctx()
    set_knob(h, "mie_lanes", lanes)
    n = x.size
    d_x = _lib.to_dev(x)
    eps = _lib.cplx_dev(np.full(n, (1.55 + 0.003j) ** 2))
    off = torch.empty(n + 1, dtype=torch.int64, device="cuda")
    L, s = _lib.lib(), _lib.stream()
    check(L.gm_coef_offsets(h, n, ptr(d_x), ptr(off), s))
    total = int(off[-1])
    an = torch.zeros(2 * total, dtype=torch.float64, device="cuda")
    bn, props = torch.zeros_like(an), torch.zeros(6 * n, dtype=torch.float64, device="cuda")
    check(L.gm_mie_batch(h, n, ptr(d_x), None, ptr(eps), None, None, float(x.max()), ptr(off),
                         ptr(an), ptr(bn), ptr(props), None, _lib.GM_MIE_SORT, s))
    return an, bn, props.view(6, n)


# a few long points among short ones (every lane-split length from the bound up),
# a single one, and a batch whose even share is above every point (no split)
@pytest.mark.parametrize("long", [(330.0, 2000.0, 40), (1500.0, 1500.0, 1), (100.0, 900.0, N // 4)])
def test_long_points_match_serial(gpu, long):
    lo, hi, k = long
    rng = np.random.default_rng(k)
    x = 10 ** rng.uniform(-1.5, 1.2, N)
    x[rng.choice(N, k, replace=False)] = np.linspace(lo, hi, k)
    got, ref = _run(x, 0), _run(x, 1)
    for a, b in zip(got[:2], ref[:2]):
        assert float((a - b).abs().max()) <= 1e-9
    for q in (0, 1, 4):
        d = (got[2][q] - ref[2][q]).abs() / ref[2][q].abs()
        assert float(d.max()) <= 1e-9, q
