"""gm_psd_contract on either side of its column and row bounds (16 columns: one
MFMA tile; 8 rows: the few-row kernel) against numpy: sums of n_pts products in
another order, within n_pts * 2^-53 of the sum of their magnitudes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_psd,n_pts,n_cols", [(1, 1, 1), (1, 257, 13), (8, 40000, 13),
                                                (8, 255, 16), (8, 300, 17), (9, 513, 13),
                                                (17, 256, 16)])
def test_contract(gpu, n_psd, n_pts, n_cols):
    import torch
    from geosmie_amd import _lib
    from geosmie_amd._lib import check, ptr
    rng = np.random.default_rng(n_pts)
    w, v = rng.uniform(0, 1, (n_psd, n_pts)), rng.standard_normal((n_pts, n_cols))
    d_w, d_v = _lib.to_dev(w), _lib.to_dev(v)
    out = torch.empty((n_psd, n_cols), dtype=torch.float64, device="cuda")
    check(_lib.lib().gm_psd_contract(_lib.ctx(), n_psd, n_pts, n_cols, ptr(d_w), ptr(d_v), ptr(out),
                                     _lib.stream()))
    bound = n_pts * 2.0 ** -53 * (w @ np.abs(v))
    assert (np.abs(out.cpu().numpy() - w @ v) <= 2 * bound + 1e-300).all()
