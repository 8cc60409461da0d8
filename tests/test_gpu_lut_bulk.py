"""gm_lut_bulk at the edges of its tiles (slabs per XCD turn, 16- and 48-row PSD
tiles, features sharing a 64-column block with P11, moments in one or two halves
of a wavefront) against FP64 sums of the same planes in numpy and the oracle's
GSF expansion.  Rows are float32: 2e-6 relative (of max |alpha1| for moments)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_slab,n_r,n_ang,n_psd,n_mom,per_slab",
                         [(1, 7, 61, 1, 32, False), (9, 8, 60, 16, 33, False),
                          (3, 13, 130, 17, 32, False), (8, 5, 64, 49, 64, False),
                          (2, 9, 70, 3, 5, True), (1, 6, 70, 17, 32, True)])
def test_bulk_rows(gpu, n_slab, n_r, n_ang, n_psd, n_mom, per_slab):
    import torch
    from geosmie_amd import _lib
    from geosmie_amd._lib import check, ptr
    from oracle import gsf as G
    ng = 70
    rng = np.random.default_rng(n_ang + n_psd)
    ang = np.linspace(0.0, 180.0, n_ang)
    p11 = rng.uniform(0.5, 2.0, (n_slab, n_r, n_ang))
    x = rng.uniform(0.1, 9.0, (n_slab, n_r))
    lam = rng.uniform(0.3, 2.0, n_slab)
    props = rng.uniform(0.2, 0.9, (6, n_slab * n_r))
    w = rng.uniform(0.1, 1.0, ((n_slab,) if per_slab else ()) + (n_psd, n_r))
    d = [_lib.to_dev(v.copy()) for v in (w, x, lam, props, p11)]
    out = torch.empty((n_slab, n_psd, 3 + n_mom), dtype=torch.float32, device="cuda")
    check(_lib.lib().gm_lut_bulk(_lib.ctx(), n_slab, n_r, n_ang, n_psd, ptr(d[0]), int(per_slab),
                                 ptr(d[1]), ptr(d[2]), ptr(d[3]), ptr(d[4]),
                                 ang.ctypes.data_as(ctypes.c_void_p), ng, n_mom, ptr(out),
                                 _lib.stream()), "gm_lut_bulk")
    got = out.cpu().numpy().astype(np.float64)
    for s in range(n_slab):
        ww = w[s] if per_slab else w
        r2 = (x[s] * lam[s] / (2 * np.pi)) ** 2
        qe, qs, g = (props[k].reshape(n_slab, n_r)[s] for k in (0, 1, 4))
        ref = np.stack([ww @ (qe * r2) / (ww @ r2), ww @ (qs * r2) / (ww @ (qe * r2)),
                        ww @ (g * qs * r2) / (ww @ (qs * r2))], 1)
        np.testing.assert_allclose(got[s, :, :3], ref, rtol=2e-6)
        pb = ww @ p11[s]
        for k in range(n_psd):
            a, _ = G.expand(ang, *[pb[k]] * 6, ng=ng, quantize=False)
            a = a[0, :n_mom]
            assert np.abs(got[s, k, 3:] - a).max() <= 2e-6 * np.abs(a).max()
