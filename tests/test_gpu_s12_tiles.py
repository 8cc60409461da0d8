"""FP64 and FP32 S1/S2 tiles (16 points x 16 to 128 angles per wavefront, angle tables
paired or read as they are, units in point order or longest first) against the
same sums by dense FP64 products of the same coefficients and tables.

The kernel adds the K terms in groups of four, the reference in torch's order:
both are FP64 sums of n_max <= 60 terms, so they agree within n_max * 2^-53 of
the sum of the terms' magnitudes; 1e-13 of max|S| (S at 0 degrees is that sum
up to a factor of a few) leaves an order of magnitude.  P11 and the row sums
are quadratic in S: twice that of their largest value.  FP32 rounds 2^29 times
coarser, operands, products and sums alike: 2^29 times those bounds.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _setup(n, n_ang, cap):
    import torch
    from geosmie_amd.lut import _DevMie
    from geosmie_amd.s12 import angle_tables_dev
    rng = np.random.default_rng(n + n_ang)
    dm = _DevMie(10 ** rng.uniform(-1.5, 1.5, n), complex(1.5, 0.01))
    cost = np.cos(np.radians(np.linspace(0.0, 180.0, n_ang))) if n_ang > 1 else np.array([0.3])
    pi_t, tau_t = angle_tables_dev(cost, max(cap, dm.nmax_max))
    k = dm.nmax_max
    idx = torch.arange(k, device="cuda")
    live = idx[None, :] < dm.d_nmax[:, None]
    at = (dm.d_off[:-1, None] + idx[None, :]).clamp(max=dm.d_an.numel() // 2 - 1)
    a, b = (torch.where(live, torch.view_as_complex(c.view(-1, 2))[at], 0) for c in
            (dm.d_an, dm.d_bn))

    def mul(c, t):
        return torch.complex(c.real.contiguous() @ t[:k], c.imag.contiguous() @ t[:k])
    return dm, pi_t, tau_t, mul(a, pi_t) + mul(b, tau_t), mul(a, tau_t) + mul(b, pi_t)


# one point and angle; ragged tiles; FP64: wavefronts of 16, 32 and 64 angles; 4100 points
# for the paired tables; 17000 with a 520-row table for the sorted order; FP32: of 32,
# 64 and 128 angles, and sorted
@pytest.mark.parametrize("n,n_ang,cap,prec", [
    (1, 1, 0, 0), (15, 17, 0, 0), (17, 371, 0, 0), (4100, 16, 0, 0), (4100, 371, 0, 0),
    (4097, 1801, 0, 0), (17000, 130, 520, 0), (1, 1, 0, 1), (17, 31, 0, 1), (4100, 371, 0, 1),
    (60001, 181, 0, 1), (90000, 371, 0, 1), (17000, 130, 520, 1)])
def test_amplitudes_and_p11(gpu, n, n_ang, cap, prec):
    import torch
    from geosmie_amd import _lib
    from geosmie_amd._lib import check, ptr
    dm, pi_t, tau_t, s1, s2 = _setup(n, n_ang, cap)
    L, ulp = _lib.lib(), 2.0 ** 29 if prec else 1.0
    args = (_lib.ctx(), n, ptr(dm.d_off), ptr(dm.d_nmax), ptr(dm.d_an), ptr(dm.d_bn), n_ang,
            ptr(pi_t), ptr(tau_t), int(pi_t.shape[0]))
    d1 = torch.empty(2 * n * n_ang, dtype=torch.float64, device="cuda")
    d2 = torch.empty_like(d1)
    check(L.gm_mie_s12(*args, ptr(d1), ptr(d2), prec, _lib.stream()), "gm_mie_s12")
    scale = max(float(s1.abs().max()), float(s2.abs().max()))
    for d, s in ((d1, s1), (d2, s2)):
        got = torch.view_as_complex(d.view(n, n_ang, 2))
        assert float((got - s).abs().max()) <= 1e-13 * ulp * scale
    p11 = torch.empty((n, n_ang), dtype=torch.float64, device="cuda")
    check(L.gm_s12_p11(*args, ptr(p11), prec, _lib.stream()), "gm_s12_p11")
    ref = (s1.abs() ** 2 + s2.abs() ** 2) / 2
    assert float((p11 - ref).abs().max()) <= 2e-13 * ulp * float(ref.max())
    mul = torch.empty((n, 4, n_ang), dtype=torch.float64, device="cuda")
    check(L.gm_s12_mueller(*args, ptr(mul), prec, _lib.stream()), "gm_s12_mueller")
    c = s1 * s2.conj()
    for e, v in enumerate((ref, (s2.abs() ** 2 - s1.abs() ** 2) / 2, c.real, c.imag)):
        assert float((mul[:, e] - v).abs().max()) <= 2e-13 * ulp * float(ref.max()), e


# rows with their own ranges and rows sharing one (1, 2 and 4 sums per group), one
# tile per chunk and several (short series, many points), sorted chunks
@pytest.mark.parametrize("n,n_ang,cap,share,prec", [
    (33, 19, 0, 1, 0), (5000, 371, 0, 2, 0), (60000, 371, 0, 1, 0), (60000, 371, 0, 4, 0),
    (17000, 130, 520, 2, 0), (33, 19, 0, 1, 1), (5000, 371, 0, 4, 1), (60000, 371, 0, 1, 1),
    (60000, 371, 0, 2, 1), (60000, 371, 0, 4, 1), (17000, 130, 520, 2, 1)])
def test_row_sums(gpu, n, n_ang, cap, share, prec):
    import torch
    from geosmie_amd import _lib
    from geosmie_amd._lib import check, ptr
    dm, pi_t, tau_t, s1, s2 = _setup(n, n_ang, cap)
    cut = n // 3 + 1
    ranges = [(0, cut)] * share + [(cut, n - cut)] * share
    w = torch.zeros((len(ranges), n), dtype=torch.float64, device="cuda")
    gen = torch.Generator(device="cuda").manual_seed(n)
    for r, (a, c) in enumerate(ranges):
        w[r, a:a + c] = torch.rand(c, generator=gen, dtype=torch.float64, device="cuda")
    k = len(ranges)
    out = torch.empty((k, 4, n_ang), dtype=torch.float64, device="cuda")
    st = (ctypes.c_int64 * k)(*[a for a, _ in ranges])
    ct = (ctypes.c_int64 * k)(*[c for _, c in ranges])
    coef = None
    if prec:
        coef = torch.empty(4 * dm.d_an.numel() // 2, dtype=torch.float32, device="cuda")
        check(_lib.lib().gm_s12_split_coef(_lib.ctx(), dm.d_an.numel() // 2, ptr(dm.d_an),
                                           ptr(dm.d_bn), prec, ptr(coef), _lib.stream()))
    check(_lib.lib().gm_s12_contract_rows(_lib.ctx(), n, ptr(dm.d_off), ptr(dm.d_nmax),
                                          ptr(dm.d_an), ptr(dm.d_bn), n_ang, ptr(pi_t), ptr(tau_t),
                                          int(pi_t.shape[0]), k, st, ct, ptr(w), ptr(out), prec,
                                          None if coef is None else ptr(coef),
                                          _lib.stream()), "gm_s12_contract_rows")
    a1, a2, c = s1.abs() ** 2, s2.abs() ** 2, s1 * s2.conj()
    for e, v in enumerate(((a1 + a2) / 2, (a2 - a1) / 2, c.real, c.imag)):
        ref = w @ v.contiguous()
        bound = 2e-13 * (2.0 ** 29 if prec else 1.0) * float((w @ ((a1 + a2) / 2)).max())
        assert float((out[:, e] - ref).abs().max()) <= bound, e
