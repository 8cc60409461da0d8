"""Small coated batches with 16, 32 or 64 lanes per point, against the shell
combination in extended precision (64-bit mantissa) on a sample of the points.

The kernel's largest errors on these points are 1.8e-11 in a_n, b_n (rounded m x, m y
next to a resonance) and 4.7e-13 in the efficiencies and g; asserted are 1e-10 and
5e-12: |a_n|, |b_n| <= 1 absolute, efficiencies relative, g absolute.  Against the same
points one per lane: the same points are NaN (series that overflow, tiny cores in
large shells), and the other classes are unchanged.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _nmax(y):
    return np.rint(2 + y + 4 * np.cbrt(y)).astype(int)


def _dn(z, start, nmax):
    D, d = np.zeros(nmax + 1, np.clongdouble), np.clongdouble(0)
    for k in range(start - 1, 0, -1):
        r = (k + 1) / z
        d = r - 1 / (d + r)
        if k <= nmax:
            D[k] = d
    return D[1:]


def _rb(z, nmax):
    """psi_n, chi_n (n = 0..nmax): psi upward to |z|, by downward ratios above."""
    az = float(abs(z))
    psi, chi = (np.zeros(nmax + 1, np.clongdouble) for _ in range(2))
    psi[0], chi[0] = np.sin(z), np.cos(z)
    R, t = np.zeros(nmax + 1, np.clongdouble), np.clongdouble(0)
    for k in range(nmax + 30 + 8 * int(np.ceil(np.cbrt(az))), 0, -1):
        it = 1 / (t + k / z)
        if k <= nmax:
            R[k] = it
        t = k / z - it
    pp, cp = np.cos(z), -np.sin(z)
    for n in range(1, nmax + 1):
        f = (2 * n - 1) / z
        psi[n] = f * psi[n - 1] - pp if n <= int(az) else psi[n - 1] * R[n]
        chi[n] = f * chi[n - 1] - cp
        pp, cp = psi[n - 1], chi[n - 1]
    return psi, chi


def _exact(x, y, e1, e2):
    """a_n, b_n with the reference's start index of the downward D_n."""
    m1, m2 = np.sqrt(np.clongdouble(e1)), np.sqrt(np.clongdouble(e2))
    x, y = np.longdouble(x), np.longdouble(y)
    m, u, v, w = m2 / m1, m1 * x, m2 * x, m2 * y
    nmax = int(_nmax(float(y)))
    nmx = int(np.rint(max(nmax, float(max(abs(m1 * y), abs(w)))) + 16))
    far = nmx + 40 + 16 * int(np.ceil(np.cbrt(float(abs(w)))))
    du = _dn(u, nmx, nmax)
    ddv, ddw = (_dn(z, nmx, nmax) - _dn(z, far, nmax) for z in (v, w))
    (pv, cv), (pw, cw), (py, cy) = (_rb(z, nmax) for z in (v, w, np.clongdouble(y)))
    n = np.arange(1, nmax + 1).astype(np.longdouble)
    dpv, dpw = pv[:-1] - n / v * pv[1:], pw[:-1] - n / w * pw[1:]
    dcw = cw[:-1] - n / w * cw[1:]
    t, cc = du * pv[1:], ddv * pv[1:]
    U, V = m * t - dpv - cc, t / m - dpv - cc
    A, B = pw[1:] * cv[1:] - cw[1:] * pv[1:], dpw * cv[1:] - dcw * pv[1:]
    Dd, Dg = pw[1:] + U * A, pw[1:] + V * A
    Nd, Ng = dpw + U * B + ddw * Dd, dpw + V * B + ddw * Dg
    xi, xi1 = py[1:] - 1j * cy[1:], py[:-1] - 1j * cy[:-1]
    Pa, Pb, Ma = Nd + m2 * Dd * n / y, m2 * Ng + Dg * n / y, m2 * Dd
    return ((Pa * py[1:] - Ma * py[:-1]) / (Pa * xi - Ma * xi1),
            (Pb * py[1:] - Dg * py[:-1]) / (Pb * xi - Dg * xi1))


def _run(h, x, y, m1, m2, sort):
    import torch
    from geosmie_amd import _lib
    from geosmie_amd._lib import check, ptr
    L, s, n = _lib.lib(), _lib.stream(), x.size
    dx, dy = _lib.to_dev(x), _lib.to_dev(y)
    e1, e2 = _lib.cplx_dev(m1 ** 2), _lib.cplx_dev(m2 ** 2)
    off = torch.empty(n + 1, dtype=torch.int64, device="cuda")
    check(L.gm_coef_offsets(h, n, ptr(dy), ptr(off), s))
    an = torch.zeros(2 * int(off[-1]), dtype=torch.float64, device="cuda")
    bn, props = torch.zeros_like(an), torch.zeros(6 * n, dtype=torch.float64, device="cuda")
    check(L.gm_mie_batch(h, n, ptr(dx), ptr(dy), ptr(e1), None, ptr(e2), float(y.max()), ptr(off),
                         ptr(an), ptr(bn), ptr(props), None, _lib.GM_MIE_SORT if sort else 0, s))
    return an, bn, props.view(6, n)


# 1024 / 2048 points are the last with 64 / 32 lanes; the largest shells and the
# smallest cores of a batch; series of one to three rows a lane and of many; points
# of the other classes between (equal radii, absorbing shells); input order
@pytest.mark.parametrize("n, y_hi, q_lo, sort", [
    (1, 0.01, 0.5, True), (1, 900.0, 0.5, True), (77, 3.0, 0.05, True), (1024, 209.0, 0.3, True),
    (1025, 60.0, 1e-4, True), (2048, 400.0, 0.3, False), (2049, 1000.0, 0.3, True),
    (6144, 15.0, 0.01, True)])
def test_lanes_per_point(gpu, n, y_hi, q_lo, sort):
    import torch
    from geosmie_amd import _lib
    from geosmie_amd.autotune import set_knob
    rng = np.random.default_rng(n)
    y = np.exp(np.linspace(np.log(y_hi), np.log(min(y_hi, 0.01)), n))
    x = y * np.exp(rng.uniform(np.log(q_lo), np.log(0.99), n))
    m1 = np.where(np.arange(n) % 3 == 0, 1.95 + 0.79j, 1.45 + 1e-4j)
    m2 = np.where(np.arange(n) % 2 == 0, 1.33 + 0j, 1.5 + 0.5e-3j)
    if n > 100:
        x[5::50] = y[5::50]
        m2[7::50] = 1.6 + 0.4j
    h, ref = _lib.private_ctx(), _lib.private_ctx()
    set_knob(ref, "coated_lanes", 1)
    got, want = _run(h, x, y, m1, m2, sort), _run(ref, x, y, m1, m2, sort)
    assert all(torch.equal(torch.isnan(a), torch.isnan(b)) for a, b in zip(got, want))
    coated = (x != y) & (m2.imag * y <= 1.0)
    rest = torch.from_numpy(~coated).to(got[2].device)
    same = torch.nan_to_num(got[2][:, rest]) == torch.nan_to_num(want[2][:, rest])
    assert bool(same.all())
    an, bn = (t.cpu().numpy().view(complex) for t in got[:2])
    props = got[2].cpu().numpy()
    off = np.concatenate([[0], np.cumsum(_nmax(y))])
    pick = np.flatnonzero(coated)
    for i in pick[::max(1, pick.size // 24)]:
        a, b = _exact(x[i], y[i], (m1 ** 2)[i], (m2 ** 2)[i])
        for z, r in ((an, a), (bn, b)):
            d = np.abs(z[off[i]:off[i + 1]] - r)
            assert np.all(np.isnan(d) | (d <= 1e-10)), i
        if np.isnan(props[0, i]):
            continue
        k = np.arange(1, a.size + 1)
        ext = 2 * ((2 * k + 1) * (a + b).real).sum() / y[i] ** 2
        sca = 2 * ((2 * k + 1) * (abs(a) ** 2 + abs(b) ** 2)).sum() / y[i] ** 2
        asy = (((2 * k + 1) / (k * (k + 1)) * (a * b.conj()).real).sum()
               + (k * (k + 2) / (k + 1) * (a * np.append(a[1:], 0).conj()
                                           + b * np.append(b[1:], 0).conj()).real).sum())
        assert abs(props[0, i] - ext) <= 5e-12 * ext and abs(props[1, i] - sca) <= 5e-12 * sca, i
        assert abs(props[4, i] - 4 * asy / (sca * y[i] ** 2)) <= 5e-12, i


# above 24576 points one per lane: the split of the longest (skewed sizes; 16 and, from
# 1200 rows on, 64 lanes) and of every point (uniform long series); more than 512k
# points, which only look for a split where series reach 512 rows
@pytest.mark.parametrize("n, y_lo, y_hi, skew", [
    (24577, 0.02, 209.0, True), (24577, 600.0, 700.0, False), (24577, 1.0, 2000.0, None),
    (512 * 1024 + 1, 1.0, 600.0, None)])
def test_long_points_of_a_batch(gpu, n, y_lo, y_hi, skew):
    got, want = _both(n, y_lo, y_hi, skew)
    # an absorbing core needs no start correction: both forms hold 1e-9
    for a, b in zip(got, want):
        assert _torch().equal(_torch().isnan(a), _torch().isnan(b))
    for a, b in zip(got[:2], want[:2]):
        assert float(_torch().nan_to_num(a - b).abs().max()) <= 2e-9
    for q in (0, 1, 4):
        rel = _torch().nan_to_num((got[2][q] - want[2][q]) / want[2][q])
        assert float(rel.abs().max()) <= 2e-9, q


# no split where it would not pay: short series, and sizes whose longest chain costs
# about what splitting it would (then every point is serial: the same bits)
@pytest.mark.parametrize("n, y_lo, y_hi, skew", [(24577, 1.0, 20.0, False),
                                                 (250000, 0.02, 400.0, True)])
def test_batches_that_stay_whole(gpu, n, y_lo, y_hi, skew):
    got, want = _both(n, y_lo, y_hi, skew)
    assert all(_torch().equal(_torch().nan_to_num(a), _torch().nan_to_num(b))
               for a, b in zip(got, want))


def _torch():
    import torch
    return torch


def _both(n, y_lo, y_hi, skew):
    """The batch with its lanes chosen by size and with one point per lane; skew: sizes
    log-distributed, None: a few of the longest among short ones."""
    from geosmie_amd import _lib
    from geosmie_amd.autotune import set_knob
    rng = np.random.default_rng(int(y_hi))
    y = (np.exp(rng.uniform(np.log(y_lo), np.log(y_hi), n)) if skew
         else rng.uniform(y_lo, y_hi if skew is False else 20.0, n))
    if skew is None:
        y[::400] = np.linspace(0.65 * y_hi, y_hi, y[::400].size)
    x = y * rng.uniform(0.3, 0.9, n)
    m1, m2 = np.full(n, 1.95 + 0.79j), np.full(n, 1.4 + 0j)
    x[5::500] = y[5::500]
    h, ref = _lib.private_ctx(), _lib.private_ctx()
    set_knob(ref, "coated_lanes", 1)
    return _run(h, x, y, m1, m2, True), _run(ref, x, y, m1, m2, True)


# the lanes per point set by hand, on a batch that runs one per lane by itself
@pytest.mark.parametrize("lanes", [16, 32, 64])
def test_lanes_set_by_hand(gpu, lanes):
    from geosmie_amd import _lib
    from geosmie_amd.autotune import get, set_knob
    n = 30001
    rng = np.random.default_rng(lanes)
    y = np.exp(rng.uniform(np.log(0.02), np.log(60.0), n))
    x = y * rng.uniform(0.3, 0.9, n)
    m1, m2 = np.full(n, 1.95 + 0.79j), np.full(n, 1.4 + 0j)
    h, ref = _lib.private_ctx(), _lib.private_ctx()
    set_knob(h, "coated_lanes", lanes)
    set_knob(ref, "coated_lanes", 1)
    assert get(h, "coated_lanes") == lanes
    got, want = _run(h, x, y, m1, m2, True), _run(ref, x, y, m1, m2, True)
    for a, b in zip(got[:2], want[:2]):
        assert _torch().equal(_torch().isnan(a), _torch().isnan(b))
        assert float(_torch().nan_to_num(a - b).abs().max()) <= 2e-9
    for q in (0, 1, 4):
        rel = _torch().nan_to_num((got[2][q] - want[2][q]) / want[2][q])
        assert float(rel.abs().max()) <= 2e-9, q
