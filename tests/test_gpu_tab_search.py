"""The temperature search of con2prim on a table: its result does not depend
on the temperature it starts from, whatever the table and the zone's Ye."""
import ctypes as C

import numpy as np
import pytest

import oracle
from asterx_amd import abi, tabeos, zones

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def _zigzag(shape):
    """log(eps + shift) falling from every third T node to the next, by 0.3;
    steep everywhere, so that T and p stay well determined by eps."""
    tab = tabeos.build(*shape)
    n = tab["data"].shape[1]
    lev = np.cumsum(np.where(np.arange(n) % 3 == 2, -0.3, 0.4))
    tab["data"][..., 1] = lev[None, :, None] + np.linspace(-2, 1, shape[0])[None, None, :]
    eps = np.exp(tab["data"][..., 1]) - tab["shift"]
    tab["eps_min"], tab["eps_max"] = max(float(eps.min()), 1e-15), float(eps.max())
    return tab


def _par(tab):
    return tab.attach(abi.params(
        c2p_prime="Palenzuela", c2p_second="None", use_temperature=1, use_press_atmo=0,
        thermal_eos_atmo=1, t_atmo=0.01, Ye_atmo=0.3, c2p_tol=1e-10, max_iter=100, vw_lim=1e3,
        B_lim=1e3, ye_min=0.035, ye_max=0.55, rho_abs_min=1e-15))


def _solve(par, cons, g, seed):
    torch = _torch()
    from asterx_amd import lib
    nz = cons.shape[1]
    cd, gd, sd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (cons, g, seed))
    out = torch.empty((9, nz), dtype=torch.float64, device="cuda")
    flag = torch.empty(nz, dtype=torch.float64, device="cuda")
    it = torch.empty(nz, dtype=torch.int32, device="cuda")
    abi.check("asx_c2p_batch_ye", lib.lib().asx_c2p_batch_ye(
        nz, cd.data_ptr(), gd.data_ptr(), sd.data_ptr(), out.data_ptr(), flag.data_ptr(),
        it.data_ptr(), C.byref(par), None))
    torch.cuda.synchronize()
    return out.cpu().numpy(), flag.cpu().numpy(), it.cpu().numpy()


def _points(par, rho, eps, ye):
    """asx_eos_from_rho_eps: T, p, eps after the clamps."""
    torch = _torch()
    from asterx_amd import lib
    n = len(rho)
    r, e, y = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (rho, eps, ye))
    out = torch.empty((3, n), dtype=torch.float64, device="cuda")
    abi.check("asx_eos_from_rho_eps", lib.lib().asx_eos_from_rho_eps(
        n, r.data_ptr(), e.data_ptr(), y.data_ptr(), out.data_ptr(), C.byref(par), None))
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("shape", [(3, 4, 2), (20, 31, 5)])
def test_table_not_monotone_in_T(shape):
    """eps(T) falls here and there, so that several cells hold a root: every
    solve takes the one that asx_eos_from_rho_eps takes."""
    _torch()
    host = _zigzag(shape)
    dtab, htab = tabeos.Table(host, device="cuda"), tabeos.Table(host, device=None)
    par, par_h = _par(dtab), _par(htab)
    nz = 3000
    prim, g = zones.make_batch_ye(nz, 41, (1e-12, 1e-4), (0.05, 80.0), (0.06, 0.5), W_max=2.0)
    cons, thermo = np.zeros((9, nz)), np.zeros((2, nz))
    abi.check("orc_prim2con_batch_ye", oracle.lib().orc_prim2con_batch_ye(
        nz, prim.ctypes.data, g.ctypes.data, cons.ctypes.data, thermo.ctypes.data,
        C.byref(par_h)))
    ref = None
    for temp in (prim[1], np.full(nz, 0.0), np.full(nz, 1e300), prim[1, ::-1]):
        seed = np.stack([prim[0], thermo[0], prim[3], prim[4], prim[5], prim[2], temp])
        got = _solve(par, cons, g, seed)
        if ref is None:
            ref = got
        for a, b in zip(got, ref):
            assert np.array_equal(a, b, equal_nan=True)
    out, flag, _ = ref
    ok = flag == 1
    assert ok.mean() > 0.5
    rho, eps, press, ye = out[0, ok], out[1, ok], out[2, ok], out[8, ok]
    pts = _points(par, rho, eps, ye)
    # zones that the floors have not moved to another (T, eps): there p is
    # the table's at T.  log eps is good to a few ulps of its |log| < 16
    # (2e-15 each), and a cell's log p spans less than 30 times its log eps
    same = np.abs(pts[2] - eps) <= 1e-14 * (np.abs(eps) + host["shift"])
    assert same.mean() > 0.9
    assert (np.abs(pts[1] / press - 1)[same] <= 1e-12).all()


def test_ye_outside_the_table():
    """Beyond the Ye axis the interpolant is extrapolated and need not grow
    with T: the result still does not depend on the starting temperature."""
    _torch()
    host = tabeos.build(20, 31, 5)
    # cold energy that falls steeply with Ye, differently at each T
    host["data"][..., 1] += np.linspace(0, 1, 5)[:, None, None] * np.sin(
        np.arange(31))[None, :, None] * 0.05
    dtab = tabeos.Table(host, device="cuda")
    par = _par(dtab)
    par_h = _par(tabeos.Table(host, device=None))
    nz = 3000
    prim, g = zones.make_batch_ye(nz, 43, (1e-12, 1e-4), (0.05, 80.0), (0.06, 0.5), W_max=2.0)
    cons, thermo = np.zeros((9, nz)), np.zeros((2, nz))
    abi.check("orc_prim2con_batch_ye", oracle.lib().orc_prim2con_batch_ye(
        nz, prim.ctypes.data, g.ctypes.data, cons.ctypes.data, thermo.ctypes.data,
        C.byref(par_h)))
    cons[8] = cons[0] * np.random.default_rng(2).choice([-3.0, 2.0, 8.0, 40.0], nz)
    ref = None
    for temp in (prim[1], np.full(nz, 0.0), np.full(nz, 1e300)):
        seed = np.stack([prim[0], thermo[0], prim[3], prim[4], prim[5], prim[2], temp])
        got = _solve(par, cons, g, seed)
        if ref is None:
            ref = got
        for a, b in zip(got, ref):
            assert np.array_equal(a, b, equal_nan=True)
