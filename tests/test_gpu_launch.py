"""Launches that cover several axes or directions at once, against the forms
that take them one by one, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import oracle
from asterx_amd import abi
from asterx_amd.patch import Patch
from states import make_state

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return torch


def _lib():
    from asterx_amd import lib
    return lib.lib()


BC_FIELDS = ["rho", "dBx_stag", "dBy_stag", "dBz_stag", "Avec_x", "Avec_y", "Avec_z", "Psi"]


@pytest.mark.parametrize("kind", ["linear", "periodic", "copy"])
@pytest.mark.parametrize("n,ng", [((2, 2, 2), 1), ((3, 4, 3), 3), ((17, 5, 9), 3),
                                  ((5, 3, 70), 2), ((130, 2, 3), 2), ((1, 1, 1), 3)])
def test_boundary_fill(n, ng, kind):
    """One launch for every axis of every centering against the oracle's fill,
    axis after axis; the single-field entry point too."""
    torch = _torch()
    if kind == "linear" and min(n) < 2 or kind == "periodic" and min(n) < ng:
        pytest.skip("refused: too few points for this kind")
    rng = np.random.default_rng(3)
    h = Patch(n, ng, (0, 0, 0), (0.1, 0.2, 0.3), slots=BC_FIELDS)
    for name in BC_FIELDS:
        h[name] = rng.normal(size=h.shape(name))
    many, one = h.to("cuda"), h.to("cuda")
    L, k = _lib(), abi.BC[kind]
    slots = (C.c_int32 * len(BC_FIELDS))(*[abi.SLOT[m] for m in BC_FIELDS])
    abi.check("asx_bc_fill_many", L.asx_bc_fill_many(
        C.byref(many.struct()), len(BC_FIELDS), slots, k, None))
    for name in BC_FIELDS:
        abi.check("asx_bc_fill", L.asx_bc_fill(C.byref(one.struct()), abi.SLOT[name], k, None))
        abi.check("orc_bc_fill", oracle.lib().orc_bc_fill(
            C.byref(h.struct()), abi.SLOT[name], k))
    torch.cuda.synchronize()
    for name in BC_FIELDS:
        assert np.array_equal(many.numpy(name), h.numpy(name)), name
        assert np.array_equal(one.numpy(name), h.numpy(name)), name


@pytest.mark.parametrize("n", [(4, 5, 6), (16, 15, 7), (33, 31, 30)])
@pytest.mark.parametrize("recon", ["wenoz", "mp5", "ppm", "minmod"])
@pytest.mark.parametrize("halo", [0, 1])
def test_faces_in_one_launch(n, recon, halo):
    """The faces of every direction and the auxiliaries in one launch against
    one launch per direction in other tile shapes."""
    torch = _torch()
    L = _lib()
    par = abi.params(reconstruction_method=recon, flux_type="HLLE", loworder_method="minmod")
    names = abi.FLUX + abi.AUX + abi.UCT
    got = []
    kcs = [abi.KCLASS["face_" + c] for c in "xyz"]
    try:
        for v in (0, 1):
            for kc in kcs:
                abi.check("asx_set_variant", L.asx_set_variant(kc, v))
            d = make_state(n=n, curved=True, zero_entropy_block=True).to("cuda")
            for name in names:
                d[name].fill_(0.0)
            abi.check("asx_fluxes", L.asx_fluxes(C.byref(d.struct()), C.byref(par), halo, None,
                                                 None))
            torch.cuda.synchronize()
            got.append({m: d.numpy(m) for m in names})
    finally:
        for kc in kcs:
            abi.check("asx_set_variant", L.asx_set_variant(kc, 0))
    for m in names:
        assert np.array_equal(got[0][m], got[1][m]), m


@pytest.mark.parametrize("n", [(62, 4, 3), (64, 17, 16), (130, 3, 33)])
@pytest.mark.parametrize("recon", ["wenoz", "ppm"])
def test_long_row_faces(n, recon):
    """The tiles of long rows (variant 8: 64 x 4 x 1 in x, 16 x 1 x 16 in z) at
    and beside whole rows, one direction at a time, against the one launch."""
    torch = _torch()
    L = _lib()
    par = abi.params(reconstruction_method=recon, flux_type="HLLE", loworder_method="minmod")
    kcs = [abi.KCLASS["face_" + c] for c in "xyz"]
    got = []
    try:
        for pick in (None, 0, 1, 2):
            for d, kc in enumerate(kcs):
                abi.check("asx_set_variant", L.asx_set_variant(kc, 8 if d == pick else 0))
            p = make_state(n=n, curved=True, zero_entropy_block=True).to("cuda")
            for name in abi.FLUX:
                p[name].fill_(0.0)
            abi.check("asx_fluxes", L.asx_fluxes(C.byref(p.struct()), C.byref(par), 1, None,
                                                 None))
            torch.cuda.synchronize()
            got.append({m: p.numpy(m) for m in abi.FLUX})
    finally:
        for kc in kcs:
            abi.check("asx_set_variant", L.asx_set_variant(kc, 0))
    for g in got[1:]:
        for m in abi.FLUX:
            assert np.array_equal(got[0][m], g[m]), m


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("n,nz", [((160, 90, 130), 9), ((40, 20, 60), 1), ((5, 3, 17), 4)])
def test_tmunu_runs(order, n, nz):
    """The tensor does not depend on the length of the runs along z, which the
    number of tiles sets: a patch against a slab of it."""
    torch = _torch()
    L, ng = _lib(), 2
    par = abi.params(tmunu_interp_order=order)
    fields = abi.PRIMS + abi.ADM[:10]
    gen = torch.Generator(device="cuda").manual_seed(8)
    p = Patch(n, ng, (0, 0, 0), (1, 1, 1), slots=fields + abi.TMUNU, device="cuda")
    z0 = n[2] // 3
    q = Patch((n[0], n[1], nz), ng, (0, 0, 0), (1, 1, 1), slots=fields + abi.TMUNU,
              device="cuda")
    for name in fields:
        p[name].copy_(torch.rand(p.shape(name), dtype=torch.float64, device="cuda",
                                 generator=gen) * 0.1)
        if name in ("alp", "gxx", "gyy", "gzz"):
            p[name].add_(1.0)
        q[name].copy_(p[name][z0:z0 + q.shape(name)[0]])
    for d in (p, q):
        abi.check("asx_tmunu", L.asx_tmunu(C.byref(d.struct()), C.byref(par), None))
    torch.cuda.synchronize()
    for name in abi.TMUNU:
        a = p[name][ng + z0:ng + z0 + nz + 1, ng:ng + n[1] + 1, ng:ng + n[0] + 1]
        assert torch.equal(a, q[name][q.interior(name)]), name
        assert bool((a != 0).all())
    p["eTtt"][p.interior("eTtt")].zero_()
    assert bool((p["eTtt"] == 0).all())  # nothing outside the interior


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("n", [(15, 15, 15), (16, 17, 18), (63, 31, 30), (64, 31, 31)])
def test_update_with_every_load_in_flight(n, order):
    """The small-patch update (16 x 2 x 2 tiles up to 1024 of them) against the
    tiled one, on either side of that line, bit for bit."""
    torch = _torch()
    from asterx_amd.patch import StateBuf
    L, kc = _lib(), abi.KCLASS["update"]
    par = abi.params(reconstruction_method="wenoz", flux_type="HLLE", local_spatial_order=order)
    d = make_state(n=n, curved=True).to("cuda")
    u0 = StateBuf(d)
    for name in abi.STATE:
        u0.arr[name] = d[name].clone() * 1.01
    got = []
    try:
        for v in (0, 1):
            abi.check("asx_set_variant", L.asx_set_variant(kc, v))
            out = StateBuf(d, fill=0.0)
            abi.check("asx_substep", L.asx_substep(
                C.byref(d.struct()), C.byref(u0.struct()), C.byref(out.struct()), 0.75, 0.25,
                0.0025, C.byref(par), None))
            torch.cuda.synchronize()
            got.append({m: out.arr[m].cpu().numpy() for m in abi.STATE})
    finally:
        abi.check("asx_set_variant", L.asx_set_variant(kc, 0))
    for m in abi.STATE:
        assert np.array_equal(got[0][m], got[1][m]), m
