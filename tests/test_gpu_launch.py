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
