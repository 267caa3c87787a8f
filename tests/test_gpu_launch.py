"""Launches that cover several axes or directions at once, against the forms
that take them one by one, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import oracle
from asterx_amd import abi
from asterx_amd.patch import Patch

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

