"""Evolution with a program's own sync(names), which may put other arrays in
the patch: the calls after it see them."""
import numpy as np
import pytest

import oracle
from asterx_amd import abi
from asterx_amd.driver import Evolution, all_slots
from states import make_state


class Exchange(Evolution):
    """A SYNC that fills new arrays and drops the old ones' contents."""
    calls = 0

    def sync(self, names):
        self.calls += 1
        super().sync(names)
        for n in names:
            if n in self.p:
                old = self.p.arr[n]
                self.p.arr[n] = old.copy()
                old[...] = np.nan


def _run(cls, instance):
    par = abi.params(reconstruction_method="ppm", flux_type="HLLE", gl_gamma=5.0 / 3.0)
    p = make_state(n=(6, 5, 7), curved=True, seed=3)
    for n in all_slots():
        if n not in p:
            p.alloc(n)
    ev = cls(oracle.backend(), p, par)
    if instance:
        fill = ev.sync
        ev.sync = lambda names: fill(names)
    ev.rhs()
    ev.poststep()
    return ev, {n: p.numpy(n).copy() for n in p.arr}


@pytest.mark.parametrize("instance", [False, True])
def test_sync_of_the_program(instance):
    _, want = _run(Evolution, False)
    ev, got = _run(Exchange, instance)
    assert ev.calls == 7  # three in the right-hand side, four after the step
    for n in want:
        assert np.array_equal(got[n], want[n], equal_nan=True), n
