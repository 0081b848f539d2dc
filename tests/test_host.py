"""CPU checks of the host library on a HIP runtime without a device
(tests/fake_hip.py): what a call launches and what it does when an allocation
is refused.  The child_* functions run in a process of their own."""
import ctypes as C
import os

import numpy as np
import pytest

from tests import fake_hip
from tests.common import nested_hierarchy

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PLUGIN = os.path.join(ROOT, "tests", "plugin", "libshallow_water.so")


def run(child, *args):
    fake_hip.run("tests.test_host", child, *args)


def flat_states(nvar):
    return lambda rng, shape: 1.0 + rng.random(shape + (nvar,))


@pytest.mark.skipif(not os.path.exists(PLUGIN), reason="plug-in not built")
def test_courant_read_back_with_a_plugin_table():
    """A registered table's qad launcher owes the library the registers only: a
    level step reads its own Courant maxima back also when the launcher is
    not the one AMRGPU_DEFINE_SOLVER makes."""
    run("child_plugin_courant")


def child_plugin_courant(fake):
    from amrclaw_amd import capi
    ops, keep = capi.load_solver_plugin(PLUGIN, "amrgpu_plugin_shallow_water")
    calls = []
    fn = C.CFUNCTYPE(C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p)
    qad = fn(lambda esize, a, ph, st: calls.append(esize) or 0)
    ops.qad = C.cast(qad, C.c_void_p)
    H = nested_hierarchy(np.random.default_rng(1), flat_states(3), 3, nlev=2, dt1=0.004)
    capi.init(capi.make_config(capi.register_solver(ops), nvar=3, mwaves=3))
    capi.load_hierarchy(H)
    for level in (1, 2):
        fake.clear()
        capi.advance_level(level)
        assert len(fake.launches("copy_u64")) == 1, level
    assert calls == [8]
    capi.finalize()
