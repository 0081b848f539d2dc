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


def test_refused_allocation_leaves_levels_whole():
    """A level whose arrays cannot be allocated is left without grids, and the
    pinned Courant array that the other levels' steps write stays theirs."""
    run("child_refused_level")


def child_refused_level(fake):
    from amrclaw_amd import capi
    H = nested_hierarchy(np.random.default_rng(1), flat_states(4), 4, nlev=2, dt1=0.004)
    many = [(8 * i, 8 * i + 3, 0, 3) for i in range(200)]
    capi.init(capi.make_config(capi.EULER))
    for kind in (fake_hip.PINNED, fake_hip.DEVICE):
        capi.load_hierarchy(H)
        capi.set_level(2, [], 0.01, 0.01)
        live = fake.live(fake_hip.DEVICE)
        for n in range(1, 100):
            fake.refuse(kind, n)
            try:
                capi.set_level(2, many, 0.01, 0.01)
            except capi.AmrgpuError:
                pass
            else:
                break
            assert fake.live(fake_hip.DEVICE) == live, (kind, n)
            fake.clear()
            dt, cfl = capi.sweep_level(2, 1e-3)[::-1]
            assert cfl == 0.0 and not fake.launches("sweep"), (kind, n)
            capi.sweep_level(1, 1e-3)
            assert [x[2] != 0 for x in fake.launches("copy_u64")] == [True], (kind, n)
        assert n > 1, kind
        fake.refuse(kind, 0)
        for bad in ((0, 3, 4, 3), (0, 30000, 0, 3)):     # an empty grid, too large a one
            with pytest.raises(capi.AmrgpuError):
                capi.set_level(2, many + [bad], 0.01, 0.01)
            with pytest.raises(capi.AmrgpuError):
                capi.put_grid(2, 0, np.ones((8, 8, 4)))
    capi.finalize()
    assert fake.live(fake_hip.DEVICE) == fake.live(fake_hip.PINNED) == 0


def test_refused_batch_is_not_kept():
    """amrgpu3_stepgrid keeps its one-grid batch for the next call of the same
    shape, but not one whose arrays could not all be allocated."""
    run("child_refused_batch")


def child_refused_batch(fake):
    from amrclaw_amd import capi, capi3
    q = np.ones((9, 8, 10, 5))
    for precision in (capi.FP64, capi.FP32):
        capi3.init3(capi3.make_config3(capi.EULER, precision=precision))
        refused = 0
        for n in range(1, 100):
            capi3.set_patches3([(3, 3, 3)])
            fake.refuse(fake_hip.DEVICE, n)
            try:
                capi3.set_patches3([(6, 4, 5)])
            except capi.AmrgpuError:
                refused += 1
                with pytest.raises(capi.AmrgpuError):
                    capi3.get_patch3(0, q.shape)
                with pytest.raises(capi.AmrgpuError):
                    fake.refuse(fake_hip.DEVICE, 1)
                    capi3.stepgrid3(q, 0.1, 0.1, 0.1, 0.01)
            else:
                break
        fake.refuse(fake_hip.DEVICE, 0)
        assert refused >= 8
        capi3.stepgrid3(q, 0.1, 0.1, 0.1, 0.01)
        allocs = fake.allocs(fake_hip.DEVICE)
        capi3.stepgrid3(q, 0.1, 0.1, 0.1, 0.01)     # the batch at hand
        assert fake.allocs(fake_hip.DEVICE) == allocs
        capi3.finalize3()
        assert fake.live(fake_hip.DEVICE) == fake.live(fake_hip.PINNED) == 0


def test_steps3_without_memory_take_the_phase_kernels():
    """The 3-D steps that need memory of their own (the two-pass FP64 step, the
    fused FP32 step of a level) give way to the phase kernels where any part of it
    is refused."""
    run("child_steps3_without_memory")


def child_steps3_without_memory(fake):
    from amrclaw_amd import capi, capi3
    from tests.common3 import nested_hierarchy3, smooth_euler3
    phases, passes, tiles = "sweep3_phase", "pass3_solve", "sweep3_tile"

    def step():
        fake.clear()
        capi3.step_patches3(0.1, 0.1, 0.1, 0.01)
        return bool(fake.launches(phases)), bool(fake.launches(passes))

    capi3.init3(capi3.make_config3(capi.EULER))
    sizes = [(6, 5, 4), (8, 3, 7)]
    capi3.set_patches3(sizes)
    n0 = fake.allocs(fake_hip.DEVICE)
    assert step() == (False, True)
    nstep = fake.allocs(fake_hip.DEVICE) - n0
    for n in range(1, nstep + 1):
        capi3.finalize3()
        capi3.init3(capi3.make_config3(capi.EULER))
        capi3.set_patches3(sizes)
        before = fake.live(fake_hip.DEVICE)
        fake.refuse(fake_hip.DEVICE, n)
        assert step() == (True, False) == step(), n       # and the steps after it
        assert fake.live(fake_hip.DEVICE) == before, n
        capi3.set_patches3(sizes)
        assert step() == (False, True), n                 # a new layout asks again
    capi3.finalize3()

    H = nested_hierarchy3(np.random.default_rng(3), smooth_euler3, 5, nlev=2)
    survived = 0
    for n in range(1, 200):
        capi3.init3(capi3.make_config3(capi.EULER, precision=capi.FP32))
        capi3.load_hierarchy3(H)
        n0 = fake.allocs(fake_hip.DEVICE)
        fake.refuse(fake_hip.DEVICE, n)
        fake.clear()
        try:
            for level in (1, 2):
                capi3.advance_level3(level)
        except capi.AmrgpuError:
            pass
        else:
            used = fake.allocs(fake_hip.DEVICE) - n0
            survived += used >= n
            assert len(fake.launches(tiles)) == (1 if used >= n else 2), n
            assert bool(fake.launches(phases)) == (used >= n), n
        fake.refuse(fake_hip.DEVICE, 0)
        capi3.finalize3()
        if n > fake.allocs(fake_hip.DEVICE) - n0:
            break
    assert survived == 5      # tiles and marks of either level, the finest's second buffer
    assert fake.live(fake_hip.DEVICE) == fake.live(fake_hip.PINNED) == 0


def test_march_tables_without_memory():
    """A level that marches because it is faster does without where the march's
    tables (its waves; with a finer level the map and entries of fluxsv) are
    refused: the tile sweep steps it."""
    run("child_march_tables")


def child_march_tables(fake):
    from amrclaw_amd import capi
    boxes = [(100 * i, 100 * i + 99, 100 * j, 100 * j + 99) for j in range(8) for i in range(8)]
    fine = [(220, 259, 220, 259), (300, 339, 300, 349)]

    def load():
        capi.set_geometry([800, 1600], [800, 1600], [2, 2], [2, 2], [1 / 800, 1 / 1600],
                          [1 / 800, 1 / 1600])
        capi.set_level(1, boxes, 1 / 800, 1 / 800)
        capi.set_level(2, fine, 1 / 1600, 1 / 1600)
        for level in (1, 2):
            capi.set_time(level, 0.0, 1e-4 / level)

    survived = 0
    for n in range(0, 200):
        capi.init(capi.make_config(capi.EULER))
        n0 = fake.allocs(fake_hip.DEVICE)
        fake.refuse(fake_hip.DEVICE, n)
        fake.clear()
        try:
            load()
            capi.advance_level(1)
        except capi.AmrgpuError:
            pass
        else:
            used = fake.allocs(fake_hip.DEVICE) - n0
            marched = bool(fake.launches("sweep_march"))
            assert marched == (n == 0 or used < n), n
            assert marched or fake.launches("sweep_kernel"), n
            survived += not marched
        fake.refuse(fake_hip.DEVICE, 0)
        total = fake.allocs(fake_hip.DEVICE) - n0
        capi.finalize()
        assert fake.live(fake_hip.DEVICE) == 0, n
        if n > total:
            break
    assert survived == 4      # the waves, the map, its cells, the entries


def test_tile_caps_bind():
    """The caps of amrgpu_set_tiling are the caller's also on levels of few grids;
    only the library's own are narrowed there."""
    run("child_tile_caps")


def child_tile_caps(fake):
    from amrclaw_amd import capi
    boxes = [(28 * i, 28 * i + 27, 0, 27) for i in range(4)]

    def tiles(call):
        fake.clear()
        call()
        return [x[1] for x in fake.launches("sweep_kernel")]

    one = lambda: capi.stepgrid_noalloc(28, 28, 1, 1, 0.01, 0.01, 1e-3)
    level = lambda: capi.sweep_level(1, 1e-3)
    for solver in (capi.EULER, capi.ACOUSTICS):
        for mode in (capi.LAUNCH_BATCHED, capi.LAUNCH_PER_PATCH):
            capi.init(capi.make_config(solver, precision=capi.MIXED))
            capi.set_launch_mode(mode)
            capi.set_level(1, boxes, 0.01, 0.01)
            batched = mode == capi.LAUNCH_BATCHED
            assert tiles(level) == ([4 * 9] if batched else [1] * 4)
            assert tiles(one) == [9]
            capi.set_tiling(0, 0)                     # nothing asked for
            assert sum(tiles(level)) == (4 * 9 if batched else 4) and tiles(one) == [9]
            capi.set_tiling(28, 28)
            assert sum(tiles(level)) == 4 and tiles(one) == [1]
            capi.set_tiling(0, 16)
            assert sum(tiles(level)) == 8 and tiles(one) == [2]
            capi.set_level(1, boxes[:3], 0.01, 0.01)
            assert sum(tiles(level)) == 6
            capi.finalize()
    capi.init(capi.make_config(capi.EULER, precision=capi.MIXED))
    capi.set_level(1, boxes, 0.01, 0.01)
    assert tiles(level) == [4 * 9]                    # a new context's caps are its own again
    capi.finalize()


def test_regrid_copies_run_side_by_side():
    """The copies of old grids into a new one touch no cell of each other or of the
    interpolation: each has a workgroup of its own."""
    run("child_regrid_units")


def child_regrid_units(fake):
    from amrclaw_amd import capi
    old = [(32 + 16 * i, 47 + 16 * i, 32 + 16 * j, 47 + 16 * j) for j in range(4) for i in range(4)]
    new = [(34, 97, 34, 97)]
    capi.init(capi.make_config(capi.EULER))
    capi.set_geometry([64, 128], [64, 128], [2, 2], [2, 2], [1 / 64, 1 / 128], [1 / 64, 1 / 128])
    capi.set_level(1, [(0, 63, 0, 63)], 1 / 64, 1 / 64)
    capi.set_level(2, old, 1 / 128, 1 / 128)
    fake.clear()
    capi.regrid_level(2, new, 0.0)
    # 16 copies; the coarse patch and the interpolation out of it together
    assert [x[1] for x in fake.launches("fill_kernel")] == [17]
    capi.finalize()


@pytest.mark.parametrize("sizes,transverse,passes", [
    ([(40, 40, 40)] * 8, 22, True), ([(40, 40, 40)] * 8, 0, True),
    ([(40, 40, 40)] * 64, 0, False), ([(16, 16, 16)] * 512, 22, False),
    ([(16, 16, 16)] * 512, 0, False), ([(6, 7, 5)] * 512, 22, True), ([(1, 1, 1)], 22, True)])
def test_route_of_fp64_advection_steps(sizes, transverse, passes):
    """Batches that fill the chip keep the phase kernels where these are the
    faster ones: the advection solver's (Euler always takes the passes)."""
    run("child_advection_route", sizes, transverse, passes)


def child_advection_route(fake, sizes, transverse, passes):
    from amrclaw_amd import capi, capi3
    for solver, want in ((capi.ADVECTION, passes), (capi.EULER, True)):
        capi3.init3(capi3.make_config3(solver, transverse=transverse))
        capi3.set_patches3(sizes[:200])
        capi3.set_patches3(sizes)                      # the route is the layout's
        fake.clear()
        capi3.step_patches3(0.1, 0.1, 0.1, 0.01)
        assert bool(fake.launches("pass3_solve")) == want, solver
        assert bool(fake.launches("sweep3_phase")) == (not want), solver
        capi3.finalize3()


@pytest.mark.parametrize("n,transverse,fused", [(8, 22, True), (12, 22, False), (14, 11, False),
                                                (16, 22, True), (46, 22, True), (12, 0, False),
                                                (8, 0, True), (46, 0, True)])
def test_route_of_fp32_advection_levels(n, transverse, fused):
    """A level's fused step where it is the faster one: not for the advection
    solver on few grids that make one large tile each."""
    run("child_advection_levels", n, transverse, fused)


def child_advection_levels(fake, n, transverse, fused):
    from amrclaw_amd import capi, capi3
    from amrclaw_amd.hierarchy import Hier3
    for solver, nvar, want in ((capi.ADVECTION, 1, fused), (capi.EULER, 5, True)):
        H = Hier3(nvar)
        H.add_level([(0, n - 1) * 3], (1 / n,) * 3, 0.1 / n, 0.0, (n, n, n))
        H.add_level([(4, 11) * 3], (0.5 / n,) * 3, 0.05 / n, 0.0, (2 * n, 2 * n, 2 * n))
        capi3.init3(capi3.make_config3(solver, precision=capi.FP32, transverse=transverse))
        capi3.load_hierarchy3(H)
        fake.clear()
        capi3.advance_level3(1)
        assert bool(fake.launches("sweep3_tile")) == want, solver
        assert bool(fake.launches("sweep3_phase")) == (not want), solver
        capi3.finalize3()


@pytest.mark.parametrize("solver", ["acoustics", "euler"])
@pytest.mark.parametrize("ngrids,small", [(9, True), (135, False)])
def test_cut_of_few_grids(solver, ngrids, small):
    """The levels of test_gpu_sweep.py::test_small_tiles_bit_exact: cut into 12x12
    tiles at most, or by the library's caps, and swept by tiles either way."""
    run("child_cut", solver, ngrids, small)


def child_cut(fake, solver, ngrids, small):
    from amrclaw_amd import capi
    from tests.common import SOLVERS
    from tests.test_gpu_sweep import SMALL_TILE_SIZES
    sizes = [SMALL_TILE_SIZES[k % len(SMALL_TILE_SIZES)] for k in range(ngrids)]
    boxes, x = [], 0
    for mx, my in sizes:
        boxes.append((x, x + mx - 1, 0, my - 1))
        x += mx
    n = {}
    for mode in (capi.LAUNCH_BATCHED, capi.LAUNCH_PERSISTENT):
        capi.init(capi.make_config(SOLVERS[solver]))
        capi.set_launch_mode(mode)
        capi.set_level(1, boxes, 1 / 64, 1 / 48)
        fake.clear()
        capi.sweep_level(1, 0.002)
        assert not fake.launches("sweep_march")
        (launch,) = fake.launches("sweep_kernel") or fake.launches("sweep_persist")
        n[mode] = launch[1]
        capi.finalize()
    cut = lambda size, cap: -(-size // cap)
    twelve = sum(cut(mx, 12) * cut(my, 12) for mx, my in sizes)
    caps = sum(cut(mx, 28) * cut(my, 12) for mx, my in sizes)
    assert caps < twelve and n[capi.LAUNCH_BATCHED] == (twelve if small else caps)


@pytest.mark.parametrize("solver,precision,grids,marches", [
    ("euler", "FP64", [(100, 100)] * 60, True), ("euler", "FP64", [(30, 30)] * 20, False),
    ("euler", "MIXED", [(100, 100)] * 60, False), ("euler", "FP32", [(100, 100)] * 60, False),
    ("acoustics", "FP64", [(100, 100)] * 60, False)])
def test_sweep_of_the_default_launch(solver, precision, grids, marches):
    run("child_default_sweep", solver, precision, grids, marches)


def child_default_sweep(fake, solver, precision, grids, marches):
    from amrclaw_amd import capi
    from tests.common import SOLVERS
    boxes, x = [], 0
    for mx, my in grids:
        boxes.append((x, x + mx - 1, 0, my - 1))
        x += mx
    capi.init(capi.make_config(SOLVERS[solver], precision=getattr(capi, precision)))
    capi.set_level(1, boxes, 0.01, 0.01)
    fake.clear()
    capi.sweep_level(1, 1e-3)
    assert bool(fake.launches("sweep_march")) == marches
    assert bool(fake.launches("sweep_kernel")) == (not marches)
    capi.finalize()
