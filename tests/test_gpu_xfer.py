"""Transfers of grids between the host heap and the device (xfer.hpp): a ring
of pinned slots (2 MiB, eight of them) that a transfer may wrap, host copies by
several threads from 8 MiB on, grids that straddle slots.  A put followed by a
get returns the values bit for bit (FP32 storage: rounded to FP32), at the
caller's offsets only; whole-level and single-grid transfers agree."""
import numpy as np
import pytest

from amrclaw_amd import capi, capi3

pytestmark = pytest.mark.gpu

# grids of a level by their total size: one small grid; a little under and over
# one slot (65,536 cells of 4 components); several slots, one thread; threads,
# once and several times round the ring
LEVELS = {
    "small": [(3, 5)],
    "slot-": [(251, 252)],
    "slot+": [(252, 252), (1, 1)],
    "serial": [(120, 77), (64, 200), (255, 255), (9, 1)],
    "threads": [(500, 300), (7, 900), (640, 480), (1, 1), (33, 1000)],
    "wrap": [(900, 800), (1100, 700), (17, 23), (800, 901)],
}


@pytest.mark.parametrize("precision", [capi.FP64, capi.FP32])
@pytest.mark.parametrize("name", list(LEVELS))
def test_level_round_trip(gpu, name, precision):
    rng = np.random.default_rng(3)
    boxes, x0 = [], 0
    for mx, my in LEVELS[name]:
        boxes.append((x0, x0 + mx - 1, 0, my - 1))
        x0 += mx
    shapes = [(b[3] + 5, b[1] - b[0] + 5, 4) for b in boxes]
    sizes = [int(np.prod(s)) for s in shapes]
    # gaps between the grids' blocks, which a transfer must not touch
    offs = np.cumsum([11] + [n + 13 for n in sizes[:-1]]).astype(np.int64)
    heap = rng.normal(size=int(offs[-1]) + sizes[-1] + 17)
    print("level round trip", name, precision, sum(sizes), flush=True)
    capi.init(capi.make_config(capi.EULER, precision=precision))
    try:
        capi.set_level(1, boxes, 0.1, 0.1)
        L = capi.lib()
        for which in (0, 1, 0):       # three transfers: the ring goes on where it was
            capi._check(L.amrgpu_put_level(1, which, heap, offs))
            back = np.full(heap.size, -7.0)
            capi._check(L.amrgpu_get_level(1, which, back, offs))
            ref = np.full(heap.size, -7.0)
            for o, n in zip(offs, sizes):
                v = heap[o:o + n]
                ref[o:o + n] = v if precision == capi.FP64 else v.astype(np.float32)
            assert np.array_equal(back, ref)
        for k, (o, n, s) in enumerate(zip(offs, sizes, shapes)):
            assert np.array_equal(capi.get_grid(1, k, s).ravel(), ref[o:o + n]), k
        q = rng.normal(size=shapes[-1])
        capi.put_grid(1, len(shapes) - 1, q, which=1)
        got = capi.get_grid(1, len(shapes) - 1, shapes[-1], which=1)
        assert np.array_equal(got, q if precision == capi.FP64 else q.astype(np.float32))
    finally:
        capi.finalize()


@pytest.mark.parametrize("precision", [capi3.FP64, capi3.FP32])
def test_stepgrid3_reuses_its_batch(gpu, precision):
    """stepgrid3 calls in a row, the shape kept and changed in between, give
    what a fresh batch gives, and the flags of the call before are forgotten."""
    rng = np.random.default_rng(5)
    cfg = capi3.make_config3(capi3.EULER, precision=precision)

    def grid(mx, my, mz):
        sh = (mz + 4, my + 4, mx + 4)
        rho, p = 0.8 + 0.4 * rng.random(sh), 0.8 + 0.4 * rng.random(sh)
        u = [0.2 * rng.normal(size=sh) for _ in range(3)]
        return np.stack([rho] + [rho * w for w in u] +
                        [p / 0.4 + 0.5 * rho * sum(w * w for w in u)], -1)
    qs = [grid(9, 7, 6), grid(9, 7, 6), grid(5, 8, 6), grid(9, 7, 6)]
    fresh = []
    for q in qs:
        capi3.init3(cfg)
        fresh.append(capi3.stepgrid3(q, 0.1, 0.1, 0.1, 0.01, want_fluxes=True))
        capi3.finalize3()
    capi3.init3(cfg)
    try:
        for q, (qf, ff, cf, df) in zip(qs, fresh):
            qn, fl, c, d = capi3.stepgrid3(q, 0.1, 0.1, 0.1, 0.01, want_fluxes=True)
            assert np.array_equal(qn, qf) and c == cf and d == df
            assert all(np.array_equal(a, b) for a, b in zip(fl, ff))
            with pytest.raises(capi3.AmrgpuError):
                capi3.get_flags3(0, q.shape[:3])      # no flags of this batch yet
            capi3.flag_patches3(0.05)
            capi3.get_flags3(0, q.shape[:3])
    finally:
        capi3.finalize3()
