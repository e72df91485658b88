"""Every form of the resident loops (csrc/eio_resident.h) that a call can be given: tiles of 64 rows by 16 R
columns, the NL forward up to R = 6, its free-surface and decimating forms to R = 6 and 5, the adjoint to 5, both Born passes to
R = 4, half of that or less in FP64; and that the calls ran resident, which results alone do not show.
A single shot takes the smallest R whose tiles fit the 256 compute units.
Bars: those of the launched kernels, FP32 1e-5 and FP64 1e-11 relative L2 against the FP64 oracle (gradients
2e-5 and 1e-10); forwards of either form give the same bits where the updates' sums are spelled out."""
import numpy as np
import pytest

import oracle as O

from helpers import GRID_OF_COMP, random_traces, rel_l2
from test_resident_gpu import _check, _ctx, _forward_case, _model, _positions

pytestmark = pytest.mark.gpu

GRAD_TOL = {np.float32: 2e-5, np.float64: 1e-10}


def _r(nz, nx):
    """The smallest R whose 64 x 16 R tiles of an nz x nx grid fit 256 compute units."""
    return next(r for r in range(1, 100) if -(-(nz - 8) // 64) * -(-(nx - 8) // (16 * r)) <= 256)


class _Resident:
    """Asserts the cooperative launches of a block, with no wait given up and none refused."""

    def __init__(self, ctx, launches):
        self.ctx, self.launches = ctx, launches

    def __enter__(self):
        self.before = self.ctx.resident_info()

    def __exit__(self, *exc):
        if exc[0] is None:
            after = self.ctx.resident_info()
            assert after[0] - self.before[0] == self.launches and after[1:] == self.before[1:], (self.before, after)


@pytest.mark.parametrize("dtype,nz,nx,r,nts,sub", [
    (np.float32, 139, 61, 1, 51, 2), (np.float32, 281, 967, 2, 34, 3), (np.float32, 563, 1103, 3, 92, 1),
    (np.float32, 601, 1593, 4, 51, 2), (np.float32, 683, 1503, 5, 51, 2), (np.float32, 1025, 1500, 6, 51, 2),
    (np.float64, 139, 61, 1, 51, 2), (np.float64, 391, 1200, 2, 34, 3)])
def test_forward_bits_launched_and_resident(dtype, nz, nx, r, nts, sub):
    """The NL forward of each R against the oracle, and its launched form (FP32: two steps per launch on the
    streamed stage, odd step counts and sub-samplings among them; FP64: one) bit for bit."""
    assert _r(nz, nx) == r
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, nts, sub, nz + nx)
    rng = np.random.default_rng(nz * nx + 10)
    shot, keep, rec, ref = _forward_case(ctx, mid, g, med, rng, dtype, 40, 90)
    with _Resident(ctx, 1):
        ctx.nl_forward([shot])
    _check(rec, ref, dtype)
    first = [x.copy() for x in rec]
    if dtype == np.float32:
        ctx.set_time_block(2, 12)
    else:
        ctx.set_variant(0)
    with _Resident(ctx, 0):
        ctx.nl_forward([shot])
    for k in range(5):
        assert np.array_equal(first[k], rec[k]), k
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,r", [
    (np.float32, 139, 61, 1), (np.float32, 281, 967, 2), (np.float32, 563, 1103, 3), (np.float32, 601, 1593, 4),
    (np.float32, 683, 1503, 5), (np.float32, 1025, 1500, 6), (np.float64, 139, 61, 1), (np.float64, 391, 1200, 2)])
def test_free_surface_tiles(dtype, nz, nx, r):
    """The free-surface forward of each R, sources and receivers on every row, the surface and the rows above it
    among them; the launched form to the same bar."""
    assert _r(nz, nx) == r
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, 51, 2, nz + nx, surface=1)
    rng = np.random.default_rng(nz * nx + 11)
    spos, rpos = _positions(rng, g, 40), _positions(rng, g, 90)
    top = np.array([x * nz + z for x in range(4, nx - 4, max(1, nx // 40)) for z in (4, 7, 8, 9)], np.int32)
    rpos = [np.unique(np.concatenate([p, top])).astype(np.int32) for p in rpos]
    spos = [np.unique(np.concatenate([p, top[1::7]])).astype(np.int32) for p in spos]
    src = random_traces(rng, spos, g.nts, np.float64)
    ref = O.nl_fwd_reg(g, med, spos, src, rpos, np.float64)
    rec = [np.zeros((rpos[GRID_OF_COMP[k]].size, g.nts), dtype) for k in range(5)]
    shot, keep = ctx.make_shot(mid, spos, rpos, [np.ascontiguousarray(s, dtype) for s in src], rec)
    with _Resident(ctx, 1):
        ctx.nl_forward([shot])
    _check(rec, ref, dtype)
    ctx.set_variant(0)
    with _Resident(ctx, 0):
        ctx.nl_forward([shot])
    _check(rec, ref, dtype)
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,r", [
    (np.float32, 500, 480, 1), (np.float32, 281, 967, 2), (np.float32, 563, 1103, 3), (np.float32, 601, 1593, 4),
    (np.float32, 683, 1503, 5), (np.float64, 139, 90, 1), (np.float64, 391, 1200, 2)])
def test_adjoint_runs_resident(dtype, nz, nx, r):
    assert _r(nz, nx) == r
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, 51, 2, nz + nx)
    rng = np.random.default_rng(nz * nx + 12)
    spos, rpos = _positions(rng, g, 30), _positions(rng, g, 60)
    dat = random_traces(rng, rpos, g.nts, np.float64)
    src = [np.zeros((spos[GRID_OF_COMP[k]].size, g.nts), dtype) for k in range(5)]
    shot, keep = ctx.make_shot(mid, spos, rpos, src, [np.ascontiguousarray(s, dtype) for s in dat])
    with _Resident(ctx, 1):
        ctx.nl_adjoint([shot])
    _check(src, O.nl_adj_reg(g, med, spos, rpos, dat, np.float64), dtype)
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,r,nts,sub", [
    (np.float32, 300, 700, 1, 70, 4),     # three launches of 32, 32 and 5 intervals
    (np.float32, 300, 700, 1, 34, 5),     # one interval over a launch, an odd sub-sampling
    (np.float32, 281, 967, 2, 66, 3),     # one interval over two launches: a state saved at an odd step
    (np.float32, 563, 1103, 3, 40, 4), (np.float32, 601, 1593, 4, 40, 3),
    (np.float64, 300, 500, 1, 70, 3), (np.float64, 391, 1200, 2, 40, 4)])
def test_born_runs_resident(dtype, nz, nx, r, nts, sub):
    """All passes of the Born forward and adjoint of one shot resident: the source pass in one launch, the
    others in launches of 32 coarse intervals."""
    assert _r(nz, nx) == r
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, nts, sub, nz + nx)
    rng = np.random.default_rng(nz * nx + 13)
    spos, rpos = _positions(rng, g, 10), _positions(rng, g, 90)
    src = [O.time_interp(s, g.dts, sub) for s in random_traces(rng, spos, nts, np.float64)]
    dat = random_traces(rng, rpos, nts, np.float64)
    dmod = np.zeros((5, nx, nz))
    dmod[:, 4:-4, 4:-4] = rng.standard_normal((5, nx - 8, nz - 8)) * np.abs(med).reshape(5, -1).max(1)[:, None, None]
    srcd, datd = [np.ascontiguousarray(s, dtype) for s in src], [np.ascontiguousarray(s, dtype) for s in dat]
    launches = 1 + -(-(nts - 1) // 32)
    dm = np.zeros((5, nx, nz), dtype)
    shot, keep = ctx.make_shot(mid, spos, rpos, srcd, datd)
    with _Resident(ctx, launches):
        ctx.born_adjoint([shot], dm)
    ref = O.born_adj_reg(g, med, spos, src, rpos, dat, np.float64)
    assert rel_l2(dm, ref) < GRAD_TOL[dtype], rel_l2(dm, ref)
    rec = [np.zeros_like(d) for d in datd]
    shot, keep = ctx.make_shot(mid, spos, rpos, srcd, rec)
    with _Resident(ctx, launches):
        ctx.born_forward([shot], np.ascontiguousarray(dmod, dtype))
    _check(rec, O.born_fwd_reg(g, med, spos, src, dmod, rpos, np.float64), dtype)
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,r,segment", [
    (np.float32, 281, 967, 2, 0), (np.float32, 601, 1593, 4, 21), (np.float32, 683, 1503, 5, 0), (np.float32, 683, 1503, 5, 21),
    (np.float64, 391, 1200, 2, 21)])
def test_fwi_runs_resident(dtype, nz, nx, r, segment):
    """FWI forward and two gradients, the second recomputing every segment: the forward and the recompute of each
    R (the receiver pass stays launched above R = 4), data and gradients against the oracle, the two gradients
    bit for bit."""
    assert _r(nz, nx) == r
    nts, sub = 42, 3 if segment else 2     # segments from an odd fine step on
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, nts, sub, nz + nx)
    rng = np.random.default_rng(nz * nx + 14)
    spos, rpos = _positions(rng, g, 10), _positions(rng, g, 60)
    src = random_traces(rng, spos, nts, np.float64)
    dat = random_traces(rng, rpos, nts, np.float64)
    srcd, datd = [np.ascontiguousarray(s, dtype) for s in src], [np.ascontiguousarray(s, dtype) for s in dat]
    rec = [np.zeros_like(d) for d in datd]
    nseg = 1 if not segment else -(-(nts - 1) // segment)
    receiver = 2 if r <= 4 else 0          # launches of 32 and 9 intervals
    shot, keep = ctx.make_shot(mid, spos, rpos, srcd, rec)
    with _Resident(ctx, nseg):
        h = ctx.fwi_forward([shot], segment if segment else nts - 1)
    _check(rec, O.nl_fwd_reg(g, med, spos, src, rpos, np.float64), dtype)
    ref = O.born_adj_reg(g, med, spos, [O.time_interp(s, g.dts, sub) for s in src], rpos, dat, np.float64)
    grads = []
    for recomputed in (nseg - 1, nseg):
        shot, keep = ctx.make_shot(mid, spos, rpos, srcd, datd)
        dm = np.zeros((5, nx, nz), dtype)
        with _Resident(ctx, recomputed + receiver):
            ctx.fwi_gradient(h, [shot], dm)
        assert rel_l2(dm, ref) < GRAD_TOL[dtype], rel_l2(dm, ref)
        grads.append(dm)
    assert np.array_equal(grads[0], grads[1])
    ctx.fwi_release(h)
    ctx.close()


def test_born_batch_runs_resident():
    """Eight shots of one grid in groups of several R: every pass of every group resident."""
    ctx = _ctx(np.float32)
    nz, nx, nts, sub = 281, 473, 40, 4
    mid, g, med = _model(ctx, nz, nx, nts, sub, 71)
    rng = np.random.default_rng(72)
    shots, keeps, ref = [], [], 0.0
    for i in range(8):
        spos, rpos = _positions(rng, g, 5), _positions(rng, g, 40)
        src = [O.time_interp(s, g.dts, sub) for s in random_traces(rng, spos, nts, np.float64)]
        dat = random_traces(rng, rpos, nts, np.float64)
        ref = ref + O.born_adj_reg(g, med, spos, src, rpos, dat, np.float64)
        shot, keep = ctx.make_shot(mid, spos, rpos, [np.ascontiguousarray(s, np.float32) for s in src],
                                   [np.ascontiguousarray(s, np.float32) for s in dat])
        shots.append(shot)
        keeps.append(keep)
    before = ctx.resident_info()
    dm = np.zeros((5, nx, nz), np.float32)
    ctx.born_adjoint(shots, dm)
    after = ctx.resident_info()
    # at least two groups, whose receiver passes take two launches each, and the source pass
    assert after[0] - before[0] >= 1 + 2 * 2 and after[1:] == before[1:], (before, after)
    assert rel_l2(dm, ref) < GRAD_TOL[np.float32], rel_l2(dm, ref)
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,nshot,nts,resident", [
    (np.float32, 72, 24, 1, 51, True),       # one tile: no exchange
    (np.float32, 72, 1500, 1, 101, True),    # one row of tiles
    (np.float32, 139, 61, 1, 51, True),      # 12 tiles, two an XCD
    (np.float32, 200, 200, 1, 120, False),   # 36 tiles that all trade across XCDs: launched steps are faster
    (np.float32, 200, 200, 4, 120, True),    # four of them: most of a shot on one XCD
    (np.float32, 200, 200, 2, 120, True),    # two: nine tiles an XCD, three whole columns
    (np.float32, 200, 330, 1, 120, False),   # 63 tiles, not whole columns, 66,000 cells
    (np.float32, 500, 480, 1, 120, True),    # enough cells for a step of its own length
    (np.float64, 200, 200, 1, 120, False), (np.float64, 200, 200, 4, 120, True), (np.float64, 280, 472, 1, 120, True)])
def test_forward_takes_the_faster_form(dtype, nz, nx, nshot, nts, resident):
    """The rule between resident and launched steps on small grids, either form against the oracle."""
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, nts, 2, nz + nx)
    rng = np.random.default_rng(nz * nx + 15)
    cases = [_forward_case(ctx, mid, g, med, rng, dtype, 10, 20) for _ in range(nshot)]
    with _Resident(ctx, int(resident)):
        ctx.nl_forward([c[0] for c in cases])
    for _, _, rec, ref in cases:
        _check(rec, ref, dtype)
    ctx.close()


def test_born_groups_pay_for_every_launch():
    """Sixteen small shots: the receiver pass takes one group of R = 4, whose three launches of 32 intervals are set
    up three times, not two groups of R = 2, which are six and slower for it."""
    ctx = _ctx(np.float32)
    nz, nx, nts, sub = 92, 434, 70, 4
    mid, g, med = _model(ctx, nz, nx, nts, sub, 73)
    rng = np.random.default_rng(74)
    shots, keeps, ref = [], [], 0.0
    for i in range(16):
        spos, rpos = _positions(rng, g, 4), _positions(rng, g, 20)
        src = [O.time_interp(s, g.dts, sub) for s in random_traces(rng, spos, nts, np.float64)]
        dat = random_traces(rng, rpos, nts, np.float64)
        ref = ref + O.born_adj_reg(g, med, spos, src, rpos, dat, np.float64)
        shot, keep = ctx.make_shot(mid, spos, rpos, [np.ascontiguousarray(s, np.float32) for s in src],
                                   [np.ascontiguousarray(s, np.float32) for s in dat])
        shots.append(shot)
        keeps.append(keep)
    dm = np.zeros((5, nx, nz), np.float32)
    with _Resident(ctx, 1 + 3):              # the source pass in one launch of R = 4
        ctx.born_adjoint(shots, dm)
    assert rel_l2(dm, ref) < GRAD_TOL[np.float32], rel_l2(dm, ref)
    ctx.close()


def test_born_source_pass_takes_the_form_of_the_others():
    """One shot of 200 x 200: the receiver pass of the Born adjoint is resident and so is the source pass beside it; the
    scattered pass of the Born forward is launched (intervals of 64 steps) and so is its source pass."""
    ctx = _ctx(np.float32)
    nz, nx, nts, sub = 200, 200, 150, 2
    mid, g, med = _model(ctx, nz, nx, nts, sub, 75)
    rng = np.random.default_rng(76)
    spos, rpos = _positions(rng, g, 10), _positions(rng, g, 60)
    src = [O.time_interp(s, g.dts, sub) for s in random_traces(rng, spos, nts, np.float64)]
    dat = random_traces(rng, rpos, nts, np.float64)
    dmod = np.zeros((5, nx, nz))
    dmod[:, 4:-4, 4:-4] = rng.standard_normal((5, nx - 8, nz - 8)) * np.abs(med).reshape(5, -1).max(1)[:, None, None]
    srcd, datd = [np.ascontiguousarray(s, np.float32) for s in src], [np.ascontiguousarray(s, np.float32) for s in dat]
    dm = np.zeros((5, nx, nz), np.float32)
    shot, keep = ctx.make_shot(mid, spos, rpos, srcd, datd)
    with _Resident(ctx, 1 + 5):
        ctx.born_adjoint([shot], dm)
    ref = O.born_adj_reg(g, med, spos, src, rpos, dat, np.float64)
    assert rel_l2(dm, ref) < GRAD_TOL[np.float32], rel_l2(dm, ref)
    rec = [np.zeros_like(d) for d in datd]
    shot, keep = ctx.make_shot(mid, spos, rpos, srcd, rec)
    with _Resident(ctx, 0):
        ctx.born_forward([shot], np.ascontiguousarray(dmod, np.float32))
    _check(rec, O.born_fwd_reg(g, med, spos, src, dmod, rpos, np.float64), np.float32)
    ctx.close()
