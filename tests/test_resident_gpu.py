"""Resident time loops (csrc/eio_resident.h: one cooperative launch, the state on the chip) against
the FP64 oracle, at the sizes where their tiles can go wrong: 64 rows by 16 R columns, R = 1..5,
with remainders of one to four rows and columns, tiles that end on the grid's edge, more devices than
a wave keeps in registers, uneven batches, and the repeat with launched kernels after a wait is given up.
Bars: those of the launched kernels, FP32 1e-5 and FP64 1e-11 relative L2."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle as O
from elastic_isotropic_operators_amd import _capi
from elastic_isotropic_operators_amd import workloads as W

from helpers import GRID_OF_COMP, random_traces, rel_l2, scattered_positions

pytestmark = pytest.mark.gpu

TOL = {np.float32: 1e-5, np.float64: 1e-11}


def _ctx(dtype):
    ctx = _capi.Context(0, dtype)
    if dtype == np.float32:
        ctx.set_time_block(2, _capi.VARIANT_AUTO)
        ctx.set_adjoint_time_block(2, _capi.VARIANT_AUTO)
    return ctx


def _model(ctx, nz, nx, nts, sub, seed, surface=0, pad=12):
    """A padded grid of exactly nz x nx cells; (model id, oracle grid, media)."""
    rng = np.random.default_rng(seed)
    vp = 2200.0 + 900.0 * rng.random((1, nz)) + 60.0 * rng.random((nx, nz))
    vs = vp / 1.8
    rho = 1800.0 + 300.0 * rng.random((nx, 1)) + 0.0 * vp
    g = O.grid(nz, nx, nts, sub, 10.0, 10.0, 0.0008 * sub / 2, pad, surface=surface)
    med = O.media(g, np.stack([rho, rho * (vp * vp - 2 * vs * vs), rho * vs * vs]), np.float64)
    mid = ctx.model_add(nz, nx, nts, sub, g.dz, g.dx, g.dts, pad, med, g.alphaCos, surface=surface)
    return mid, g, med


def _positions(rng, g, n, below=4):
    p = scattered_positions(rng, g.nz, g.nx, n)
    return [q[q % g.nz >= below] for q in p]


def _forward_case(ctx, mid, g, med, rng, dtype, nsrc, nrec, below=4):
    spos, rpos = _positions(rng, g, nsrc, below), _positions(rng, g, nrec, below)
    src = random_traces(rng, spos, g.nts, np.float64)
    ref = O.nl_fwd_reg(g, med, spos, src, rpos, np.float64)
    rec = [np.zeros((rpos[GRID_OF_COMP[k]].size, g.nts), dtype) for k in range(5)]
    shot, keep = ctx.make_shot(mid, spos, rpos, [np.ascontiguousarray(s, dtype) for s in src], rec)
    return shot, keep, rec, ref


def _check(rec, ref, dtype):
    for k in range(5):
        assert np.linalg.norm(ref[k]) > 0
        assert rel_l2(rec[k], ref[k]) < TOL[dtype], (k, rel_l2(rec[k], ref[k]))


@pytest.mark.parametrize("dtype,nz,nx,nsrc,nrec", [
    (np.float32, 72, 24, 10, 20),       # one full tile of R = 1
    (np.float32, 73, 25, 10, 20),       # one row and one column over
    (np.float32, 76, 28, 10, 20),       # the four halo rows and columns exactly
    (np.float32, 40, 90, 300, 700),     # more entries than a wave keeps in registers
    (np.float32, 139, 61, 20, 40),
    (np.float32, 281, 967, 40, 60),     # R = 2
    (np.float32, 563, 1103, 40, 60),    # R = 3
    (np.float32, 601, 1593, 40, 60),    # R = 4
    (np.float32, 683, 1503, 40, 60),    # R = 5
    (np.float64, 73, 25, 10, 20),
    (np.float64, 40, 90, 300, 700),
    (np.float64, 281, 967, 40, 60),     # R = 2
])
def test_forward_tiles(dtype, nz, nx, nsrc, nrec):
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, 51, 2, nz + nx)
    rng = np.random.default_rng(nz * nx)
    shot, keep, rec, ref = _forward_case(ctx, mid, g, med, rng, dtype, nsrc, nrec)
    ctx.nl_forward([shot])
    assert ctx.last_timing()[1] == 1          # one launch
    _check(rec, ref, dtype)
    first = [r.copy() for r in rec]
    ctx.nl_forward([shot])                     # the buffers of the first call are reused
    for k in range(5):
        assert np.array_equal(first[k], rec[k]), k
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_forward_uneven_batch(dtype):
    """Shots of several grids, lengths and sub-samplings in one launch, odd counts among them."""
    ctx = _ctx(dtype)
    rng = np.random.default_rng(5)
    cases = []
    for i, (nz, nx, nts, sub) in enumerate([(90, 130, 50, 2), (150, 90, 27, 4), (61, 200, 33, 3), (75, 75, 90, 1)]):
        mid, g, med = _model(ctx, nz, nx, nts, sub, 50 + i)
        cases.append(_forward_case(ctx, mid, g, med, rng, dtype, 8, 20))
    ctx.nl_forward([c[0] for c in cases])
    for _, _, rec, ref in cases:
        _check(rec, ref, dtype)
    ctx.close()


def test_forward_many_groups():
    """More tiles than compute units: groups one after the other, each with its own inboxes."""
    ctx = _ctx(np.float32)
    rng = np.random.default_rng(6)
    models = [_model(ctx, 200 + 3 * i, 700 + 50 * i, 50 + i, 2, 60 + i) for i in range(3)]
    cases = [_forward_case(ctx, *models[i % 3], rng, np.float32, 5, 15) for i in range(9)]
    ctx.nl_forward([c[0] for c in cases])
    assert ctx.last_shot_groups() >= 2
    for _, _, rec, ref in cases:
        _check(rec, ref, np.float32)
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx", [(np.float32, 73, 25), (np.float32, 330, 601), (np.float64, 139, 90)])
def test_forward_free_surface(dtype, nz, nx):
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, 51, 2, 7, surface=1)
    rng = np.random.default_rng(8)
    shot, keep, rec, ref = _forward_case(ctx, mid, g, med, rng, dtype, 20, 40, below=9)
    ctx.nl_forward([shot])
    assert ctx.last_timing()[1] == 1
    _check(rec, ref, dtype)
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_given_up_wait_repeats_with_launched_kernels(dtype):
    """A spin limit of one poll ends the resident launch (every workgroup leaves at its next wait); the
    call then runs its loop with launched kernels."""
    ctx = _ctx(dtype)
    ctx.set_persistent(0, 1)
    mid, g, med = _model(ctx, 281, 301, 51, 2, 9)
    rng = np.random.default_rng(10)
    shot, keep, rec, ref = _forward_case(ctx, mid, g, med, rng, dtype, 20, 40)
    ctx.nl_forward([shot])
    assert ctx.last_timing()[1] > 1
    _check(rec, ref, dtype)
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,segment", [(np.float32, 139, 90, 0), (np.float32, 281, 967, 0), (np.float32, 563, 1103, 26),
                                                 (np.float64, 139, 90, 0), (np.float64, 281, 967, 26)])
def test_fwi_record_and_checkpoints(dtype, nz, nx, segment):
    """FWI forward and gradient with the forward (whole record, or checkpoints whose segments are long enough
    for a resident launch) and the recompute resident: data and gradient against the oracle, a second gradient
    (which recomputes every segment) bit for bit, and both again after a given-up wait."""
    ctx = _ctx(dtype)
    nts, sub = 80, 4
    mid, g, med = _model(ctx, nz, nx, nts, sub, 11)
    rng = np.random.default_rng(12)
    spos, rpos = _positions(rng, g, 10), _positions(rng, g, 30)
    src = random_traces(rng, spos, nts, np.float64)
    dat = random_traces(rng, rpos, nts, np.float64)
    fine = [O.time_interp(s, g.dts, sub) for s in src]
    ref = O.nl_fwd_reg(g, med, spos, src, rpos, np.float64)
    ref_dm = O.born_adj_reg(g, med, spos, fine, rpos, dat, np.float64)
    srcd = [np.ascontiguousarray(s, dtype) for s in src]
    datd = [np.ascontiguousarray(s, dtype) for s in dat]
    grads = []
    for limit in (0, 1):
        if limit:
            ctx.set_persistent(0, limit)
        rec = [np.zeros((rpos[GRID_OF_COMP[k]].size, nts), dtype) for k in range(5)]
        shot, keep = ctx.make_shot(mid, spos, rpos, srcd, rec)
        h = ctx.fwi_forward([shot], segment if segment else nts - 1)
        _check(rec, ref, dtype)
        for _ in range(2):
            shot, keep2 = ctx.make_shot(mid, spos, rpos, srcd, datd)
            dm = np.zeros((5, nx, nz), dtype)
            ctx.fwi_gradient(h, [shot], dm)
            assert rel_l2(dm, ref_dm) < (2e-5 if dtype == np.float32 else 1e-10), rel_l2(dm, ref_dm)
            grads.append(dm)
        ctx.fwi_release(h)
    assert np.array_equal(grads[0], grads[1])
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,nts,sub,nsrc,nrec", [
    (np.float32, 72, 24, 51, 2, 10, 20),       # one full tile of R = 1
    (np.float32, 73, 25, 50, 3, 10, 20),       # one row and one column over, an odd sub-sampling
    (np.float32, 76, 28, 90, 1, 10, 20),
    (np.float32, 40, 90, 51, 2, 700, 700),     # more entries than a wave keeps in registers
    (np.float32, 281, 967, 51, 2, 40, 60),     # R = 2
    (np.float32, 563, 1103, 51, 2, 40, 60),    # R = 3
    (np.float32, 601, 1593, 51, 2, 40, 60),    # R = 4
    (np.float32, 683, 1503, 51, 2, 40, 60),    # R = 5
    (np.float64, 73, 25, 50, 3, 10, 20),
    (np.float64, 40, 90, 51, 2, 700, 700),
    (np.float64, 281, 967, 51, 2, 40, 60),     # R = 2
])
def test_adjoint_tiles(dtype, nz, nx, nts, sub, nsrc, nrec):
    """The NL adjoint, then again with its waits given up (launched kernels): both against the oracle, and
    the resident one again into buffers of the call before."""
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, nts, sub, nz + nx)
    rng = np.random.default_rng(nz * nx + 1)
    spos, rpos = _positions(rng, g, nsrc), _positions(rng, g, nrec)
    dat = random_traces(rng, rpos, nts, np.float64)
    ref = O.nl_adj_reg(g, med, spos, rpos, dat, np.float64)
    datd = [np.ascontiguousarray(s, dtype) for s in dat]
    out = []
    for limit in (0, 0, 1):
        if limit:
            ctx.set_persistent(0, limit)
        src = [np.full((spos[GRID_OF_COMP[k]].size, nts), 7, dtype) for k in range(5)]
        shot, keep = ctx.make_shot(mid, spos, rpos, src, datd)
        ctx.nl_adjoint([shot])
        _check(src, ref, dtype)
        out.append(src)
    for k in range(5):
        assert np.array_equal(out[0][k], out[1][k]), k
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_adjoint_batch(dtype):
    """Shots of several grids (one step count) in one launch, and a step limit that ends inside a coarse
    sample: the same as the launched kernels."""
    ctx = _ctx(dtype)
    rng = np.random.default_rng(15)
    shots, outs, refs, keeps = [], [], [], []
    for i, (nz, nx) in enumerate([(90, 130), (150, 90), (61, 200)]):
        mid, g, med = _model(ctx, nz, nx, 50, 4, 70 + i)
        spos, rpos = _positions(rng, g, 8), _positions(rng, g, 20)
        dat = random_traces(rng, rpos, g.nts, np.float64)
        refs.append(O.nl_adj_reg(g, med, spos, rpos, dat, np.float64))
        src = [np.zeros((spos[GRID_OF_COMP[k]].size, g.nts), dtype) for k in range(5)]
        shot, keep = ctx.make_shot(mid, spos, rpos, src, [np.ascontiguousarray(s, dtype) for s in dat])
        shots.append(shot)
        outs.append(src)
        keeps.append(keep)
    ctx.nl_adjoint(shots)
    for src, ref in zip(outs, refs):
        _check(src, ref, dtype)
    ctx.set_step_limit(186)
    ctx.nl_adjoint(shots)
    part = [[s.copy() for s in src] for src in outs]
    ctx.set_persistent(0, 1)
    ctx.nl_adjoint(shots)
    for src, p in zip(outs, part):
        for k in range(5):
            assert np.any(p[k]) and rel_l2(p[k], src[k]) < TOL[dtype], k
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,nts,sub", [
    (np.float32, 73, 25, 70, 3),      # R = 1, one row and one column over, three launches of 32 coarse intervals
    (np.float32, 76, 28, 34, 4),      # one interval over a launch
    (np.float32, 139, 90, 33, 4),     # exactly one launch
    (np.float32, 281, 967, 40, 2),    # R = 2
    (np.float32, 563, 1103, 40, 2),   # R = 3
    (np.float32, 601, 1593, 40, 2),   # R = 4
    (np.float64, 73, 25, 70, 3),
    (np.float64, 281, 967, 40, 2),    # R = 2
])
def test_born_adjoint_tiles(dtype, nz, nx, nts, sub):
    """Both Born passes resident for a batch of two shots, twice in the same buffers, and with every wait given
    up; the gradient against the oracle's, summed over the shots."""
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, nts, sub, nz + nx)
    rng = np.random.default_rng(nz * nx + 2)
    shots, keeps, ref = [], [], 0.0
    for i in range(2 if nz * nx < 400000 else 1):
        spos, rpos = _positions(rng, g, 10), _positions(rng, g, 80)
        src = [O.time_interp(s, g.dts, sub) for s in random_traces(rng, spos, nts, np.float64)]
        dat = random_traces(rng, rpos, nts, np.float64)
        ref = ref + O.born_adj_reg(g, med, spos, src, rpos, dat, np.float64)
        shot, keep = ctx.make_shot(mid, spos, rpos, [np.ascontiguousarray(s, dtype) for s in src],
                                   [np.ascontiguousarray(s, dtype) for s in dat])
        shots.append(shot)
        keeps.append(keep)
    grads = []
    for limit in (0, 0, 1):
        if limit:
            ctx.set_persistent(0, limit)
        dm = np.zeros((5, nx, nz), dtype)
        ctx.born_adjoint(shots, dm)
        assert rel_l2(dm, ref) < (2e-5 if dtype == np.float32 else 1e-10), rel_l2(dm, ref)
        grads.append(dm)
    assert np.array_equal(grads[0], grads[1])
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx,nts,sub", [
    (np.float32, 73, 25, 70, 3),      # R = 1, one row and one column over, three launches of 32 coarse intervals
    (np.float32, 76, 28, 34, 4),      # one interval over a launch
    (np.float32, 139, 90, 33, 4),     # exactly one launch
    (np.float32, 281, 967, 40, 2),    # R = 2
    (np.float32, 563, 1103, 40, 2),   # R = 3
    (np.float32, 601, 1593, 40, 2),   # R = 4
    (np.float64, 73, 25, 70, 3),
    (np.float64, 281, 967, 40, 2),    # R = 2
])
def test_born_forward_tiles(dtype, nz, nx, nts, sub):
    """Both passes of the Born forward resident for a batch of two shots, twice in the same buffers, and with
    every wait given up; the data against the oracle's."""
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, nts, sub, nz + nx)
    rng = np.random.default_rng(nz * nx + 3)
    dm = np.zeros((5, nx, nz))
    dm[:, 4:-4, 4:-4] = rng.standard_normal((5, nx - 8, nz - 8)) * np.abs(med).reshape(5, -1).max(1)[:, None, None]
    shots, keeps, recs, refs = [], [], [], []
    for i in range(2 if nz * nx < 400000 else 1):
        spos, rpos = _positions(rng, g, 10), _positions(rng, g, 300)
        src = [O.time_interp(s, g.dts, sub) for s in random_traces(rng, spos, nts, np.float64)]
        refs.append(O.born_fwd_reg(g, med, spos, src, dm, rpos, np.float64))
        rec = [np.zeros((rpos[GRID_OF_COMP[k]].size, nts), dtype) for k in range(5)]
        shot, keep = ctx.make_shot(mid, spos, rpos, [np.ascontiguousarray(s, dtype) for s in src], rec)
        shots.append(shot)
        keeps.append(keep)
        recs.append(rec)
    dmd = np.ascontiguousarray(dm, dtype)
    first = None
    for limit in (0, 0, 1):
        if limit:
            ctx.set_persistent(0, limit)
        ctx.born_forward(shots, dmd)
        for rec, ref in zip(recs, refs):
            _check(rec, ref, dtype)
        if first is None:
            first = [[r.copy() for r in rec] for rec in recs]
        elif not limit:
            assert all(np.array_equal(a, b) for x, y in zip(first, recs) for a, b in zip(x, y))
    ctx.close()


_CHILD = """
import sys
import numpy as np
from elastic_isotropic_operators_amd import _capi
import test_resident_gpu as t
out = t._second_process_case()
np.save(sys.argv[1], out)
"""


def _second_process_case():
    """Data of an NL forward, an NL adjoint and both Born passes of one shot, in one row."""
    ctx = _ctx(np.float32)
    mid, g, med = _model(ctx, 139, 90, 90, 2, 21)
    rng = np.random.default_rng(22)
    spos, rpos = _positions(rng, g, 10), _positions(rng, g, 20)
    src = [np.ascontiguousarray(s, np.float32) for s in random_traces(rng, spos, g.nts, np.float64)]
    fine = [np.ascontiguousarray(O.time_interp(s.astype(np.float64), g.dts, 2), np.float32) for s in src]
    dat = [np.ascontiguousarray(s, np.float32) for s in random_traces(rng, rpos, g.nts, np.float64)]
    rec = [np.zeros_like(d) for d in dat]
    back = [np.zeros_like(s) for s in src]
    dm = np.zeros((5, g.nx, g.nz), np.float32)
    lin = [np.zeros_like(d) for d in dat]
    keep = []

    def shot(s, r):
        sh, k = ctx.make_shot(mid, spos, rpos, s, r)
        keep.append(k)
        return [sh]

    ctx.nl_forward(shot(src, rec))
    ctx.nl_adjoint(shot(back, dat))
    ctx.born_adjoint(shot(fine, dat), dm)
    ctx.born_forward(shot(fine, lin), np.ascontiguousarray(dm / np.abs(dm).max()))
    h = ctx.fwi_forward(shot(src, rec), 44)
    ctx.fwi_gradient(h, shot(src, dat), dm)
    ctx.fwi_release(h)
    ctx.close()
    parts = rec + back + [dm] + lin
    return np.concatenate([p.ravel() / np.linalg.norm(p) for p in parts])


def test_second_process(tmp_path):
    """Another process that uses the device while this one holds its cooperative queue: the same results, with
    launched kernels where it gets no cooperative launch."""
    mine = _second_process_case()
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([here, os.path.dirname(here)] + sys.path))
    out = str(tmp_path / "out.npy")
    subprocess.run([sys.executable, "-c", _CHILD, out], check=True, env=env, timeout=90)
    theirs = np.load(out)
    assert theirs.shape == mine.shape and rel_l2(theirs, mine) < 1e-5, rel_l2(theirs, mine)
