"""Calls whose resident loops (csrc/eio_resident.h) give up a wait, are refused or run out of memory, or
that ask for launched steps: the launched kernels take over with the same answers.
Bars: those of the launched kernels, FP32 1e-5 and FP64 1e-11 relative L2 (gradients twice that and ten
times that, as sums over many products)."""
import ctypes
import importlib.util
import os
import shutil
import subprocess
import threading
import time

import numpy as np
import pytest

import oracle as O
from elastic_isotropic_operators_amd import _capi

from helpers import GRID_OF_COMP, random_traces, rel_l2
from test_resident_gpu import _check, _ctx, _forward_case, _model, _positions

pytestmark = pytest.mark.gpu

GRAD_TOL = {np.float32: 2e-5, np.float64: 1e-10}
ILLEGAL_STATE, LAUNCH_FAILURE = 401, 719   # hipErrorIllegalState (a held queue), hipErrorLaunchFailure


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    """(shim, the C ABI's binding on a copy of the library that calls the HIP runtime through it)."""
    d = tmp_path_factory.mktemp("shim")
    so, lib = str(d / "hip_shim.so"), str(d / "libeio_copy.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-o", so, os.path.join(os.path.dirname(__file__), "hip_shim.c"),
                    "-L/opt/rocm/lib", "-Wl,--no-as-needed", "-lamdhip64"], check=True)
    shutil.copy(_capi.LIB_PATH, lib)
    s = ctypes.CDLL(so, mode=ctypes.RTLD_GLOBAL)
    s.shim_capacity.argtypes = [ctypes.c_size_t]
    s.shim_live.restype = ctypes.c_size_t
    spec = importlib.util.spec_from_file_location("eio_capi_shimmed", _capi.__file__)
    capi = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(capi)
    capi.LIB_PATH = lib
    capi.lib()
    return s, capi


@pytest.fixture
def shimmed(shim):
    yield shim
    shim[0].shim_launches(0, 0, 0)
    shim[0].shim_capacity(2 ** 64 - 1)


def _shim_ctx(capi, dtype):
    ctx = capi.Context(0, dtype)
    if dtype == np.float32:
        ctx.set_time_block(2, capi.VARIANT_AUTO)
        ctx.set_adjoint_time_block(2, capi.VARIANT_AUTO)
    return ctx


@pytest.mark.parametrize("change", ["given_up", "graph"])
@pytest.mark.parametrize("dtype,sub", [(np.float32, 3), (np.float64, 3), (np.float64, 4)])
def test_launched_recompute_from_resident_checkpoints(dtype, sub, change):
    """A store made by resident loops whose segments are recomputed by launched steps, because the gradient
    gives up its waits or runs in graph mode: a segment may start at an odd fine step (odd sub-sampling and
    segment), where the launched steps expect the levels in the other order."""
    nts, segment, nz, nx = 80, 61, 139, 90      # a second segment from fine step 183 (244 with sub 4) on
    ctx = _ctx(dtype)
    mid, g, med = _model(ctx, nz, nx, nts, sub, 31)
    rng = np.random.default_rng(32)
    spos, rpos = _positions(rng, g, 10), _positions(rng, g, 30)
    src = random_traces(rng, spos, nts, np.float64)
    dat = random_traces(rng, rpos, nts, np.float64)
    ref = O.nl_fwd_reg(g, med, spos, src, rpos, np.float64)
    ref_dm = O.born_adj_reg(g, med, spos, [O.time_interp(s, g.dts, sub) for s in src], rpos, dat, np.float64)
    srcd = [np.ascontiguousarray(s, dtype) for s in src]
    datd = [np.ascontiguousarray(s, dtype) for s in dat]
    rec = [np.zeros((rpos[GRID_OF_COMP[k]].size, nts), dtype) for k in range(5)]
    shot, keep = ctx.make_shot(mid, spos, rpos, srcd, rec)
    before = ctx.resident_info()[0]
    h = ctx.fwi_forward([shot], segment)
    assert ctx.resident_info()[0] == before + 2
    _check(rec, ref, dtype)
    if change == "given_up":
        ctx.set_persistent(0, 1)
    else:
        ctx.set_graph(True)
    shot, keep = ctx.make_shot(mid, spos, rpos, srcd, datd)
    for _ in range(2):      # the first finds the last segment in the ring of the forward
        dm = np.zeros((5, nx, nz), dtype)
        ctx.fwi_gradient(h, [shot], dm)
        assert rel_l2(dm, ref_dm) < GRAD_TOL[dtype], rel_l2(dm, ref_dm)
    ctx.fwi_release(h)
    ctx.close()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_refused_launch_is_tried_again(shimmed, dtype):
    """A refused cooperative launch costs its call, and a growing count of the calls after it, the resident
    form, not the context's life; each call's data are right."""
    shim, capi = shimmed
    ctx = _shim_ctx(capi, dtype)
    mid, g, med = _model(ctx, 500, 480, 101, 2, 41)
    rng = np.random.default_rng(42)
    shot, keep, rec, ref = _forward_case(ctx, mid, g, med, rng, dtype, 10, 20)

    def form():
        for r in rec:
            r[...] = 7
        before = ctx.resident_info()[0]
        ctx.nl_forward([shot])
        resident = ctx.resident_info()[0] > before
        assert (ctx.last_timing()[1] == 1) == resident
        _check(rec, ref, dtype)
        return "RL"[not resident]

    def refused(launches, pause):
        """Refuses the next launches; the calls of the next `pause` seconds do not try, those after it do."""
        shim.shim_launches(ILLEGAL_STATE, launches, 0)
        for _ in range(launches):
            n = ctx.resident_info()[2]
            begin = time.monotonic()
            assert form() == "L" and ctx.resident_info()[1:] == (0, n + 1, ILLEGAL_STATE)
            again = form()
            if time.monotonic() < begin + pause:
                assert again == "L" and ctx.resident_info()[2] == n + 1
            time.sleep(pause + 32 * (time.monotonic() - begin))
            pause *= 2

    assert form() + form() == "RR"
    refused(1, 0.25)
    assert form() + form() == "RR"
    refused(2, 0.25)              # twice in a row: the second pause is twice as long
    assert form() == "R"
    refused(1, 0.25)              # a call that ran resident has ended the row
    assert form() == "R"
    ctx.close()


def test_other_launch_errors_are_raised(shimmed):
    """An error that is no refusal reaches the caller; the context runs resident afterwards."""
    shim, capi = shimmed
    ctx = _shim_ctx(capi, np.float32)
    mid, g, med = _model(ctx, 500, 480, 101, 2, 43)
    rng = np.random.default_rng(44)
    shot, keep, rec, ref = _forward_case(ctx, mid, g, med, rng, np.float32, 10, 20)
    shim.shim_launches(LAUNCH_FAILURE, 1, 0)
    with pytest.raises(capi.EioError, match="hipLaunchCooperativeKernel"):
        ctx.nl_forward([shot])
    assert ctx.resident_info()[:3] == (0, 0, 0)
    ctx.nl_forward([shot])
    assert ctx.resident_info()[0] == 1
    _check(rec, ref, np.float32)
    ctx.close()


def test_given_up_wait_is_not_paid_on_every_call():
    """After a call that gave up a wait, those of the next quarter of a second do not try."""
    ctx = _ctx(np.float32)
    ctx.set_persistent(0, 1)
    mid, g, med = _model(ctx, 500, 480, 51, 2, 45)
    rng = np.random.default_rng(46)
    shot, keep, rec, ref = _forward_case(ctx, mid, g, med, rng, np.float32, 10, 20)
    for given_up in (1, 2):
        begin = time.monotonic()
        ctx.nl_forward([shot])
        assert ctx.resident_info()[1] == given_up
        _check(rec, ref, np.float32)
        ctx.nl_forward([shot])
        if time.monotonic() < begin + 0.25:
            assert ctx.resident_info()[1] == given_up
        _check(rec, ref, np.float32)
        time.sleep(0.25 + 32 * (time.monotonic() - begin))
    ctx.close()


def _passes(ctx, mid, g, dtype):
    """One call of each entry point on one shot: which of them ran resident."""
    rng = np.random.default_rng(52)
    spos, rpos = _positions(rng, g, 5), _positions(rng, g, 5)
    nt = {"src": np.ones((1, g.nts), dtype), "fine": np.ones((1, (g.nts - 1) * g.sub + 1), dtype)}

    def traces(pos, key):
        return [np.repeat(nt[key], pos[GRID_OF_COMP[k]].size, 0) for k in range(5)]

    src, fine, dat = traces(spos, "src"), traces(spos, "fine"), traces(rpos, "src")
    dm = np.ones((5, g.nx, g.nz), dtype)

    def gradient(s):
        h = ctx.fwi_forward(s(src), g.nts - 1)
        ctx.fwi_gradient(h, s(src), dm)
        ctx.fwi_release(h)

    calls = {"nl_forward": lambda s: ctx.nl_forward(s(src)), "nl_adjoint": lambda s: ctx.nl_adjoint(s(src))}
    if not g.surface:
        calls.update(born_forward=lambda s: ctx.born_forward(s(fine), dm), born_adjoint=lambda s: ctx.born_adjoint(s(fine), dm),
                     fwi=gradient)
    out, keep = {}, []

    def shot(tr):
        sh, k = ctx.make_shot(mid, spos, rpos, tr, dat)
        keep.append(k)
        return [sh]

    for name, call in calls.items():
        before = ctx.resident_info()[0]
        call(shot)
        out[name] = ctx.resident_info()[0] > before
    return out


@pytest.mark.parametrize("dtype,sub,surface", [(np.float32, 2, 1), (np.float32, 3, 0), (np.float64, 2, 0), (np.float64, 2, 1),
                                               (np.float32, 2, 0)])
def test_explicit_variant_keeps_launched_steps(dtype, sub, surface):
    """A one-step variant that the caller sets is run where a pass would be launched one step at a time;
    FP32 passes that take two steps a launch have variants of their own, which stay automatic here."""
    ctx = _ctx(dtype)
    nts = 102 if sub == 3 else 201           # 303 fine steps are an odd count for the NL adjoint
    mid, g, med = _model(ctx, 300, 700, nts, sub, 51, surface=surface)
    auto = _passes(ctx, mid, g, dtype)
    assert auto["nl_forward"] and (surface or all(auto.values())), auto
    ctx.set_variant(3)
    fixed = _passes(ctx, mid, g, dtype)
    if dtype == np.float32 and sub == 2 and not surface:
        assert fixed == auto
    elif dtype == np.float32 and sub == 3:
        assert fixed == {k: k == "nl_forward" for k in fixed}, fixed
    else:
        assert not any(fixed.values()), fixed
    ctx.set_variant(_capi.VARIANT_AUTO)
    assert _passes(ctx, mid, g, dtype) == auto
    ctx.close()


@pytest.mark.parametrize("dtype,nz,nx", [(np.float32, 300, 500), (np.float64, 300, 500)])
def test_born_ring_on_a_full_card(shimmed, dtype, nz, nx):
    """The ring of the Born passes: the same bits whatever memory is free, kept where there is plenty, given back
    at the call's end where there is little and when another allocation needs it, and done without (launched
    passes) where there is none."""
    shim, capi = shimmed
    nts, sub = 70, 4
    size = np.dtype(dtype).itemsize
    ring = 33 * 5 * nz * nx * size
    rng = np.random.default_rng(61)
    grads, data, fit, ref = [], [], [], None
    # what is left when the call has all but the ring: plenty, half a ring more than it, half a ring
    for spare in (100.0, 1.5, 0.5):
        shim.shim_capacity(2 ** 64 - 1)
        ctx = _shim_ctx(capi, dtype)
        mid, g, med = _model(ctx, nz, nx, nts, sub, 62)
        if ref is None:
            spos, rpos = _positions(rng, g, 10), _positions(rng, g, 80)
            src = [O.time_interp(s, g.dts, sub) for s in random_traces(rng, spos, nts, np.float64)]
            dat = random_traces(rng, rpos, nts, np.float64)
            dmod = np.zeros((5, nx, nz))
            dmod[:, 4:-4, 4:-4] = rng.standard_normal((5, nx - 8, nz - 8)) * np.abs(med).reshape(5, -1).max(1)[:, None, None]
            ref = (O.born_adj_reg(g, med, spos, src, rpos, dat, np.float64), O.born_fwd_reg(g, med, spos, src, dmod, rpos, np.float64))
        srcd, datd, dmd = ([np.ascontiguousarray(t, dtype) for t in src], [np.ascontiguousarray(t, dtype) for t in dat],
                           np.ascontiguousarray(dmod, dtype))

        def call():
            dm = np.zeros((5, nx, nz), dtype)
            sh, keep = ctx.make_shot(mid, spos, rpos, srcd, datd)
            ctx.born_adjoint([sh], dm)
            rec = [np.zeros_like(t) for t in datd]
            sh, keep = ctx.make_shot(mid, spos, rpos, srcd, rec)
            ctx.born_forward([sh], dmd)
            assert rel_l2(dm, ref[0]) < GRAD_TOL[dtype]
            _check(rec, ref[1], dtype)
            return dm, rec

        call()
        fit.append(shim.shim_live() - ring)      # every buffer of the two calls but the ring
        if spare < 100:
            ctx.release_workspace()
            shim.shim_capacity(int(fit[-1] + spare * ring))
        before = ctx.resident_info()[0]
        for _ in range(2):
            dm, rec = call()
            grads.append(dm)
            data.append(rec)
        launches = ctx.resident_info()[0] - before
        if spare > 1:
            # source pass and three launches of 32 intervals each, twice the pair of calls
            assert launches == 2 * 2 * 4, launches
            assert np.array_equal(grads[0], dm) and all(np.array_equal(a, b) for a, b in zip(data[0], rec))
        else:
            assert launches == 2 * 2, launches    # the source passes only
            assert shim.shim_live() <= fit[-1]
        if spare > 1:
            assert shim.shim_live() == fit[-1] + (ring if spare > 3 else 0)
        if spare == 100.0:     # a model whose media (33 x 5 fields of the grid) only the ring's memory can hold
            shim.shim_capacity(fit[-1] + ring + ring // 4)
            _model(ctx, nz, 33 * nx, nts, sub, 63)
            assert fit[-1] + ring <= shim.shim_live() < fit[-1] + ring + 4096
        ctx.close()
        assert shim.shim_live() == 0


@pytest.mark.parametrize("dtype,nz,nx", [(np.float32, 300, 700), (np.float64, 300, 500)])
def test_refused_in_the_middle_of_a_pass(shimmed, dtype, nz, nx):
    """A refusal after some launches of a scattered or receiver pass or of a checkpointed gradient: what they left
    in the outputs, the ring and the record is made again, launched."""
    shim, capi = shimmed
    nts, sub, segment = 70, 3, 23
    rng = np.random.default_rng(82)
    g = None

    def context():
        ctx = _shim_ctx(capi, dtype)
        return (ctx,) + _model(ctx, nz, nx, nts, sub, 81)

    ctx, mid, g, med = context()
    ctx.close()
    spos, rpos = _positions(rng, g, 10), _positions(rng, g, 80)
    src = random_traces(rng, spos, nts, np.float64)
    fine = [O.time_interp(s, g.dts, sub) for s in src]
    dat = random_traces(rng, rpos, nts, np.float64)
    dmod = np.zeros((5, nx, nz))
    dmod[:, 4:-4, 4:-4] = rng.standard_normal((5, nx - 8, nz - 8)) * np.abs(med).reshape(5, -1).max(1)[:, None, None]
    ref_dm = O.born_adj_reg(g, med, spos, fine, rpos, dat, np.float64)
    ref_lin = O.born_fwd_reg(g, med, spos, fine, dmod, rpos, np.float64)
    srcd, fined, datd = ([np.ascontiguousarray(t, dtype) for t in tr] for tr in (src, fine, dat))

    def born_adjoint(ctx, mid, after):
        shim.shim_launches(ILLEGAL_STATE, 1, after)
        dm = np.zeros((5, nx, nz), dtype)
        shot, keep = ctx.make_shot(mid, spos, rpos, fined, datd)
        ctx.born_adjoint([shot], dm)
        assert rel_l2(dm, ref_dm) < GRAD_TOL[dtype], (after, rel_l2(dm, ref_dm))

    def born_forward(ctx, mid, after):
        shim.shim_launches(ILLEGAL_STATE, 1, after)
        rec = [np.full_like(t, 7) for t in datd]
        shot, keep = ctx.make_shot(mid, spos, rpos, fined, rec)
        ctx.born_forward([shot], np.ascontiguousarray(dmod, dtype))
        _check(rec, ref_lin, dtype)

    def fwi_gradient(ctx, mid, after):
        shot, keep = ctx.make_shot(mid, spos, rpos, srcd, [np.zeros_like(t) for t in datd])
        h = ctx.fwi_forward([shot], segment)
        assert ctx.resident_info()[0] == 3
        shim.shim_launches(ILLEGAL_STATE, 1, after)
        for _ in range(2):
            dm = np.zeros((5, nx, nz), dtype)
            shot, keep = ctx.make_shot(mid, spos, rpos, srcd, datd)
            ctx.fwi_gradient(h, [shot], dm)
            assert rel_l2(dm, ref_dm) < GRAD_TOL[dtype], (after, rel_l2(dm, ref_dm))
        ctx.fwi_release(h)

    for call in (born_adjoint, born_forward, fwi_gradient):
        for after in (0, 1, 2, 3):
            ctx, mid, _, _ = context()
            call(ctx, mid, after)
            assert ctx.resident_info()[1:] == (0, 1, ILLEGAL_STATE), (call, after)
            ctx.close()


def test_two_threads_run_resident():
    """Two contexts on two threads of one process at once, each on its own stream: both resident, their launches one
    after the other on the device, with the data of each alone."""
    def case(seed):
        ctx = _ctx(np.float32)
        mid, g, med = _model(ctx, 500, 480, 101, 2, seed)
        rng = np.random.default_rng(seed)
        return (ctx,) + _forward_case(ctx, mid, g, med, rng, np.float32, 10, 20)

    cases = [case(91), case(92)]
    alone = []
    for ctx, shot, keep, rec, ref in cases:
        ctx.nl_forward([shot])
        _check(rec, ref, np.float32)
        alone.append([r.copy() for r in rec])
    ready = threading.Barrier(2)

    def run(case):
        ctx, shot, keep, rec, ref = case
        ready.wait()
        for _ in range(20):
            ctx.nl_forward([shot])

    threads = [threading.Thread(target=run, args=(c,)) for c in cases]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for (ctx, shot, keep, rec, ref), first in zip(cases, alone):
        assert ctx.resident_info() == (21, 0, 0, 0)
        assert all(np.array_equal(a, b) for a, b in zip(rec, first))
        ctx.close()
