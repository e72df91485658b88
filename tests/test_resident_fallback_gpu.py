"""Calls whose resident loops (csrc/eio_resident.h) give up a wait, are refused or run out of memory, or
that ask for launched steps: the launched kernels take over with the same answers.
Bars: those of the launched kernels, FP32 1e-5 and FP64 1e-11 relative L2 (gradients twice that and ten
times that, as sums over many products)."""
import numpy as np
import pytest

import oracle as O

from helpers import GRID_OF_COMP, random_traces, rel_l2
from test_resident_gpu import _check, _ctx, _model, _positions

pytestmark = pytest.mark.gpu

GRAD_TOL = {np.float32: 2e-5, np.float64: 1e-10}


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
    h = ctx.fwi_forward([shot], segment)
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
