"""The work that users have this framework do, as cases to be timed.

  nl      the nonlinear shot operator of the drop-in layer (Elastic_iso_{float,double}_prop), forward or
          adjoint: host model vector in, host data vector out
  born    the Born shot operator of the same layer, forward or adjoint
  batch   eio_nl_forward through the C ABI on shots of uneven grids and lengths, traces resident on the GPU
  fwi     ElasticFwi: misfit and gradient of a shot batch, in shot groups with the whole coarse record
          (misfit_and_gradient) or through torch autograd with checkpoints

Sizes are those of a padded grid (sponge and FAT halo included).  Models are layered, sources are
Ricker wavelets at the surface, receivers lie on a line at the surface, as in the workloads of the
benchmark.  Every device sits on a node of the centre grid, so a component on a staggered grid is the mean of its
two or four nearest nodes.
"""
import math

import numpy as np
import torch

FAT = 4
SURF = 8            # free surface: its row
GRID_OF_COMP = (1, 2, 0, 0, 3)
FD = (1.196289062541883, -0.079752604188901, 0.009570312506634, -6.975446437140719e-04)
DX = 10.0
# (node offsets along x, along z) of the points a component averages
OFFSETS = (((0, 0), (1, 0)), ((0, 0), (0, 1)), ((0, 0),), ((0, 0),), ((0, 0), (0, 1), (1, 0), (1, 1)))


def listed():
    return [
        # one tiny shot: what a dot test or a first trial of a script runs; launch latency and host work
        dict(name="nl_small", kind="nl", real="float", adjoint=False, surface=0, nz=72, nx=88, nts=120, sub=1,
             nexp=1, nrec=30, pad=10),
        # the plain NL example: one shot of a 200 x 400 model with a 30-cell sponge
        dict(name="nl_single", kind="nl", real="float", adjoint=False, surface=0, nz=280, nx=472, nts=1000, sub=1,
             nexp=1, nrec=200, pad=30),
        # the adjoint of a shot line on the same grid
        dict(name="nl_adjoint", kind="nl", real="float", adjoint=True, surface=0, nz=280, nx=472, nts=500, sub=1,
             nexp=8, nrec=200, pad=30),
        # land acquisition: free surface instead of the top sponge
        dict(name="nl_free_surface", kind="nl", real="float", adjoint=False, surface=1, nz=328, nx=600, nts=400,
             sub=1, nexp=2, nrec=250, pad=30),
        # the double-precision operator (reference results, dot tests at full size)
        dict(name="nl_double", kind="nl", real="double", adjoint=False, surface=0, nz=280, nx=472, nts=400, sub=1,
             nexp=2, nrec=200, pad=30),
        # modelling of a survey: shots of uneven grids and trace lengths in one call
        dict(name="nl_batch", kind="batch", nz0=381, nz1=680, nx0=680, nx1=1880, nts0=250, nts1=400, sub=2, nexp=8,
             nrec=300, pad=40),
        # one shot of a large model
        dict(name="nl_large", kind="batch", nz0=1028, nz1=1028, nx0=3028, nx1=3028, nts0=200, nts1=200, sub=2,
             nexp=1, nrec=1500, pad=10),
        # linearised modelling of a shot line, and its adjoint (one migration, one gradient)
        dict(name="born_forward", kind="born", real="float", adjoint=False, nz=280, nx=472, nts=600, sub=1, nexp=8,
             nrec=200, pad=30),
        dict(name="born_adjoint", kind="born", real="float", adjoint=True, nz=280, nx=472, nts=600, sub=1, nexp=8,
             nrec=200, pad=30),
        dict(name="born_adjoint_double", kind="born", real="double", adjoint=True, nz=168, nx=248, nts=250, sub=1,
             nexp=2, nrec=100, pad=20),
        # the FWI gradient on a field-sized grid, in shot groups
        dict(name="fwi_gradient", kind="fwi", checkpoint=False, nz=600, nx=1592, nts=500, sub=2, nexp=2, nrec=700,
             pad=40),
        # the FWI gradient of any torch loss, with checkpoints, on a smaller grid
        dict(name="fwi_checkpointed", kind="fwi", checkpoint=True, nz=280, nx=472, nts=500, sub=1, nexp=4, nrec=200,
             pad=30),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: grids of the operators are 16 m + 8 cells along each axis (their block size),
    those of the C ABI anything."""
    kind = rng.choice(("nl", "nl", "nl", "born", "born", "batch", "fwi"))
    sub = rng.choice((1, 1, 2))
    pad = rng.choice((10, 20, 30, 40))
    if kind == "batch":
        nz, nx = rng.randint(150, 700), rng.randint(200, 1900)
        c = dict(kind=kind, nz0=nz, nz1=nz + rng.randint(0, 150), nx0=nx, nx1=nx + rng.randint(0, 400),
                 nts0=rng.randint(120, 300), nts1=rng.randint(300, 450), sub=sub, nexp=_log(rng, 1, 10),
                 nrec=rng.randint(20, 70), pad=pad)
    else:
        nz, nx = 16 * _log(rng, 5, 38) + 8, 16 * _log(rng, 6, 99) + 8
        pad = min(pad, nz // 4, nx // 4)
        c = dict(kind=kind, nz=nz, nx=nx, nts=rng.randint(100, 700), sub=sub, nexp=_log(rng, 1, 9),
                 nrec=rng.randint(8, (nx - 8 - 2 * pad) // 2), pad=pad)
        if kind == "nl":
            c.update(real=rng.choice(("float", "float", "double")), adjoint=rng.random() < 0.4,
                     surface=int(rng.random() < 0.25))
        elif kind == "born":
            c.update(real=rng.choice(("float", "float", "double")), adjoint=rng.random() < 0.5)
        else:
            c.update(checkpoint=rng.random() < 0.5)
    most = 3.0e9 if c.get("real") == "double" else 6.0e9   # cell-updates: the largest listed case has 7.6e9
    if c.get("real") == "double" and kind == "born":
        most = 1.0e9
    while work(c)["flops"] / FLOPS > most:
        if c["nexp"] > 1:
            c["nexp"] -= 1
        elif kind == "batch":
            c["nts0"] = max(2, c["nts0"] // 2)
            c["nts1"] = max(2, c["nts1"] // 2)
        else:
            c["nts"] //= 2
    return c


# ------------------------------------------------------------------ what a pass cannot do without
FLOPS = 117  # of one cell-update: eight 8-point derivatives, five updates with the sponge


def _batch_shapes(case):
    """(nz, nx, nts) of each shot of an uneven batch, spread over the case's ranges."""
    n = case["nexp"]
    out = []
    for e in range(n):
        f = (e * 0.381966) % 1.0 if n > 1 else 0.0
        g = (e * 0.618034 + 0.25) % 1.0 if n > 1 else 0.0
        out.append((int(case["nz0"] + f * (case["nz1"] - case["nz0"])), int(case["nx0"] + g * (case["nx1"] - case["nx0"])),
                    int(case["nts1"] - g * (case["nts1"] - case["nts0"]))))
    return out


def work(case):
    size = 8 if case.get("real") == "double" else 4
    sub = 2 * case["sub"]
    if case["kind"] == "batch":
        shapes = _batch_shapes(case)
        cells = sum((z - 8) * (x - 8) * (t - 1) * sub for z, x, t in shapes)
        io = sum(5 * z * x + (5 * case["nrec"] + 2) * t for z, x, t in shapes)
        return {"bytes": 4 * io, "flops": FLOPS * cells}
    n, nt, ns = case["nz"] * case["nx"], case["nts"], case["nexp"]
    steps = (nt - 1) * sub
    cells = ns * (case["nz"] - 8) * (case["nx"] - 8)
    traces = ns * 5 * (case["nrec"] + 1) * nt
    if case["kind"] == "nl":
        return {"bytes": size * (5 * n + traces), "flops": FLOPS * cells * steps}
    # Born: two passes and an imaging condition (45 flops a cell) each coarse sample; the gradient: the same
    return {"bytes": size * (8 * n + traces), "flops": cells * (2 * FLOPS * steps + 45 * nt)}


# ------------------------------------------------------------------ inputs, from the seed alone
def _rng(seed, *more):
    return np.random.default_rng([int(seed)] + [int(m) for m in more])


def _elastic(r, nz, nx, vmin=1700.0, vmax=3700.0):
    """(3, nx, nz) rho, lambda, mu of a layered model with a smooth lateral variation, float32."""
    nl = int(r.integers(5, 12))
    depth = np.sort(r.integers(1, nz, nl - 1))
    vp_l = np.sort(r.uniform(vmin, vmax, nl))[r.permutation(nl)]
    layer = np.searchsorted(depth, np.arange(nz), side="right")
    lat = 1.0 + 0.04 * np.sin(2.0 * np.pi * (np.arange(nx) / nx * r.uniform(0.5, 3.0) + r.uniform()))
    vp = np.clip(vp_l[layer][None, :] * lat[:, None], vmin, vmax)
    vs = vp / r.uniform(1.65, 2.1, nl)[layer][None, :]
    rho = 310.0 * vp ** 0.25
    return np.stack([rho, rho * (vp * vp - 2.0 * vs * vs), rho * vs * vs]).astype(np.float32)


def _ricker(nts, dts, f, t0):
    a = (np.pi * f) ** 2 * (np.arange(nts) * dts - t0) ** 2
    return (1.0 - 2.0 * a) * np.exp(-a)


def _wavelet(r, nts, dts):
    """Explosive source: the same Ricker on sxx and szz, (5, nts)."""
    m = np.zeros((5, nts), np.float32)
    f = r.uniform(9.0, 14.0)
    m[2] = m[3] = _ricker(nts, dts, f, 1.1 / f) * r.uniform(0.8, 1.2)
    return m


def _data(r, ns, nrec, nts, dts):
    """(ns, 5, nrec, nts) recorded events: hyperbolic arrivals, velocities scaled by an impedance."""
    t = np.arange(nts) * dts
    x = np.arange(nrec) / max(1, nrec - 1)
    out = np.zeros((ns, 5, nrec, nts), np.float32)
    for e in range(ns):
        for k in range(5):
            for _ in range(3):
                t0, dip, xs, f = r.uniform(0.1, 0.9) * nts * dts, r.uniform(0.1, 0.6), r.uniform(), r.uniform(8.0, 14.0)
                arr = np.sqrt(t0 ** 2 + (dip * (x - xs)) ** 2)
                a = (np.pi * f * (t[None, :] - arr[:, None])) ** 2
                out[e, k] += (r.uniform(0.3, 1.0) * (1.0 - 2.0 * a) * np.exp(-a)).astype(np.float32)
    out[:, :2] *= 2e-7
    return out


def _devices(case):
    """Node indices (iz, ix) of the sources (one a shot) and of the receivers."""
    pad, ns, nrec = case["pad"], case["nexp"], case["nrec"]
    inner = case["nx"] - 8 - 2 * pad
    top = FAT + (FAT if case.get("surface") else pad)
    sx = [FAT + pad + min(inner - 2, (2 * e + 1) * inner // (2 * ns)) for e in range(ns)]
    step = max(1, (inner - 2) // nrec)
    return top + 2, sx, top + 1, [FAT + pad + 1 + step * i for i in range(nrec)], step


def _inputs(case, seed):
    """Everything a pass reads, in numpy."""
    r = _rng(seed, 1)
    dts = 0.001
    if case["kind"] == "batch":
        shots = []
        for e, (nz, nx, nts) in enumerate(_batch_shapes(case)):
            q = _rng(seed, 2, e)
            pad, nrec = case["pad"], case["nrec"]
            inner = nx - 8 - 2 * pad
            step = max(1, (inner - 2) // nrec)
            src = (FAT + pad + inner // 2) * nz + FAT + pad + 2
            rec = np.array([(FAT + pad + 1 + step * i) * nz + FAT + pad + 1 for i in range(min(nrec, inner - 2))],
                           np.int32)
            shots.append(dict(nz=nz, nx=nx, nts=nts, elastic=_elastic(q, nz, nx), src=src, rec=rec,
                              wavelet=_wavelet(q, nts, dts)))
        return dict(shots=shots, dts=dts)
    nz, nx, nts = case["nz"], case["nx"], case["nts"]
    d = dict(dts=dts, elastic=_elastic(r, nz, nx), wavelet=_wavelet(r, nts, dts))
    if case["kind"] == "fwi" or case.get("adjoint"):
        d["data"] = _data(r, case["nexp"], case["nrec"], nts, dts)
        if case["kind"] == "fwi":
            d["data"] *= 1e-2     # the size of the modelled data
    if case["kind"] == "born" and not case["adjoint"]:
        # a smooth 5 % perturbation inside the sponge
        p = case["pad"] + FAT
        f = sum(r.normal() * np.outer(np.sin(2 * np.pi * (r.uniform(1, 25) * np.arange(nx) / nx + r.uniform())),
                                      np.sin(2 * np.pi * (r.uniform(1, 15) * np.arange(nz) / nz + r.uniform())))
                for _ in range(12))
        f[:p] = f[nx - p:] = 0.0
        f[:, :p] = f[:, nz - p:] = 0.0
        d["perturbation"] = (d["elastic"] * (0.05 * f / np.abs(f).max())[None]).astype(np.float32)
    return d


# ------------------------------------------------------------------ a user's program
def _operator(case, inp):
    from elastic_isotropic_operators_amd.sep import Hypercube, SepVector, genericIO
    if case["real"] == "double":
        from elastic_isotropic_operators_amd import Elastic_iso_double_prop as P
    else:
        from elastic_isotropic_operators_amd import Elastic_iso_float_prop as P
    storage = "dataDouble" if case["real"] == "double" else "dataFloat"
    nz, nx, nts, ns, pad = case["nz"], case["nx"], case["nts"], case["nexp"], case["pad"]
    zm = FAT if case.get("surface") else pad
    zs, sx, zr, rx, step = _devices(case)
    sp = sx[1] - sx[0] if ns > 1 else 1
    par = dict(nts=nts, dts=inp["dts"], sub=case["sub"], nz=nz, nx=nx, dz=DX, dx=DX, fMax=20.0, mod_par=0,
               zPadMinus=zm, zPadPlus=pad, xPadMinus=pad, xPadPlus=pad, nExp=ns, zSource=zs - zm - FAT + 1,
               xSource=sx[0] - pad - FAT + 1, spacingShots=sp, nReceiver=case["nrec"], depthReceiver=zr - zm - FAT + 1,
               oReceiver=rx[0] - pad - FAT + 1, dReceiver=step, iGpu=0, blockSize=16,
               surfaceCondition=case.get("surface", 0))
    par = genericIO.io(params=["%s=%s" % kv for kv in par.items()])
    axis, cube = Hypercube.axis, Hypercube.hypercube
    oz, ox = -(FAT + zm) * DX, -(FAT + pad) * DX
    elastic = SepVector.getSepVector(cube(axes=[axis(n=nz, o=oz, d=DX), axis(n=nx, o=ox, d=DX), axis(n=3)]),
                                     storage=storage)
    elastic.getNdArray()[...] = inp["elastic"]
    sc, sxg, sz, sxz, saxis = P.buildSourceGeometry(par, elastic)
    rc, rxg, rz, rxz, raxis = P.buildReceiversGeometry(par, elastic)
    t = axis(n=nts, o=0.0, d=inp["dts"])
    data = SepVector.getSepVector(cube(axes=[t, raxis, axis(n=5), saxis]), storage=storage)
    if "data" in inp:
        data.getNdArray()[...] = inp["data"]
    geometry = (sc, sxg, sz, sxz, rc, rxg, rz, rxz)
    if case["kind"] == "nl":
        model = SepVector.getSepVector(cube(axes=[t, axis(n=1), axis(n=5), axis(n=1)]), storage=storage)
        model.getNdArray()[0, :, 0, :] = inp["wavelet"]
        op = P.nonlinearPropElasticShotsGpu(model, data, elastic, par, *geometry)
    else:
        signal = SepVector.getSepVector(cube(axes=[t, axis(n=1), axis(n=5)]), storage=storage)
        signal.getNdArray()[:, 0, :] = inp["wavelet"]
        model = elastic.clone()
        if "perturbation" in inp:
            model.getNdArray()[...] = inp["perturbation"]
        op = P.BornElasticShotsGpu(model, data, elastic, par, [signal], *geometry)
    return dict(op=op, model=model, data=data, adjoint=case["adjoint"])


def _source_rows(case):
    """Shot spacing may leave the last shots off _devices' even spread: the operator's are evenly spaced."""
    zs, sx, zr, rx, step = _devices(case)
    sp = sx[1] - sx[0] if len(sx) > 1 else 1
    return zs, [sx[0] + e * sp for e in range(len(sx))], zr, rx


def prepare(case, seed):
    inp = _inputs(case, seed)
    if case["kind"] in ("nl", "born"):
        return _operator(case, inp)
    if case["kind"] == "batch":
        from elastic_isotropic_operators_amd import _capi
        ctx = _capi.Context(0, np.float32)
        ctx.set_time_block(2, _capi.VARIANT_AUTO)
        shots, keep, recs = [], [], []
        sub = 2 * case["sub"]
        empty = np.zeros(0, np.int32)
        for s in inp["shots"]:
            dtw = inp["dts"] / sub
            media = torch.from_numpy(_media(s["elastic"].astype(np.float64), dtw).astype(np.float32)).cuda()
            n = s["nz"] * s["nx"] * 4
            mid = ctx.model_add(s["nz"], s["nx"], s["nts"], sub, DX, DX, inp["dts"], case["pad"], None,
                                device_ptrs=[media.data_ptr() + k * n for k in range(5)])
            src = torch.from_numpy(s["wavelet"] * np.float32(2.0 * dtw / (DX * DX))).cuda()
            rec = torch.empty((5, s["rec"].size, s["nts"]), dtype=torch.float32, device="cuda")
            shot, k = ctx.make_shot(mid, [np.array([s["src"]], np.int32), empty, empty, empty], [s["rec"]] * 4,
                                    [0, 0, src[2].data_ptr(), src[3].data_ptr(), 0],
                                    [rec[c].data_ptr() for c in range(5)])
            shots.append(shot)
            recs.append(rec)
            keep.append((k, src))
        torch.cuda.synchronize()
        return dict(ctx=ctx, shots=shots, keep=keep, recs=recs)
    from elastic_isotropic_operators_amd.fwi import ElasticFwi
    zs, sx, zr, rx = _source_rows(case)
    pad = case["pad"]
    o = -(FAT + pad) * DX
    grid = dict(nz=case["nz"], nx=case["nx"], dz=DX, dx=DX, oz=o, ox=o, nts=case["nts"], dts=inp["dts"],
                sub=case["sub"], minPad=pad, alphaCos=0.99)
    eng = ElasticFwi(grid, np.full((len(sx), 1), o + zs * DX), np.array([[o + x * DX] for x in sx]),
                     inp["wavelet"][:, None, :], np.full(len(rx), o + zr * DX), np.array([o + x * DX for x in rx]),
                     segment=int(math.ceil(math.sqrt(case["nts"] - 1))) if case["checkpoint"] else 0)
    return dict(eng=eng, model=torch.from_numpy(inp["elastic"]).cuda(), d_obs=torch.from_numpy(inp["data"]).cuda(),
                checkpoint=case["checkpoint"])


def run(state):
    if "op" in state:
        if state["adjoint"]:
            state["op"].adjoint(False, state["model"], state["data"])
            return state["model"].getNdArray()
        state["op"].forward(False, state["model"], state["data"])
        return state["data"].getNdArray()
    if "ctx" in state:
        state["ctx"].nl_forward(state["shots"], device_ptrs=True)
        return state["recs"]
    if state["checkpoint"]:
        m = state["model"].clone().requires_grad_(True)
        phi = state["eng"].misfit(m, state["d_obs"])
        phi.backward()
        return [phi.detach(), m.grad]
    phi, grad = state["eng"].misfit_and_gradient(state["model"], state["d_obs"])
    return [phi, grad]


# ------------------------------------------------------------------ the same in 64 bits, from the equations
def _sadj(f, ax):
    """Mean with the previous node along ax (ends as the operators have them)."""
    n = f.shape[ax]
    f = np.moveaxis(f, ax, 0)
    o = np.empty_like(f)
    o[1:n - 1] = 0.5 * (f[1:n - 1] + f[:n - 2])
    o[0] = 0.5 * f[0]
    o[n - 1] = f[n - 1] + 0.5 * f[n - 2]
    return np.moveaxis(o, 0, ax)


def _sfwd(f, ax):
    """Its transpose as the operators have it: mean with the next node."""
    n = f.shape[ax]
    f = np.moveaxis(f, ax, 0)
    o = np.empty_like(f)
    o[:n - 1] = 0.5 * (f[:n - 1] + f[1:])
    o[n - 1] = f[n - 1]
    return np.moveaxis(o, 0, ax)


def _media(el, dtw):
    rho, lam, mu = el
    return np.stack([2 * dtw / _sadj(rho, 0), 2 * dtw / _sadj(rho, 1), 2 * dtw * (lam + 2 * mu), 2 * dtw * lam,
                     2 * dtw * _sadj(_sadj(mu, 0), 1)])


class _Exact:
    """Time loops of `ns` shots of one grid in float64 torch."""

    def __init__(self, el, nts, sub, dts, pad, ns, surface=0):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.nx, self.nz = el.shape[1:]
        self.ns, self.nts, self.sub, self.dts, self.surface = ns, nts, sub, dts, surface
        self.dtw = dts / sub
        self.nstep = (nts - 1) * sub
        self.media_np = _media(el.astype(np.float64), self.dtw)
        self.med = torch.from_numpy(self.media_np).to(self.dev)
        x, z = np.arange(self.nx)[:, None], np.arange(self.nz)[None, :]
        d = np.minimum(np.minimum(x - FAT, self.nx - 1 - FAT - x), self.nz - 1 - FAT - z)
        if not surface:
            d = np.minimum(d, z - FAT)
        t = 0.99 + 0.01 * np.cos(np.pi / max(pad, 1) * (pad - d))
        t = np.where((d < pad) & (d >= 0), t, 1.0)
        self.damp = torch.from_numpy(t).to(self.dev)
        self.c = [f / DX for f in FD]
        s = 1.0 / math.sqrt((self.nstep + 1) / nts)
        i = np.arange(sub + 1)
        self.fa, self.fb = (1.0 - i / sub) * s, i / sub * s
        self.iu = (slice(None), slice(FAT, self.nx - FAT), slice(FAT, self.nz - FAT))
        self.mi = [m[FAT:-FAT, FAT:-FAT] for m in self.med]
        self.di = self.damp[FAT:-FAT, FAT:-FAT]
        if surface:
            row = torch.arange(FAT, self.nz - FAT, device=self.dev)
            self.on, self.below = (row == SURF).double(), (row > SURF).double()

    def state(self):
        return torch.zeros((5, self.ns, self.nx, self.nz), dtype=torch.float64, device=self.dev)

    def der(self, q, ax, plus):
        """Staggered derivative along x (1) or z (2) on the update region."""
        q = q.narrow(3 - ax, FAT, q.shape[3 - ax] - 2 * FAT)
        n = q.shape[ax] - 2 * FAT
        out = None
        for k in range(4):
            hi, lo = (FAT + 1 + k, FAT - k) if plus else (FAT + k, FAT - 1 - k)
            t = q.narrow(ax, hi, n) - q.narrow(ax, lo, n)
            out = t.mul_(self.c[k]) if out is None else out.add_(t, alpha=self.c[k])
        return out

    def forward_terms(self, u):
        m = self.mi
        if self.surface:
            S = SURF
            u[3][..., S] = 0.0
            u[3][..., S - 4:S] = -u[3][..., S + 1:S + 5].flip(-1)
            u[4][..., S - 3:S + 1] = -u[4][..., S + 1:S + 5].flip(-1)
            u[0][..., S - 4:S] = 0.0
            u[1][..., S - 4:S + 1] = 0.0
        ax = m[0] * (self.der(u[2], 1, False) + self.der(u[4], 2, True))
        az = m[1] * (self.der(u[3], 2, False) + self.der(u[4], 1, True))
        vxx, vzz = self.der(u[0], 1, True), self.der(u[1], 2, True)
        a2, a3 = m[2] * vxx + m[3] * vzz, m[3] * vxx + m[2] * vzz
        a4 = m[4] * (self.der(u[0], 2, False) + self.der(u[1], 1, False))
        if self.surface:
            on, b = self.on, self.below
            ax = ax * (on + b)
            a2 = a2 * b + on * (m[2] - m[3] * m[3] / m[2]) * vxx
            az, a3, a4 = az * b, a3 * b, a4 * b
        return ax, az, a2, a3, a4

    def adjoint_terms(self, u):
        m = self.med
        s0, s1, s6 = m[0] * u[0], m[1] * u[1], m[4] * u[4]
        a, b = m[2] * u[2] + m[3] * u[3], m[3] * u[2] + m[2] * u[3]
        return (-(self.der(a, 1, False) + self.der(s6, 2, True)), -(self.der(b, 2, False) + self.der(s6, 1, True)),
                -self.der(s0, 1, True), -self.der(s1, 2, True), -(self.der(s0, 2, False) + self.der(s1, 1, False)))

    def points(self, rows):
        """Flat node indices (5 lists of (ns, points) tensors) of devices given as (iz, ix) per shot."""
        out = []
        for k in range(5):
            out.append([torch.tensor([[e * self.nx * self.nz + (ix + ox) * self.nz + iz + oz for iz, ix in rows[e]]
                                      for e in range(self.ns)], device=self.dev) for ox, oz in OFFSETS[k]])
        return out

    def loop(self, steps, terms, extra=None, inject=None, after=None):
        """new = d (d old + terms(cur) + extra) + d s, from rest, over the fine steps `steps`."""
        old, cur = self.state(), self.state()
        for k in steps:
            t = terms(cur)
            e = extra(k) if extra else None
            for f in range(5):
                v = self.di * old[f][self.iu] + t[f]
                if e is not None:
                    v = v + e[f]
                old[f][self.iu] = self.di * v
            if inject:
                inject(k, old)
            if after:
                after(k, old)
            old, cur = cur, old

    def injector(self, pts, weight, series):
        """Adds d * weight * series[f][step] (ns, devices) of each component at its points."""
        d = self.damp.reshape(-1).repeat(self.ns)

        def inject(k, u):
            for f in range(5):
                if series[f] is None:
                    continue
                s = series[f][k]
                for p in pts[f]:
                    w = weight(f, p) / len(pts[f])
                    u[f].view(-1).index_add_(0, p.reshape(-1), (d[p] * w * s).reshape(-1))
        return inject

    def recorder(self, pts, count):
        rec = torch.zeros((5, self.nstep, self.ns, count), dtype=torch.float64, device=self.dev)

        def record(k, u):
            for f in range(5):
                flat = u[f].view(-1)
                rec[f, k] = sum(flat[p] for p in pts[f]) / len(pts[f])
        return rec, record

    def fine(self, tr):
        """Coarse series (..., nts) -> value injected at forward step k, (nstep, ...)."""
        fa, fb = (torch.from_numpy(a[:self.sub]).to(self.dev) for a in (self.fa, self.fb))
        v = tr[..., :-1, None] * fa + tr[..., 1:, None] * fb
        return v.reshape(tr.shape[:-1] + (self.nstep,)).movedim(-1, 0)

    def coarse(self, rec):
        """Fine records (nstep, ...) at weights of it2 = 1..sub -> (..., nts)."""
        fa, fb = (torch.from_numpy(a[1:]).to(self.dev) for a in (self.fa, self.fb))
        v = rec.movedim(0, -1).reshape(rec.shape[1:] + (self.nts - 1, self.sub))
        out = torch.zeros(rec.shape[1:] + (self.nts,), dtype=torch.float64, device=self.dev)
        out[..., :-1] += (v * fa).sum(-1)
        out[..., 1:] += (v * fb).sum(-1)
        return out

    def source_weight(self, f, p):
        """rhoxDtw, rhozDtw at the nodes, or 2 dtw; all by the cell's area."""
        if f < 2:
            return self.med[f].reshape(-1)[p % (self.nx * self.nz)] / (DX * DX)
        return 2.0 * self.dtw / (DX * DX)

    def series(self, wavelet):
        w = torch.from_numpy(wavelet.astype(np.float64)).to(self.dev)
        return [self.fine(w[f])[:, None, None].expand(-1, self.ns, 1) if bool((w[f] != 0).any()) else None
                for f in range(5)]

    def modelled(self, src, wavelet, rec, keep=None, scaled=True):
        """Data (ns, 5, nrec, nts) of an explosive source."""
        sp, rp = self.points(src), self.points(rec)
        out, record = self.recorder(rp, len(rec[0]))
        weight = self.source_weight if scaled else (lambda f, p: 1.0)

        def after(k, u):
            record(k, u)
            if keep is not None:
                j, i = k // self.sub, k % self.sub + 1
                keep[:, j] += u[:2] * self.fa[i]
                keep[:, j + 1] += u[:2] * self.fb[i]
        self.loop(range(self.nstep), self.forward_terms, None, self.injector(sp, weight, self.series(wavelet)), after)
        return torch.stack([self.coarse(out[f]) for f in range(5)], dim=1)

    def adjoint_steps(self):
        """Reverse step k -> (coarse index, it2)."""
        return [(self.nts - 2 - k // self.sub, self.sub - 1 - k % self.sub) for k in range(self.nstep)]

    def data_series(self, data):
        """Injected values of the adjoint loop, per component (nstep, ns, nrec)."""
        d = torch.from_numpy(np.ascontiguousarray(data, np.float64)).to(self.dev) if isinstance(data, np.ndarray) else data
        return [torch.stack([d[:, f, :, j] * self.fa[i + 1] + d[:, f, :, j + 1] * self.fb[i + 1]
                             for j, i in self.adjoint_steps()]) for f in range(5)]

    def wavefield(self):
        return torch.zeros((2, self.nts, self.ns, self.nx, self.nz), dtype=torch.float64, device=self.dev)

    def strain(self, W, j):
        u = W[:, j]
        return (self.der(u[0], 1, True), self.der(u[1], 2, True),
                self.der(u[0], 2, False) + self.der(u[1], 1, False))

    def rate(self, W, j):
        lo = W[:, j - 1][(slice(None),) + self.iu] if j > 0 else 0.0
        hi = W[:, j + 1][(slice(None),) + self.iu] if j < self.nts - 1 else 0.0
        return (lo - hi) / (2.0 * self.dts)

    def born_forward(self, src, wavelet, rec, pert):
        W = self.wavefield()
        self.modelled(src, wavelet, rec, keep=W)
        p = pert.astype(np.float64)
        dm = np.stack([_sadj(p[0], 0) * self.media_np[0], _sadj(p[0], 1) * self.media_np[1], 2 * self.dtw * p[1],
                       2 * self.dtw * p[2], 2 * self.dtw * _sadj(_sadj(p[2], 0), 1)])
        dm = [torch.from_numpy(a[FAT:-FAT, FAT:-FAT].copy()).to(self.dev) for a in dm]
        slot = {}

        def secondary(j):
            if j not in slot:
                xx, zz, xz = self.strain(W, j)
                t = self.rate(W, j)
                dl = dm[2] * (xx + zz)
                slot.pop(j - 2, None)
                slot[j] = (dm[0] * t[0], dm[1] * t[1], dl + 2 * dm[3] * xx, dl + 2 * dm[3] * zz, dm[4] * xz)
            return slot[j]

        def extra(k):
            j, i = k // self.sub, k % self.sub
            return [a * self.fa[i] + b * self.fb[i] for a, b in zip(secondary(j), secondary(j + 1))]
        out, record = self.recorder(self.points(rec), len(rec[0]))
        self.loop(range(self.nstep), self.forward_terms, extra, None, record)
        return torch.stack([self.coarse(out[f]) for f in range(5)], dim=1)

    def image(self, W, rec, data):
        """Imaging condition of the adjoint wavefield of `data`, stacked over shots: (drho, dlambda, dmu)."""
        acc = torch.zeros((5, self.nx - 8, self.nz - 8), dtype=torch.float64, device=self.dev)
        slot = {j: self.state() for j in (self.nts - 1, self.nts - 2)}
        where = self.adjoint_steps()

        def use(j):
            s = slot.pop(j)
            a = [s[f][self.iu] for f in range(5)]
            xx, zz, xz = self.strain(W, j)
            t = self.rate(W, j)
            acc[0] += (a[0] * t[0]).sum(0)
            acc[1] += (a[1] * t[1]).sum(0)
            acc[2] += ((a[2] + a[3]) * (xx + zz)).sum(0)
            acc[3] += 2.0 * (xx * a[2] + zz * a[3]).sum(0)
            acc[4] += (a[4] * xz).sum(0)

        def after(k, u):
            j, i = where[k]
            if j not in slot:
                use(j + 2)
                slot[j] = self.state()
            slot[j].add_(u, alpha=float(self.fa[i]))
            slot[j + 1].add_(u, alpha=float(self.fb[i]))
        self.loop(range(self.nstep), self.adjoint_terms, None,
                  self.injector(self.points(rec), lambda f, p: 1.0, self.data_series(data)), after)
        use(1)
        use(0)
        a = np.zeros((5, self.nx, self.nz))
        a[:, FAT:-FAT, FAT:-FAT] = acc.cpu().numpy()
        a[0] *= self.media_np[0]
        a[1] *= self.media_np[1]
        a[2:] *= 2.0 * self.dtw
        return np.stack([_sfwd(a[0], 0) + _sfwd(a[1], 1), a[2], a[3] + _sfwd(_sfwd(a[4], 1), 0)])

    def nl_adjoint(self, src, rec, data):
        sp = self.points(src)
        out = torch.zeros((5, self.nts), dtype=torch.float64, device=self.dev)
        where = self.adjoint_steps()
        fine = torch.zeros((5, self.nstep), dtype=torch.float64, device=self.dev)

        def after(k, u):
            for f in range(5):
                flat = u[f].view(-1)
                fine[f, k] = sum((flat[p] * self.source_weight(f, p)).sum() for p in sp[f]) / len(sp[f])
        self.loop(range(self.nstep), self.adjoint_terms if not self.surface else None, None,
                  self.injector(self.points(rec), lambda f, p: 1.0, self.data_series(data)), after)
        v = fine.reshape(5, self.nts - 1, self.sub)
        j = torch.tensor([w[0] for w in where[::self.sub]], device=self.dev)
        i = [w[1] for w in where[:self.sub]]
        out.index_add_(1, j, (v * torch.from_numpy(self.fa[i]).to(self.dev)).sum(-1))
        out.index_add_(1, j + 1, (v * torch.from_numpy(self.fb[i]).to(self.dev)).sum(-1))
        return out


def exact(case, seed):
    # the adjoint with a free surface is the transpose of the forward, which these equations do not spell out;
    # of the rest, what 64 bits would take more than about 20 seconds for has no value either
    if case.get("surface") and case.get("adjoint"):
        return None
    steps = sum(t * 2 * case["sub"] for _, _, t in _batch_shapes(case)) if case["kind"] == "batch" else \
        2 * case["nts"] * case["sub"] * (3 if case["kind"] != "nl" else 1)
    if steps * 0.9e-3 + work(case)["flops"] / FLOPS * 0.9e-9 > 18.0:
        return None
    if case["kind"] not in ("nl", "batch") and case["nexp"] * case["nz"] * case["nx"] * case["nts"] * 16 > 60e9:
        return None
    inp = _inputs(case, seed)
    sub = 2 * case["sub"]
    if case["kind"] == "batch":
        out = []
        for s in inp["shots"]:
            x = _Exact(s["elastic"], s["nts"], sub, inp["dts"], case["pad"], 1)
            ent = [[(int(p) % s["nz"], int(p) // s["nz"]) for p in s["rec"]]]
            pts = x.points(ent)
            pts = [[p[0]] for p in pts]
            rec, record = x.recorder(pts, len(ent[0]))
            sp = [[p[0]] for p in x.points([[(s["src"] % s["nz"], s["src"] // s["nz"])]])]
            inj = x.injector(sp, lambda f, p: 2.0 * x.dtw / (DX * DX), x.series(s["wavelet"]))
            x.loop(range(x.nstep), x.forward_terms, None, inj, record)
            out.append(torch.stack([x.coarse(rec[f])[0] for f in range(5)]))
        return out
    zs, sx, zr, rx = _source_rows(case)
    ns = case["nexp"]
    src = [[(zs, x)] for x in sx]
    rec = [[(zr, x) for x in rx]] * ns
    x = _Exact(inp["elastic"], case["nts"], sub, inp["dts"], case["pad"], ns, case.get("surface", 0))
    if case["kind"] == "nl":
        if case["adjoint"]:
            return x.nl_adjoint(src, rec, inp["data"]).cpu().numpy()[None, :, None, :]
        return x.modelled(src, inp["wavelet"], rec).cpu().numpy()
    if case["kind"] == "born" and not case["adjoint"]:
        return x.born_forward(src, inp["wavelet"], rec, inp["perturbation"]).cpu().numpy()
    W = x.wavefield()
    data = x.modelled(src, inp["wavelet"], rec, keep=W)
    if case["kind"] == "born":
        return x.image(W, rec, inp["data"])
    res = data - torch.from_numpy(inp["data"].astype(np.float64)).to(x.dev)
    phi = 0.5 * float((res * res).sum())
    grad = torch.from_numpy(x.image(W, rec, res))
    # in the order and types of run(): the autograd path returns a tensor for the misfit
    return [torch.tensor(phi, dtype=torch.float64) if case["checkpoint"] else phi, grad]
