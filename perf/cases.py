"""The measured cases of the em2d library: whole steps, its stage entry
points, batches, the learned current filter and its training, and the
diagnostics, each through the entry points a program calls.

A step's kernels go on the library's own stream; fields come back as views
of the library's device buffers.  A species' particles stay on the device
during a run, and with the default (order-free) sort their order inside a
tile is not part of what the sort promises, so a step's cases return the
fields, which every particle's push, move, deposit and place in the sort
enter; the stage case uses the reference order, which is promised, and
returns every particle array as well.

`exact` states the same step in 64 bits on global periodic grids: linear
interpolation of the staggered fields, the Boris rotation, the
charge-conserving deposit of paths split at cell edges, the filter and the
leapfrog field update.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PACKAGE = os.path.join(ROOT, "zpic-parallel_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

import pyzpic as zp  # noqa: E402

DT = float(np.float32(0.07))
DX = 0.1
UTH, UZ = 0.1, 0.6
GL, GU = 1, 2  # guard cells of the field grids
NPARAM = 8835


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the high-ppc box that runs beside a production run with the learned
        # filter, every step of it: few, small tiles, many particles in each
        dict(name="shadow64", kind="step", ntx=8, nty=8, nx=8, ny=8, px=16, py=16, filter="none", order=1),
        # the reference's own Weibel problem
        dict(name="weibel128", kind="step", ntx=8, nty=8, nx=16, ny=16, px=8, py=8, filter="none", order=1),
        # a wide box of few particles per cell, strongly filtered, in tiles
        # that are not square: the grid's share of the step is large
        dict(name="weibel1056x720", kind="step", ntx=33, nty=45, nx=32, ny=16, px=2, py=2, filter="compensated",
             order=4),
        # the production size: 537 million particles
        dict(name="weibel2048", kind="load", ntx=128, nty=128, nx=16, ny=16, px=8, py=8, filter="binomial", order=1),
        # laser wakefield, window moving through plasma: five steps, in four
        # of which the window moves
        dict(name="lwfa4096x512", kind="lwfa", ntx=256, nty=32, nx=16, ny=16, px=4, py=2),
        # a parameter scan: uneven instances, one launch per stage, or one
        # persistent launch per step, replayed from a graph
        dict(name="scan12", kind="batch", n=12, scan=4, persistent=False),
        dict(name="scan12_persistent", kind="batch", n=12, scan=4, persistent=True),
        # a program with its own device buffers: the stages one by one, the
        # reference's particle order, ragged tiles, a filter along y
        dict(name="stages_ragged", kind="stages", ntx=19, nty=23, nx=24, ny=10, px=5, py=3, order=2),
        # the production run of the learned current filter
        dict(name="learned512", kind="learned", ntx=32, nty=32, nx=16, ny=16, px=2, py=2),
        # training that filter: Adam steps on stored pairs
        dict(name="train512", kind="train", H=512, W=512, pairs=6, steps=8),
        # what a run reports every few steps
        dict(name="report768", kind="report", ntx=48, nty=48, nx=16, ny=16, px=4, py=4, bx=128, bu=96),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "lwfa", "batch", "stages", "learned", "train", "report"])
    if kind == "lwfa":
        return dict(kind=kind, ntx=_log_int(rng, 24, 256), nty=_log_int(rng, 4, 32), nx=16, ny=16,
                    px=rng.randint(1, 4), py=rng.randint(1, 3))
    if kind == "batch":
        while True:
            c = dict(kind=kind, n=rng.randint(2, 12), scan=rng.randint(5, 10 ** 6), persistent=rng.random() < 0.5)
            if sum(_cells(i) * i["px"] * i["py"] for i in _instances(c)) < 25_000_000:
                return c
    if kind == "train":
        return dict(kind=kind, H=_log_int(rng, 48, 640), W=32 * _log_int(rng, 2, 20), pairs=rng.randint(1, 6),
                    steps=rng.randint(2, 10))
    if kind == "learned":
        t = rng.choice([8, 16, 32])
        return dict(kind=kind, ntx=32 // t * _log_int(rng, 3, 24), nty=_log_int(rng, 64, 768) // t + 1, nx=t, ny=t,
                    px=rng.randint(1, 3), py=rng.randint(1, 3))
    nx, ny = rng.randint(8, 32), rng.randint(8, 32)
    ntx, nty = max(1, _log_int(rng, 48, 1024) // nx), max(1, _log_int(rng, 48, 1024) // ny)
    px, py = rng.randint(1, 12), rng.randint(1, 12)
    cells = ntx * nx * nty * ny
    while cells * px * py > 12_000_000:
        px, py = max(1, px - 1), max(1, py - 1)
    c = dict(kind=kind, ntx=ntx, nty=nty, nx=nx, ny=ny, px=px, py=py)
    if kind == "step":
        c["filter"], c["order"] = rng.choice(["none", "binomial", "compensated"]), rng.randint(1, 4)
    elif kind == "stages":
        c["order"] = rng.randint(1, 3)
    else:
        # the reference's field energy sums ny x ny cells of a tile
        c["nx"], c["ntx"] = ny, max(1, cells // (ny * ny * nty))
        c["bx"], c["bu"] = rng.randint(16, 256), rng.randint(16, 256)
    return c


# ----------------------------------------------------------------- the inputs
def _gen(seed, k=0):
    return torch.Generator(device="cuda").manual_seed(1000003 * (int(seed) % (1 << 40)) + k)


def _plasma(c, seed, k, uz, uth=UTH):
    """Species k as it is in the middle of a run: particles anywhere in the
    box, thermal with a drift, in no order inside their tiles (tile by tile;
    counts per tile, cells inside the tile, positions, momenta)."""
    g = _gen(seed, 10 + k)
    n = c["ntx"] * c["nx"] * c["nty"] * c["ny"] * c["px"] * c["py"]
    tiles = c["ntx"] * c["nty"]
    tile = torch.sort(torch.randint(tiles, (n,), generator=g, device="cuda", dtype=torch.int32)).values
    count = torch.bincount(tile, minlength=tiles).int()
    ix = torch.stack([torch.randint(c["nx"], (n,), generator=g, device="cuda", dtype=torch.int32),
                      torch.randint(c["ny"], (n,), generator=g, device="cuda", dtype=torch.int32)], 1)
    x = torch.rand(n, 2, generator=g, device="cuda") - 0.5
    u = torch.randn(n, 3, generator=g, device="cuda") * uth
    u[:, 2] += uz
    return count, ix, x, u


def _waves(c, seed, k, amp):
    """A global (rows, columns, 3) field of a few long waves."""
    rng = np.random.RandomState((int(seed) * 7 + k) % (1 << 32))
    H, W = c["nty"] * c["ny"], c["ntx"] * c["nx"]
    y = torch.arange(H, device="cuda", dtype=torch.float64)[:, None] / H
    x = torch.arange(W, device="cuda", dtype=torch.float64)[None, :] / W
    f = torch.zeros(H, W, 3, device="cuda", dtype=torch.float64)
    for j in range(3):
        for _ in range(4):
            kx, ky = rng.randint(-6, 7, 2)
            f[..., j] += amp * rng.uniform(0.3, 1) * torch.sin(2 * math.pi * (kx * x + ky * y + rng.uniform()))
    return f.float()


def _tile_index(c, gl=GL, gu=GU):
    """Global row and column of every element of the tile-major grid, and the
    padded elements per tile."""
    ex, ey = gl + c["nx"] + gu, gl + c["ny"] + gu
    H, W = c["nty"] * c["ny"], c["ntx"] * c["nx"]
    rows = (torch.arange(c["nty"])[:, None] * c["ny"] + torch.arange(ey)[None, :] - gl) % H
    cols = (torch.arange(c["ntx"])[:, None] * c["nx"] + torch.arange(ex)[None, :] - gl) % W
    r = rows[:, None, :, None].expand(c["nty"], c["ntx"], ey, ex).reshape(-1, ey * ex)
    q = cols[None, :, None, :].expand(c["nty"], c["ntx"], ey, ex).reshape(-1, ey * ex)
    return r.cuda(), q.cuda(), (ex * ey + 3) & ~3


def _tiled(c, f):
    """The tile-major grid, guards included, of a global periodic field."""
    r, q, vol = _tile_index(c)
    out = torch.zeros(r.shape[0], vol, 3, device="cuda", dtype=f.dtype)
    out[:, :r.shape[1]] = f[r, q]
    return out.reshape(-1, 3)


def _instances(c):
    """The instances of a scan: grid, particles per cell."""
    rng = random.Random(c["scan"])
    got = []
    for _ in range(c["n"]):
        n, p = rng.choice([64, 128, 256, 512]), rng.choice([2, 4, 8])
        got.append(dict(ntx=n // 16, nty=n // 16, nx=16, ny=16, px=p, py=p, filter="none", order=1))
    return got


def _drifts(c, seed):
    rng = random.Random(int(seed))
    return [(rng.uniform(0.2, 0.9), rng.uniform(0.02, 0.2)) for _ in range(c["n"])]


def _box(c):
    return np.float32(c["ntx"] * c["nx"] * DX), np.float32(c["nty"] * c["ny"] * DX)


def _sim(c, seed, uz=UZ, uth=UTH):
    """A simulation of electrons and positrons in the middle of a run."""
    filt = (c["filter"], 0, c["order"]) if c.get("filter", "none") != "none" else None
    sim = zp.Simulation((c["ntx"], c["nty"]), (c["nx"], c["ny"]), _box(c), DT, filter=filt)
    for k, s in enumerate((-1.0, 1.0)):
        sim.add_species(zp.Species("species%d" % k, s, (c["px"], c["py"])))
        sim.species[k].set_particles(*(t.cpu().numpy() for t in _plasma(c, seed, k, -s * uz, uth)))
    for k, name in enumerate("EB"):
        sim.set_field(name, _tiled(c, _waves(c, seed, k, 0.05)).cpu().numpy())
    return sim


def _denoiser(c, seed=None, pairs=0):
    """The network of the weights that the package ships, or a new one."""
    H, W = (c["H"], c["W"]) if "H" in c else (c["nty"] * c["ny"], c["ntx"] * c["nx"])
    if seed is None:
        return zp.Denoiser.load(os.path.join(PACKAGE, "weights", "denoiser_weibel.npz"), H, W)
    return zp.Denoiser(H, W, pairs, params=_params(seed).astype(np.float32), scale=0.02)


def _params(seed):
    rng = np.random.RandomState((int(seed) + 3) % (1 << 32))
    p = np.zeros(NPARAM)
    for off, n, fan in ((0, 1200, 75), (1216, 6400, 400), (7632, 1200, 400)):
        p[off:off + n] = rng.normal(0, math.sqrt(2.0 / fan), n)
    return p.astype(np.float32)


def _pairs(c, seed):
    """Noisy and smooth currents."""
    t = dict(ntx=1, nty=1, nx=c["W"], ny=c["H"])
    got = []
    for k in range(c["pairs"]):
        tgt = _waves(t, seed, 100 + k, 0.02)
        noise = torch.randn(c["H"], c["W"], 3, generator=_gen(seed, 100 + k), device="cuda") * 0.02
        got.append((tgt + noise, tgt))
    return got


class _View:
    """A device buffer of the library as torch sees it."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(shape=(n, 3), typestr="<f4", data=(ptr, False), version=3)


def _fields(s, sim):
    """E, B and J of a simulation where they are now (the current has two
    buffers that change places)."""
    L, views = s["lib"], s["views"]
    out = {}
    for k, name in enumerate("EBJ"):
        ptr, periodic = ctypes.c_void_p(), (ctypes.c_int * 2)()
        if L.zpic_field_device(sim.h, k, ctypes.byref(ptr), ctypes.byref(sim.geom), periodic):
            raise RuntimeError(L.zpic_last_error().decode())
        if ptr.value not in views:
            views[ptr.value] = torch.as_tensor(_View(ptr.value, sim.ntiles * sim.geom.tile_vol), device="cuda")
        out[name] = views[ptr.value]
    return out


class _Particles(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("np", "offset", "ix", "x", "u")] + [("max_part", ctypes.c_uint32)]


class _Sort(ctypes.Structure):
    _fields_ = [(n, ctypes.c_void_p) for n in ("idx", "npt", "new_np", "seg", "tmp_np", "total", "nmove", "stage_ix",
                                               "stage_x", "stage_u")]


def _lib():
    L = zp.lib()
    p, i, f = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
    for name, args in (("zpic_field_device", [p, i, p, p, p]),
                       ("zpic_species_get_phasespace", [p, i, f, f, i, i, f, f, i, p]),
                       ("zpic_fill", [p, ctypes.c_size_t, f, p]),
                       ("zpic_push_move_deposit", [p] * 5 + [f] * 6 + [p, p, i, p]),
                       ("zpic_tile_sort", [p] * 3 + [i] * 6 + [p]),
                       ("zpic_current_advance", [p, p] + [i] * 5 + [p]),
                       ("zpic_yee", [p] * 4 + [f] * 3 + [i, i, p])):
        getattr(L, name).restype = i
        getattr(L, name).argtypes = args
    return L


def _stage_state(c, seed):
    """One species in buffers of the program's own, on a stream of its own."""
    L = _lib()
    g = zp.Geom()
    if L.zpic_geom_init(ctypes.byref(g), c["ntx"], c["nty"], c["nx"], c["ny"], GL, GU):
        raise RuntimeError(L.zpic_last_error().decode())
    count, ix, x, u = _plasma(c, seed, 0, UZ)
    n, tiles = ix.shape[0], count.shape[0]
    room = n + n // 5

    def full(t):
        out = torch.zeros(room, t.shape[1], dtype=t.dtype, device="cuda")
        out[:n] = t
        return out

    new = lambda *shape, d=torch.int32: torch.zeros(*shape, dtype=d, device="cuda")  # noqa: E731
    t = dict(np=count, offset=(torch.cumsum(count, 0) - count).int(), ix=full(ix), x=full(x), u=full(u))
    w = dict(np=new(tiles), offset=new(tiles), ix=new(room, 2), x=new(room, 2, d=torch.float32),
             u=new(room, 3, d=torch.float32))
    s = dict(idx=new(room), npt=new(9 * tiles), new_np=new(tiles), seg=new(16 * tiles), tmp_np=new(tiles),
             total=new(1), nmove=new(1, d=torch.int64))
    ptr = lambda d: {k: v.data_ptr() for k, v in d.items()}  # noqa: E731
    E, B = (_tiled(c, _waves(c, seed, k, 0.05)) for k in (0, 1))
    J = torch.zeros_like(E)
    return dict(kind="stages", lib=L, c=c, g=g, P=_Particles(**ptr(t), max_part=room),
                T=_Particles(**ptr(w), max_part=room), S=_Sort(**ptr(s)), n=n, t=t, w=w, s=s, E=E, B=B, J=J,
                energy=new(tiles, d=torch.float64), stream=torch.cuda.Stream())


def _lwfa(c, seed):
    """The window in the middle of the plasma, the pulse inside."""
    rng = random.Random(int(seed))
    W, H = c["ntx"] * c["nx"], c["nty"] * c["ny"]
    box = (np.float32(W * 0.05), np.float32(H * 0.2))
    sim = zp.Simulation((c["ntx"], c["nty"]), (c["nx"], c["ny"]), box, float(np.float32(0.04)),
                        filter=("compensated", 0, 4))
    dens = zp.Density.ramp("x", 0.01, 0.0, float(box[0]) * rng.uniform(0.1, 0.15))
    sim.add_species(zp.Species("electrons", -1.0, (c["px"], c["py"]), "cold", density=dens))
    sim.species[0].set_bc(("periodic", "periodic"), ("open", "open"))
    sim.set_emf_bc(("periodic", "periodic"), ("absorbing", "absorbing"))
    sim.set_current_bc(("periodic", "periodic"), ("none", "none"))
    front = float(box[0]) - 4.8
    pol = rng.uniform(0, 2 * math.pi)
    sim.add_laser(zp.Gaussian(start=front, fwhm=4.0, a0=rng.uniform(1.8, 2.2), omega0=10.0,
                              W0=min(8.0, float(box[1]) / 6), focus=front + 14.8, axis=float(box[1]) / 2,
                              cos_pol=math.cos(pol), sin_pol=math.sin(pol)))
    sim.set_moving_window()
    return sim


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind, c=case, lib=_lib(), views={})
    if kind == "step":
        s["sim"] = _sim(case, seed)
    elif kind == "load":
        s["sim"] = zp.weibel(ntiles=(case["ntx"], case["nty"]), nx=(case["nx"], case["ny"]),
                             ppc=(case["px"], case["py"]), box=_box(case), dt=DT, uth=(UTH,) * 3, ufl=(0.0, 0.0, UZ),
                             filter=(case["filter"], 0, case["order"]), seed=1 + int(seed) % 1000003)
    elif kind == "learned":
        s["sim"] = _sim(case, seed)
        s["sim"].set_learned_filter(_denoiser(case))
    elif kind == "lwfa":
        s["sim"] = _lwfa(case, seed)
    elif kind == "batch":
        s["sims"] = [_sim(c, int(seed) + 100 * k, uz, uth)
                     for k, (c, (uz, uth)) in enumerate(zip(_instances(case), _drifts(case, seed)))]
        s["batch"] = zp.Batch(s["sims"], graph=True, persistent=case["persistent"])
    elif kind == "stages":
        s = _stage_state(case, seed)
    elif kind == "train":
        s["net"] = _denoiser(case, seed, case["pairs"])
        tile = dict(ntx=case["W"] // 32, nty=1, nx=32, ny=case["H"])
        box = (np.float32(case["W"] * DX), np.float32(case["H"] * DX))
        with_j = [zp.Simulation((tile["ntx"], tile["nty"]), (tile["nx"], tile["ny"]), box, DT) for _ in range(2)]
        for pair in _pairs(case, seed):
            for sim, f in zip(with_j, pair):
                sim.set_field("J", _tiled(tile, f).cpu().numpy())
            with_j[0].add_pair_to(s["net"], with_j[1])
        for sim in with_j:
            sim.close()
        s["seed"] = int(seed) % 1000
    else:
        s["sim"] = _sim(case, seed)
        s["x_range"] = float(_box(case)[0])
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------- one pass
def _ok(s, rc):
    if rc:
        raise RuntimeError(s["lib"].zpic_last_error().decode())


def run(state):
    s, kind = state, state["kind"]
    if kind in ("step", "load", "learned"):
        s["sim"].advance()
        return _fields(s, s["sim"])
    if kind == "lwfa":
        s["sim"].advance(5)
        return _fields(s, s["sim"])
    if kind == "batch":
        s["batch"].advance()
        return [_fields(s, sim) for sim in s["sims"]]
    if kind == "train":
        losses = s["net"].train(s["c"]["steps"], lr=1e-3, seed=s["seed"])
        return {"losses": losses, "params": s["net"].params()}
    if kind == "stages":
        return _run_stages(s)
    return _run_report(s)


def _run_stages(s):
    c, L, g = s["c"], s["lib"], s["g"]
    st = s["stream"].cuda_stream
    q = -1.0 / (c["px"] * c["py"])
    E, B, J = (s[k].data_ptr() for k in "EBJ")
    P, T, S, G = (ctypes.byref(s[k]) for k in ("P", "T", "S", "g"))
    _ok(s, L.zpic_fill(J, s["J"].numel(), 0.0, st))
    _ok(s, L.zpic_push_move_deposit(P, G, E, B, J, -0.5 * DT, DT / DX, DT / DX, q, q * DX / DT, q * DX / DT,
                                    s["energy"].data_ptr(), S, 0, st))
    _ok(s, L.zpic_tile_sort(P, T, S, c["ntx"], c["nty"], c["nx"], c["ny"], 1, 1, st))
    _ok(s, L.zpic_current_advance(J, G, 1, 1, c["order"], 1, 1, st))
    _ok(s, L.zpic_yee(E, B, J, G, DT / DX, DT / DX, DT, 1, 1, st))
    t, n = s["t"], s["n"]
    return dict(np=t["np"], offset=t["offset"], ix=t["ix"][:n], x=t["x"][:n], u=t["u"][:n], energy=s["energy"],
                E=s["E"], B=s["B"], J=s["J"])


def _run_report(s):
    sim, c, L = s["sim"], s["c"], s["lib"]
    eE, eB = sim.emf_energy()
    out = dict(eE=eE, eB=eB)
    for k, sp in enumerate(sim.species):
        out["charge%d" % k] = sp.charge()
        x_ux = np.zeros((c["bu"], c["bx"]), np.float32)
        uz = np.zeros(c["bu"], np.float32)
        _ok(s, L.zpic_species_get_phasespace(sp.h, 0, 0.0, s["x_range"], c["bx"], 2, -0.6, 0.6, c["bu"],
                                             x_ux.ctypes.data))
        _ok(s, L.zpic_species_get_phasespace(sp.h, 4, -1.2, 1.2, c["bu"], 0, 0.0, 1.0, 0, uz.ctypes.data))
        out["x_ux%d" % k], out["uz%d" % k] = x_ux, uz
    return out


# ----------------------------------------------------------- what a pass needs
def _cells(c):
    return c["ntx"] * c["nx"] * c["nty"] * c["ny"]


def _step_work(c, species=2):
    """Particles read and written (28 bytes each way), E and B read and
    written, J written; about 220 operations per particle (interpolation,
    rotation, move, deposit) and 40 per cell, 15 more per filter pass."""
    n, cells = _cells(c) * c["px"] * c["py"] * species, _cells(c)
    passes = {"none": 0, "binomial": c.get("order", 1), "compensated": c.get("order", 1) + 1}[c.get("filter", "none")]
    return dict(bytes=56 * n + 60 * cells, flops=220 * n + (40 + 15 * passes) * cells)


def work(case):
    c, kind = case, case["kind"]
    if kind in ("step", "load"):
        return _step_work(c)
    if kind == "stages":
        return _step_work(dict(c, filter="binomial"), 1)
    if kind == "lwfa":
        w = _step_work(dict(c, filter="compensated", order=4), 1)
        return {k: 5 * v for k, v in w.items()}
    if kind == "batch":
        each = [_step_work(i) for i in _instances(c)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    macs = 25 * (3 * 16 + 16 * 16 + 16 * 3)  # one application of the network to a cell
    if kind == "learned":
        w = _step_work(c)
        return dict(bytes=w["bytes"], flops=w["flops"] + 2 * macs * _cells(c))
    if kind == "train":
        # forward, weight gradients, and input gradients of two layers
        cells = c["H"] * c["W"]
        return dict(bytes=c["steps"] * (24 * cells + 28 * NPARAM),
                    flops=c["steps"] * cells * 2 * (2 * macs + 25 * (16 * 16 + 16 * 3)))
    n = 2 * _cells(c) * c["px"] * c["py"]
    return dict(bytes=(16 + 20 + 12) * n + 24 * _cells(c) + 2 * 4 * (_cells(c) + c["bx"] * c["bu"] + c["bu"]),
                flops=60 * n + 12 * _cells(c))


# ------------------------------------------------------------------ in 64 bits
def _interpolate(E, B, gx, gy, x):
    H, W, _ = E.shape
    hx, hy = (x[:, 0] < 0).long(), (x[:, 1] < 0).long()
    # on the cell's corners, or half a cell off along an axis
    w = {0: (0.5 - x[:, 0], 0.5 + x[:, 0]), 1: ((1 - hx) - x[:, 0], hx + x[:, 0])}
    v = {0: (0.5 - x[:, 1], 0.5 + x[:, 1]), 1: ((1 - hy) - x[:, 1], hy + x[:, 1])}
    i, j = {0: gx, 1: gx - hx}, {0: gy, 1: gy - hy}

    def at(F, comp, a, b):
        f = F[..., comp]
        x0, x1, y0, y1 = i[a] % W, (i[a] + 1) % W, j[b] % H, (j[b] + 1) % H
        return (f[y0, x0] * w[a][0] + f[y0, x1] * w[a][1]) * v[b][0] + \
               (f[y1, x0] * w[a][0] + f[y1, x1] * w[a][1]) * v[b][1]

    e = torch.stack([at(E, 0, 1, 0), at(E, 1, 0, 1), at(E, 2, 0, 0)], 1)
    b = torch.stack([at(B, 0, 0, 1), at(B, 1, 1, 0), at(B, 2, 1, 1)], 1)
    return e, b


def _push(u, e, b, alpha):
    """Half an electric kick, the rotation, half a kick; and u^2 / (gamma + 1)
    in the middle."""
    u = u + alpha * e
    usq = (u * u).sum(1, keepdim=True)
    g = torch.sqrt(1 + usq)
    t = alpha / g * b
    u1 = u + torch.cross(u, t, dim=1)
    u2 = u + torch.cross(u1, 2 * t / (1 + (t * t).sum(1, keepdim=True)), dim=1)
    return u2 + alpha * e, (usq / (g + 1))[:, 0]


def _segment(J, gx, gy, a, b, qnx, qny, qvz):
    """The current of straight paths from a to b, each inside one cell."""
    H, W, _ = J.shape
    jx, jy = qnx * (b[:, 0] - a[:, 0]), qny * (b[:, 1] - a[:, 1])
    A = {0: 0.5 - a, 1: 0.5 + a}
    Z = {0: 0.5 - b, 1: 0.5 + b}

    def add(comp, dx, dy, v):
        J.view(-1).index_add_(0, (((gy + dy) % H) * W + (gx + dx) % W) * 3 + comp, v)

    for k in (0, 1):
        add(0, 0, k, jx * 0.5 * (A[k][:, 1] + Z[k][:, 1]))
        add(1, k, 0, jy * 0.5 * (A[k][:, 0] + Z[k][:, 0]))
        for m in (0, 1):
            ax, zx, ay, zy = A[m][:, 0], Z[m][:, 0], A[k][:, 1], Z[k][:, 1]
            add(2, m, k, qvz * (ax * ay + zx * zy + (ax * zy - zx * ay) / 2))


def _deposit(J, gx, gy, x0, x1, qnx, qny, qvz):
    """Paths that leave their cell along an axis are cut at its edge, along x
    first."""
    def cut(gx, gy, a, b, qvz, axis):
        out = (b[:, axis] >= 0.5).long() - (b[:, axis] < -0.5).long()
        whole, part = out == 0, out != 0
        yield gx[whole], gy[whole], a[whole], b[whole], qvz[whole]
        gx, gy, a, b, qvz, out = gx[part], gy[part], a[part], b[part], qvz[part], out[part]
        edge = 0.5 * out
        f = (edge - a[:, axis]) / (b[:, axis] - a[:, axis])
        mid = a + (b - a) * f[:, None]
        mid[:, axis] = edge
        yield gx, gy, a, mid, qvz * f
        start, end = mid.clone(), b.clone()
        start[:, axis] = -edge
        end[:, axis] -= out
        if axis == 0:
            yield gx + out, gy, start, end, qvz * (1 - f)
        else:
            yield gx, gy + out, start, end, qvz * (1 - f)

    def inside(gx, gy, a, b, qvz):
        # a piece that starts beyond an edge along y belongs to the next row
        over = (a[:, 1] >= 0.5).long() - (a[:, 1] < -0.5).long()
        a, b = a.clone(), b.clone()
        a[:, 1] -= over
        b[:, 1] -= over
        return gx, gy + over, a, b, qvz

    for p in cut(gx, gy, x0, x1, qvz, 0):
        for r in cut(*inside(*p), 1):
            _segment(J, *r[:4], qnx, qny, r[4])


def _pass3(J, axis, a, b, c):
    return torch.roll(J, 1, axis) * a + J * b + torch.roll(J, -1, axis) * c


def _filtered(J, name, order, axis=1):
    if name == "none":
        return J
    for _ in range(order):
        J = _pass3(J, axis, 0.25, 0.5, 0.25)
    if name == "compensated":
        b = (4.0 + 2.0 * order) / order
        J = _pass3(J, axis, -1 / (b - 2), b / (b - 2), -1 / (b - 2))
    return J


def _fields_step(E, B, J):
    d = DT / DX

    def half():
        B[..., 0] -= d / 2 * (torch.roll(E[..., 2], -1, 0) - E[..., 2])
        B[..., 1] += d / 2 * (torch.roll(E[..., 2], -1, 1) - E[..., 2])
        B[..., 2] += d / 2 * ((torch.roll(E[..., 0], -1, 0) - E[..., 0]) - (torch.roll(E[..., 1], -1, 1) - E[..., 1]))

    half()
    E[..., 0] += d * (B[..., 2] - torch.roll(B[..., 2], 1, 0)) - DT * J[..., 0]
    E[..., 1] += -d * (B[..., 2] - torch.roll(B[..., 2], 1, 1)) - DT * J[..., 1]
    E[..., 2] += d * ((B[..., 1] - torch.roll(B[..., 1], 1, 1)) - (B[..., 0] - torch.roll(B[..., 0], 1, 0))) - \
        DT * J[..., 2]
    half()


def _layers(p):
    out, o = [], 0
    for co, ci in ((16, 3), (16, 16), (3, 16)):
        w = p[o:o + co * ci * 25].reshape(co, ci, 25)
        o += co * ci * 25
        out.append((w, p[o:o + co]))
        o += co
    return out


def _network(p, x):
    """The network on a (rows, columns, 3) field, 5x5 taps, periodic."""
    layers = _layers(p)
    for k, (w, b) in enumerate(layers):
        z = b
        for t in range(25):
            z = z + torch.roll(x, (2 - t // 5, 2 - t % 5), (0, 1)) @ w[:, :, t].T
        x = torch.relu(z) if k < 2 else z
    return x


def _global_cells(c, count, ix):
    tile = torch.repeat_interleave(torch.arange(count.shape[0], device="cuda"), count.long())
    return tile, (tile % c["ntx"]) * c["nx"] + ix[:, 0], (tile // c["ntx"]) * c["ny"] + ix[:, 1]


def _step64(c, seed, species, axis=1, net=None):
    """E, B, J (tile-major) and the tiles' energy sums after one step;
    species: (charge sign, drift, thermal spread) each."""
    E, B = (_waves(c, seed, k, 0.05).double() for k in (0, 1))
    J = torch.zeros_like(E)
    energy = torch.zeros(c["ntx"] * c["nty"], dtype=torch.float64, device="cuda")
    for k, (sign, uz, uth) in enumerate(species):
        count, ix, x, u = _plasma(c, seed, k, uz, uth)
        tile, gx, gy = _global_cells(c, count, ix)
        q = sign / (c["px"] * c["py"])
        for at in torch.arange(x.shape[0], device="cuda").split(1 << 22):
            xx = x[at].double()
            e, b = _interpolate(E, B, gx[at], gy[at], xx)
            v, en = _push(u[at].double(), e, b, 0.5 * DT * sign)
            energy.index_add_(0, tile[at], en)
            rg = 1 / torch.sqrt(1 + (v * v).sum(1))
            x1 = xx + DT / DX * rg[:, None] * v[:, :2]
            _deposit(J, gx[at], gy[at], xx, x1, q * DX / DT, q * DX / DT, q * v[:, 2] * rg * 0.5)
    if net is not None:
        p, scale = net
        J = scale * _network(p, J / scale)
    else:
        J = _filtered(J, c.get("filter", "none"), c.get("order", 1), axis)
    _fields_step(E, B, J)
    return dict(E=_tiled(c, E), B=_tiled(c, B), J=_tiled(c, J)), energy


def _pair_of_species(uz=UZ, uth=UTH):
    return [(-1.0, uz, uth), (1.0, -uz, uth)]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("load", "lwfa"):
        return None
    if kind == "step":
        return _step64(c, seed, _pair_of_species())[0]
    if kind == "learned":
        d = np.load(os.path.join(PACKAGE, "weights", "denoiser_weibel.npz"), allow_pickle=False)
        net = torch.from_numpy(d["params"].astype(np.float64)).cuda(), float(d["scale"])
        return _step64(c, seed, _pair_of_species(), net=net)[0]
    if kind == "batch":
        return [_step64(i, int(seed) + 100 * k, _pair_of_species(uz, uth))[0]
                for k, (i, (uz, uth)) in enumerate(zip(_instances(c), _drifts(c, seed)))]
    if kind == "stages":
        f, energy = _step64(dict(c, filter="binomial"), seed, [(-1.0, UZ, UTH)], axis=0)
        return dict(np=None, offset=None, ix=None, x=None, u=None, energy=energy, **f)
    if kind == "train":
        return _train64(c, seed)
    return _report64(c, seed)


def _picks(n, steps, seed):
    """The pairs that the training's seed picks, step by step: words of the
    32-bit Mersenne twister scaled to [0, n) by the high word of word * n,
    drawn again where the low word falls in the uneven rest."""
    r = np.random.RandomState(seed)  # the same generator and seeding
    got = []
    while len(got) < steps:
        m = int.from_bytes(r.bytes(4), "little") * n
        if (m & 0xFFFFFFFF) >= (1 << 32) % n:
            got.append(m >> 32)
    return got


def _train64(c, seed):
    p = torch.from_numpy(_params(seed).astype(np.float64)).cuda().requires_grad_()
    scale = float(np.float32(0.02))
    pairs = [(a.double(), b.double()) for a, b in _pairs(c, seed)]
    opt = torch.optim.Adam([p], lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    losses = []
    for k in _picks(c["pairs"], c["steps"], int(seed) % 1000):
        opt.zero_grad()
        a, b = pairs[k]
        loss = ((scale * _network(p, a / scale) - b) ** 2).mean()
        loss.backward()
        opt.step()
        losses.append(float(loss))
    return {"losses": np.array(losses), "params": p.detach().cpu().numpy()}


def _report64(c, seed):
    E, B = (_waves(c, seed, k, 0.05).double() for k in (0, 1))
    out = dict(eE=(E * E).sum((0, 1)).cpu().numpy(), eB=(B * B).sum((0, 1)).cpu().numpy())
    for k, sign in enumerate((-1.0, 1.0)):
        count, ix, x, u = _plasma(c, seed, k, -sign * UZ)
        x, u = x.double(), u.double()
        _, gx, gy = _global_cells(c, count, ix)
        q = sign / (c["px"] * c["py"])
        out["charge%d" % k] = None  # a guard element keeps its tile's share alone
        norm = DX * DX * abs(q)

        def bins(v, lo, hi, n):
            s = (v - lo) * (n / (hi - lo)) - 0.5
            i = torch.trunc(s + 1).long() - 1
            return [(i, 1 - (s - i)), (i + 1, s - i)], n / (hi - lo)

        (xb, xn) = bins((gx + x[:, 0] + 0.5) * DX, 0.0, float(_box(c)[0]), c["bx"])
        (ub, un) = bins(u[:, 0], -0.6, 0.6, c["bu"])
        (zb, zn) = bins(u[:, 2], -1.2, 1.2, c["bu"])
        x_ux = torch.zeros(c["bu"] * c["bx"], dtype=torch.float64, device="cuda")
        for i, wi in xb:
            for j, wj in ub:
                # an axis' last bin stays empty
                m = (i >= 0) & (i < c["bx"] - 1) & (j >= 0) & (j < c["bu"] - 1)
                x_ux.index_add_(0, (j * c["bx"] + i)[m], (wi * wj)[m] * norm * xn * un)
        uz = torch.zeros(c["bu"], dtype=torch.float64, device="cuda")
        for i, wi in zb:
            m = (i >= 0) & (i < c["bu"] - 1)
            uz.index_add_(0, i[m], wi[m] * norm * zn)
        out["x_ux%d" % k] = x_ux.reshape(c["bu"], c["bx"]).cpu().numpy()
        out["uz%d" % k] = uz.cpu().numpy()
    return out

