"""The fast mode's diagnostic deposits against the deterministic mode's
(bit-exact with the reference): phase spaces whose bins a workgroup sums in
LDS or not, ranges that cut particles off, grouped tiles; charge; and the
field energy's sums in the reference's order."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def phasespace(zp, sp, q0, r0, n0, q1=0, r1=(0.0, 1.0), n1=0):
    L = zp.lib()
    f, i = ctypes.c_float, ctypes.c_int
    L.zpic_species_get_phasespace.restype = i
    L.zpic_species_get_phasespace.argtypes = [ctypes.c_void_p, i, f, f, i, i, f, f, i, ctypes.c_void_p]
    out = np.zeros((max(n1, 1), n0), np.float32)
    assert L.zpic_species_get_phasespace(sp.h, q0, r0[0], r0[1], n0, q1, r1[0], r1[1], n1, out.ctypes.data) == 0
    return out


@pytest.fixture(scope="module", params=[((3, 2), (16, 16), (3, 3)), ((70, 40), (4, 5), (2, 1)), ((1, 9), (23, 7), (4, 2))])
def pair(request):
    import pyzpic as zp
    ntiles, nx, ppc = request.param
    sims = [zp.weibel(ntiles=ntiles, nx=nx, ppc=ppc, deterministic=det) for det in (False, True)]
    sims[1].advance(4)
    for k, s in enumerate(sims[1].species):
        p = s.particles()
        sims[0].species[k].set_particles(*(p[n] for n in ("np", "ix", "x", "u")))
    for name in "EB":
        sims[0].set_field(name, sims[1].field(name))
    yield zp, sims
    for sim in sims:
        sim.close()


def close(a, b):
    # terms of at most the largest bin's size, each rounded to FP32 and summed
    # in another order: some thousand of them stay within 1e-5 of it
    assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()


@pytest.mark.parametrize("axes", [
    (0, (0.0, 1.0), 64),                              # x over part of the box
    (1, (0.1, 3.0), 7),
    (4, (-1.0, 1.2), 200),
    (2, (-0.05, 0.02), 9),                            # most particles outside
    (0, (-0.3, 40.0), 128, 2, (-0.4, 0.4), 96),
    (1, (0.0, 6.0), 50, 4, (-1.0, 1.0), 33),
    (0, (0.0, 8.0), 90, 1, (0.0, 8.0), 110),
    (2, (-0.3, 0.3), 128, 4, (-0.9, 0.9), 96),        # the most bins that fit
    (2, (-0.3, 0.3), 128, 4, (-0.9, 0.9), 97),        # more
    (2, (-0.3, 0.3), 91, 3, (-0.3, 0.3), 91),
    (2, (-0.3, 0.3), 3, 3, (-0.9, 0.9), 4),
])
def test_phasespace(pair, axes):
    zp, (fast, det) = pair
    for k in range(2):
        close(phasespace(zp, fast.species[k], *axes), phasespace(zp, det.species[k], *axes))


def test_charge(pair):
    zp, (fast, det) = pair
    for k in range(2):
        close(fast.species[k].charge(), det.species[k].charge())


def test_field_energy_order(pair):
    zp, (fast, det) = pair
    g = fast.geom
    if g.ny > g.nx:
        pytest.skip("the reference's loop leaves the tile's interior")
    for which, got in zip("EB", fast.emf_energy()):
        f = fast.field(which).reshape(fast.ntiles, g.tile_vol, 3)[:, :g.ext_x * g.ext_y]
        f = f.reshape(fast.ntiles, g.ext_y, g.ext_x, 3)[:, 1:1 + g.ny, 1:1 + g.ny]
        sq = (f * f).reshape(fast.ntiles, -1, 3).astype(np.float64)
        tiles = np.add.accumulate(sq, axis=1)[:, -1]
        assert np.array_equal(np.add.accumulate(tiles, axis=0)[-1], got)


@pytest.mark.parametrize("n", [64, 100, 127])
def test_charge_of_large_tiles(n):
    """Tiles up to the largest that the charge takes (128 KiB of LDS), larger
    than a particle pass's, through the stage entry point."""
    import pyzpic as zp
    import torch

    class Particles(ctypes.Structure):
        _fields_ = [(k, ctypes.c_void_p) for k in ("np", "offset", "ix", "x", "u")] + [("max_part", ctypes.c_uint32)]

    L = zp.lib()
    L.zpic_deposit_charge.restype = ctypes.c_int
    L.zpic_deposit_charge.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_float, ctypes.c_int, ctypes.c_void_p]
    g = zp.Geom()
    assert L.zpic_geom_init(ctypes.byref(g), 2, 1, n, n, 0, 1) == 0
    rng = np.random.default_rng(n)
    count = 6000
    t = dict(np=torch.tensor([count, count], dtype=torch.int32), offset=torch.tensor([0, count], dtype=torch.int32),
             ix=torch.from_numpy(rng.integers(0, n, (2 * count, 2)).astype(np.int32)),
             x=torch.from_numpy((rng.random((2 * count, 2)) - 0.5).astype(np.float32)), u=torch.zeros(2 * count, 3))
    t = {k: v.cuda() for k, v in t.items()}
    p = Particles(*(t[k].data_ptr() for k in ("np", "offset", "ix", "x", "u")), max_part=2 * count)
    out = []
    for det in (0, 1):
        rho = torch.zeros(2 * g.tile_vol, device="cuda")
        torch.cuda.synchronize()
        assert L.zpic_deposit_charge(ctypes.byref(p), ctypes.byref(g), rho.data_ptr(), -0.25, det, None) == 0
        torch.cuda.synchronize()
        out.append(rho.cpu().numpy())
    assert np.abs(out[1]).max() > 0
    close(*out)
