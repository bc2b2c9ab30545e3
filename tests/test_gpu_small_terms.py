"""The current of particles whose terms are far from the unit: slow ones (a
cold species at its start, a small seed) against 64-bit sums, and positions
outside their cell or momenta that are no number, which reach no further than
their own cells, against the deterministic mode."""
import numpy as np
import pytest

from gridutil import gather

pytestmark = pytest.mark.gpu

DT = float(np.float32(0.07))
DX = 0.1


def simulation(zp, ntiles, nx, deterministic=False):
    box = tuple(np.float32(n * m * DX) for n, m in zip(ntiles, nx))
    sim = zp.Simulation(ntiles, nx, box, DT, deterministic=deterministic)
    sim.add_species(zp.Species("electrons", -1.0, (16, 16)))
    return sim


def interior(sim, ntiles, nx, name="J"):
    g = sim.geom
    return gather(sim.field(name), ntiles, nx, g.ext_x, g.tile_vol, g.offset)


@pytest.mark.parametrize("v", [1e-7, 1e-9, 1e-13, 1e-25])
@pytest.mark.parametrize("count", [40, 1024, 16384])
def test_slow_particles(v, count):
    """uz alone, then ux alone of particles in the middle of their cells
    (whose float positions hold a displacement of any size): a term takes at
    most eight FP32 roundings of 2^-24, the sum in doubles none."""
    import pyzpic as zp
    ntiles, nx = (2, 1), (8, 8)
    rng = np.random.default_rng(count)
    n = 2 * count
    ix = np.stack([rng.integers(0, nx[0], n), rng.integers(0, nx[1], n)], 1).astype(np.int32)
    gx = ix[:, 0] + np.repeat([0, nx[0]], count)
    H, W = nx[1], ntiles[0] * nx[0]
    for comp in (2, 0):
        x = (rng.random((n, 2)) - 0.5).astype(np.float32)
        if comp == 0:
            x[:, 0] = 0
        u = np.zeros((n, 3), np.float32)
        u[:, comp] = v * (0.5 + rng.random(n))
        sim = simulation(zp, ntiles, nx)
        sim.species[0].set_particles([count, count], ix, x, u)
        sim.advance()
        got = interior(sim, ntiles, nx)[..., comp].astype(np.float64)
        sim.close()
        ref = np.zeros((H, W))
        xx, vel = x.astype(np.float64), u[:, comp].astype(np.float64)
        for j in (0, 1):
            wy = 0.5 + (2 * j - 1) * xx[:, 1]
            for i in ((0, 1) if comp == 2 else (0,)):
                # Jx of a path inside a cell belongs to the cell's own column;
                # its displacement over dt is the velocity
                wx = 0.5 + (2 * i - 1) * xx[:, 0] if comp == 2 else 1.0
                np.add.at(ref, ((ix[:, 1] + j) % H, (gx + i) % W), -vel * wx * wy / 256)
        assert np.linalg.norm(got - ref) <= 8 * 2.0 ** -24 * np.linalg.norm(ref), (comp, v, count)


@pytest.mark.parametrize("count", [3, 5000])   # a tile of one part, and one in parts
@pytest.mark.parametrize("what", ["nan", "outside", "far"])
def test_ill_particles(what, count):
    import pyzpic as zp
    ntiles, nx = (3, 2), (8, 8)
    rng = np.random.default_rng(7)
    np_ = np.array([5, 0, 2000, 40, count, 1], np.int32)
    n = int(np_.sum())
    ix = rng.integers(0, 8, (n, 2)).astype(np.int32)
    x = (rng.random((n, 2)) - 0.5).astype(np.float32)
    u = rng.normal(0, 0.3, (n, 3)).astype(np.float32)
    bad = int(np_[:4].sum()) + count // 2
    ix[bad] = 3, 5
    if what == "nan":
        u[bad, 1] = np.nan
    else:
        x[bad] = (0.9, -0.7) if what == "outside" else (3.7, 2.2)
    u[bad, 0] = 0.3
    out = []
    for det in (False, True):
        sim = simulation(zp, ntiles, nx, det)
        sim.species[0].set_particles(np_, ix, x, u)
        sim.advance()
        out.append((interior(sim, ntiles, nx), interior(sim, ntiles, nx, "E")))
        sim.close()
    for fast, ref in zip(*out):
        assert np.array_equal(np.isnan(fast), np.isnan(ref))
        assert np.isnan(ref).any() == (what == "nan") and not np.isnan(ref).all()
        # (paths cut outside their cell: terms of some tens, each to 2^-24)
        ok = ~np.isnan(ref)
        assert np.abs(fast - ref)[ok].max() <= 1e-5 * np.abs(ref[ok]).max()


@pytest.mark.parametrize("count", [3, 5000])
@pytest.mark.parametrize("where", [(np.nan, 0.1), (0.2, -7.0), (3e4, 2e4)])
def test_charge_of_ill_positions(where, count):
    """The charge of a position that is no number, or outside its cell: the
    same elements as in the deterministic mode, nothing lost beside them."""
    import pyzpic as zp
    ntiles, nx = (3, 2), (8, 8)
    rng = np.random.default_rng(8)
    np_ = np.array([5, 0, 2000, 40, count, 1], np.int32)
    n = int(np_.sum())
    ix = rng.integers(0, 8, (n, 2)).astype(np.int32)
    x = (rng.random((n, 2)) - 0.5).astype(np.float32)
    bad = int(np_[:4].sum()) + count // 2
    ix[bad], x[bad] = (3, 5), where
    out = []
    for det in (False, True):
        sim = simulation(zp, ntiles, nx, det)
        sim.species[0].set_particles(np_, ix, x, np.zeros((n, 3), np.float32))
        out.append(sim.species[0].charge())
        sim.close()
    fast, ref = out
    assert np.array_equal(np.isnan(fast), np.isnan(ref))
    assert np.isnan(ref).any() == bool(np.isnan(where[0])) and not np.isnan(ref).all()
    # (each element to 1e-5 of its own, the particles of an element being a
    # few hundred terms of one sign; those of the bad cell to 1e-5 of its terms)
    ok = ~np.isnan(ref)
    size = np.abs(ref[ok])
    assert (np.abs(fast - ref)[ok] <= 1e-5 * np.where(size > 100, size.max(), size + 1e-3)).all()
