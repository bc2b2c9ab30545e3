"""Crowded tiles in the fast-mode particle pass: a tile's particles shared by
several workgroups, at the counts where the cut changes, against the
deterministic mode (one wavefront per tile, bit-exact with the oracle)."""
import numpy as np
import pytest

from conftest import same_tile_multisets

pytestmark = pytest.mark.gpu


def crowded(ntiles, nx, counts, seed):
    """Particles of `counts` per tile, anywhere in the tile, fast enough that
    every direction out of it occurs."""
    rng = np.random.default_rng(seed)
    n = int(np.sum(counts))
    ix = np.stack([rng.integers(0, nx[0], n), rng.integers(0, nx[1], n)], 1).astype(np.int32)
    x = (rng.random((n, 2)) - 0.5).astype(np.float32)
    u = rng.normal(0, 0.8, (n, 3)).astype(np.float32)
    return np.asarray(counts, np.int32), ix, x, u


@pytest.mark.parametrize("ntiles,nx,threads,counts", [
    ((1, 1), (16, 16), 256, [5000]),
    ((3, 2), (8, 8), 256, [0, 1, 1023, 1024, 1025, 2048]),
    ((3, 2), (8, 8), 64, [2049, 0, 14 * 1024, 64, 16000, 3]),
    ((3, 2), (8, 8), 256, [2047, 2048, 2049, 4096, 4097, 1]),
    ((3, 2), (8, 8), 64, [14 * 2048, 14 * 2048 + 1, 0, 40000, 13 * 2048, 6143]),
    ((2, 2), (32, 32), 512, [30000, 1, 0, 1100]),
    ((33, 32), (8, 8), 256, [3] * 1055 + [5000]),   # more than one tile per thread of the scan
    ((32, 32), (8, 8), 256, [1] * 1000 + [0] * 23 + [9000]),
    ((64, 64), (4, 4), 256, [2] * 4090 + [0] * 5 + [3000]),
    ((2, 2), (36, 36), 256, [20000, 3, 0, 1025]),   # the largest tiles: two workgroups of the pass per CU
    ((2, 2), (38, 38), 512, [20000, 3, 0, 1025]),   # and one
    ((1, 1), (38, 38), 64, [5000]),
    ((241, 17), (4, 5), 256, [1] * 4096 + [3000]),  # more tiles than the cut is used for
])
def test_crowded_tiles(ntiles, nx, threads, counts):
    import pyzpic as zp
    total = int(np.sum(counts))
    ppc = max(1, int(np.ceil(np.sqrt(total / (ntiles[0] * ntiles[1] * nx[0] * nx[1])))))
    old = zp.get_threads_per_tile()
    sims = []
    try:
        zp.set_threads_per_tile(threads)
        for det in (False, True):
            sim = zp.weibel(ntiles=ntiles, nx=nx, ppc=(ppc, ppc), deterministic=det)
            for k, s in enumerate(sim.species):
                s.set_particles(*crowded(ntiles, nx, counts if k == 0 else counts[::-1], 5 + k))
            sims.append(sim)
        for step in range(3):  # the cut follows the counts, which follow the crowd as it spreads
            fast, det = sims
            state = [s.particles() for s in fast.species]
            for k, s in enumerate(det.species):
                s.set_particles(*(state[k][n] for n in ("np", "ix", "x", "u")))
            for f in "EB":
                det.set_field(f, fast.field(f))
            for sim in sims:
                sim.advance()
            for k in range(2):
                assert same_tile_multisets(fast.species[k].particles(), det.species[k].particles()), (step, k)
            for f in "JEB":
                a, b = fast.field(f).astype(np.float64), det.field(f).astype(np.float64)
                assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b), (step, f)
            np.testing.assert_allclose(fast.energies(), det.energies(), rtol=1e-5)
    finally:
        zp.set_threads_per_tile(old)
        for sim in sims:
            sim.close()


def test_species_of_different_sizes():
    """Species side by side whose lists of parts differ in length, one of them
    empty."""
    import pyzpic as zp
    sims = []
    for det in (False, True):
        sim = zp.Simulation((5, 4), (8, 8), (np.float32(4.0), np.float32(3.2)), 0.07, deterministic=det)
        for k, ppc in enumerate([(1, 1), (20, 20), (2, 1)]):
            sim.add_species(zp.Species(f"s{k}", (-1.0, 1.0, 4.0)[k], ppc))
        sims.append(sim)
    for sim in sims:
        for k, counts in enumerate([[3] * 19 + [700], [1200] * 20, [0] * 20]):
            sim.species[k].set_particles(*crowded((5, 4), (8, 8), counts, 11 + k))
        sim.advance()
    fast, det = sims
    for k in range(3):
        assert same_tile_multisets(fast.species[k].particles(), det.species[k].particles()), k
    for f in "JEB":
        a, b = fast.field(f).astype(np.float64), det.field(f).astype(np.float64)
        assert np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b), f
    for sim in sims:
        sim.close()
