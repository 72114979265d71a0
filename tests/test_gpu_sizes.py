"""The kernels whose form depends on the size of the system, at the sizes where
the form changes and at ragged ones, against the CPU oracle."""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _fluid(n, rho, seed):
    """n sites of a jittered simple-cubic lattice in a cubic box, Maxwell velocities"""
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1.0 / 3.0)))
    L = max((n / rho) ** (1.0 / 3.0), 3.0)
    k = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[rng.permutation(m ** 3)[:n]]
    x = (k + 0.5 + rng.uniform(-0.1, 0.1, (n, 3))) * (L / m)
    return L, x, rng.standard_normal((n, 3))


# the force kernel takes 32, 16, 8, 4 or 2 lanes per local (2: full lists only)
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("n,ntypes", [(1, 1), (2, 1), (3, 2), (33, 1), (517, 3), (4095, 1), (4097, 2), (12287, 4),
                                      (12289, 1), (39999, 1), (40001, 3), (99999, 1), (100003, 2)])
def test_lj_run_vs_oracle_at_size_edges(n, ntypes, half):
    """bit-identical state after runs of 1, 6 and 25 steps (rebuilds every 10,
    a thermo step among them), some particles fixed"""
    from pairs_amd import md
    L, x, v = _fluid(n, 0.75, n)
    rng = np.random.default_rng(n + 1)
    types = rng.integers(0, ntypes, n).astype(np.int32)
    flags = np.where(rng.random(n) < 0.02, 4, 0).astype(np.int32)
    v[flags == 4] = 0.0
    eps = 1.0 - 0.1 * np.abs(np.subtract.outer(np.arange(ntypes), np.arange(ntypes))).ravel()
    sig6 = (1.0 - 0.03 * np.add.outer(np.arange(ntypes), np.arange(ntypes)).ravel()) ** 6
    kw = dict(half=half, ntypes=ntypes, reneighbor_every=10, thermo_every=15)
    cap = 4 * n + 40000 if n < 4000 else 3 * n
    g = md.LJSystem([(0.0, L)] * 3, particle_capacity=cap, send_capacity=cap, neighbor_capacity=120, epsilon=eps,
                    sigma6=sig6, **kw)
    o = po.OracleMD([(0.0, L)] * 3, cap, ncap=160, ccap=128, send_cap=cap, eps=eps, sig6=sig6, **kw)
    g.upload(x, v, types=types, flags=flags)
    o.set_particles(x, v, types=types, flags=flags)
    o.setup_cells()
    # (the oracle integrates into step ts at its start, as a continued run does)
    for a, b in ((0, 1), (1, 7), (7, 32)):
        g.run(a, b, 100)
        o.run(a, b)
        assert g.nlocal == o.nlocal and g.nghost == o.nghost
        for name, p, q in (("position", g.positions(True), o.positions(True)),
                           ("velocity", g.velocities(), o.velocities()), ("force", g.forces(), o.forces())):
            assert np.array_equal(p, q), f"{name} after step {b}: max |diff| {np.abs(p - q).max()}"
