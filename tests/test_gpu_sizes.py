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


@pytest.mark.parametrize("n", [100, 5000, 13000, 45000, 110000])
def test_forces_beside_a_particle_at_infinity(n):
    """a particle that has left for infinity, in the last slot of an open system,
    leaves the forces of the others as they are without it"""
    from pairs_amd import md, mlp
    L, x, v = _fluid(n, 0.8, n)
    m = mlp.MLPModel(seed=2)
    out = []
    for far in (False, True):
        g = md.LJSystem([(0.0, L)] * 3, particle_capacity=n + 8, send_capacity=64, neighbor_capacity=120,
                        periodic=(0, 0, 0))
        g.upload(np.concatenate([x, np.full((1, 3), np.inf)]) if far else x,
                 np.concatenate([v, np.zeros((1, 3))]) if far else v)
        g.exchange()
        g.borders()
        g.build_cell_lists()
        g.build_neighbor_lists()
        g.lennard_jones()
        got = [g.forces()[:n], g.numneighs()[:n]]
        mlp.forces(g, m)
        out.append(got + [g.forces()[:n]])
    for p, q in zip(*out):
        assert np.array_equal(p, q)


def test_lj_run_in_arrays_of_many_slots():
    """a small system in arrays of 38.5 million slots: a list row's offset passes 4 GiB"""
    from pairs_amd import md
    L, x, v = _fluid(500, 0.8, 1)
    out = []
    for cap in (8000, 38500000):
        g = md.LJSystem([(0.0, L)] * 3, particle_capacity=cap, send_capacity=8000, neighbor_capacity=128)
        g.upload(x, v)
        g.run(0, 30, 100)
        out.append((g.positions(True), g.velocities(), g.forces()))
        assert g.numneighs().min() > 28
        del g
    for p, q in zip(*out):
        assert np.array_equal(p, q)


def _spheres(case):
    """uid, radius, position, velocity of a few spheres, domain, half-spaces"""
    rng = np.random.default_rng(len(case))
    d = 0.0029
    planes = [(100000, (0.0, 0.0, 0.0), (0.0, 0.0, 1.0), 13)]
    if case.startswith("pile"):  # a loose pile of n spheres
        n = int(case[4:])
        m = int(np.ceil(n ** (1.0 / 3.0)))
        k = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
        x = (k + 0.5) * 0.97 * d + rng.uniform(-0.02, 0.02, (n, 3)) * d
        r = 0.5 * d * rng.uniform(0.95, 1.05, n)
        dom = (max(0.012, m * 0.97 * d + 0.001), max(0.012, m * 0.97 * d + 0.001), max(0.02, m * d + 0.01))
    elif case == "crowd":  # one sphere with 30 small ones around it: more partners than the search keeps
        u = rng.standard_normal((30, 3))
        u /= np.linalg.norm(u, axis=1)[:, None]
        x = np.concatenate([[[0.01, 0.01, 0.01]], 0.01 + u * 0.00198])
        r = np.concatenate([[0.0016], np.full(30, 0.0004)])
        dom = (0.02, 0.02, 0.02)
    elif case == "dense":  # many small spheres per cell: more candidates than a lane's mask holds
        k = np.stack(np.meshgrid(*[np.arange(9)] * 3, indexing="ij"), -1).reshape(-1, 3)
        x = 0.002 + (k + 0.5) * 0.0008 + rng.uniform(-1e-5, 1e-5, (729, 3))
        r = np.full(729, 0.00041)
        dom = (0.02, 0.02, 0.02)
    elif case == "image":  # a partner and its periodic image touch the same sphere
        x = np.array([[0.0004, 0.006, 0.006], [0.0019, 0.0082, 0.006], [0.0011, 0.006, 0.0088]])
        r = np.full(3, 0.00145)
        dom = (0.0031, 0.012, 0.012)
    else:  # half-spaces in cells of their own, among spheres
        k = np.stack(np.meshgrid(*[np.arange(3)] * 3, indexing="ij"), -1).reshape(-1, 3)
        x = 0.004 + (k + 0.5) * 0.98 * d
        r = np.full(27, 0.5 * d)
        planes += [(7, (0.0055, 0.0052, 0.0046), (0.0, 0.0, 1.0), 12), (900, (0.0055, 0.0052, 0.012), (0.0, 0.6, -0.8), 12)]
        dom = (0.02, 0.02, 0.02)
    return np.arange(1, len(r) + 1) + 10, r, x, rng.uniform(-0.05, 0.05, x.shape), dom, planes


@pytest.mark.parametrize("case", ["pile1", "pile7", "pile9", "pile33", "pile257", "crowd", "dense", "image", "walls"])
def test_dem_contacts_vs_oracle(case):
    """contacts, history and trajectory of small arrangements that take every
    form of the contact kernels, 30 steps against the oracle"""
    from pairs_amd import dem
    uid, r, x, v, dom, planes = _spheres(case)
    g = dem.DEMSystem(dom, particle_capacity=16384, contact_capacity=48)
    o = po.OracleDEM(dom, cap=16384, ccap=48, cellcap=256)
    g.add_spheres(uid, r, x, v)
    for k in range(len(r)):
        o.add_sphere(int(uid[k]), r[k], x[k], v[k])
    for s in (g, o):
        for u, pos, nrm, fl in planes:
            s.add_halfspace(u, pos, nrm, flags=fl)
        s.setup()
    for a, b in ((0, 1), (1, 4), (4, 30)):
        g.run(a, b)
        o.run(a, b)
        assert g.nlocal == o.nlocal and g.nghost == o.nghost, b
        assert np.array_equal(g.get("uid"), o.get("uid")), b
        nc, cl, sk, tsd, iv = g.contacts()
        onc, ocl, osk, otsd, oiv = o.contacts()
        assert np.array_equal(nc, onc), b
        for i in range(len(nc)):
            m = nc[i]
            assert np.array_equal(cl[i, :m], ocl[i, :m]) and np.array_equal(sk[i, :m], osk[i, :m]), (b, i)
        # sin and cos of the rotation update differ in their last bits: 1e-10, as the DEM tests
        for name, p, q in [(k, g.get(k), o.get(k)) for k in ("position", "linear_velocity", "angular_velocity",
                                                              "force", "torque")]:
            assert np.abs(p - q).max() <= 1e-10 * max(np.abs(q).max(), 1e-300), (b, name)


def test_dem_phase_times_add_up():
    """the phases that are part of the contact kernel read zero, and the others make
    up the time of the contact kernels"""
    from pairs_amd import dem
    uid, r, x, v, dom, planes = _spheres("pile257")
    s = dem.DEMSystem(dom, particle_capacity=4096)
    s.add_spheres(uid, r, x, v)
    for u, pos, nrm, fl in planes:
        s.add_halfspace(u, pos, nrm, flags=fl)
    s.setup()
    s.set_timing(2)
    s.run(0, 20)
    phases, (contact, launches) = s.phase_times(), s.contact_kernel_time()
    assert launches == 10 and phases[2] == phases[4] == 0.0
    assert all(phases[k] > 0.0 for k in (0, 1, 3, 5))
    # (event times are rounded to 1e-7 ms in float)
    assert abs(phases[1] + phases[3] - contact) < 1e-5 * contact + 1e-6


@pytest.mark.parametrize("flags", [0, 8])
def test_dem_unfixed_halfspaces_vs_oracle(flags):
    """half-spaces without the FIXED flag look for contacts themselves, as points
    of radius 0; a sphere of negative radius is a sphere all the same"""
    from pairs_amd import dem
    uid, r, x, v, dom, planes = _spheres("walls")
    uid, r = np.append(uid, 500), np.append(r, -0.0004)
    x, v = np.concatenate([x, x[:1] - [0.0, 0.0, 0.0008]]), np.concatenate([v, [[0.0, 0.01, 0.0]]])
    g = dem.DEMSystem(dom, particle_capacity=16384, contact_capacity=48)
    o = po.OracleDEM(dom, cap=16384, ccap=48, cellcap=256)
    g.add_spheres(uid, r, x, v)
    for k in range(len(r)):
        o.add_sphere(int(uid[k]), r[k], x[k], v[k])
    for s in (g, o):
        for u, pos, nrm, fl in planes:
            s.add_halfspace(u, pos, nrm, flags=fl if fl == 13 else flags)
        s.setup()
    for a, b in ((0, 1), (1, 4), (4, 30)):
        g.run(a, b)
        o.run(a, b)
        assert np.array_equal(g.get("uid"), o.get("uid")), b
        nc, cl, sk, _, _ = g.contacts()
        onc, ocl, osk, _, _ = o.contacts()
        assert np.array_equal(nc, onc), b
        for i in range(len(nc)):
            m = nc[i]
            assert np.array_equal(cl[i, :m], ocl[i, :m]) and np.array_equal(sk[i, :m], osk[i, :m]), (b, i)
        if b == 1:
            assert (nc[g.get("shape") == 1] > 0).sum() == 2 and nc[g.get("uid") == 500] > 0
        for name, p, q in [(k, g.get(k), o.get(k)) for k in ("position", "linear_velocity", "angular_velocity",
                                                              "force", "torque")]:
            assert np.abs(p - q).max() <= 1e-10 * max(np.abs(q).max(), 1e-300), (b, name)


# k_mlp_eval takes workgroups of 4 waves below 8192 rows, of 16 from there; past
# 65536 rows a wave walks several tiles
@pytest.mark.parametrize("n", [1, 15, 17, 8191, 8192, 8193, 65537, 131089])
def test_mlp_eval_vs_oracle_at_size_edges(n):
    """energies and dE/dG against the BF16-emulating oracle at the tolerance of
    the 1000-row test, on 300 rows drawn from all of them, and the first and
    last 20; equal descriptors give equal results wherever their row lies"""
    from oracle import mlp_oracle as mo
    from pairs_amd import mlp
    rng = np.random.default_rng(n)
    p = mo.xavier(7).astype(np.float32)
    sc = np.concatenate([rng.uniform(0.0, 3.0, 16), rng.uniform(0.3, 2.0, 16), [-5.5, 0.7]]).astype(np.float32)
    m = mlp.MLPModel(seed=1)
    m.set_params(p, sc)
    base = rng.uniform(0.0, 4.0, (1000, 16)).astype(np.float32)
    pick = rng.integers(0, 1000, n)
    E, D = m.eval(base[pick])
    Eb, Db = mo.forward_bf16(p, sc, base)
    rows = np.unique(np.concatenate([np.arange(min(n, 20)), np.arange(max(n - 20, 0), n), rng.integers(0, n, 300)]))
    err = np.sqrt(np.mean((E[rows] - Eb[pick[rows]]) ** 2))
    assert err < 5e-3 * Eb.std(), err
    ref = Db[pick[rows]]
    assert np.sqrt(np.mean((D[rows] - ref) ** 2)) < 5e-3 * np.sqrt(np.mean(ref ** 2))
    E0, D0 = m.eval(base)
    assert np.array_equal(E, E0[pick]) and np.array_equal(D, D0[pick])


# a partial's tiles are taken four at a time: 1, 3, 4, 5 and 9 of them
@pytest.mark.parametrize("tiles", [1, 3, 4, 5, 9])
def test_mlp_energy_grad_vs_oracle_by_tiles(tiles):
    """k_mlp_grad on a minibatch of 64 partials of `tiles` 16-row tiles, at the
    tolerance of the one-tile test"""
    from oracle import mlp_oracle as mo
    from pairs_amd import mlp
    import test_gpu_mlp as tm
    rng = np.random.default_rng(tiles)
    rows, batch, seed, step = 3000, 1024 * tiles, 11, 5
    G = rng.uniform(0.0, 4.0, (rows, 16)).astype(np.float32)
    lab = rng.normal(-5.0, 0.8, rows).astype(np.float32)
    p, sc = mo.xavier(5).astype(np.float32), tm._scale().astype(np.float32)
    m = mlp.MLPModel(seed=1, dataset_capacity=rows)
    m.set_params(p, sc)
    assert m.add_rows(G, lab) == rows
    g, loss = m.energy_grad(step, batch=batch, seed=seed)
    idx = np.array([tm._splitmix64(seed ^ (step << 32) ^ j) % rows for j in range(batch)])
    Lr, ref = mo.energy_loss_grad(p.astype(np.float64), sc.astype(np.float64), G[idx].astype(np.float64),
                                  lab[idx].astype(np.float64))
    assert abs(loss - Lr) <= 2e-2 * Lr, (loss, Lr)
    tm._check_grad(g, ref, f"{tiles} tiles")


# 864 to 5324 atoms: 1 to 6 tiles in a partial of k_mlp_cgrad, ragged ones among them
@pytest.mark.parametrize("cells", [6, 9, 10, 11])
def test_mlp_config_grad_vs_oracle_by_tiles(cells):
    from oracle import mlp_oracle as mo
    from pairs_amd import mlp
    import test_gpu_mlp as tm
    s, L = tm._state(cells, 40)
    x = s.positions()
    El, Fl = mo.lj_atom_energy(x, L), mo.lj_forces(x, L)
    G = mo.descriptors(x, L)
    sc = np.concatenate([G.mean(0), 1.0 / G.std(0), [El.mean(), El.std()]]).astype(np.float32)
    p = mo.xavier(5).astype(np.float32)
    m = mlp.MLPModel(seed=1, dataset_capacity=16)
    m.set_params(p, sc)
    g, (le, lf) = m.config_grad(s, 0.5, 1.0)
    _, le_r, lf_r, ref = mo.config_loss_grad(p.astype(np.float64), sc.astype(np.float64), x, L, El, Fl, 0.5, 1.0)
    assert abs(le - le_r) <= 3e-2 * le_r and abs(lf - lf_r) <= 3e-2 * lf_r
    tm._check_grad(g, ref, f"{len(x)} atoms")


# 6912 and 8788 atoms: either side of k_mlp_eval's rule, with its writes to ghost images
@pytest.mark.parametrize("cells", [12, 13])
def test_mlp_forces_vs_oracle_at_size_edges(cells):
    from oracle import mlp_oracle as mo
    from pairs_amd import mlp
    import test_gpu_mlp as tm
    s, L = tm._state(cells, 40)
    x = s.positions()
    G = mo.descriptors(x, L)
    p = mo.xavier(5).astype(np.float32)
    sc = np.concatenate([G.mean(0), 1.0 / G.std(0), [-5.5, 0.7]]).astype(np.float32)
    m = mlp.MLPModel(seed=1)
    m.set_params(p, sc)
    e, _ = mlp.forces(s, m)
    Fx, Ex = mo.forces(p, sc, x, L)
    assert tm._rel_rms(s.forces(), Fx) < 3e-2
    assert abs(e - Ex.sum()) < 1e-3 * abs(Ex.sum())


def test_mlp_forces_after_module_rebuild_with_many_images():
    """a run whose locals have 7 images each, then a rebuild by modules after which
    half of them have 11, more than the image table holds, those that the table
    leaves out inside the cutoff of others: forces as those of a system that
    starts there"""
    from pairs_amd import md, mlp
    L = 5.04  # less than two cell spacings
    x = 1.2 + 3.7 * np.stack(np.meshgrid(*[np.arange(2)] * 3, indexing="ij"), -1).reshape(-1, 3)
    x += np.random.default_rng(8).uniform(-0.02, 0.02, x.shape)
    v = np.zeros((8, 3))
    v[:4, 0] = (2.27 - x[:4, 0]) / 0.005  # within a spacing of both faces in one step
    m = mlp.MLPModel(seed=3)

    def system(x, v):
        s = md.LJSystem([(0.0, L)] * 3, particle_capacity=4000, send_capacity=4000, neighbor_capacity=120)
        s.upload(x, v)
        return s
    g = system(x, v)
    g.run(0, 1, 0)
    g.euler()
    for s in (g, None):
        s = s or system(g.positions(), g.velocities())
        s.exchange()
        s.borders()
        s.build_cell_lists()
        s.build_neighbor_lists()
        e, w = mlp.forces(s, m)
        out = (e, w, s.nghost, s.positions(True), s.forces())
        if s is g:
            got = out
    assert got[2] == out[2] == 4 * 7 + 4 * 11
    assert got[0] == out[0] and got[1] == out[1]
    assert np.array_equal(got[3], out[3]) and np.array_equal(got[4], out[4])


def test_second_upload_starts_without_images():
    """an upload into a system that has run: the first rebuild is checked before the
    steps behind it, as a new system's, and the run is the same"""
    from pairs_amd import md, native
    out = []
    for first in (700, 0):
        g = md.LJSystem([(0.0, 14.0)] * 3, particle_capacity=16000, send_capacity=12000, neighbor_capacity=120)
        if first:
            _, x, v = _fluid(first, first / 14.0 ** 3, 1)
            g.upload(x, v)
            g.run(0, 3, 100)
        _, x, v = _fluid(2300, 2300 / 14.0 ** 3, 2)
        g.upload(x, v)
        g.run(0, 23, 100)
        out.append((g.positions(True), g.velocities(), g.forces(), g.count(native.REBUILDS_DEFERRED)))
    for p, q in zip(*out):
        assert np.array_equal(p, q)


# exchange and borders: 0 to 3 periodic dimensions; the leavers of a step fit the
# list that the integration keeps (1024) or do not; a box narrower than two
# cell widths, whose particles have images on both sides; a cell grid whose
# block totals do not fit the fill kernel's scan (2048 * 1024 cells)
@pytest.mark.parametrize("pairs,periodic,dom,speed", [
    (300, (True, True, False), (0.03, 0.02, 0.03), 20.0),
    (300, (False, True, False), (0.03, 0.02, 0.03), 20.0),
    (300, (True, True, True), (0.03, 0.02, 0.03), 20.0),
    (300, (False, False, False), (0.03, 0.02, 0.03), 20.0),
    (2500, (True, True, False), (0.06, 0.06, 0.06), 300.0),
    (2500, (True, False, True), (0.06, 0.06, 0.06), 300.0),
    (2500, (True, True, True), (0.06, 0.06, 0.06), 300.0),
    (40, (True, True, True), (0.0045, 0.03, 0.0041), 20.0),
    (200, (True, True, False), (0.41, 0.41, 0.41), 400.0),
])
def test_dem_exchange_and_borders_vs_oracle(pairs, periodic, dom, speed):
    """touching pairs that fly through the faces together, their order, ghosts
    and contact history against the oracle, with a run cut into chunks"""
    from pairs_amd import dem
    rng = np.random.default_rng(pairs)
    dom = np.asarray(dom)
    r = 0.0001
    x = rng.uniform(0.0006, 1.0, (pairs, 3)) * (dom - 0.0012) + 0.0003
    u = rng.standard_normal((pairs, 3))
    u *= 1.94 * r / np.linalg.norm(u, axis=1)[:, None]
    v = rng.uniform(-speed, speed, (pairs, 3)) * np.asarray(periodic)
    pos, vel = np.concatenate([x, x + u]), np.concatenate([v, v + rng.uniform(-0.05, 0.05, v.shape)])
    order = rng.permutation(2 * pairs)
    pos, vel = pos[order], vel[order]
    uid = np.arange(1, 2 * pairs + 1)
    cells = int(np.prod(np.ceil(dom / 0.0025) + 4)) + 2
    g = dem.DEMSystem(tuple(dom), periodic=periodic, particle_capacity=40000, contact_capacity=6, send_capacity=30000,
                      ncells_capacity=cells)
    o = po.OracleDEM(tuple(dom), periodic=periodic, cap=40000, ccap=6, cellcap=16 if cells > 1000000 else 256,
                     send_cap=30000, ncells_cap=cells)
    g.add_spheres(uid, np.full(2 * pairs, r), pos, vel)
    for k in range(2 * pairs):
        o.add_sphere(int(uid[k]), r, pos[k], vel[k])
    for s in (g, o):
        s.setup()
    for a, b in ((0, 1), (1, 3), (3, 8)):
        g.run(a, b)
        o.run(a, b)
        assert g.nlocal == o.nlocal and g.nghost == o.nghost, b
        assert np.array_equal(g.get("uid", ghosts=True), o.get("uid", ghosts=True)), b
        nc, cl, sk, tsd, iv = g.contacts()
        onc, ocl, osk, otsd, oiv = o.contacts()
        assert np.array_equal(nc, onc), b
        for i in range(len(nc)):
            m = nc[i]
            assert np.array_equal(cl[i, :m], ocl[i, :m]) and np.array_equal(sk[i, :m], osk[i, :m]), (b, i)
            if m:
                assert np.abs(tsd[i, :m] - otsd[i, :m]).max() <= 1e-9 * np.abs(otsd).max(), (b, i)
        for name in ("position", "linear_velocity"):
            p, q = g.get(name, ghosts=True), o.get(name, ghosts=True)
            assert np.abs(p - q).max() <= 1e-10 * np.abs(q).max(), (b, name)
    assert nc.max() > 0


# exchange and borders of a rebuild: 0 to 3 periodic dimensions; leavers that are
# one per thread of the one-workgroup exchange (1024), several, or do not fit its
# list (4096; then, from the next rebuild on, the wide kernels run); a box narrower than two cell spacings; more
# than one border tile (1024 reference indices)
@pytest.mark.parametrize("n,periodic,edge,speed", [
    (1, (1, 1, 1), 39.0, 300.0), (1023, (1, 1, 1), 21.0, 200.0), (1025, (1, 1, 1), 22.0, 200.0),
    (6000, (1, 1, 1), 39.0, 200.0), (6000, (1, 1, 1), 39.0, 2500.0), (6000, (0, 1, 1), 39.0, 3500.0),
    (6000, (1, 1, 1), 39.0, 7000.0),
    (6000, (1, 1, 0), 39.0, 200.0), (6000, (1, 0, 1), 39.0, 200.0), (3000, (0, 1, 0), 31.0, 200.0),
    (3000, (0, 0, 1), 31.0, 200.0), (3000, (1, 0, 0), 31.0, 200.0), (3000, (0, 0, 0), 31.0, 200.0),
    (100, (1, 1, 1), 5.04, 100.0), (3000, (1, 1, 1), 100.0, 300.0)])  # (54873 cells: several rounds of the scan)
def test_lj_exchange_and_borders_vs_oracle(n, periodic, edge, speed):
    """free flight through the faces with a rebuild after every step: order,
    ghosts, maps and lists against the oracle"""
    from pairs_amd import md
    import test_gpu_md as tm
    rng = np.random.default_rng(n + int(speed))
    box = [(0.0, edge)] * 3
    x = rng.uniform(0.0, edge, (n, 3))
    v = rng.uniform(-speed, speed, (n, 3)) * np.asarray(periodic)
    flags = np.where(rng.random(n) < 0.02, 4, 0).astype(np.int32)
    flags[rng.random(n) < 0.01] = 8
    g = md.LJSystem(box, particle_capacity=40000, neighbor_capacity=200, send_capacity=30000, periodic=periodic)
    o = po.OracleMD(box, 40000, ncap=200, ccap=256, send_cap=30000, periodic=periodic)
    g.upload(x, v, flags=flags)
    o.set_particles(x, v, flags=flags)
    o.setup_cells()
    for step in range(4):
        g.euler()
        o.euler()
        g.exchange()
        g.borders()
        g.build_cell_lists()
        g.build_neighbor_lists()
        o.rebuild()
        assert o.overflow == 0
        assert np.array_equal(g.nsend(), o.nsend()), step
        assert np.array_equal(g.positions(True), o.positions(True)), step
        assert np.array_equal(g.velocities(), o.velocities()), step
        tm._compare_lists(g, o, step)


@pytest.mark.parametrize("half", [False, True])
def test_lj_long_columns_vs_oracle(half):
    """a sparse system of columns of 953 cells, whose table of cells takes most of a
    build workgroup's LDS"""
    from pairs_amd import md
    rng = np.random.default_rng(9)
    n, box = 300, [(0.0, 8.4), (0.0, 8.4), (0.0, 2660.0)]
    x = rng.uniform(0.0, 1.0, (n, 3)) * [8.4, 8.4, 1.0]
    x[:, 2] = (np.arange(n) // 10 + 0.5) * 88.0 + 1.1 * (np.arange(n) % 10)  # strings of ten
    v = rng.standard_normal((n, 3))
    g = md.LJSystem(box, particle_capacity=8000, neighbor_capacity=100, send_capacity=6000, half=half)
    o = po.OracleMD(box, 8000, ncap=100, ccap=64, send_cap=6000, half=half)
    g.upload(x, v)
    o.set_particles(x, v)
    o.setup_cells()
    for a, b in ((0, 1), (1, 23)):
        g.run(a, b, 100)
        o.run(a, b)
        assert o.overflow == 0
        for name, p, q in (("position", g.positions(True), o.positions(True)),
                           ("velocity", g.velocities(), o.velocities()), ("force", g.forces(), o.forces())):
            assert np.array_equal(p, q), (name, b)
    assert g.numneighs().max() > 0


# large systems of one type take the timestep's forces from LDS tiles; two types
# with the same parameters do not, and give the same bits
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("sites,spacing,every", [
    ((59, 59, 59), 1.06, 10),     # the LJ fluid; a last column of cells nearly empty
    ((26, 29, 271), 1.06, 12),    # long columns
    ((61, 61, 55), 0.93, 10),     # dense: tiles that do not fit, the 32-bit lists instead
    ((130, 130, 12), 1.06, 10)])  # short columns: no tiles
def test_lj_tiles_vs_gathers(half, sites, spacing, every):
    from pairs_amd import md
    rng = np.random.default_rng(sum(sites))
    k = np.stack(np.meshgrid(*[np.arange(m) for m in sites], indexing="ij"), -1).reshape(-1, 3)
    n = len(k)
    k = k[rng.permutation(n)]
    box = [(0.0, m * spacing) for m in sites]
    x = (k + 0.5 + rng.uniform(-0.08, 0.08, k.shape)) * spacing
    v = rng.standard_normal(k.shape)
    flags = np.where(rng.random(n) < 0.02, 4, 0).astype(np.int32)
    v[flags == 4] = 0.0
    out = []
    for nt in (1, 2):
        g = md.LJSystem(box, particle_capacity=2 * n, send_capacity=n, neighbor_capacity=140, half=half, ntypes=nt,
                        reneighbor_every=every, thermo_every=16, ncells_capacity=200000)
        g.upload(x, v, flags=flags, types=np.arange(n, dtype=np.int32) % nt)
        got = []
        for a, b in ((0, 1), (1, 6), (6, 27)):
            g.run(a, b, 100)
            got += [g.positions(True), g.velocities(), g.forces()]
        out.append(got)
    for p, q in zip(*out):
        assert np.array_equal(p, q)


def test_lj_tiles_of_a_slab_with_a_gap_vs_gathers():
    """columns no longer than a group, particles below the open lower face, and empty
    columns: runs of a group's candidate cells that begin at one slot"""
    from pairs_amd import md
    rng = np.random.default_rng(12)
    k = np.stack(np.meshgrid(np.arange(220), np.arange(65), np.arange(14), indexing="ij"), -1).reshape(-1, 3)
    n = len(k)
    x = (k + 0.5 + rng.uniform(-0.06, 0.06, k.shape)) * [0.95, 0.95, 1.0]
    x[:, 1] += 4.0
    x[:, 2] -= 1.0
    v = rng.standard_normal(k.shape)
    out = []
    for nt in (1, 2):
        g = md.LJSystem([(0.0, 209.0), (0.0, 70.25), (0.0, 13.9)], particle_capacity=2 * n, send_capacity=n,
                        neighbor_capacity=160, ntypes=nt, reneighbor_every=10, periodic=(1, 1, 0))
        g.upload(x, v, types=np.arange(n, dtype=np.int32) % nt)
        got = []
        for a, b in ((0, 1), (1, 12)):
            g.run(a, b, 100)
            got += [g.positions(True), g.velocities(), g.forces()]
        out.append(got)
    for p, q in zip(*out):
        assert np.array_equal(p, q)


def test_lj_forces_before_a_build():
    """a large system's forces where no build has made tiles yet: after an upload,
    after another one, after the lists have grown, in a run that starts between
    two rebuilds; two types with the same parameters take no tiles"""
    from pairs_amd import md
    rng = np.random.default_rng(3)
    m, a = 59, 1.06
    k = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    n = len(k)
    x = (k + 0.5 + rng.uniform(-0.08, 0.08, k.shape)) * a
    v = rng.standard_normal(k.shape)
    y = x[rng.permutation(n)]
    out = []
    for nt in (1, 2):
        t = np.arange(n, dtype=np.int32) % nt
        g = md.LJSystem([(0.0, m * a)] * 3, particle_capacity=2 * n, send_capacity=n, neighbor_capacity=120,
                        ntypes=nt, reneighbor_every=10)
        g.upload(x, v, types=t)
        g.lennard_jones()
        assert not g.forces().any()
        g.run(1, 3, 100)
        got = [g.positions(), g.velocities()]
        g.run(3, 25, 100)
        got.append(g.forces())
        g.upload(y, v, types=t)  # (the lists are those of the run)
        g.lennard_jones()
        got.append(g.forces())
        g._call("pairs_hip_reserve", 0, 200, 0)
        g.lennard_jones()
        assert not g.forces().any()
        g.run(0, 12, 100)
        got += [g.positions(True), g.velocities(), g.forces()]
        out.append(got)
    for p, q in zip(*out):
        assert np.array_equal(p, q, equal_nan=True)


def test_tiles_come_back():
    """the tile arrays of a large system (more than 100 MB here) are given back while
    an MLP potential is attached and while a configuration is too dense for
    them, and are there again after a detach and after the next upload; the
    trajectory is that of a system that never was without"""
    import ctypes
    from pairs_amd import md, mlp
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value / 1e6
    rng = np.random.default_rng(7)
    m, a = 59, 1.06
    k = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    n = len(k)
    x = (k + 0.5 + rng.uniform(-0.08, 0.08, k.shape)) * a
    v = rng.standard_normal(k.shape)
    model = mlp.MLPModel(seed=1)
    out = []
    for attach in (False, True):
        g = md.LJSystem([(0.0, m * a)] * 3, particle_capacity=3 * n, send_capacity=2 * n, neighbor_capacity=256,
                        reneighbor_every=10)
        g.upload(x, v)
        g.run(0, 12, 100)
        if attach:
            f0 = free()
            mlp.attach(g, model, -1.0)
            f1 = free()
            mlp.detach(g)
            f2 = free()
            assert f2 < f1 - 100, (f0, f1, f2)
            g.lennard_jones()
        g.run(12, 33, 100)
        out.append((g.positions(True), g.velocities(), g.forces()))
    for p, q in zip(*out):
        assert np.array_equal(p, q)
    # a density of 1.59: the tiles of many groups do not fit
    f0 = free()
    dense = (np.stack(np.meshgrid(*[np.arange(73)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5) * (m * a / 73)
    g.upload(dense, np.zeros(dense.shape))
    g.exchange()
    g.borders()
    g.build_cell_lists()
    g.build_neighbor_lists()
    assert free() > f0 + 100, (f0, free())
    g.upload(x, v)
    assert abs(free() - f0) < 100, (f0, free())
    g.run(0, 12, 100)
    g.run(12, 33, 100)
    for p, q in zip(out[0], (g.positions(True), g.velocities(), g.forces())):
        assert np.array_equal(p, q)


def test_tiles_off_behind_a_build_given_up():
    """a clump whose cells' candidates no build workgroup can hold: the build fails,
    the forces behind it do without tiles, and the next upload starts anew"""
    import ctypes
    from pairs_amd import md, native
    hip = ctypes.CDLL("libamdhip64.so")

    def free():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
        return a.value / 1e6
    rng = np.random.default_rng(11)
    m, a = 59, 1.06
    k = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    n = len(k)
    x = (k + 0.5 + rng.uniform(-0.08, 0.08, k.shape)) * a
    v = rng.standard_normal(k.shape)
    y = x.copy()
    y[:60000] = 26.0 + rng.uniform(0.0, 8.4, (60000, 3))
    g = md.LJSystem([(0.0, m * a)] * 3, particle_capacity=3 * n, send_capacity=2 * n, neighbor_capacity=256,
                    reneighbor_every=10)
    g.upload(x, v)
    g.run(0, 2, 100)
    first = g.forces()
    g.upload(y, v)
    g.exchange()
    g.borders()
    g.build_cell_lists()
    before = free()
    with pytest.raises(native.PairsHipError):
        g.build_neighbor_lists()
    assert free() > before + 100, (before, free())
    g.lennard_jones()
    g.upload(x, v)
    g.run(0, 2, 100)
    assert np.array_equal(first, g.forces())


def test_upload_without_room_for_tiles():
    """lists that take three quarters of the device's memory leave no room for their
    16-bit copies: the system is uploaded and runs all the same"""
    import ctypes
    from pairs_amd import md
    rng = np.random.default_rng(6)
    m, a = 59, 1.06
    k = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    n = len(k)
    x = (k + 0.5 + rng.uniform(-0.08, 0.08, k.shape)) * a
    v = rng.standard_normal(k.shape)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert md.nat.lib() and ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    out = []
    for ncap in (120, int(0.75 * free.value / (4 * 2 * n))):
        g = md.LJSystem([(0.0, m * a)] * 3, particle_capacity=2 * n, send_capacity=n, neighbor_capacity=ncap,
                        reneighbor_every=10)
        g.upload(x, v)
        g.run(0, 12, 100)
        out.append((g.positions(True), g.velocities(), g.forces()))
        del g
    for p, q in zip(*out):
        assert np.array_equal(p, q)


# a large system's steps behind a rebuild that overflowed and is repeated: the
# ghosts outgrow the send map, or a segment's tile outgrows what the build stages
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("what", ["send", "tile"])
def test_lj_tiles_behind_failed_rebuilds(what, half):
    from pairs_amd import md, native
    rng = np.random.default_rng(5)
    m, a = 59, 1.06
    k = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
    n = len(k)
    # (the third layer from each lower face straddles the ghost layer's edge)
    x = (k + 0.64 + rng.uniform(-0.08, 0.08, k.shape)) * a
    v = -(10.0 if what == "send" else 16.0) * np.sin(2.0 * np.pi * x / (m * a))  # towards the faces
    out = []
    for nt in (1, 2):
        t = np.arange(n, dtype=np.int32) % nt
        kw = dict(particle_capacity=3 * n, neighbor_capacity=300, half=half, ntypes=nt, reneighbor_every=10)
        g = md.LJSystem([(0.0, m * a)] * 3, send_capacity=n, **kw)
        g.upload(x, v, types=t)
        g.run(0, 1, 100)
        if what == "send":  # (room for the ghosts of the first rebuild, hardly more)
            ghosts = g.nghost
            g = md.LJSystem([(0.0, m * a)] * 3, send_capacity=ghosts + 64, **kw)
            g.upload(x, v, types=t)
        g.run(0, 37, 100)
        assert g.count(native.REBUILD_ROLLBACKS) > 0
        out.append([g.positions(True), g.velocities(), g.forces()])
    for p, q in zip(*out):
        assert np.array_equal(p, q)


# downloads come in blocks of 1 MiB: 43690 rows of three doubles, 131072 doubles, 262144 words
@pytest.mark.parametrize("n", [1, 43690, 43691, 87381, 131073, 262145])
def test_downloads_at_block_edges(n):
    from pairs_amd import dem, md
    rng = np.random.default_rng(n)
    L = 2.0 * n ** (1.0 / 3.0)
    x, v = rng.uniform(0.0, L, (n, 3)), rng.standard_normal((n, 3))
    t, fl = rng.integers(0, 3, n).astype(np.int32), rng.integers(0, 2, n).astype(np.int32) * 4
    g = md.LJSystem([(0.0, L)] * 3, particle_capacity=n, send_capacity=16, neighbor_capacity=16, ntypes=3)
    g.upload(x, v, types=t, flags=fl)
    assert np.array_equal(g.positions(), x) and np.array_equal(g.velocities(), v) and np.array_equal(g.types(), t)
    s = dem.DEMSystem((L, L, L), particle_capacity=n + 1, contact_capacity=4, send_capacity=16, cell_width=L / 4,
                      ncells_capacity=1000)
    r = rng.uniform(0.1, 0.2, n)
    s.add_spheres(np.arange(n) + 5, r, x, v)
    assert np.array_equal(s.get("position"), x) and np.array_equal(s.get("linear_velocity"), v)
    assert np.array_equal(s.get("uid"), np.arange(n) + 5) and np.array_equal(s.get("radius"), r)
