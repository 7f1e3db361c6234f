"""GPU parity of the reciprocal sums over the mesh (mesh.hip), which take over
from the ion-by-ion sums where they cost less, and the choice between the two
(read back from the kernel families that were timed).

Reference: the oracle for everything but the reciprocal terms (it is given no
reciprocal cells), plus the reciprocal sums term by term in numpy's FP64
(Potentials.f90:1428-2249 as matrix products).

Tolerance 1e-12 of the largest value: a phase 2 pi k.u carries a rounding of
2 pi K eps = 4e-14 at the largest K = 54 here in either sum, and 25 times that
covers the mesh's weights and the sums' order.
"""
import numpy as np
import pytest

from helpers import rel_maxnorm

pytestmark = pytest.mark.gpu
EPS = 0.00552635
TOL = 1e-12


def kcells(cell, kc):
    rec = 2 * np.pi * np.linalg.inv(cell).T
    vol = rec[0] @ np.cross(rec[1], rec[2])
    return [int(kc * np.linalg.norm(np.cross(rec[(a + 1) % 3], rec[(a + 2) % 3])) / vol + 0.5)
            for a in range(3)]


def reciprocal(pos, qs, cell, K, kc, sigma):
    """(energy, forces, absolute-position virial, field subtracted from chi)."""
    inv = np.linalg.inv(cell)
    b = 2 * np.pi * inv.T
    u = pos @ inv
    k = [np.arange(-K[0], K[0] + 1), np.arange(-K[1], K[1] + 1), np.arange(0, K[2] + 1)]
    ex = []
    for a in range(3):
        ph = u[:, a:a + 1] * k[a]
        ex.append(np.exp(2j * np.pi * (ph - np.rint(ph))))
    inv2v = 1.0 / (2.0 * abs(np.linalg.det(cell)) * EPS)
    n = len(pos)
    energy, field, grad = 0.0, np.zeros(n), np.zeros((n, 3))
    for a, k1 in enumerate(k[0]):
        kv = (k1 * b[0] + k[1][:, None, None] * b[1] + k[2][None, :, None] * b[2])
        k2 = (kv * kv).sum(2)
        on = (k2 < kc * kc) & (k2 > 0)
        w = np.where(k[2] == 0, 1.0, 2.0)[None, :]
        c = np.where(on, inv2v * w * np.exp(-sigma ** 2 * k2 / 2) / np.where(on, k2, 1.0), 0.0)
        e12 = ex[0][:, a:a + 1] * ex[1]
        s = (qs[:, None] * e12).T @ ex[2]
        energy += float((c * np.abs(s) ** 2).sum())
        z = 2.0 * c * s
        back = ex[2].conj()

        def at(y):
            return ((back @ y.T) * e12.conj()).sum(1)
        field += at(z).real
        for d in range(3):
            grad[:, d] += (at(z * kv[..., d]) * -1j).real
    f = -qs[:, None] * grad
    st = np.array([pos[:, x] @ f[:, y] for x, y in
                   ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2), (0, 1))])
    return energy, f, st, field


def ions(case):
    rng = np.random.default_rng(case["seed"])
    n = case["n"]
    u = rng.random((n, 3))
    # a jittered lattice of distinct sites, so that no two ions coincide
    m = int(np.ceil(n ** (1 / 3)))
    site = np.array([(i, j, k) for i in range(m) for j in range(m) for k in range(m)])[:n]
    u = (site + 0.5 + 0.3 * (u - 0.5)) / m * np.array(case.get("part", (1.0, 1.0, 1.0)))
    u += rng.integers(-case.get("out", 0), case.get("out", 0) + 1, (n, 3))
    cell = np.array(case["cell"], dtype=float)
    if cell.ndim == 1:
        cell = np.diag(cell)
    q = rng.choice([-1.0, 1.0], n) * rng.uniform(0.5, 2.0, n)
    scaler = rng.uniform(0.5, 1.5, n) if case.get("scaled") else None
    return u @ cell, q, cell, scaler


CASES = [
    # a cube, K = 29: tiles of 128 x 120 x 120 points
    dict(n=3000, cell=(36.0, 36.0, 36.0), kc=5.0, seed=1),
    # three different axes, K = 48, 24, 12, more ions than one chunk per tile
    dict(n=9000, cell=(60.0, 30.0, 15.0), kc=5.0, seed=2),
    # sheared, ions up to three cells outside, scaled charges that do not cancel
    dict(n=3500, cell=((36.0, 0.0, 0.0), (9.0, 34.0, 0.0), (-7.0, 5.0, 33.0)), kc=5.2, seed=3,
         out=3, scaled=True),
    # everything in one corner: empty tiles and crowded ones
    dict(n=3001, cell=(40.0, 40.0, 40.0), part=(0.3, 0.35, 0.4), kc=4.6, seed=4),
    # a flat cell: the smallest mesh an axis can have (24 points)
    dict(n=8000, cell=(68.0, 64.0, 7.0), kc=5.0, seed=5),
    # some 45 ions in each tile of a corner, none in the others
    dict(n=12000, cell=(60.0, 60.0, 60.0), part=(0.3, 0.35, 0.4), kc=4.6, seed=6),
    # the sum has barely decayed at the mesh's band edge: 1.0e-4 there
    dict(n=3000, cell=(36.0, 36.0, 36.0), kc=5.0, seed=7, sigma=4.292 / 5.0),
]
# everything in one corner of a smaller cell: the crowded tiles cost more
DIRECT = {3}


def went_over_the_mesh(eng, call):
    """Whether the reciprocal sums of call() went over the mesh."""
    eng.timing(True)
    call()
    families = eng.timing_read()
    eng.timing(False)
    assert "ewald_sk" in families
    return "ewald_mesh_place" in families


@pytest.mark.parametrize("k", range(len(CASES)))
def test_mesh_matches_term_by_term(oracle, k):
    from pysic_amd.engine import Engine
    case = CASES[k]
    pos, q, cell, scaler = ions(case)
    n, kc, sigma, rc = len(pos), case["kc"], case.get("sigma", 1.2), 3.0
    K = kcells(cell, kc)
    print("mesh case %d: n=%d K=%s" % (k, n, K), flush=True)
    sp = np.zeros(n, np.int32)
    eng = Engine(0)
    eng.create_atoms(sp, pos, charges=q)
    eng.create_cell(cell)
    eng.set_potentials(np.zeros((0, 12)))
    eng.set_bond_order_factors(np.zeros((0, 14)))
    eng.set_ewald(rc, kc, K, sigma, EPS, scaler=scaler)
    eng.generate_neighbor_lists(np.full(n, rc + 0.2))
    nl = oracle.neighbor_list(pos, cell, [1, 1, 1], np.full(n, rc + 0.2))
    qs = q if scaler is None else q * scaler
    ew0 = [1, rc, kc, 0, 0, 0, sigma, EPS]
    none = np.zeros((0, 12))

    def reference(p):
        args = (sp, p, q, cell, nl, none, None, ew0, scaler)
        er, fr, sr, field = reciprocal(p, qs, cell, K, kc, sigma)
        f, s = oracle.evaluate("forces", *args)
        return (oracle.evaluate("energy", *args) + er, f + fr, s + sr,
                oracle.evaluate("enegs", *args) - field)

    def compare(p, order):
        e0, f0, s0, x0 = reference(p)
        for what in order:
            if what == "e":
                assert abs(eng.energy() - e0) <= TOL * abs(e0)
            elif what == "f":
                f, s = eng.forces()
                print("  forces %.1e" % rel_maxnorm(f, f0), flush=True)
                assert rel_maxnorm(f, f0) <= TOL
                # the virial sums n terms r F that may cancel
                assert np.abs(s - s0).max() <= TOL * np.abs(p).max() * np.abs(f0).sum()
            else:
                assert rel_maxnorm(eng.electronegativities(), x0) <= TOL

    compare(pos, "efx")
    # moved ions: nothing of the old places or structure factors is left
    moved = pos + np.random.default_rng(9).normal(0.0, 0.02, pos.shape)
    eng.update_coordinates(moved)
    compare(moved, "fex")
    assert went_over_the_mesh(eng, eng.electronegativities) == (k not in DIRECT)
    eng.close()


def test_relaxation_steps_over_the_mesh():
    """The relaxation keeps the ions' places on the mesh over its steps: its
    charges are those of the same steps driven from outside, where every
    electronegativity call places them again."""
    from pysic_amd.engine import Engine
    pos, _, cell, _ = ions(CASES[0])
    n = len(pos)
    pd = np.array([[2, 1, 0, 0, 10.0, 2.0, 0, 0, -1, 0, 0, 0]])
    eng = Engine(0)
    eng.create_atoms(np.zeros(n, np.int32), pos, charges=np.zeros(n))
    eng.create_cell(cell)
    eng.set_potentials(pd)
    eng.set_bond_order_factors(np.zeros((0, 14)))
    eng.set_ewald(3.0, 5.0, kcells(cell, 5.0), 1.2, EPS)
    eng.generate_neighbor_lists(np.full(n, 3.2))
    q0 = np.random.default_rng(3).normal(0.0, 0.1, n)
    dt, fr = 0.02, 4.0
    got, rate, steps, _ = eng.relax_charges(q0, np.zeros(n), 4, dt, 1.0, fr, 1e-14)
    assert steps == 4
    q, v = q0.copy(), np.zeros(n)

    def force():
        eng.update_charges(q)
        x = eng.electronegativities()
        return x - x.mean()
    f = force()
    for _ in range(4):
        q = q + v * dt + (f - fr * v) * dt * dt
        v = (1 - 0.5 * fr * dt) * v + 0.5 * f * dt
        f = force()
        v = (v + 0.5 * f * dt) / (1 + 0.5 * fr * dt)
    assert rel_maxnorm(got, q) <= TOL and rel_maxnorm(rate, v) <= TOL
    assert went_over_the_mesh(eng, eng.electronegativities)
    eng.close()


def _engine(pos, q, cell, kc, sigma=1.2, rc=3.0):
    from pysic_amd.engine import Engine
    n = len(pos)
    eng = Engine(0)
    eng.create_atoms(np.zeros(n, np.int32), pos, charges=q)
    eng.create_cell(cell)
    eng.set_potentials(np.zeros((0, 12)))
    eng.set_bond_order_factors(np.zeros((0, 14)))
    eng.set_ewald(rc, kc, kcells(cell, kc), sigma, EPS)
    eng.generate_neighbor_lists(np.full(n, rc + 0.2))
    return eng


def _new_cell(eng, pos, cell, kc, sigma=1.2, rc=3.0):
    eng.create_cell(cell)
    eng.set_ewald(rc, kc, kcells(cell, kc), sigma, EPS)
    eng.update_coordinates(pos)
    eng.generate_neighbor_lists(np.full(len(pos), rc + 0.2))


def test_forces_of_long_waves():
    """Forces of disordered ions whose sum has decayed far inside the mesh's
    band, so that the longest waves carry them, against the same terms in
    extended precision.  Bound: along one axis of n = 120 points the derivative
    of the wave k = 1 is off by 1.1e-15 of it by the kernel's tail (2.6e-18 in
    its transform) and by n / (2 pi) / 2 eps / 2 = 1.0e-15 by the rounding of
    products that cancel: 1.5e-15; the other two components of its gradient,
    which vanish, by as much: sqrt(3) of it, 2.6e-15, for the longest wave and
    less for the others.  (A kernel of a tail of 1.8e-17 gave 8.4e-15.)"""
    n, edge, kc = 3000, 36.0, 5.0
    pos, q = _ions_of(n, (edge,) * 3, (1, 1, 1))
    q -= q.mean()
    sigma = 27.0 / kc     # 1e-18 at a third of the band
    eng = _engine(pos, q, np.eye(3) * edge, kc, sigma, 1e-3)
    f = eng.forces()[0]
    assert went_over_the_mesh(eng, eng.electronegativities)
    eng.close()
    ld = np.longdouble
    pi, K = 4 * np.arctan(ld(1)), 10
    b = 2 * pi / ld(edge)
    k = [np.arange(-K, K + 1), np.arange(-K, K + 1), np.arange(0, K + 1)]
    ex = []
    for a in range(3):
        turn = (pos[:, a].astype(ld) / ld(edge))[:, None] * k[a]
        ex.append(np.exp(2j * pi * (turn - np.rint(turn))))
    want = np.zeros((n, 3), ld)
    for x, k1 in enumerate(k[0]):
        k2 = b * b * (k1 * k1 + k[1][:, None] ** 2 + k[2][None] ** 2)
        on = k2 > 0
        c = np.where(on, np.where(k[2] == 0, 1, 2)[None] * np.exp(-ld(sigma) ** 2 * k2 / 2) /
                     np.where(on, k2, 1), 0) / (2 * ld(edge) ** 3 * ld(EPS))
        e12 = ex[0][:, x:x + 1] * ex[1]
        z = 2 * c * np.einsum("ij,ik->jk", q[:, None] * e12, ex[2])
        at = np.einsum("ik,jk->ij", ex[2].conj(), z) * e12.conj()
        at3 = np.einsum("ik,jk->ij", ex[2].conj() * (k[2] * b), z) * e12.conj()
        for d, y in enumerate((at.sum(1) * (k1 * b), (at * (k[1] * b)).sum(1), at3.sum(1))):
            want[:, d] -= q * (y * -1j).real
    error = float(np.sqrt(((f - want) ** 2).sum() / (want ** 2).sum()))
    print("long waves: relative error %.2e" % error, flush=True)
    assert error <= 2.6e-15


def test_tables_follow_the_cell():
    """The transforms' tables are kept while the k-vector counts stay and
    shared by equal axes: over a strain, new counts, axes of other lengths and
    back, one handle gives what a new handle gives, bit for bit."""
    u = np.random.default_rng(4).permutation(ions(CASES[1])[0] / np.array(CASES[1]["cell"]))
    n = len(u)
    q = np.random.default_rng(5).choice([-1.0, 1.0], n)
    cube = np.eye(3) * 36.0
    strain = np.array([[1.001, 0.002, 0.0], [0.0, 0.999, 0.001], [0.0, 0.0, 1.0005]])
    eng, seen, way = None, set(), set()
    for k, cell in enumerate((cube, cube @ strain, cube @ strain @ strain, np.diag([60.0, 30.0, 15.0]),
                              np.diag([30.0, 15.0, 60.0]), cube * 0.9, cube)):
        pos = u @ cell
        seen.add(tuple(kcells(cell, 5.0)))
        print("cell %d K=%s" % (k, kcells(cell, 5.0)), flush=True)
        fresh = _engine(pos, q, cell, 5.0)
        if eng is None:
            eng = _engine(pos, q, cell, 5.0)
        else:
            _new_cell(eng, pos, cell, 5.0)
        for e in (eng, fresh):   # both from their own sorted order
            e.generate_neighbor_lists(np.full(n, 3.2))
        assert eng.energy() == fresh.energy()
        for a, b in zip(eng.forces(), fresh.forces()):
            assert np.array_equal(a, b)
        assert np.array_equal(eng.electronegativities(), fresh.electronegativities())
        way.add(went_over_the_mesh(eng, eng.electronegativities))
        fresh.close()
    assert len(seen) == 4   # the strained cubes have the cube's counts
    assert way == {True}
    eng.close()


def test_first_evaluation_in_a_new_cell_is_quick():
    """A strained cell with the same k-vector counts, as every step of a cell
    relaxation brings: its first evaluation takes at most 0.4 ms more than a
    repeated one (8,000 ions: 0.12; forming the tables again took 1.0)."""
    import time
    from pysic_amd import structures as st
    s = st.rocksalt((10, 10, 10), sigma=0.08, seed=3)
    eng = _engine(s.positions, s.charges, s.cell, 2.5713, 2.0443, 10.0)
    times = {True: [], False: []}
    for k in range(24):
        new = k % 2 == 0
        f = 1.0 + 1e-5 * (k % 7)
        t = time.perf_counter()
        if new:
            _new_cell(eng, s.positions * f, s.cell * f, 2.5713, 2.0443, 10.0)
        else:
            eng.update_coordinates(s.positions * f)
            eng.generate_neighbor_lists(np.full(len(s), 10.2))
        eng.energy()
        eng.forces()
        times[new].append(time.perf_counter() - t)
    assert went_over_the_mesh(eng, eng.electronegativities)
    extra = 1e6 * (np.median(times[True][2:]) - np.median(times[False][2:]))
    print("a new cell: %.0f us more" % extra, flush=True)
    assert extra <= 400.0
    eng.close()


# the choice: (ions, cell edges, part of the cell they fill, k_c, sigma, mesh)
CHOICE = [
    (8000, (56.4,) * 3, (1, 1, 1), 2.5713, 2.0443, True),
    (4096, (45.1,) * 3, (1, 1, 1), 2.5713, 2.0443, False),     # few pairs
    (500, (180.5,) * 3, (0.25, 0.25, 0.05), 2.5713, 2.0443, False),   # mesh for few ions
    (4000, (100.0,) * 3, (1, 1, 0.2), 2.5713, 2.0443, True),   # a slab worth its mesh
    (262144, (180.5,) * 3, (1, 1, 1), 0.5, 10.0, False),       # a thousand ions a tile
    (32000, (200.0,) * 3, (0.2, 0.2, 0.2), 1.3, 3.6, False),   # a particle: crowded tiles
    (32000, (200.0,) * 3, (1, 1, 1), 1.3, 3.6, True),          # the same ions spread out
    (8000, (56.4,) * 3, (1, 1, 1), 2.5713, 1.6, False),        # not decayed: 2e-4
]


def _ions_of(n, edge, part):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3) - 1e-9))
    site = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    u = (site + 0.5 + 0.3 * (rng.random((n, 3)) - 0.5)) / m * np.array(part)
    return u * np.array(edge), rng.choice([-1.0, 1.0], n)


@pytest.mark.parametrize("k", range(len(CHOICE)))
def test_the_cheaper_way_is_taken(k):
    n, edge, part, kc, sigma, mesh = CHOICE[k]
    print("choice %d: n=%d" % (k, n), flush=True)
    pos, q = _ions_of(n, edge, part)
    eng = _engine(pos, q, np.diag(edge), kc, sigma, 5.0)
    assert went_over_the_mesh(eng, eng.electronegativities) == mesh
    eng.close()


def test_one_handle_changes_its_way(oracle):
    """Through new cells and atom counts from the direct sums to the mesh and
    back, each time what a new handle gives, bit for bit; the reciprocal parts
    of a mesh and a direct evaluation against the sums term by term."""
    steps = [(2000, 30.0, False), (3000, 36.0, True), (2999, 36.0, True), (3000, 30.0, False),
             (1500, 36.0, False), (3000, 36.0, True)]
    eng = None
    for n, edge, mesh in steps:
        print("step n=%d edge=%g" % (n, edge), flush=True)
        pos, q = _ions_of(n, (edge,) * 3, (1, 1, 1))
        cell = np.eye(3) * edge
        fresh = _engine(pos, q, cell, 5.0)
        if eng is None:
            eng = _engine(pos, q, cell, 5.0)
        elif n != eng_n:
            eng.create_atoms(np.zeros(n, np.int32), pos, charges=q)
            _new_cell(eng, pos, cell, 5.0)
        else:
            eng.update_charges(q)
            _new_cell(eng, pos, cell, 5.0)
        eng_n = n
        for e in (eng, fresh):   # both from their own sorted order
            e.generate_neighbor_lists(np.full(n, 3.2))
        got = eng.energy(), eng.forces()[0], eng.electronegativities()
        want = fresh.energy(), fresh.forces()[0], fresh.electronegativities()
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
        assert went_over_the_mesh(eng, eng.electronegativities) == mesh
        nl = oracle.neighbor_list(pos, cell, [1, 1, 1], np.full(n, 3.2))
        args = (np.zeros(n, np.int32), pos, q, cell, nl, np.zeros((0, 12)), None,
                [1, 3.0, 5.0, 0, 0, 0, 1.2, EPS], None)
        er, fr, _, field = reciprocal(pos, q, cell, kcells(cell, 5.0), 5.0, 1.2)
        f, _ = oracle.evaluate("forces", *args)
        assert abs(got[0] - oracle.evaluate("energy", *args) - er) <= TOL * abs(got[0])
        assert rel_maxnorm(got[1], f + fr) <= TOL
        assert rel_maxnorm(got[2], oracle.evaluate("enegs", *args) - field) <= TOL
        fresh.close()
    eng.close()
