"""Edges of the COMB kernels' work split against the oracle (FP64 on both
sides; the engine sums each pair from both ends, so results agree to
rounding: 1e-9 relative, as the other COMB tests).

  * general pair kind: the entries within the cutoff, compacted 48 at a time
    in batches of 32 list rows: 12, 42, 54 and 134 of them per atom;
  * bond-order slots: 32 atoms a block, 16 of an atom's slots staged:
    2.2 g/cm^3 (about 7 slots) and 5.0 (about 16, many beyond the stage),
    atom counts around the block;
  * angle legs: only pairs that some row's angle can use, with a third
    species, legs of two different species and an asymmetric row.
"""
import numpy as np
import pytest

from helpers import assert_same_pairs, comb_charges, rel_maxnorm
from pysic_amd import structures as st
from pysic_amd.interactions import (Potential, ProductPotential, build_descriptors, comb_sio2)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from pysic_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


def check(eng, oracle, s, model, reach, q=None):
    names = sorted(set(s.symbols))
    pd, bd, _ = build_descriptors(model, {x: k for k, x in enumerate(names)})
    sp = np.array([names.index(x) for x in s.symbols], np.int32)
    n, cut = len(s), np.full(len(s), reach)
    eng.create_atoms(sp, s.positions, charges=q)
    eng.create_cell(s.cell, (True, True, True))
    eng.set_potentials(pd)
    eng.set_bond_order_factors(bd)
    eng.ewald_off()
    eng.generate_neighbor_lists(cut)
    nl = oracle.neighbor_list(s.positions, s.cell, [1, 1, 1], cut)
    assert_same_pairs(eng, nl)
    args = (sp, s.positions, q, s.cell, nl, pd, bd)
    e_ref = oracle.evaluate("energy", *args)
    f_ref, w_ref = oracle.evaluate("forces", *args)
    e = eng.energy()
    f, w = eng.forces()
    print("  n %d |dE|/N %.2e  rel|dF| %.2e  rel|dW| %.2e" % (
        n, abs(e - e_ref) / n, rel_maxnorm(f, f_ref), rel_maxnorm(w, w_ref)), flush=True)
    assert abs(e - e_ref) / n <= 1e-9 * max(1.0, abs(e_ref) / n)
    assert rel_maxnorm(f, f_ref) <= 1e-9
    assert rel_maxnorm(w, w_ref) <= 1e-9


@pytest.mark.parametrize("cutoff", [4.0, 6.0, 7.0, 9.2])
def test_general_pairs_within_the_cutoff(eng, oracle, cutoff):
    print("case: general pairs, cutoff %g" % cutoff, flush=True)
    s = st.fcc((4, 4, 4), a=5.26, sigma=0.05, seed=4)
    model = [ProductPotential([
        Potential("Buckingham", symbols=[["Ar", "Ar"]], parameters=[500.0, 5e3, 0.35],
                  cutoff=cutoff, cutoff_margin=0.5),
        Potential("power", symbols=[["Ar", "Ar"]], parameters=[1.0, 4.0, 0.5])])]
    check(eng, oracle, s, model, 9.7)


@pytest.mark.parametrize("n_si,density", [(8, 2.2), (11, 2.2), (21, 5.0), (43, 5.0)])
def test_bond_order_slots(eng, oracle, n_si, density):
    print("case: bond-order slots, %d Si at %g" % (n_si, density), flush=True)
    s = st.amorphous_sio2(n_si, density, seed=12)
    check(eng, oracle, s, comb_sio2(), 3.55, comb_charges(s.symbols, seed=5))


@pytest.mark.parametrize("rows", [[["Si", "O", "Si"]], [["Si", "O", "Ar"]],
                                  [["Si", "O", "Ar"], ["O", "O", "Si"], ["O", "Ar", "O"]]])
def test_angle_legs(eng, oracle, rows):
    print("case: angle legs %s" % rows, flush=True)
    s = st.random_mixture(350, 17.0, 1.7, ["Si", "O", "Ar", "O"], seed=8)
    model = [Potential("bond_bend", symbols=[r], cutoff=3.0 + 0.2 * k, cutoff_margin=0.5,
                       parameters=[1.0 + k, 1.8 + 0.2 * k, 1 + k % 2, 2])
             for k, r in enumerate(rows)]
    check(eng, oracle, s, model, 4.0, np.zeros(len(s)))


def test_streams_beside_the_main_one():
    """A handle's third evaluation, or its dynamics, put the angles and the
    bond-order pairs on streams of their own: the same bits before and after,
    and with the kernels timed, where all is serial again."""
    from pysic_amd.engine import Engine
    s = st.amorphous_sio2(200, 2.2, seed=8)
    st.maxwell_boltzmann(s, 300.0, 5)
    q = comb_charges(s.symbols, 9)
    n = len(s)
    pd, bd, _ = build_descriptors(comb_sio2(), {"O": 0, "Si": 1})
    sp = np.array([("O", "Si").index(x) for x in s.symbols], np.int32)

    def handle():
        e = Engine(0)
        e.create_atoms(sp, s.positions, masses=s.masses, charges=q, momenta=s.momenta)
        e.create_cell(s.cell, (True, True, True))
        e.set_potentials(pd)
        e.set_bond_order_factors(bd)
        e.ewald_off()
        e.set_neighbor_capacity(48)
        e.generate_neighbor_lists(np.full(n, 3.55))
        return e

    a, b = handle(), handle()
    first = a.energy(), a.forces()                       # serial
    for timed in (False, False, True, False):            # streams
        a.timing(timed)
        again = a.energy(), a.forces()
        assert again[0] == first[0]
        assert all(np.array_equal(x, y) for x, y in zip(again[1], first[1]))
    # dynamics of a handle that has evaluated and of one that has not
    for e in (a, b):
        e.md_run(6, 0.02, rebuild=1)
    for x, y in zip(a.state(), b.state()):
        assert np.array_equal(x, y)
    for e in (a, b):
        e.md_run(5, 0.02, rebuild=2)                     # eager steps
    for x, y in zip(a.state(), b.state()):
        assert np.array_equal(x, y)
    a.close()
    b.close()
