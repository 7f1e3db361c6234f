"""Per-atom arrays between host and device (transfer.hip): every row arrives,
bit for bit, in the caller's order, at the sizes where the way changes (the
small slots hold 10,922 rows of 3 or 32,768 scalars; the large ones 131,072
rows of 3 or 393,216 scalars, in chunks over several threads), and with
several handles moving data at once, and whatever the process sets as the
default kind of pinned memory."""
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 10922, 10923, 32768, 32769, 131072, 131073, 393217, 1000003]


def system(n, seed):
    """n atoms on a jittered lattice whose order is shuffled, so that the
    device's cell order is far from the caller's; charges alone interact."""
    from pysic_amd.engine import Engine
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3) - 1e-9))
    k = rng.permutation(m ** 3)[:n]
    site = np.stack([k % m, k // m % m, k // (m * m)], axis=1)
    pos = (site + 0.5 + rng.uniform(-0.2, 0.2, (n, 3))) * 3.0
    mom = rng.normal(size=(n, 3))
    e = Engine(0)
    e.create_atoms(np.zeros(n, np.int32), pos, charges=np.zeros(n), momenta=mom)
    e.create_cell(np.eye(3) * max(3.0 * m, 9.0))
    # E = q^2: chi = -2 q exactly
    e.set_potentials(np.array([[2, 1, 0, 0, 1.0, 2.0, 0, 0, -1, 0, 0, 0]]))
    e.set_bond_order_factors(np.zeros((0, 14)))
    e.ewald_off()
    e.generate_neighbor_lists(np.full(n, 1.0))
    return e, pos, mom, rng


def roundtrip(n, seed):
    e, pos, mom, rng = system(n, seed)
    got = e.state()
    assert np.array_equal(got[0], pos) and np.array_equal(got[1], mom)
    moved = pos + 0.25
    e.update_coordinates(moved)              # momenta kept
    got = e.state()
    assert np.array_equal(got[0], moved) and np.array_equal(got[1], mom)
    e.update_coordinates(pos, 2.0 * mom)
    got = e.state()
    assert np.array_equal(got[0], pos) and np.array_equal(got[1], 2.0 * mom)
    for _ in range(3):                       # uploads in a row share two slots
        q = rng.normal(size=n)
        e.update_charges(q)
    assert np.array_equal(e.electronegativities(), -2.0 * q)
    assert abs(e.energy() - float((q * q).sum())) <= 1e-12 * n * float((q * q).max())
    f, w = e.forces()
    assert not f.any() and not w.any()
    e.close()


@pytest.mark.parametrize("n", SIZES)
def test_roundtrip(n):
    roundtrip(n, n)


def test_handles_on_several_threads():
    failed = []

    def work(k):
        try:
            for n in (5000, 140000, 12000):
                roundtrip(n + k, 100 * k)
        except BaseException as exc:   # reported below, with the thread's number
            failed.append((k, repr(exc)))
    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed


@pytest.mark.parametrize("coherent", ["0", "1"])
def test_default_kind_of_pinned_memory(coherent):
    """The rows of the large downloads and the errors that end a relaxation
    are read after events: they need coherent memory, also in a process
    whose default is the other kind."""
    code = """
import numpy as np
import test_gpu_small_systems as small
import test_gpu_transfer as t
t.roundtrip(1000003, 3)
print("rows arrive", flush=True)
eng = small.Engine(0)
q0, v0 = small._relaxation_case(eng, 1500)
q, v, steps, err, errs = small._driven(eng, q0, v0, 200, 0.05, 4.0, 1e-6)
for _ in range(3):
    got, rate, k, e = eng.relax_charges(q0, v0, 200, 0.05, 1.0, 4.0, 1e-6)
    assert k == steps and 3 < k < 200, (k, steps)
    assert abs(e - err) <= 1e-3 * abs(err) and np.abs(got - q).max() <= 1e-10
eng.close()
print("errors arrive", flush=True)
"""
    here = os.path.dirname(os.path.abspath(__file__))
    code = "import sys; sys.path[:0] = [%r, %r]\nfrom pysic_amd.engine import Engine\n" % (
        here, os.path.dirname(here)) + code.replace("small.Engine", "Engine")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=110,
                         env=dict(os.environ, HIP_HOST_COHERENT=coherent))
    assert out.returncode == 0, out.stdout + out.stderr
    assert "errors arrive" in out.stdout
