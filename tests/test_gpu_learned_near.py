"""Corrector stages over the neighbors kept by the descriptor pass.

An atom with up to 128 neighbors within the descriptor cutoff (6 A) reads
them from the kept rows, one with more walks its full list: SiO2 at 2.2
g/cm^3 has 47 to 72, at 4.6 114 to 133 (both kinds in one wave) and at 6.0
more than 150 (only the second).  One stage and four
stages against the oracle's (at the higher densities the trained stages diverge).

Tolerance: a stage's dq is a sum of FP32 Gaussians (2e-5 of the largest
feature, as the descriptors) times FP64 differences, so a stage is off by at
most 2e-5 of the largest change it and the stages before it make.
"""
import os
import sys

import numpy as np
import pytest

from conftest import ROOT

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import mlp_oracle as MO  # noqa: E402

from pysic_amd import structures as st  # noqa: E402

pytestmark = pytest.mark.gpu

MODEL = os.path.join(ROOT, "pysic_amd", "data", "sio2_eem_mlp.npz")


@pytest.mark.skipif(not os.path.exists(MODEL), reason="trained model not present")
@pytest.mark.parametrize("density", [2.2, 4.6, 6.0])
def test_stages_over_kept_and_full_rows(density):
    from pysic_amd.learned import ChargePredictor, DESC_ETA, DESC_MU, DESC_RC, EEMSystem, SPECIES
    from test_gpu_learned import _oracle_chi_setup
    print("case: kept neighbors density=%g" % density, flush=True)
    p = ChargePredictor.load(MODEL, 0)
    eem = EEMSystem(0)
    s = st.amorphous_sio2(96, density, 5)
    n = len(s)
    sp = np.array([SPECIES.index(x) for x in s.symbols], np.int32)
    eem.load(s)
    f, _ = p.descriptors(eem.eng)
    ref = MO.descriptors(s.positions, s.cell, [True] * 3, sp, 2, DESC_RC, DESC_MU, DESC_ETA)
    assert np.abs(f[:, :ref.shape[1]] - ref).max() <= 2e-5 * np.abs(ref).max()
    q = p.warm_start(eem.eng, 0)
    chi_of, _ = _oracle_chi_setup(s)
    d, moved = np.zeros(n), 0.0
    for k, c in enumerate(p.corrector):
        dq = MO.corrector_stage(s.positions, s.cell, [True] * 3, sp, DESC_RC, DESC_MU, DESC_ETA,
                                chi_of(q), d, c)
        q, d, moved = q + dq, dq, moved + np.abs(dq).max()
        if k in (0, 3):
            err = np.abs(p.warm_start(eem.eng, k + 1) - q).max()
            print("  stages %d: |q - q_oracle| max %.2e of %.2e" % (k + 1, err, moved), flush=True)
            assert err <= 2e-5 * moved
    eem.close()
    p.close()
