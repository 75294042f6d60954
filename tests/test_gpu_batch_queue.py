"""The pair queue of the batched driver's FP64 form against the oracle's
trajectory: a skewed cell (no neighbour lists), separate LJ and Coulomb cutoffs
either way round, uncharged molecules, frameworks of less than one wave step,
one atom more, and more than the workgroup's 512 lanes, and frameworks that
leave no room for the queue in LDS or that LDS does not hold.  The same FP64
terms summed in another order: energy changes to 1e-10 of their size."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_fw,cell,species,cut", [
    (63, (25.0, 26.0, 25.5, 3.0, -2.0, 1.5), ("CO2", "N2"), (12.0, 12.0)),
    (65, (24.0, 24.0, 24.0, 0, 0, 0), ("CO2",), (11.0, 12.0)),
    (513, (36.0, 30.0, 26.0, 0, 0, 0), ("N2",), (12.0, 10.0)),
    (300, (27.0, 27.0, 27.0, 0, 0, 0), ("methane",), (12.0, 12.0)),
    # LDS holds the framework and the neighbour lists but no queue; the
    # framework alone; or lists and queue, the framework read from memory
    (3000, (56.0, 56.0, 56.0, 0, 0, 0), ("CO2",), (12.0, 12.0)),
    (3500, (56.0, 56.0, 56.0, 0, 0, 0), ("CO2",), (12.0, 12.0)),
    (3900, (56.0, 56.0, 56.0, 0, 0, 0), ("CO2",), (12.0, 12.0)),
    (3000, (56.0, 56.0, 56.0, 3.0, -2.0, 1.5), ("CO2",), (12.0, 12.0)),
])
def test_fp64_batch_matches_oracle(engine_mod, n_fw, cell, species, cut):
    from graspa_amd import synth
    from test_gpu_batch import ENERGY_KEYS, _engine_batch, _oracle_run, _same_sequence
    s = synth.build(n_fw=n_fw, L=cell[0], species=species, mol_fraction=[1.0 / len(species)] * len(species), seed=n_fw,
                    T=300.0, P=5e6, cycles=10, cutoff=cut[0],
                    probs=dict(translation=1.0, rotation=1.0, swap=2.0, reinsertion=1.0))
    s.cell = np.array([cell[0], 0.0, 0.0, cell[3], cell[1], 0.0, cell[4], cell[5], cell[2]], dtype=np.float64)
    s.fw_pos = s.fw_pos * np.array([1.0, cell[1] / cell[0], cell[2] / cell[0]])
    s.cut_coul = cut[1]
    s.setup_ewald()
    o, mc, otr = _oracle_run(s, seed=77, stream=3, cycles=8)
    boxes, bt, moves = _engine_batch(engine_mod, [s], [77], [3], 8, engine_mod.GRASPA_FP64)
    gtr = bt.trace(0)
    bt.close()
    assert moves == len(otr)
    _same_sequence(otr, gtr)
    assert sum(a.accepted for a in otr) > 5
    for i, (a, b) in enumerate(zip(otr, gtr)):
        for k in ENERGY_KEYS:
            x, y = getattr(a.de, k), getattr(b.de, k)
            assert abs(x - y) <= 1e-9 + 1e-10 * abs(x), (i, k, x, y)
