"""The finish kernel of the Widom pipeline (orientation selection and Fourier
term, four insertions per wave; one per wave for molecules of more than four
sites) against the FP64 oracle for every molecule size it is built for, more
orientations than a 16-lane row holds, and cells whose k-vectors fill less and
more than one chunk of 64 rows.  Both sides are FP64 sums of the same terms in
other orders, so energies agree to 1e-10 of their size as everywhere in these
tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _species(m):
    """A rigid charged chain of m sites, 1.1 A apart, neutral for m > 1."""
    q = np.linspace(-0.4, 0.4, m) if m > 1 else np.array([0.3])
    return dict(name="rod%d" % m, names=["r%d_%d" % (m, i) for i in range(m)], eps=[60.0 + i for i in range(m)],
                sig=[2.9] * m, charge=[float(x) for x in q], mass=[10.0] * m,
                atoms=[(i, (0.1 * i * i, 0.0, 1.1 * i)) for i in range(m)])


@pytest.mark.parametrize("m,K,O,L,n_fw,n", [(1, 10, 10, 24.0, 400, 200), (2, 10, 20, 24.0, 400, 200),
                                            (3, 7, 16, 24.0, 400, 300), (4, 10, 17, 34.0, 900, 150),
                                            (5, 16, 12, 24.0, 300, 150), (8, 5, 9, 24.0, 300, 200)])
def test_finish_matches_oracle(engine_mod, monkeypatch, m, K, O, L, n_fw, n):
    from graspa_amd import synth
    from oracle import binding as ob
    monkeypatch.setitem(synth.SPECIES, "rod", lambda: _species(m))
    s = synth.build(n_fw=n_fw, L=L, species=("rod",), seed=m, K=K, O=O, probs=dict(widom=1.0))
    o = ob.OracleSystem(s)
    _, skf, ska, _, _, _ = o.ewald_total()
    ref = ob.widom_records_to_numpy(o.widom_batch(1, ska, skf, seed=5, n_insert=n))
    print("widom finish", m, K, O, L, flush=True)
    box = engine_mod.Box(s, precision=engine_mod.GRASPA_FP64)
    box.init_ewald()
    intra, selfe = o.exclusion(1)
    res, _ = box.widom_batch(1, n, seed=5, excl=intra + selfe)
    got = engine_mod.widom_results_to_numpy(res)
    box.close()
    assert ref["ok"].sum() > 5
    assert np.array_equal(got["ok"], ref["ok"])
    ok = ref["ok"] == 1
    assert np.array_equal(got["first_bead"][ok], ref["first_bead"][ok])
    assert np.array_equal(got["orientation"][ok], ref["orientation"][ok])
    for k in ("energy", "ewald"):
        err = np.abs(got[k][ok] - ref[k][ok])
        assert np.all(err <= 1e-8 + 1e-10 * np.abs(ref[k][ok])), (k, err.max())
