"""The pair kernel's block lists (cells wider than the cutoff sphere) against
the FP64 oracle: cells where a block is in reach through two images and where
it is not, cubic, orthorhombic and skewed, a last block of one atom, more
blocks in reach than a list holds, and separate LJ and Coulomb cutoffs.  FP64
sums of the same terms in another order agree to 1e-10 of their size; the fast
form keeps its stated 1e-3 internal units per insertion."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(cell, n_fw, species, cut, K):
    from graspa_amd import synth
    s = synth.build(n_fw=n_fw, L=float(cell[0]), species=(species,), seed=n_fw, K=K, cutoff=cut[0],
                    probs=dict(widom=1.0))
    s.cell = np.array([cell[0], 0.0, 0.0, cell[3], cell[1], 0.0, cell[4], cell[5], cell[2]], dtype=np.float64)
    s.fw_pos = s.fw_pos * np.array([1.0, cell[1] / cell[0], cell[2] / cell[0]])
    s.cut_coul = cut[1]
    s.eps = s.eps * 0.2
    if species == "methane":      # (small atoms: a framework this dense leaves no room otherwise)
        s.sig = s.sig * 0.5
    s.setup_ewald()
    return s


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("cell,n_fw,species,cut", [
    ((28.0, 28.0, 28.0, 0, 0, 0), 513, "CO2", (12.0, 12.0)),
    ((44.0, 30.0, 26.0, 0, 0, 0), 900, "CO2", (12.0, 12.0)),
    ((31.0, 33.0, 32.0, 4.0, -3.0, 2.5), 801, "N2", (12.0, 12.0)),
    ((48.0, 48.0, 48.0, 0, 0, 0), 2500, "CO2", (10.0, 12.0)),
    ((40.0, 40.0, 40.0, 0, 0, 0), 9000, "methane", (16.0, 16.0)),
])
def test_block_lists_match_oracle(engine_mod, form, cell, n_fw, species, cut):
    from oracle import binding as ob
    s = _system(cell, n_fw, species, cut, 10)
    n = 120
    o = ob.OracleSystem(s)
    _, skf, ska, _, _, _ = o.ewald_total()
    ref = ob.widom_records_to_numpy(o.widom_batch(1, ska, skf, seed=5, n_insert=n))
    print("widom blocks", form, cell, n_fw, cut, flush=True)
    box = engine_mod.Box(s, precision=engine_mod.GRASPA_FP64 if form == "fp64" else engine_mod.GRASPA_MIXED)
    box.init_ewald()
    intra, selfe = o.exclusion(1)
    res, _ = box.widom_batch(1, n, seed=5, excl=intra + selfe)
    got = engine_mod.widom_results_to_numpy(res)
    shaped = []
    for shape in ((12, 0, 0), (4, 1, 1)):      # the framework from memory; other workgroups
        box.set_eval_shape(*shape)
        shaped.append(engine_mod.widom_results_to_numpy(box.widom_batch(1, n, seed=5, excl=intra + selfe)[0]))
    box.close()
    assert ref["ok"].sum() > 20
    assert np.array_equal(got["ok"], ref["ok"])
    ok = ref["ok"] == 1
    assert np.array_equal(got["first_bead"][ok], ref["first_bead"][ok])
    assert np.array_equal(got["orientation"][ok], ref["orientation"][ok])
    err = np.abs(got["energy"][ok] - ref["energy"][ok])
    assert np.all(err <= (1e-8 + 1e-10 * np.abs(ref["energy"][ok]) if form == "fp64" else 1e-3)), err.max()
    for other in shaped:
        assert np.array_equal(got["energy"], other["energy"]) and np.array_equal(got["rosen"], other["rosen"])


def test_right_angled_form_with_entries_below_the_diagonal(engine_mod):
    """Cells are taken as right-angled when the entries above the diagonal
    (cell[3], cell[6], cell[7]) vanish, and images are then found from the
    diagonal alone, whatever the entries below it: the pair kernel finds the
    same images as the oracle in such a cell too (small atoms, so that no
    overlap screen decides a trial)."""
    from graspa_amd import synth
    from oracle import binding as ob
    s = synth.build(n_fw=300, L=30.0, species=("CO2",), seed=3, probs=dict(widom=1.0))
    s.eps, s.sig = s.eps * 0.1, s.sig * 0.3
    s.cell = np.array([30.0, 3.0, 0.0, 0.0, 30.0, 2.0, 0.0, 0.0, 30.0])
    n = 60
    o = ob.OracleSystem(s)
    _, skf, ska, _, _, _ = o.ewald_total()
    ref = ob.widom_records_to_numpy(o.widom_batch(1, ska, skf, seed=5, n_insert=n))
    print("widom blocks, entries below the diagonal", flush=True)
    box = engine_mod.Box(s, precision=engine_mod.GRASPA_FP64)
    box.init_ewald()
    intra, selfe = o.exclusion(1)
    got = engine_mod.widom_results_to_numpy(box.widom_batch(1, n, seed=5, excl=intra + selfe)[0])
    box.close()
    assert ref["ok"].sum() > 20
    assert np.array_equal(got["ok"], ref["ok"])
    ok = ref["ok"] == 1
    assert np.array_equal(got["first_bead"][ok], ref["first_bead"][ok])
    assert np.array_equal(got["orientation"][ok], ref["orientation"][ok])
    err = np.abs(got["energy"][ok] - ref["energy"][ok])
    assert np.all(err <= 1e-8 + 1e-10 * np.abs(ref["energy"][ok])), err.max()
