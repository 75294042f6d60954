"""The pair kernel's block lists (cells wider than the cutoff sphere) against
the FP64 oracle, in each case after checking that the box took them or not:
cells where a block is in reach through two images and where it is not, cubic,
orthorhombic and skewed, a last block of one atom, more blocks in reach than a
list holds, separate LJ and Coulomb cutoffs, guests in LDS and in memory.  FP64
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


def _check(engine_mod, form, s, cut, lists, n=120):
    """n insertions against the oracle; `lists`: whether the box takes block lists."""
    from oracle import binding as ob
    o = ob.OracleSystem(s)
    _, skf, ska, _, _, _ = o.ewald_total()
    ref = ob.widom_records_to_numpy(o.widom_batch(1, ska, skf, seed=5, n_insert=n))
    print("widom blocks", form, list(s.cell), len(s.fw_type), cut, flush=True)
    box = engine_mod.Box(s, precision=engine_mod.GRASPA_FP64 if form == "fp64" else engine_mod.GRASPA_MIXED, capacity=256)
    box.init_ewald()
    intra, selfe = o.exclusion(1)
    box.timing_enable("widom_list")
    res, _ = box.widom_batch(1, n, seed=5, excl=intra + selfe)
    launches = box.timing_read()[1]
    box.timing_enable("widom_list", False)
    assert (launches > 0) == lists, launches
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


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("cell,n_fw,species,cut,share", [
    ((28.0, 28.0, 28.0, 0, 0, 0), 513, "CO2", (12.0, 12.0), 1.02),
    ((44.0, 30.0, 26.0, 0, 0, 0), 900, "CO2", (12.0, 12.0), 0.63),
    ((31.0, 33.0, 32.0, 4.0, -3.0, 2.5), 801, "N2", (12.0, 12.0), 0.70),
    ((48.0, 48.0, 48.0, 0, 0, 0), 2500, "CO2", (10.0, 12.0), 0.21),
    ((40.0, 40.0, 40.0, 0, 0, 0), 9000, "methane", (16.0, 16.0), 0.46),
])
def test_block_lists_match_oracle(engine_mod, form, cell, n_fw, species, cut, share):
    """`share`: the mean share of the cell within reach of a block.  The FP64
    form takes lists in all of these cells, the fast form under 0.42."""
    _check(engine_mod, form, _system(cell, n_fw, species, cut, 10), cut, form == "fp64" or share < 0.42)


@pytest.mark.parametrize("form", ["fp64", "mixed"])
@pytest.mark.parametrize("cell,n_fw,species,cut,n_guest", [
    # a block in reach through two images of the short axis, guests in LDS (share 0.37)
    ((44.0, 40.0, 27.0, 0, 0, 0), 3000, "CO2", (12.0, 12.0), 60),
    # more than 512 guest atoms: read from memory
    ((44.0, 40.0, 27.0, 0, 0, 0), 3000, "CO2", (12.0, 12.0), 180),
    # skewed, two images, the larger cutoff the LJ one (share 0.43)
    ((36.0, 33.0, 34.0, 4.0, -3.0, 2.5), 3001, "N2", (12.0, 11.0), 20),
    # about 240 of 875 blocks in reach: more than a list holds (share 0.28)
    ((48.0, 48.0, 48.0, 0, 0, 0), 14000, "methane", (16.0, 16.0), 5),
])
def test_block_lists_of_both_forms_match_oracle(engine_mod, form, cell, n_fw, species, cut, n_guest):
    """Cells in which both forms take lists, with guest molecules (on a
    lattice, turned at random)."""
    s = _system(cell, n_fw, species, cut, 10)
    rng = np.random.default_rng(n_fw + n_guest)
    c = s.components[0]
    grid = np.stack(np.meshgrid(*[np.arange(int(x // 5.0)) for x in cell[:3]], indexing="ij"), -1).reshape(-1, 3) * 5.0
    at = grid[rng.permutation(len(grid))[:n_guest]] + 2.0
    assert len(at) == n_guest
    rel = np.asarray(c.template_pos) - np.asarray(c.template_pos)[0]
    turn = np.stack([np.linalg.qr(rng.normal(size=(3, 3)))[0] for _ in range(n_guest)])
    c.init_pos = (at[:, None, :] + np.einsum("nij,aj->nai", turn, rel)).reshape(-1, 3)
    c.init_molid = np.repeat(np.arange(n_guest), c.molsize).astype(np.int64)
    _check(engine_mod, form, s, cut, True)


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
