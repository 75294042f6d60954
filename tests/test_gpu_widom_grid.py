"""The screening grid of a Widom batch (one workgroup per CU down to eight
insertions each, whole wave steps above): batches at the edges of its rules
give, insertion by insertion, the records of one large batch bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("rosen", "energy", "vdw", "real", "ewald", "first_bead", "orientation", "ok")


@pytest.fixture(scope="module")
def whole(engine_mod):
    from graspa_amd import synth
    s = synth.config1(n_fw=500)
    box = engine_mod.Box(s, precision=engine_mod.GRASPA_MIXED)
    box.init_ewald()
    intra, selfe = engine_mod.exclusion_energy(s, 1)
    res, _ = box.widom_batch(1, 100000, seed=19, excl=intra + selfe)
    yield box, intra + selfe, engine_mod.widom_results_to_numpy(res)
    box.close()


@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 2047, 2048, 2049, 6145, 98304, 98305])
def test_batches_of_any_size_give_the_same_records(engine_mod, whole, n):
    box, excl, ref = whole
    print("widom grid", n, flush=True)
    res, summ = box.widom_batch(1, n, seed=19, first_index=100000 - n, excl=excl)
    got = engine_mod.widom_results_to_numpy(res)
    assert summ.n == n and summ.n_ok == ref["ok"][100000 - n:].sum()
    for k in FIELDS:
        assert np.array_equal(got[k], ref[k][100000 - n:]), k
