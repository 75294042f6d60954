"""Whole-box energies (a workgroup per guest atom, 256 threads over the atoms)
against the FP64 oracle: no guests at all, one molecule, atom counts on both
sides of the 256-thread stride, one- and two-species boxes.  Both sides sum
the same FP64 terms in different orders: n terms of size up to E lose at most
n * 1.1e-16 relative to the sum of their magnitudes, far below 1e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_fw,n_mol,species", [(255, 0, ("CO2",)), (256, 1, ("CO2",)), (257, 9, ("CO2", "N2")),
                                                (600, 30, ("CO2", "methane"))])
def test_totals_match_oracle(engine_mod, n_fw, n_mol, species):
    from graspa_amd import synth
    from oracle.binding import OracleSystem
    s = synth.build(n_fw=n_fw, L=26.0, species=species, seed=n_fw + n_mol)
    rng = np.random.default_rng(n_mol)
    grid = np.stack(np.meshgrid(*[np.arange(5)] * 3, indexing="ij"), -1).reshape(-1, 3) * 5.0 + 1.0
    pick = rng.permutation(len(grid))
    for i, c in enumerate(s.components):
        if n_mol:
            at = grid[pick[i * n_mol:(i + 1) * n_mol]]
            rel = np.asarray(c.template_pos) - np.asarray(c.template_pos)[0]
            c.init_pos = (at[:, None, :] + rel[None]).reshape(-1, 3)
            c.init_molid = np.repeat(np.arange(n_mol), c.molsize).astype(np.int64)
    print("totals", n_fw, n_mol, species, flush=True)
    box = engine_mod.Box(s, precision=engine_mod.GRASPA_FP64, capacity=64)
    f = box.init_ewald()
    e = box.total_energy()
    o = OracleSystem(s)
    ref = o.total_vdw_real()
    four = o.ewald_total()[0]
    box.close()
    for k in ("hg_vdw", "hg_real", "gg_vdw", "gg_real"):
        assert abs(getattr(e, k) - getattr(ref, k)) <= 1e-9 + 1e-10 * abs(getattr(ref, k)), k
    for k in ("gg_ewald", "hh_ewald", "hg_ewald"):
        assert abs(getattr(e, k) - getattr(four, k)) <= 1e-9 + 1e-10 * abs(getattr(four, k)), k
        assert abs(getattr(f, k) - getattr(four, k)) <= 1e-9 + 1e-10 * abs(getattr(four, k)), k


def test_totals_of_a_left_handed_cell(engine_mod):
    """A cell of negative volume has k-vectors inside the reciprocal cutoff but
    none with a coefficient the kernels use: the pair sums are the oracle's,
    the Fourier sums those of the structure-factor build."""
    from graspa_amd import synth
    from oracle.binding import OracleSystem
    s = synth.build(n_fw=300, L=26.0, species=("CO2",), seed=8)
    c = s.components[0]
    at = np.array([[4.0, 4.0, 4.0], [13.0, 13.0, 13.0], [20.0, 9.0, 17.0]])
    rel = np.asarray(c.template_pos) - np.asarray(c.template_pos)[0]
    c.init_pos = (at[:, None, :] + rel[None]).reshape(-1, 3)
    c.init_molid = np.repeat(np.arange(3), c.molsize).astype(np.int64)
    s.cell = s.cell * np.array([1.0] * 8 + [-1.0])
    print("totals, left-handed cell", flush=True)
    box = engine_mod.Box(s, precision=engine_mod.GRASPA_FP64, capacity=64)
    f = box.init_ewald()
    e = box.total_energy()
    ref = OracleSystem(s).total_vdw_real()
    box.close()
    for k in ("hg_vdw", "hg_real", "gg_vdw", "gg_real"):
        assert abs(getattr(e, k) - getattr(ref, k)) <= 1e-9 + 1e-10 * abs(getattr(ref, k)), k
    for k in ("gg_ewald", "hh_ewald", "hg_ewald"):
        assert getattr(e, k) == getattr(f, k), k
