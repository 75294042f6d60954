"""Workloads of the GCMC energy engine, as its users' programs run them.

A case names one workload by plain values; :func:`prepare` builds the boxes a
program keeps (framework, guests, structure factors) from a seed,
:func:`run` makes one pass through the public entry points of
``graspa_amd.engine``, and :func:`exact` gives what the pass returns as plain
torch computes it in 64 bits.  The workloads:

  widom   batches of CBMC test insertions (Henry coefficients, chemical
          potentials), with the per-insertion records or the sums only
  graph   the same batch captured once and replayed
  gcmc    Monte Carlo cycles of one or many boxes on the device
  parity  Monte Carlo cycles in the reference's random-number order
  move    the energy calls of one trial move, as another program's Monte
          Carlo driver makes them
  totals  energies and structure factors of a whole box (set-up of a box, and
          the drift check at the end of a run)

Frameworks are jittered lattices (graspa_amd.synth).  Boxes that hold guests
have straight channels cut through the lattice, so that the molecules placed
there interact with the walls as adsorbed molecules do.
"""
import math

import numpy as np
import torch

from graspa_amd import deck, engine, synth

CUTOFF = 12.0
WALL = 3.0       # closest approach of a placed guest site to any other atom, A


def listed():
    return [
        # one trial move of a driver that calls the engine per move: the smallest calls, all latency
        dict(name="move-2304-fp64", op="move", n_fw=2304, cell="ortho", L=40.0, species="CO2", precision="fp64",
             n_guest=26),
        # a quick Henry estimate of one structure of a screening, records kept
        dict(name="widom-1000-open", op="widom", n_fw=750, cell="cubic", L=24.0, species="CO2", precision="mixed",
             n_guest=0, n_insert=1000, K=10, O=10, records=True),
        # the stated Widom workload: 100,000 CO2 insertions into the dense 1,536-atom framework, replayed
        dict(name="graph-100k-1536", op="graph", n_fw=1536, cell="cubic", L=24.0, species="CO2", precision="mixed",
             n_guest=0, n_insert=100000, K=10, O=10, replays=2),
        # its lower-density variant, where over a third of the constructions complete
        dict(name="widom-100k-750", op="widom", n_fw=750, cell="cubic", L=24.0, species="CO2", precision="mixed",
             n_guest=0, n_insert=100000, K=10, O=10, records=False),
        # the same framework class in the plain FP64 form (reference results)
        dict(name="widom-50k-1000-fp64", op="widom", n_fw=1000, cell="cubic", L=24.0, species="CO2",
             precision="fp64", n_guest=0, n_insert=50000, K=10, O=10, records=False),
        # chemical potential at loading in a zeolite-sized orthorhombic box, records kept
        dict(name="widom-20k-loaded", op="widom", n_fw=2304, cell="ortho", L=40.0, species="CO2", precision="mixed",
             n_guest=26, n_insert=20000, K=10, O=10, records=True),
        # a replicated framework (2 x 2 x 2 cells), far wider than the cutoff
        dict(name="widom-20k-6000", op="widom", n_fw=6000, cell="cubic", L=48.0, species="CO2", precision="mixed",
             n_guest=0, n_insert=20000, K=10, O=10, records=False),
        # a skewed cell, nitrogen (a massless charged centre), odd counts and trial numbers
        dict(name="widom-9999-skewed-n2", op="widom", n_fw=2999, cell="tri", L=31.0, species="N2", precision="mixed",
             n_guest=7, n_insert=9999, K=7, O=12, records=True),
        # one GCMC box in the plain FP64 form
        dict(name="gcmc-1-fp64", op="gcmc", n_fw=2304, cell="ortho", L=40.0, species="CO2", precision="fp64",
             n_guest=26, boxes=1, cycles=10, K=10, O=10),
        # many boxes of a mixture per launch, sizes and loadings spread
        dict(name="gcmc-64-mixture", op="gcmc", n_fw=3000, cell="cubic", L=38.0, species="CO2,N2", precision="mixed",
             n_guest=40, boxes=64, cycles=20, K=10, O=10),
        # GCMC in the reference's draw order, driven move by move from the host
        dict(name="parity-2304-fp64", op="parity", n_fw=2304, cell="ortho", L=40.0, species="CO2", precision="fp64",
             n_guest=26, cycles=5, K=10, O=10),
        # set-up and drift check of a large loaded box
        dict(name="totals-6000-loaded", op="totals", n_fw=6000, cell="cubic", L=48.0, species="CO2",
             precision="fp64", n_guest=240),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["widom"] * 5 + ["graph", "gcmc", "gcmc", "parity", "move", "totals"])
    cell = rng.choice(["cubic", "cubic", "ortho", "tri"])
    # the shortest width of the cell stays above twice the cutoff
    L = rng.uniform({"cubic": 24.0, "ortho": 37.0, "tri": 28.0}[cell], 46.0)
    volume = L ** 3 * {"cubic": 1.0, "ortho": 0.67, "tri": 0.92}[cell]
    loaded = op in ("gcmc", "parity", "move", "totals") or rng.random() < 0.4
    n_fw = int(volume * (rng.uniform(0.04, 0.06) if loaded else rng.uniform(0.045, 0.11)))
    c = dict(op=op, n_fw=n_fw, cell=cell, L=L, species=rng.choice(["CO2", "CO2", "N2", "CO2,N2"]),
             precision=rng.choice(["mixed", "mixed", "fp64"]), n_guest=0)
    if loaded:
        c["n_guest"] = max(1, int(volume * rng.uniform(0.0001, 0.0009)))
    if op in ("widom", "graph", "gcmc", "parity"):
        c.update(K=rng.randint(5, 16), O=rng.randint(5, 12))
    if op in ("widom", "graph"):
        most = 100000 * 1536 // n_fw // (4 if c["precision"] == "fp64" else 2)
        c.update(n_insert=_log(rng, 300, max(400, min(100000, most))))
        if op == "graph":
            c.update(replays=rng.randint(1, 3))
        else:
            c.update(records=rng.random() < 0.5)
    elif op == "gcmc":
        c.update(boxes=_log(rng, 1, 64), cycles=rng.randint(2, 10))
        if rng.random() < 0.25:
            # united-atom butane, uncharged, grown bead by bead
            c.update(species="butane", K=16, O=8)
    elif op == "parity":
        c.update(cycles=rng.randint(1, 5))
    return c


# --------------------------------------------------------------------------
# boxes
# --------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _cell(case):
    L = case["L"]
    if case["cell"] == "tri":
        return deck.cell_from_parameters(L, L, L, 82.0, 76.0, 86.0)
    lz = 0.67 * L if case["cell"] == "ortho" else L
    return np.array([L, 0.0, 0.0, 0.0, L, 0.0, 0.0, 0.0, lz])


def _channels(n_fw, cell, rng):
    """Fractional positions of n_fw atoms of a jittered lattice with straight
    channels along c (the n_fw lattice points farthest from the channel axes,
    about 70% of the lattice), and the channel axes."""
    H = cell.reshape(3, 3)                                     # rows a, b, c
    lengths = np.linalg.norm(H, axis=1)
    pitch = (abs(np.linalg.det(H)) * 0.7 / n_fw) ** (1.0 / 3.0)
    n = np.maximum(1, np.round(lengths / pitch)).astype(int)
    while n.prod() < n_fw:
        n[np.argmax(lengths / n)] += 1
    grid = np.stack(np.meshgrid(*[np.arange(k) for k in n], indexing="ij"), -1).reshape(-1, 3)
    f = (grid + 0.5) / n
    per = [max(1, int(round(lengths[d] / 24.0))) for d in (0, 1)]
    axes = np.array([((i + 0.5) / per[0], (j + 0.5) / per[1]) for i in range(per[0]) for j in range(per[1])])
    chat = H[2] / lengths[2]
    d = f[:, None, :2] - axes[None]
    d -= np.round(d)
    v = d @ H[:2]
    v -= (v @ chat)[..., None] * chat
    dist = np.linalg.norm(v, axis=-1).min(1) + rng.normal(0.0, 0.2, len(f))
    keep = np.sort(np.argsort(-dist, kind="stable")[:n_fw])
    jit = rng.normal(0.0, 0.2, (n_fw, 3)) @ np.linalg.inv(H)
    return np.mod(f[keep] + jit, 1.0), axes


def _rotation(rng):
    q = rng.normal(size=4)
    w, x, y, z = q / np.linalg.norm(q)
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)],
                     [2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)],
                     [2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)]])


def _nearest(sites, atoms, H):
    """Distance of each site (.., 3) to the nearest of the atoms, minimum image."""
    dev = _device()
    s = torch.as_tensor(sites, dtype=torch.float64, device=dev).reshape(-1, 1, 3)
    a = torch.as_tensor(atoms, dtype=torch.float64, device=dev).reshape(1, -1, 3)
    h = torch.as_tensor(H, dtype=torch.float64, device=dev)
    d = (s - a) @ torch.linalg.inv(h)
    d = (d - torch.round(d)) @ h
    return d.square().sum(-1).amin(1).sqrt().reshape(np.shape(sites)[:-1]).cpu().numpy()


def _place(template, n, fw, cell, axes, rng, others):
    """n molecules of the template (fewer where they do not fit) at random
    places about the channel axes, every site at least WALL from the framework
    and from other molecules; `others`: the sites placed before."""
    H = cell.reshape(3, 3)
    Hi = np.linalg.inv(H)
    taken = np.empty((len(others) + n * len(template), 3))
    taken[:len(others)] = others
    k = len(others)
    out = []
    rel = template - template[0]
    for _ in range(8):
        m = 4 * n + 64
        f = np.concatenate([axes[rng.integers(0, len(axes), m)], rng.random((m, 1))], 1)
        at = f @ H + rng.normal(0.0, 2.2, (m, 3))
        sites = np.stack([at[i] + rel @ _rotation(rng).T for i in range(m)])
        for i in np.nonzero(_nearest(sites, fw, H).min(1) > WALL)[0]:
            if len(out) == n:
                break
            if k:
                d = (sites[i][:, None, :] - taken[None, :k]) @ Hi
                d = (d - np.round(d)) @ H
                if (d * d).sum(-1).min() < WALL * WALL:
                    continue
            out.append(sites[i])
            taken[k:k + len(template)] = sites[i]
            k += len(template)
    return np.array(out).reshape(-1, len(template), 3), taken[:k]


def _system(case, seed, k=0):
    """System k of a case: force field and species from graspa_amd.synth, the
    framework and the guests' places from the seed."""
    rng = np.random.default_rng([int(seed), k, 77])
    species = case["species"].split(",")
    cell = _cell(case)
    butane = species == ["butane"]
    probs = dict(widom=1.0) if case["op"] in ("widom", "graph") else dict(translation=1.0, rotation=1.0, swap=2.0)
    if case["op"] in ("gcmc", "parity") and not butane:
        probs["reinsertion"] = 1.0
    fw_seed = int(rng.integers(1 << 30))
    s = synth.build(n_fw=case["n_fw"], L=case["L"], species=species, seed=fw_seed, T=300.0, P=3e5, cutoff=CUTOFF,
                    charges=not butane, K=case.get("K", 10), O=case.get("O", 10), probs=probs)
    H = cell.reshape(3, 3)
    s.cell = cell
    if case["n_guest"]:
        f, axes = _channels(case["n_fw"], cell, rng)
        s.fw_pos = f @ H
        # independent random charges of the full width bind molecules unlike any neutral wall does
        s.fw_charge = 0.5 * s.fw_charge
    else:
        s.fw_pos = np.mod(s.fw_pos / case["L"], 1.0) @ H
    if not butane:
        s.setup_ewald()
    got = np.empty((0, 3))
    for i, c in enumerate(s.components):
        n = case["n_guest"] // len(s.components) + (1 if i < case["n_guest"] % len(s.components) else 0)
        if not n:
            continue
        mol, got = _place(np.asarray(c.template_pos), n, s.fw_pos, cell, axes, rng, got)
        if len(mol):
            c.init_pos = mol.reshape(-1, 3)
            c.init_molid = np.repeat(np.arange(len(mol)), c.molsize).astype(np.int64)
    if butane:
        s.components[0].chain = synth.butane_chain()
        s.components[0].rigid = False
    return s


def _box_case(case, i):
    """Box i of a case of several boxes: cell edges 24 A up to L, framework
    atoms and guests by volume, spread from 60% to 140% of the case's."""
    if case["boxes"] == 1 or case["cell"] != "cubic":
        return case
    t = (0.5 + i) / case["boxes"]
    t2 = math.modf(i * 0.6180339887)[0]
    L = 24.0 + (case["L"] - 24.0) * t
    vol = (L / case["L"]) ** 3
    return dict(case, L=L, n_fw=int(case["n_fw"] * vol * (0.8 + 0.4 * t2)),
                n_guest=int(case["n_guest"] * vol * (0.6 + 0.8 * math.modf(t2 * 7.0)[0])))


def _precision(case):
    return engine.GRASPA_MIXED if case["precision"] == "mixed" else engine.GRASPA_FP64


def _box(case, seed, k=0, capacity=None):
    s = _system(case, seed, k)
    b = engine.Box(s, precision=_precision(case), capacity=capacity or max(64, 2 * case["n_guest"]))
    b.init_ewald()
    return s, b


# --------------------------------------------------------------------------
# passes
# --------------------------------------------------------------------------

def _proposals(case, s, seed, n=32):
    """Moves a driver proposes: a molecule, its displacement, K first-bead
    trials anywhere in the box and O orientations about a bead in a channel."""
    rng = np.random.default_rng([int(seed), 5])
    c = s.components[0]
    H = s.cell.reshape(3, 3)
    nm = len(c.init_pos) // c.molsize
    pos = np.asarray(c.init_pos).reshape(nm, c.molsize, 3)
    rel = np.asarray(c.template_pos)[1:] - np.asarray(c.template_pos)[0]
    out = []
    for _ in range(n):
        m = int(rng.integers(nm))
        shift = rng.uniform(-0.3, 0.3, 3)
        first = rng.random((10, 3)) @ H
        bead = pos[int(rng.integers(nm))][0] + np.array([0.0, 0.0, 4.0])
        orient = np.concatenate([bead + rel @ _rotation(rng).T for _ in range(10)])
        out.append((m, shift, first, orient))
    return out


def prepare(case, seed):
    op = case["op"]
    st = dict(case=case, seed=int(seed), passes=0)
    if op == "gcmc":
        boxes = []
        for i in range(case["boxes"]):
            bc = _box_case(case, i)
            boxes.append(_box(bc, seed, i, capacity=1024)[1])
        st["boxes"] = boxes
        st["batch"] = engine.Batch(boxes, [int(seed) + 1000 + i for i in range(len(boxes))])
        return st
    s, b = _box(case, seed, capacity=1024 if op == "parity" else None)
    st.update(system=s, box=b)
    if op in ("widom", "graph"):
        intra, selfe = engine.exclusion_energy(s, 1)
        st["excl"] = intra + selfe
        # the box's first batch makes what later batches of the framework use
        b.widom_batch(1, 64, seed=int(seed) + 2, excl=st["excl"], results=False)
        b.widom_totals(reset=True)
        if op == "graph":
            b.widom_graph(1, case["n_insert"], seed=int(seed), excl=st["excl"])
    elif op == "parity":
        s.seed = int(seed) & 0xffff
        st["mc"] = engine.MonteCarlo(b)
    elif op == "move":
        c = s.components[0]
        st["pos"] = np.asarray(c.init_pos).reshape(-1, c.molsize, 3).copy()
        st["proposals"] = _proposals(case, s, seed)
    return st


_SUMS = ("sum_w", "sum_w2", "sum_we", "n", "n_first_bead", "n_ok")
_RECORD = ("rosen", "energy", "vdw", "real", "ewald", "first_bead", "orientation", "ok")


def _energy(e):
    return np.array(list(e.as_dict().values()))


def _sums(summ):
    return {q: np.float64(getattr(summ, q)) for q in _SUMS}


def _positions(box, comp, rows):
    """A species' positions in an array of `rows` rows (zeros after the last atom)."""
    out = np.zeros((rows, 3))
    pos = box.get_molecules(comp)[0]
    out[:len(pos)] = pos
    return out


def run(st):
    case = st["case"]
    op, k = case["op"], st["passes"]
    st["passes"] = k + 1
    if op == "widom":
        n = case["n_insert"]
        res, summ = st["box"].widom_batch(1, n, seed=st["seed"], first_index=k * n, excl=st["excl"],
                                          results=case["records"])
        out = _sums(summ)
        if case["records"]:
            rec = engine.widom_results_to_numpy(res)
            out.update({q: rec[q] for q in _RECORD})
        return out
    if op == "graph":
        st["box"].widom_graph_launch(case["replays"])
        summ = st["box"].widom_totals(reset=True)
        return _sums(summ)
    if op == "gcmc":
        bt = st["batch"]
        moves = bt.run(case["cycles"], production=True)
        stats = [bt.stats(i) for i in range(bt.n)]
        out = dict(moves=moves, running=np.stack([_energy(x.running) for x in stats]),
                   n_mol=np.stack([x.n_mol for x in stats]), counters=np.stack([x.counters for x in stats]),
                   load=np.stack([x.load_sum for x in stats]))
        if bt.n == 1:
            # the configuration a program writes to its restart file
            bt.sync()
            for c in st["boxes"][0].comp_ids:
                out["pos%d" % c] = _positions(st["boxes"][0], c, 4096)
        return out
    if op == "parity":
        mc = st["mc"]
        moves, _ = mc.cycles(k * case["cycles"], case["cycles"])
        e, nm, cnt, _, _ = mc.stats()
        out = dict(moves=moves, running=_energy(e), n_mol=nm, counters=cnt)
        for c in st["box"].comp_ids:
            out["pos%d" % c] = _positions(st["box"], c, 4096)
        return out
    if op == "move":
        b, c = st["box"], st["system"].components[0]
        m, shift, first, orient = st["proposals"][k % len(st["proposals"])]
        old = st["pos"][m]
        new = old + shift
        e1, o1 = b.trial_energies(first, c.types[:1], c.charges[:1], len(first), self_comp=1, self_molid=m)
        e2, o2 = b.trial_energies(orient, c.types[1:], c.charges[1:], 10, self_comp=1, self_molid=m)
        de, ov = b.single_body_delta(1, m, old, new, c.types, c.charges)
        same, cross = b.ewald_delta(old, c.charges, new, c.charges)
        b.ewald_accept()
        b.commit_move(1, m, new)
        st["pos"][m] = new
        return dict(e1=e1, o1=o1, e2=e2, o2=o2, de=_energy(de), overlap=ov, same=np.float64(same),
                    cross=np.float64(cross))
    b = st["box"]
    fourier = b.init_ewald()
    total = b.total_energy()
    sk_fw, sk_ads = b.structure_factors()
    return dict(fourier=_energy(fourier), total=_energy(total), sk_fw=sk_fw, sk_ads=sk_ads)


# --------------------------------------------------------------------------
# work
# --------------------------------------------------------------------------

def _free_fraction(case):
    """Share of random first-bead positions that no framework atom overlaps."""
    s = _system(dict(case, n_guest=0) if case["op"] in ("widom", "graph") and not case["n_guest"] else case, 0)
    rng = np.random.default_rng(3)
    H = s.cell.reshape(3, 3)
    pts = rng.random((512, 3)) @ H
    t0 = int(s.components[0].types[0])
    r = np.array([0.475 * s.sig[t, t0] for t in range(3)])     # about where LJ passes OverlapCriteria
    dead = np.zeros(len(pts), bool)
    for t in range(3):
        at = s.fw_pos[s.fw_type == t]
        dead |= _nearest(pts, at, H) < r[t]
    return max(0.002, float(1.0 - dead.mean()))


def work(case):
    """Bytes: the box's atoms, structure factors and tables once, the results
    once.  FLOP: 52 per pair inside the cutoff of the trials that no atom
    overlaps (33 uncharged), 16 per (k-vector, site) and 12 per k-vector of the
    Fourier terms."""
    s = _system(dict(case, n_guest=0), 0)
    species = s.components[0]
    M = species.molsize
    n = case["n_fw"] + case["n_guest"] * M
    near = n * min(1.0, 4.0 / 3.0 * math.pi * CUTOFF ** 3 / abs(s.volume))
    nk = 0 if s.no_charges else int(s.nvec * 0.5)
    pair = 33.0 if s.no_charges else 52.0
    box_bytes = 36.0 * n + 48.0 * nk
    op = case["op"]
    if op in ("widom", "graph"):
        f = _free_fraction(case)
        K, O = case["K"], case["O"]
        ins = case["n_insert"] * case.get("replays", 1)
        placed = 1.0 - (1.0 - f) ** K
        trials = K * f + placed * O * (M - 1) * f
        flops = ins * (trials * near * pair + placed * nk * (16.0 * M + 12.0))
        return dict(bytes=box_bytes + (64.0 if case.get("records") else 0.0) * ins, flops=flops)
    if op in ("gcmc", "parity"):
        moves = case["cycles"] * max(20, case["n_guest"] + 1) * case.get("boxes", 1)
        # translations and rotations: old and new sites; CBMC moves: the trials left
        flops = moves * (2 * M * near * pair + nk * (32.0 * M + 12.0))
        return dict(bytes=box_bytes * case.get("boxes", 1), flops=flops)
    if op == "move":
        sites = 10 + 10 * (M - 1) + 2 * M
        return dict(bytes=box_bytes, flops=sites * near * pair + nk * (32.0 * M + 12.0))
    guests = case["n_guest"] * M
    return dict(bytes=box_bytes, flops=guests * near * pair + n * nk * 16.0)


# --------------------------------------------------------------------------
# the same in 64 bits, by plain torch
# --------------------------------------------------------------------------

class _Exact:
    """Atoms, force field and Ewald set-up of a system as float64 tensors."""

    def __init__(self, s):
        dev = _device()
        self.dev, self.s = dev, s
        self.H = torch.as_tensor(s.cell.reshape(3, 3), dtype=torch.float64, device=dev)
        self.Hi = torch.linalg.inv(self.H)
        self.eps = torch.as_tensor(s.eps, dtype=torch.float64, device=dev)
        self.sig2 = torch.as_tensor(np.asarray(s.sig) ** 2, dtype=torch.float64, device=dev)
        self.shift = torch.as_tensor(s.shift, dtype=torch.float64, device=dev)
        self.fw = self._atoms(s.fw_pos, s.fw_charge, s.fw_type, np.full(len(s.fw_type), -1))
        g = [(c.init_pos, np.tile(c.charges, len(c.init_pos) // c.molsize), np.tile(c.types, len(c.init_pos) // c.molsize),
              1000000 * i + np.asarray(c.init_molid)) for i, c in enumerate(s.components) if c.init_pos is not None]
        self.guests = self._atoms(*[np.concatenate([x[j] for x in g]) for j in range(4)]) if g else None
        self._k()

    def _atoms(self, pos, q, types, mol):
        t = lambda x, d=torch.float64: torch.as_tensor(np.asarray(x), dtype=d, device=self.dev)  # noqa: E731
        return dict(pos=t(pos).reshape(-1, 3), q=t(q), type=t(types, torch.int64), mol=t(mol, torch.int64))

    def _k(self):
        s = self.s
        if s.no_charges:
            return
        kx, ky, kz = s.kmax
        g = torch.meshgrid(torch.arange(0, kx + 1, device=self.dev), torch.arange(-ky, ky + 1, device=self.dev),
                           torch.arange(-kz, kz + 1, device=self.dev), indexing="ij")
        k = torch.stack(g, -1).reshape(-1, 3).double()
        k2 = k.square().sum(-1)
        self.on = (k2 > 1e-10) & (k2 < s.recip_cut)
        v = 2.0 * math.pi * k @ self.Hi.T
        r2 = v.square().sum(-1)
        pref = s.prefactor * 2.0 * math.pi / abs(s.volume) * (1.0 + (k[:, 0] > 0).double())
        self.kvec = k
        self.ktemp = torch.where(self.on, pref * torch.exp(-0.25 / s.alpha ** 2 * r2) / r2.clamp_min(1e-300), 0.0)

    def phases(self, pos, q):
        """sum over the sites (.., M) of q e^{i k.r} at every active k."""
        f = pos @ self.Hi
        ph = 2.0 * math.pi * (f @ self.kvec[self.on].T)
        return (torch.complex(torch.cos(ph), torch.sin(ph)) * q[..., None]).sum(-2)

    def structure(self, at):
        out = torch.zeros(len(self.kvec), dtype=torch.complex128, device=self.dev)
        if at is not None:
            acc = torch.zeros(int(self.on.sum()), dtype=torch.complex128, device=self.dev)
            for i in range(0, len(at["q"]), 1024):
                acc += self.phases(at["pos"][i:i + 1024], at["q"][i:i + 1024])
            out[self.on] = acc
        return out

    def pairs(self, sites, types, q, at, skip=None, chunk=30_000_000, weight=None):
        """LJ and real-space energies of the sites against the atoms and
        whether a pair overlaps; skip: per site the molecule left out."""
        s = self.s
        n = len(sites)
        v = torch.zeros(n, dtype=torch.float64, device=self.dev)
        r = torch.zeros_like(v)
        o = torch.zeros(n, dtype=torch.bool, device=self.dev)
        step = max(1, chunk // max(1, len(at["q"])))
        for i in range(0, n, step):
            sl = slice(i, min(n, i + step))
            d = (at["pos"][None] - sites[sl, None]) @ self.Hi
            d = (d - torch.round(d)) @ self.H
            r2 = d.square().sum(-1)
            use = torch.ones_like(r2, dtype=torch.bool) if skip is None else at["mol"][None] != skip[sl, None]
            ty = types[sl, None], at["type"][None].expand(len(r2), -1)
            x = self.sig2[ty] / r2
            x = x * x * x
            e = 4.0 * self.eps[ty] * (x * (x - 1.0)) - self.shift[ty]
            near = use & (r2 < s.cut_vdw ** 2)
            e = torch.where(near, e, 0.0)
            o[sl] = (near & ((e > s.overlap) | (r2 < 0.01))).any(1)
            v[sl] = e.sum(1)
            if not s.no_charges:
                rr = r2.sqrt()
                c = s.prefactor * q[sl, None] * at["q"][None] * torch.erfc(s.alpha * rr) / rr
                r[sl] = torch.where(use & (r2 < s.cut_coul ** 2), c, 0.0).sum(1)
        return v, r, o

    def all_pairs(self, sites, types, q, skip=None):
        """hg vdw, hg real, gg vdw, gg real (n, 4) and the overlap flags."""
        v, r, o = self.pairs(sites, types, q, self.fw)
        z = torch.zeros_like(v)
        gv, gr = z, z
        if self.guests is not None:
            gv, gr, go = self.pairs(sites, types, q, self.guests, skip)
            o = o | go
        return torch.stack([v, r, gv, gr], 1), o


def _uniform(seed, index, d):
    """Philox4x32-10 uniforms of draws d of insertions `index` (stream 0): the
    generator's published round function on int64 tensors."""
    mask = 0xffffffff
    c = [index & mask, (index >> 32) & mask, (d >> 1).expand_as(index), torch.zeros_like(index)]
    k0, k1 = seed & mask, (seed >> 32) & mask
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [((p1 >> 32) & mask) ^ c[1] ^ k0, p1 & mask, ((p0 >> 32) & mask) ^ c[3] ^ k1, p0 & mask]
        k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
    odd = (d & 1).expand_as(index) == 1
    a, b = torch.where(odd, c[2], c[0]), torch.where(odd, c[3], c[1])
    return (((a << 21) | (b >> 11)).double() + 0.5) / 9007199254740992.0


def _pick(e, dead, u, beta):
    """Selected trial (-1: none) and mean Boltzmann factor of trials (n, T)."""
    lw = torch.where(dead, -math.inf, -beta * e)
    top = lw.amax(1, keepdim=True)
    w = torch.where(dead, 0.0, torch.exp(lw - torch.where(torch.isfinite(top), top, 0.0)))
    cum = w.cumsum(1)
    reach = ~dead & (cum >= (u * cum[:, -1])[:, None])
    idx = torch.arange(e.shape[1], device=e.device)
    last = torch.where(dead, -1, idx).amax(1)
    sel = torch.where(reach.any(1), reach.to(torch.int8).argmax(1), last)
    total = torch.where(dead, 0.0, torch.exp(lw)).sum(1)
    ok = ~dead.all(1) & ~(total < 1e-150)
    return torch.where(ok, sel, -1), torch.where(ok, total / e.shape[1], 0.0)


def _exact_widom(case, s, seed):
    X = _Exact(s)
    dev = X.dev
    K, O = case["K"], case["O"]
    n = case["n_insert"] * case.get("replays", 1)
    c = s.components[0]
    M = c.molsize
    types = torch.as_tensor(np.asarray(c.types), dtype=torch.int64, device=dev)
    q = torch.as_tensor(c.charges, dtype=torch.float64, device=dev)
    beta = s.beta
    diag = torch.as_tensor(s.cell[[0, 4, 8]], device=dev)
    index = torch.arange(n, dtype=torch.int64, device=dev)

    def draws(ix, first, m):
        d = torch.arange(first, first + m, dtype=torch.int64, device=dev)
        return _uniform(seed, ix[:, None].expand(-1, m), d[None])

    first = draws(index, 0, 3 * K).reshape(n, K, 3) * diag
    flat = first.reshape(-1, 3)
    e1, o1 = X.all_pairs(flat, types[0].expand(len(flat)), q[0].expand(len(flat)))
    v1, r1 = (e1[:, 0] + e1[:, 2]).reshape(n, K), (e1[:, 1] + e1[:, 3]).reshape(n, K)
    sel1, w1 = _pick(v1 + r1, o1.reshape(n, K), draws(index, 3 * K, 1)[:, 0], beta)
    placed = (sel1 >= 0) & (w1 > 1e-150)
    rec = {f: torch.zeros(n, dtype=torch.float64, device=dev) for f in ("rosen", "energy", "vdw", "real", "ewald")}
    fb = torch.full((n,), -1, dtype=torch.int64, device=dev)
    ori = fb.clone()
    at = torch.nonzero(placed)[:, 0]
    if len(at):
        bead = first[at, sel1[at]]
        u = draws(at, 3 * K + 1, 3 * O).reshape(len(at), O, 3)
        tpl = c.template_pos if c.init_pos is None else c.init_pos[:M]
        rel = torch.as_tensor(np.asarray(tpl)[1:] - np.asarray(tpl)[0], device=dev)
        a, b = torch.sqrt(1.0 - u[..., 0]), torch.sqrt(u[..., 0])
        t1, t2 = 2.0 * math.pi * u[..., 1], 2.0 * math.pi * u[..., 2]
        w, x, y, z = a * torch.sin(t1), a * torch.cos(t1), b * torch.sin(t2), b * torch.cos(t2)
        R = torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                         2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                         2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)], -1).reshape(len(at), O, 3, 3)
        sites = bead[:, None, None] + torch.einsum("noij,aj->noai", R, rel)
        m = sites.reshape(-1, 3)
        ty = types[1:].expand(len(at), O, M - 1).reshape(-1)
        e2, o2 = X.all_pairs(m, ty, q[1:].expand(len(at), O, M - 1).reshape(-1))
        v2 = (e2[:, 0] + e2[:, 2]).reshape(len(at), O, M - 1).sum(-1)
        r2 = (e2[:, 1] + e2[:, 3]).reshape(len(at), O, M - 1).sum(-1)
        sel2, w2 = _pick(v2 + r2, o2.reshape(len(at), O, M - 1).any(-1), draws(at, 3 * K + 3 * O + 1, 1)[:, 0], beta)
        done = (sel2 >= 0) & (w1[at] * w2 > 1e-150)
        ix, s2 = at[done], sel2[done]
        ev = v1[ix, sel1[ix]] + v2[done, s2]
        er = r1[ix, sel1[ix]] + r2[done, s2]
        mol = torch.cat([bead[done][:, None], sites[done, s2]], 1)
        ew = torch.zeros_like(ev)
        if not s.no_charges:
            t = X.ktemp[X.on]
            sf, sa = X.structure(X.fw)[X.on], X.structure(X.guests)[X.on]
            intra, selfe = _exclusion(s)
            for i in range(0, len(ix), 2048):
                cn = X.phases(mol[i:i + 2048], q.expand(len(mol[i:i + 2048]), M))
                same = (t * ((sa + cn).abs().square() - sa.abs().square())).sum(1)
                ew[i:i + 2048] = same - (intra + selfe) + 2.0 * (t * (sf.conj() * cn).real).sum(1)
        W = w1[ix] * w2[done] * torch.exp(-beta * ew)
        for f, v in (("rosen", W), ("energy", ev + er + ew), ("vdw", ev), ("real", er), ("ewald", ew)):
            rec[f][ix] = v
        fb[ix], ori[ix] = sel1[ix], s2
    ok = fb >= 0
    W, E = rec["rosen"], rec["energy"]
    out = dict(sum_w=W.sum(), sum_w2=W.square().sum(), sum_we=(W * E).sum(), n=np.float64(n),
               n_first_bead=placed.double().sum(), n_ok=ok.double().sum())
    if case.get("records"):
        out.update(rec, first_bead=fb.to(torch.int32), orientation=ori.to(torch.int32), ok=ok.to(torch.int32))
    return out


def _exclusion(s):
    c = s.components[0]
    pos = np.asarray(c.template_pos if c.init_pos is None else c.init_pos[:c.molsize])
    intra = 0.0
    for i in range(c.molsize):
        for j in range(i + 1, c.molsize):
            r = float(np.linalg.norm(pos[i] - pos[j]))
            intra += s.prefactor * c.charges[i] * c.charges[j] * math.erf(s.alpha * r) / r
    return intra, s.prefactor * s.alpha / math.sqrt(math.pi) * float(np.square(c.charges).sum())


def _exact_move(case, s, seed):
    X = _Exact(s)
    dev = X.dev
    c = s.components[0]
    M = c.molsize
    t = lambda x: torch.as_tensor(np.asarray(x), dtype=torch.float64, device=dev)  # noqa: E731
    m, shift, first, orient = _proposals(case, s, seed)[0]
    old = np.asarray(c.init_pos).reshape(-1, M, 3)[m]
    types = torch.as_tensor(np.asarray(c.types), dtype=torch.int64, device=dev)
    q = t(c.charges)

    def energies(pos, ty, qq):
        return X.all_pairs(t(pos).reshape(-1, 3), ty, qq, torch.full((len(ty),), m, device=dev))

    e1, o1 = energies(first, types[:1].expand(10), q[:1].expand(10))
    e2, o2 = energies(orient, types[1:].repeat(10), q[1:].repeat(10))
    en, on = energies(old + shift, types, q)
    eo, _ = energies(old, types, q)
    d = (en - eo).sum(0)
    de = torch.zeros(10, dtype=torch.float64, device=dev)
    de[1], de[4], de[2], de[5] = d[0], d[1], d[2], d[3]
    k = X.ktemp[X.on]
    sa, sf = X.structure(X.guests)[X.on], X.structure(X.fw)[X.on]
    dn = X.phases(t(old + shift), q) - X.phases(t(old), q)
    return dict(e1=e1, o1=o1.to(torch.uint8), e2=e2.reshape(10, M - 1, 4).sum(1),
                o2=o2.reshape(10, M - 1).any(1).to(torch.uint8), de=de, overlap=int(on.any()),
                same=(k * ((sa + dn).abs().square() - sa.abs().square())).sum(),
                cross=(k * (sf.conj() * dn).real).sum())


def _exact_totals(s):
    X = _Exact(s)
    sf, sa = X.structure(X.fw), X.structure(X.guests)
    k = X.ktemp
    fourier = torch.zeros(10, dtype=torch.float64, device=X.dev)
    fourier[8] = (k * sa.abs().square()).sum()
    fourier[6] = (k * sf.abs().square()).sum()
    fourier[7] = 2.0 * (k * (sf.conj() * sa).real).sum()
    total = fourier.clone()
    g = X.guests
    v, r, _ = X.pairs(g["pos"], g["type"], g["q"], X.fw)
    gv, gr, _ = X.pairs(g["pos"], g["type"], g["q"], g, g["mol"])
    total[1], total[4], total[2], total[5] = v.sum(), r.sum(), 0.5 * gv.sum(), 0.5 * gr.sum()
    flat = lambda z: torch.view_as_real(z).reshape(-1)  # noqa: E731
    return dict(fourier=fourier, total=total, sk_fw=flat(sf), sk_ads=flat(sa))


def exact(case, seed):
    """None for the Monte Carlo runs: a chain's state has no value apart from
    the accept and reject decisions that led to it."""
    op = case["op"]
    if op in ("gcmc", "parity"):
        return None
    s = _system(case, seed)
    if op == "move":
        return _exact_move(case, s, seed)
    if op == "totals":
        return _exact_totals(s)
    return _exact_widom(case, s, seed)
