"""GPU tests of the SCC's subspace path (k_sub.hip) against the full
diagonalisation in every iteration (XTBAMD_SUBSPACE=0).

The path stops when max |R| <= 1e-12 max(|A_ii|, 1), the criterion of a
finished diagonalisation, so density errors are below 1e-12 x 30 eV / gap
(a few 1e-11 at gaps above 2 eV); the SCC amplifies them by the few units by
which any rounding is amplified.  Energies (Eh) are second order in them.
Sizes: occupied and virtual counts at the edges of the 64 x 64 product tiles
and of the k-blocks of 16, and a molecule with fewer than one tile.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {"energy": 1e-9, "charges": 1e-8, "gradient": 1e-8, "wbo": 1e-8, "emo": 1e-7, "hl_gap_ev": 1e-7}


def _engine():
    import xtb_amd
    if xtb_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP runtime")
    return xtb_amd


def _both(monkeypatch, mols, solvent=None, **kw):
    xa = _engine()
    out = []
    for on in ("0", "1"):
        monkeypatch.setenv("XTBAMD_SUBSPACE", on)
        b = xa.Batch(mols, **kw)
        if solvent:
            b.set_solvent(solvent, "p16", True)
        b.run()
        out.append((b.results(), b.counters()))
        b.close()
    return out


def _check(a, b, tag):
    assert a["iterations"] == b["iterations"] and a["converged"] == b["converged"], tag
    assert a["ihomo"] == b["ihomo"], tag
    # both come from a diagonalisation of the same matrix to within TOL["emo"]
    # (and its Fermi level): |df| <= 2 spins x (2 x 1e-7 eV) / (4 kT), kT = 0.0259 eV
    # at 300 K (the lowest temperature here with fractional occupations)
    assert float(np.max(np.abs(a["focc"] - b["focc"]))) <= 4 * TOL["emo"] / (4 * 0.02585), tag
    for k, tol in TOL.items():
        d = float(np.max(np.abs(np.asarray(a[k]) - np.asarray(b[k]))))
        assert d <= tol, f"{tag} {k}: {d:.2e}"


def _halogenated(n, seed):
    from xtb_amd import workloads as w
    z, x = w.alkane(n, seed)
    z, x = z.copy(), x.copy()
    for h in np.flatnonzero(z == 1)[::5]:
        c = int(np.argmin(np.linalg.norm(x[:n] - x[h], axis=1)))
        x[h] = x[c] + (x[h] - x[c]) * (1.77 / 1.09)
        z[h] = 17
    return z, x


# (H2O)n: 4n occupied, 2n virtual; CnH(2n+2): 3n + 1 of each
@pytest.mark.parametrize("kind,n", [("water", 1), ("water", 4), ("water", 16), ("water", 17), ("water", 31),
                                    ("water", 33), ("alkane", 1), ("alkane", 5), ("alkane", 21), ("alkane", 22),
                                    ("alkane", 42), ("alkane", 43), ("halo", 3), ("halo", 12)])
def test_subspace_and_full_diagonalisation_agree(monkeypatch, kind, n):
    from xtb_amd import workloads as w
    z, x = _halogenated(n, 3) if kind == "halo" else (w.water_cluster if kind == "water" else w.alkane)(n, 3)
    (full, cf), (sub, cs) = _both(monkeypatch, [(z, x, 0.0, 0)])
    _check(full[0], sub[0], f"{kind} {n}")
    if len(x) > 40:   # the path was taken: fewer Jacobi rounds
        assert cs[1] < cf[1], (cs, cf)


@pytest.mark.parametrize("kw,solvent", [({"etemp": 0.0}, None), ({"etemp": 1000.0}, None), ({"etemp": 9000.0}, None),
                                        ({"guess": "sad"}, None), ({"accuracy": 0.01}, None), ({"maxiter": 3}, None),
                                        ({}, "water")])
def test_subspace_options_agree(monkeypatch, kw, solvent):
    """Smearing (at 9000 K every molecule keeps the full diagonalisation), the
    SAD guess, tight accuracy, a run cut off before convergence and solvent."""
    from xtb_amd import workloads as w
    mols = [w.water_cluster(9, 1), w.alkane(14, 2), w.water_cluster(1, 4), _halogenated(6, 5)]
    (full, _), (sub, _) = _both(monkeypatch, [(z, x, 0.0, 0) for z, x in mols], solvent, **kw)
    for k, (a, b) in enumerate(zip(full, sub)):
        _check(a, b, f"{kw} mol {k}")


@pytest.mark.parametrize("ratio", [0.4, 0.7, 0.8, 0.84, 0.86, 0.95, 1.05, 1.4])
def test_subspace_at_temperatures_around_the_gap_bound(monkeypatch, ratio):
    """Electronic temperatures at which 52 kT is `ratio` times the gap: on the
    path with room, at the edge where its diagonal estimate (0.85 of the gap)
    or the contraction decides, and above, where every molecule keeps the full
    diagonalisation.  The density error of whole occupations is e^-26 at the
    bound itself, so the tolerances are those of every other temperature."""
    from xtb_amd import workloads as w
    xa = _engine()
    for z, x in (w.water_cluster(9, 1), w.alkane(14, 2), w.water_cluster(30, 4)):
        gap = xa.singlepoint(z, x)["hl_gap_ev"]
        t = ratio * gap / (52 * 8.617333e-5)
        (full, cf), (sub, cs) = _both(monkeypatch, [(z, x, 0.0, 0)], etemp=t)
        _check(full[0], sub[0], f"{len(z)} atoms, {t:.0f} K")
        if ratio > 1.0:
            assert cs == cf, (cs, cf)


def test_one_workgroup_path_bitwise_at_every_workgroup_size(monkeypatch):
    """Workgroups of 64, 256 and 512 threads (largest molecule of the launch up
    to 32, 64 and more AOs) share out the same blocks of the same products: 24,
    30 and 32 AOs alone, beside 62 and 36 AOs, and beside 96 AOs on the path."""
    xa = _engine()
    from xtb_amd import workloads as w
    small = [w.water_cluster(4, 3), w.water_cluster(5, 3), w.alkane(5, 3), w.water_cluster(1, 3)]

    def run(mols):
        b = xa.Batch([(z, x, 0.0, 0) for z, x in mols])
        b.run()
        r = b.results()
        b.close()
        return r

    ref = run(small)
    mixes = [run(small + [w.alkane(10, 3), w.water_cluster(6, 3)])]
    monkeypatch.setenv("XTBAMD_SUB_WG", "128")
    mixes.append(run(small + [w.water_cluster(16, 3)]))
    for r in mixes:
        for m, a in enumerate(ref):
            assert a["iterations"] == r[m]["iterations"] and a["energy"] == r[m]["energy"], m
            for k in ("gradient", "charges", "wbo", "emo", "focc"):
                assert np.array_equal(a[k], r[m][k]), (m, k)


def test_subspace_launches_only_where_a_molecule_can_use_them(monkeypatch, capfd):
    """Steps queued per SCC iteration (XTBAMD_TRACE_ROUNDS): none in the first
    one, whose orbitals the path needs; none at all for open shells, for gaps
    far below 52 kT (9000 K) and once every molecule has given up; the second
    iteration starts with the steps of a cold start."""
    from xtb_amd import workloads as w
    xa = _engine()
    monkeypatch.setenv("XTBAMD_TRACE_ROUNDS", "1")

    def steps(mols, **kw):
        capfd.readouterr()
        b = xa.Batch(mols, **kw)
        out = []
        for _ in range(2):   # a batch run again starts anew
            b.run()
            out.append([int(ln.split()[-3]) for ln in capfd.readouterr().err.splitlines() if "subspace steps" in ln])
        b.close()
        assert len(out[0]) > 3 and out[0] == out[1], out
        return out[0]

    zw, xw = w.water_cluster(20, 3)
    za, xa_ = w.alkane(14, 3)
    s = steps([(zw, xw, 0.0, 0), (za, xa_, 0.0, 0)])
    print(s, flush=True)
    assert s[0] == 0 and s[1] >= 6 and all(k > 0 for k in s[1:]), s
    assert not any(steps([(za[:-1], xa_[:-1], 0.0, 1)]))
    assert not any(steps([(zw, xw, 0.0, 0)], etemp=9000.0))
    small = w.water_cluster(3, 3) + (0.0, 0)
    s = steps([small])
    assert s[0] == 0 and any(s[1:]), s
    assert not any(steps([small], etemp=9000.0))


def test_subspace_small_gaps_ions_and_open_shells(monkeypatch, golden):
    """Gaps of 0.7 to 3 eV (given up or never taken), charged and open-shell
    molecules beside gapped ones in one batch."""
    from xtb_amd import workloads as w
    mols = []
    for k in ("mindless01", "mindless02", "mindless05", "mindless07", "mindless09"):
        g = golden[k]
        mols.append((np.array(g["numbers"]), np.array(g["positions"]), g["charge"], g["uhf"]))
    z, x = w.water_cluster(2, 3)
    mols.append((z[:-1], x[:-1], -1.0, 0))           # HO-(H2O)
    za, xa = w.alkane(8, 3)
    mols.append((za[:-1], xa[:-1], 0.0, 1))          # radical
    mols.append((za[:-1], xa[:-1], 1.0, 0))          # cation
    mols.append((za, xa, 0.0, 2))                    # triplet
    mols.append((np.array([2]), np.zeros((1, 3)), 0.0, 0))
    mols.append((za, xa, 0.0, 0))
    (full, _), (sub, _) = _both(monkeypatch, mols)
    for k, (a, b) in enumerate(zip(full, sub)):
        _check(a, b, f"mol {k}")


@pytest.mark.parametrize("blk_min", [65, 96])
def test_blocks_on_the_blocked_eigensolver(monkeypatch, blk_min):
    """Last diagonalisation with the blocks of at least blk_min rows on the
    blocked eigensolver (both, one or neither block of a molecule)."""
    from xtb_amd import workloads as w
    monkeypatch.setenv("XTBAMD_EIG_BLK_MIN", str(blk_min))
    mols = [w.alkane(n, 3) for n in (20, 27, 33, 40)] + [w.water_cluster(k, 5) for k in (14, 23, 40)]
    (a, _), (b, _) = _both(monkeypatch, mols)
    for (z, _), x, y in zip(mols, a, b):
        _check(x, y, f"{len(z)} atoms")


@pytest.mark.parametrize("first,whole,half", [(65, 65, 1 << 30), (1 << 30, 1 << 30, 80), (200, 200, 100),
                                              (65, 1 << 30, 1 << 30), (1 << 30, 65, 1 << 30), (150, 200, 130)])
def test_lines_of_whole_matrices_and_blocks(monkeypatch, first, whole, half):
    """First and later iterations and blocks on the blocked eigensolver from
    lines of their own; each setting with and without the subspace path, whose
    absence keeps whole matrices in every iteration."""
    from xtb_amd import workloads as w
    monkeypatch.setenv("XTBAMD_EIG_BLK_MIN", str(whole))
    monkeypatch.setenv("XTBAMD_EIG_BLK_MIN_FIRST", str(first))
    monkeypatch.setenv("XTBAMD_EIG_BLK_MIN_HALF", str(half))
    mols = [w.alkane(27, 3), w.alkane(40, 3), w.water_cluster(23, 5)]
    (a, _), (b, _) = _both(monkeypatch, mols)
    for (z, _), x, y in zip(mols, a, b):
        _check(x, y, f"{len(z)} atoms")


def test_orthogonalisation_over_the_spectrum():
    """S^(-1/2) from S = I (two atoms far apart: every eigenvalue at one end of
    the interval that the scaled steps expect) to eigenvalues far below it
    (compressed molecules); the oracle diagonalises the generalised problem.
    Energies agree to cond(S) eps x 30 Eh, below 1e-9 Eh up to cond(S) = 1e5."""
    xa = _engine()
    from oracle import pyoracle as po
    h4 = np.array([[0.0, 0.0, 0.9 * k] for k in range(4)])
    mols = [(np.array([2, 2]), np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 40.0]])),
            (np.array([1, 1]), np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 0.7]])),
            (np.array([1, 1, 1, 1]), h4),
            (np.array([6, 6, 1, 1]), np.array([[0, 0, 0], [0, 0, 1.8], [0, 0, -1.6], [0, 0, 3.4]], dtype=float))]
    b = xa.Batch(mols)
    b.run()
    res = b.results()
    b.close()
    for (z, x), r in zip(mols, res):
        o = po.singlepoint(z, x)
        assert r["iterations"] == o["iterations"], z
        assert abs(r["energy"] - o["e_total"]) <= 1e-9, (z, r["energy"], o["e_total"])


@pytest.mark.parametrize("maxiter", [31, 33, 34, 36])
def test_mixing_history_around_the_lds_limit(maxiter):
    """Broyden histories of 30, 32 (the largest whose inverse is taken in LDS),
    33 and 35 earlier iterations: an accuracy that no iteration reaches keeps
    the SCC going.  Both sides are converged to rounding long before, so the
    energies agree to a few ulp of 30 Eh times the SCC's amplification."""
    xa = _engine()
    from oracle import pyoracle as po
    from xtb_amd import workloads as w
    mols = [w.water_cluster(2, 3), w.alkane(4, 3)]
    b = xa.Batch(mols, accuracy=1e-11, maxiter=maxiter)
    b.run()
    res = b.results()
    b.close()
    for (z, x), r in zip(mols, res):
        o = po.singlepoint(z, x, accuracy=1e-11, maxiter=maxiter)
        assert r["iterations"] >= maxiter - 1 and r["iterations"] == o["iterations"], (r["iterations"], o["iterations"])
        assert abs(r["energy"] - o["e_total"]) <= 1e-10, (z, r["energy"], o["e_total"])
