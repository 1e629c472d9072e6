"""Performance cases: the single points that users of xtb_amd run.

Molecules are the generic seeded systems of xtb_amd.workloads (water clusters,
all-trans alkanes) and alkanes with fluorine and chlorine in place of some
hydrogens (d shells).  A case fixes composition and sizes; the seed moves the
atoms (and picks the orientation of the waters and the halogen sites), so two
seeds of one case cost the same up to the number of SCC iterations.

Outputs are the results that xtb_singlepoint hands back: energies, gradient,
charges, multipoles, bond orders, orbital energies and occupations (and the
density matrix where matrices are asked for).  Orbital coefficients are left
out: their signs, and their rotation inside degenerate sets, are arbitrary.
"""
import math
import random

import numpy as np

import xtb_amd
from xtb_amd import engine, workloads

SCALARS = ("energy", "hl_gap_ev", "gnorm", "e_elec", "e_es", "e_aes", "e_disp", "e_rep", "e_solv")
ARRAYS = ("gradient", "charges", "qsh", "dipm", "qp", "emo", "focc", "dipole")


def listed():
    return [
        # the smallest call: one water molecule, all latency and launches
        {"name": "water1", "kind": "single", "system": "water", "units": 1},
        # an ordinary single point by the entry point for callers that may not allocate (192 AOs)
        {"name": "water32_noalloc", "kind": "noalloc", "system": "water", "units": 32},
        # an ordinary organic molecule with its density matrix (386 AOs, an odd size)
        {"name": "alkane64_density", "kind": "single", "system": "alkane", "units": 64, "matrices": True},
        # d-shell elements in implicit water (ALPB), as for a drug-like molecule
        {"name": "halo23_alpb", "kind": "single", "system": "halo", "units": 23, "solvent": "water"},
        # a radical: the open-shell occupation path
        {"name": "radical17", "kind": "single", "system": "radical", "units": 17},
        # one step of a geometry optimisation or of dynamics: restart from the last wavefunction (288 AOs)
        {"name": "water48_restart", "kind": "restart", "system": "water", "units": 48},
        # a numerical Hessian of butane: 6n displaced copies of one small molecule as one batch
        {"name": "hessian_butane", "kind": "hessian", "system": "alkane", "units": 4},
        # the benchmark's workload: 512 mixed molecules of 10-200 atoms on a kept batch
        {"name": "batch512", "kind": "batch", "system": "mixed", "count": 512, "lo": 10, "hi": 200},
        # a screening batch of small d-shell molecules in implicit water
        {"name": "batch96_halo_alpb", "kind": "batch", "system": "halo", "count": 96, "lo": 10, "hi": 60,
         "solvent": "water"},
        # serving: requests of 20-400 atoms through the continuous-batching loop of a kept server
        {"name": "server64", "kind": "server", "system": "mixed", "count": 64, "lo": 20, "hi": 400},
        # the largest single point of the benchmark, (H2O)700: 4200 AOs
        {"name": "water700", "kind": "single", "system": "water", "units": 700},
        # the eigensolver by itself on matrices that the caller holds
        {"name": "eigh3", "kind": "eigh", "n0": 193, "n1": 517, "n2": 1024},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["single", "single", "noalloc", "restart", "hessian", "batch", "batch", "server", "eigh"])
    if kind == "eigh":
        return {"kind": kind, "n0": _log(rng, 24, 300), "n1": _log(rng, 24, 700), "n2": _log(rng, 24, 1100)}
    if kind == "server":
        return {"kind": kind, "system": "mixed", "count": rng.randint(5, 72), "lo": rng.randint(12, 40),
                "hi": rng.randint(60, 400)}
    if kind == "batch":
        c = {"kind": kind, "system": rng.choice(["mixed", "mixed", "halo", "water"]), "count": _log(rng, 3, 512),
             "lo": rng.randint(6, 30), "hi": rng.randint(40, 200)}
        if c["system"] == "halo":
            c["count"] = min(c["count"], 200)
        if rng.random() < 0.4:
            c["solvent"] = rng.choice(["water", "toluene", "acetone"])
        return c
    if kind == "hessian":
        return {"kind": kind, "system": rng.choice(["water", "alkane", "halo"]), "units": rng.randint(1, 9)}
    system = rng.choice(["water", "alkane", "halo"]) if kind == "noalloc" else \
        rng.choice(["water", "alkane", "halo", "radical"])
    top = {"noalloc": 55, "restart": 120, "single": 400}[kind]
    if system in ("halo", "radical"):
        top = min(top, 36)
    c = {"kind": kind, "system": system, "units": _log(rng, 2, top)}
    if kind == "single":
        if c["units"] <= 100 and rng.random() < 0.3:
            c["matrices"] = True
        if c["units"] <= 150 and rng.random() < 0.3:
            c["solvent"] = rng.choice(["water", "toluene", "acetone"])
    return c


# --- systems ---------------------------------------------------------------

def _halogenated(ncarbon, seed):
    """An alkane with about every sixth hydrogen replaced by F or Cl (at least
    one Cl), the atom moved out to the C-X bond length."""
    z, x = workloads.alkane(ncarbon, seed)
    z, x = z.copy(), x.copy()
    rng = np.random.default_rng(seed + 1)
    hyd = np.flatnonzero(z == 1)
    for k, h in enumerate(hyd[::6]):
        c = int(np.argmin(np.linalg.norm(x[:ncarbon] - x[h], axis=1)))
        z[h], r = (17, 1.77) if k % 2 == 0 else (9, 1.36)
        d = x[h] - x[c]
        x[h] = x[c] + d / np.linalg.norm(d) * r * workloads.AATOAU + rng.uniform(-0.01, 0.01, 3)
    return z, x


def _molecule(system, units, seed):
    """(numbers, positions[bohr], charge, uhf)"""
    if system == "water":
        z, x = workloads.large_water_cluster(seed) if units == 700 else workloads.water_cluster(units, seed)
    elif system == "halo":
        z, x = _halogenated(units, seed)
    else:
        z, x = workloads.alkane(units, seed)
        if system == "radical":   # one terminal hydrogen taken off
            return z[:-1], x[:-1], 0.0, 1
    return z, x, 0.0, 0


def _sizes(case):
    """[(system, units)] of a batch: log-uniform sizes in [lo, hi] atoms; fixed
    by the case so that its cost does not depend on the seed."""
    rng = random.Random(case["count"] * 1000003 + case["lo"] * 1009 + case["hi"])
    out = []
    for _ in range(case["count"]):
        atoms = math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))
        system = case["system"]
        if system == "mixed":
            system = "water" if rng.random() < 0.5 else "alkane"
        out.append((system, max(1, round(atoms / 3 if system == "water" else (atoms - 2) / 3))))
    return out


def _molecules(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "hessian":
        z, x, q, u = _molecule(case["system"], case["units"], int(rng.integers(1 << 30)))
        mols = []
        for i in range(len(z)):
            for k in range(3):
                for s in (-0.005, 0.005):
                    y = x.copy()
                    y[i, k] += s
                    mols.append((z, y, q, u))
        return mols
    if "count" in case:
        return [_molecule(s, n, int(rng.integers(1 << 30))) for s, n in _sizes(case)]
    return [_molecule(case["system"], case["units"], int(rng.integers(1 << 30)))]


def _symmetric(n, rng):
    """A dense symmetric matrix with a spectrum like a Fock matrix in eV."""
    a = rng.standard_normal((n, n)) / math.sqrt(n)
    return np.ascontiguousarray(a + a.T + np.diag(rng.uniform(-20.0, 20.0, n)))


# --- one case --------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "eigh":
        rng = np.random.default_rng(seed)
        return {"case": case, "mats": [_symmetric(case[k], rng) for k in ("n0", "n1", "n2")]}
    state = {"case": case, "mols": _molecules(case, seed)}
    if kind in ("batch", "hessian"):
        state["batch"] = engine.Batch(state["mols"])
        if case.get("solvent"):
            state["batch"].set_solvent(case["solvent"], "p16", True)
    elif kind == "server":
        state["server"] = engine.Server(hbm_gb=24.0, max_atoms=400, max_slots=256)
    elif kind == "restart":   # the wavefunction of the last geometry
        z, x, q, u = state["mols"][0]
        state["last"] = xtb_amd.singlepoint(z, x, q, u)
        state["moved"] = x + np.random.default_rng(seed + 7).uniform(-0.02, 0.02, x.shape)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "eigh":
        pairs = engine.eigh(state["mats"])
        return {"values": [w for w, _ in pairs], "vectors": [_signed(v) for _, v in pairs]}
    if kind in ("batch", "hessian"):
        return _outputs(state["batch"].run().results())
    if kind == "server":
        srv = state["server"]
        ids = [srv.submit(z, x, q, u) for z, x, q, u in state["mols"]]
        while srv.step() > 0:
            pass
        srv.finished()
        return _outputs([srv.result(i) for i in ids])
    z, x, q, u = state["mols"][0]
    if kind == "noalloc":
        return _outputs([engine.singlepoint_noalloc(z, x, q, u)])
    if kind == "restart":
        b = engine.Batch([(z, state["moved"], q, u)])
        b.set_guess(0, state["last"]["qsh"], state["last"]["dipm"], state["last"]["qp"])
        r = b.run().result(0)
        b.close()
        return _outputs([r])
    r = xtb_amd.singlepoint(z, x, q, u, matrices=bool(case.get("matrices")), solvent=case.get("solvent"),
                            solv_kernel="p16" if case.get("solvent") else "still", alpb=bool(case.get("solvent")))
    return _outputs([r])


def _signed(v):
    """Eigenvectors (rows) with their largest component positive."""
    k = np.argmax(np.abs(v), axis=1)
    return v * np.sign(v[np.arange(len(v)), k])[:, None]


def _outputs(results):
    out = {k: np.array([r[k] for r in results]) for k in SCALARS}
    for k in ARRAYS:
        out[k] = results[0][k] if len(results) == 1 else np.concatenate([r[k] for r in results])
    out["wbo"] = results[0]["wbo"] if len(results) == 1 else np.concatenate([r["wbo"].ravel() for r in results])
    if "density" in results[0]:
        out["density"] = results[0]["density"]
    return out


# --- accounting ------------------------------------------------------------

ITERATIONS = 8   # SCC iterations of a typical single point from the EEQ guess


def _dims(case):
    """[(atoms, shells, AOs)] of the case's molecules"""
    out = []
    for z, _, _, _ in _molecules(case, 0):
        z = np.asarray(z)
        nsh = int(np.sum(np.where(z == 1, 1, np.where(z == 17, 3, 2))))
        out.append((len(z), nsh, int(np.sum(np.where(z == 1, 1, np.where(z == 17, 9, 4))))))
    return out


def work(case):
    """Inputs and results once; the dense linear algebra of one single point
    (22/3 N^3 per SCC iteration for the eigenproblem in an orthonormal basis
    and the density, 13/3 N^3 for the reduction and the energy-weighted
    density), which the parts of order N^2 do not add much to."""
    if case["kind"] == "eigh":
        ns = [case[k] for k in ("n0", "n1", "n2")]
        return {"bytes": 8.0 * sum(2 * n * n + n for n in ns), "flops": sum(9.0 * n ** 3 for n in ns)}
    nbytes = flops = 0.0
    for n, nsh, nao in _dims(case):
        nbytes += 4.0 * n + 8.0 * (3 * n + 3 * n + n + nsh + 9 * n + n * n + 2 * nao)
        if case.get("matrices"):
            nbytes += 16.0 * nao * nao
        flops += (ITERATIONS * 22.0 / 3.0 + 13.0 / 3.0) * float(nao) ** 3
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Four times what other orders of the sums and other eigensolvers of the
    same precision showed: eigenvectors 5e-13 against LAPACK (more where two
    eigenvalues happen to lie close), a single point's dipole (a sum of nearly
    cancelling terms) up to 2e-7, its other results up to 1e-8."""
    if case["kind"] == "eigh":
        return {"rel": 1e-10, "max": 1e-8}
    return {"rel": 1e-6, "max": 1e-5}


def exact(case, seed):
    """The eigenvalues and vectors by LAPACK.  A single point has no value
    beyond the 64 bits it is computed in: it is the state where a fixed-point
    iteration in 64 bits stops."""
    if case["kind"] != "eigh":
        return None
    pairs = [np.linalg.eigh(m) for m in prepare(case, seed)["mats"]]
    return {"values": [w for w, _ in pairs], "vectors": [_signed(np.ascontiguousarray(v.T)) for _, v in pairs]}
