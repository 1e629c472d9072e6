"""Project autotuner of the batched engine on one MI355X (gfx950).

Times, on the device, the choices the engine leaves open and writes them to a
tuning file that every batch reads at set-up (``tuning_gfx950.txt`` next to
``libxtb_amd.so``; environment variables ``XTBAMD_*`` override it):

* the smallest eigenproblems that go to the blocked eigensolver (Householder
  tridiagonalisation, divide and conquer, back-transformation) instead of
  block-Jacobi rounds; each line is the smallest size from which the blocked
  solver wins at every larger one:
  ``eig_blk_min_first``, the first SCC iteration (unrelated orbitals to start
  from), one-molecule single points of water clusters and alkanes, kept only
  if the 512-molecule batch is not slower with it;
  ``eig_blk_min``, the next iterations up to ``eig_blk_iters`` (2 or 4, or
  all; timed on the 700-water cluster with a diagonalisation in every
  iteration, as open shells and small gaps take it): the mean of a water
  cluster and an alkane, with a diagonalisation in every iteration and on the
  subspace path, which falls back to some;
  ``eig_blk_min_half``, the occupied and virtual blocks of the last
  diagonalisation, which start nearly diagonal (the size of the larger block).
* ``jac_lanes`` (1..3) and ``jac_cross`` (0/1): the stream lanes and the
  cross-round schedule of the block-Jacobi rounds, timed on the 512-molecule
  workload.
* ``gemm`` (mfma / valu): the batched FP64 product kernel.

    python -m xtb_amd.tune [--out DIR] [--steps K]

writes ``DIR/tuning_gfx950.txt`` and ``DIR/autotune_gfx950.md`` (the
measurements).
"""
import argparse
import os
import sys
import time

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

from xtb_amd import workloads  # noqa: E402

KEYS = ("XTBAMD_EIG_BLK_MIN", "XTBAMD_EIG_BLK_MIN_FIRST", "XTBAMD_EIG_BLK_MIN_HALF", "XTBAMD_EIG_BLK_ITERS",
        "XTBAMD_JAC_LANES", "XTBAMD_JAC_CROSS", "XTBAMD_GEMM", "XTBAMD_SUBSPACE")


def _set(env):
    for k in KEYS:
        os.environ.pop(k, None)
    os.environ["XTBAMD_TUNING"] = "off"
    for k, v in env.items():
        os.environ[k] = str(v)


def _time_batch(mols, env, steps, warmup=1):
    import xtb_amd
    _set(env)
    b = xtb_amd.Batch([(z, x, 0.0, 0) for z, x in mols])
    for _ in range(warmup):
        b.run()
    ts = []
    for _ in range(steps):
        t = time.perf_counter()
        b.run()
        ts.append(time.perf_counter() - t)
    e = [r["energy"] for r in b.results()]
    b.close()
    return float(np.median(ts)), e


def tune(steps=3, out=HERE, log=print):
    rows_iters, rows_next, rows_bins, rows_half, rows_batch = [], [], [], [], []
    off = 1 << 30
    bins = [("water", 12), ("alkane", 24), ("water", 22), ("alkane", 44), ("water", 43), ("alkane", 86),
            ("water", 64), ("water", 100), ("water", 170), ("alkane", 240), ("water", 256), ("alkane", 300),
            ("water", 300), ("water", 400), ("alkane", 500), ("water", 500), ("water", 600), ("alkane", 700),
            ("water", 700)]

    def molecule(kind, size, seed=7):
        if kind == "water" and size == 700:
            return workloads.large_water_cluster(2017 + seed)
        return workloads.water_cluster(size, seed) if kind == "water" else workloads.alkane(size, seed)

    def line(rows):
        """smallest size from which the blocked solver wins in every larger bin"""
        rows.sort()
        for i in range(len(rows)):
            if all(tb < tj for *_, tj, tb in rows[i:]):
                return rows[i][0]
        return off

    # 1. eigensolver path: iterations after the first, a diagonalisation in each
    big = [molecule("water", 700)]
    for it in (2, 4, off):
        t, _ = _time_batch(big, {"XTBAMD_SUBSPACE": 0, "XTBAMD_EIG_BLK_MIN": 65, "XTBAMD_EIG_BLK_ITERS": it}, steps)
        rows_iters.append((it, t))
        log(f"tune eig: {'every iteration' if it == off else f'first {it}'} on the blocked solver {1e3 * t:.1f} ms")
    iters = min(rows_iters, key=lambda r: r[1])[0]
    for size in (300, 400, 500, 600, 700):   # 6 AOs per water and per carbon
        tj = tb = 0.0
        for kind in ("water", "alkane"):
            z, x = molecule(kind, size)
            for sub in (0, 1):
                env = {"XTBAMD_SUBSPACE": sub, "XTBAMD_EIG_BLK_ITERS": iters, "XTBAMD_EIG_BLK_MIN_FIRST": 65,
                       "XTBAMD_EIG_BLK_MIN_HALF": off}
                tj += 0.25 * _time_batch([(z, x)], dict(env, XTBAMD_EIG_BLK_MIN=off), steps)[0]
                tb += 0.25 * _time_batch([(z, x)], dict(env, XTBAMD_EIG_BLK_MIN=65), steps)[0]
        rows_next.append((6 * size, tj, tb))
        log(f"tune eig: {6 * size} AOs first iteration blocked {1e3 * tj:.1f} ms, also the next {1e3 * tb:.1f} ms")
    cut_next = line(rows_next)
    # the first iteration (one molecule per batch)
    for kind, size in bins:
        z, x = molecule(kind, size)
        tj, ej = _time_batch([(z, x)], {"XTBAMD_EIG_BLK_MIN": off}, steps)
        tb, eb = _time_batch([(z, x)], {"XTBAMD_EIG_BLK_MIN": off, "XTBAMD_EIG_BLK_MIN_FIRST": 65}, steps)
        dE = abs(ej[0] - eb[0])
        rows_bins.append((workloads.ao_count(z), kind, size, dE, tj, tb))
        log(f"tune eig: {kind} {size} nao={rows_bins[-1][0]} jacobi {1e3 * tj:.1f} ms blocked {1e3 * tb:.1f} ms "
            f"dE={dE:.1e}")
    cut = min(line(rows_bins), cut_next)
    # the blocks of the last diagonalisation, whole matrices at their cutoff
    # (two geometries each: the rounds of a block differ by up to two times)
    cut_half = off
    if cut < off:
        env = {"XTBAMD_EIG_BLK_MIN": cut_next, "XTBAMD_EIG_BLK_MIN_FIRST": cut, "XTBAMD_EIG_BLK_ITERS": iters}
        for kind, size in (("water", 170), ("alkane", 300), ("water", 300), ("water", 400), ("alkane", 500),
                           ("water", 500), ("alkane", 700), ("water", 550), ("water", 600), ("water", 650),
                           ("alkane", 900), ("water", 700)):
            tl = th = 0.0
            for seed in (7, 8):
                z, x = molecule(kind, size, seed)
                occ = 4 * size if kind == "water" else 3 * size + 1
                block = max(occ, workloads.ao_count(z) - occ)
                tl += 0.5 * _time_batch([(z, x)], dict(env, XTBAMD_EIG_BLK_MIN_HALF=off), steps)[0]
                th += 0.5 * _time_batch([(z, x)], dict(env, XTBAMD_EIG_BLK_MIN_HALF=block), steps)[0]
            rows_half.append((block, kind, size, tl, th))
            log(f"tune blocks: {kind} {size} block of {block} rows: rounds {1e3 * tl:.1f} ms blocked {1e3 * th:.1f} ms")
        cut_half = line(rows_half)
    # 2. batch schedule on the 512-molecule workload
    mols = workloads.mixed_batch(512, seed=2024)
    best = None
    for lanes in (1, 2, 3):
        for cross in (0, 1):
            t, _ = _time_batch(mols, {"XTBAMD_JAC_LANES": lanes, "XTBAMD_JAC_CROSS": cross,
                                      "XTBAMD_EIG_BLK_MIN": off}, steps)
            rows_batch.append((f"jac_lanes={lanes} jac_cross={cross}", t))
            log(f"tune batch: lanes {lanes} cross {cross}: {1e3 * t:.1f} ms")
            if best is None or t < best[0]:
                best = (t, lanes, cross)
    _, lanes, cross = best
    base = {"XTBAMD_JAC_LANES": lanes, "XTBAMD_JAC_CROSS": cross}
    tv, _ = _time_batch(mols, dict(base, XTBAMD_GEMM="valu", XTBAMD_EIG_BLK_MIN=off), steps)
    tm, _ = _time_batch(mols, dict(base, XTBAMD_GEMM="mfma", XTBAMD_EIG_BLK_MIN=off), steps)
    rows_batch += [("gemm=valu", tv), ("gemm=mfma", tm)]
    gemm = "valu" if tv < tm else "mfma"
    # the cutoff must not slow the batch down (its largest problems are below
    # it unless the blocked path wins there too)
    if cut < off:
        tc, _ = _time_batch(mols, dict(base, XTBAMD_GEMM=gemm, XTBAMD_EIG_BLK_MIN=cut),
                            steps)
        rows_batch.append((f"eig_blk_min_first={cut}", tc))
        if tc > min(tv, tm):
            rows_batch.append((f"eig_blk_min_first={cut} rejected for the batch", tc))
            cut = max(cut, 1 + max(workloads.ao_count(z) for z, _ in mols))
    _set({})
    os.environ.pop("XTBAMD_TUNING", None)
    stamp = time.strftime("%Y-%m-%d %H:%M:%S")
    with open(os.path.join(out, "tuning_gfx950.txt"), "w") as f:
        f.write(f"# written by python -m xtb_amd.tune ({stamp}); environment variables XTBAMD_* override\n")
        f.write(f"eig_blk_min {cut_next}\neig_blk_min_first {cut}\neig_blk_min_half {cut_half}\n"
                f"eig_blk_iters {iters}\n"
                f"jac_lanes {lanes}\njac_cross {cross}\ngemm {gemm}\n")
    with open(os.path.join(out, "autotune_gfx950.md"), "w") as f:
        f.write("# Autotuner measurements (one MI355X)\n\n")
        f.write("Command: `python -m xtb_amd.tune --out <dir>` (median of "
                f"{steps} timed runs after one warm-up per configuration).\n\n")
        f.write("## SCC iterations on the blocked solver ((H2O)700, a diagonalisation in every iteration)\n\n"
                "| iterations | ms |\n|---|---:|\n")
        for it, t in rows_iters:
            f.write(f"| {'all' if it == off else f'first {it}'} | {1e3 * t:.1f} |\n")
        name = lambda kind, size: f"(H2O){size}" if kind == "water" else f"C{size}H{2 * size + 2}"
        f.write("\n## Iterations after the first, up to that number (mean of a water cluster and an alkane, with a\n"
                "diagonalisation in every iteration and on the subspace path)\n\n"
                "| AOs | block Jacobi ms | blocked ms |\n|---:|---:|---:|\n")
        for nao, tj, tb in rows_next:
            f.write(f"| {nao} | {1e3 * tj:.1f} | {1e3 * tb:.1f} |\n")
        f.write("\n## First iteration (one molecule per batch, whole single point)\n\n")
        f.write("| molecule | AOs | block Jacobi ms | blocked ms | dE (Eh) |\n|---|---:|---:|---:|---:|\n")
        for nao, kind, size, dE, tj, tb in rows_bins:
            f.write(f"| {name(kind, size)} | {nao} | {1e3 * tj:.1f} | {1e3 * tb:.1f} | {dE:.1e} |\n")
        f.write("\n## Blocks of the last diagonalisation (whole matrices at their cutoff; mean of two geometries)\n\n"
                "| larger block (rows) | molecule | block Jacobi ms | blocked ms |\n|---:|---|---:|---:|\n")
        for block, kind, size, tl, th in rows_half:
            f.write(f"| {block} | {name(kind, size)} | {1e3 * tl:.1f} | {1e3 * th:.1f} |\n")
        f.write("\n## 512-molecule batch (ms per batched step)\n\n| configuration | ms |\n|---|---:|\n")
        for conf, t in rows_batch:
            f.write(f"| {conf} | {1e3 * t:.1f} |\n")
        f.write(f"\nChosen: eig_blk_min {cut_next}, eig_blk_min_first {cut}, eig_blk_min_half {cut_half}, eig_blk_iters {iters}, "
                f"jac_lanes {lanes}, jac_cross {cross}, gemm {gemm}.\n")
    return {"eig_blk_min": cut_next, "eig_blk_min_first": cut, "eig_blk_min_half": cut_half, "eig_blk_iters": iters,
            "jac_lanes": lanes, "jac_cross": cross, "gemm": gemm}


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--out", default=HERE)
    ap.add_argument("--steps", type=int, default=3)
    a = ap.parse_args(argv)
    os.makedirs(a.out, exist_ok=True)
    r = tune(a.steps, a.out, log=lambda s: print(s, flush=True))
    print(r, flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
