"""GPU test of the three-body dispersion kernel (k_d4_atm) against the FP64
oracle, at atom counts around its steps: 64 atoms c per wave, 128 atoms b per
block held in LDS.

Both sides run the same SCC iterations in FP64, so the gradients and energies
differ by rounding only (a few 1e-12 here).  One triple of neighbouring
molecules left out or counted twice changes the gradient by more than 1e-8 and
the energy by more than 1e-9 (C9 about 1e2, distances below 10 bohr).
"""
import numpy as np
import pytest

from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def _cluster(natoms, seed):
    """`natoms` atoms of a water cluster, the last molecule cut down to H2 or
    an H2O + H2 ending (closed shells of even electron counts only)."""
    from xtb_amd import workloads as w
    nw, rest = divmod(natoms, 3)
    z, x = w.water_cluster(nw + 2, seed)
    keep = list(range(3 * nw))
    extra = []
    if rest == 2:
        extra = [np.array([0.0, 0.0, 0.0]), np.array([0.0, 0.0, 1.4])]
    elif rest == 1:
        extra = [np.array([0.0, 0.0, 0.0])]
    zz = [int(z[k]) for k in keep] + ([1] * rest if rest == 2 else [2] * rest)
    far = x[3 * nw] if nw else np.zeros(3)
    xx = [x[k] for k in keep] + [far + e for e in extra]
    return np.array(zz, dtype=np.int32), np.array(xx)


@pytest.mark.parametrize("sizes", [(1, 2, 3, 6), (63, 64, 65, 66), (126, 127, 128, 129, 130)])
def test_three_body_dispersion_against_oracle(sizes):
    import xtb_amd
    if xtb_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP runtime")
    mols = [_cluster(n, 7 + n) for n in sizes]
    b = xtb_amd.Batch(mols)
    b.run()
    res = b.results()
    b.close()
    for (z, x), r in zip(mols, res):
        assert len(z) in sizes
        o = po.singlepoint(z, x)
        assert r["iterations"] == o["iterations"], len(z)
        dg = float(np.max(np.abs(r["gradient"] - o["gradient"])))
        de = abs(r["e_disp"] - o["e_disp"])
        print(f"{len(z)} atoms: dg={dg:.2e} de={de:.2e}", flush=True)
        assert dg <= 1e-9 and de <= 1e-10, (len(z), dg, de)
