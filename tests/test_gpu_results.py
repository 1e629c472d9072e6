"""GPU test of the whole-batch results: equal to the molecules' own, bit for
bit and of the same shapes and types, for a batch of one, of unequal sizes and
in solvent; sizes-only requests fill the scalars."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count,solvent", [(1, None), (7, None), (5, "water")])
def test_batch_results_equal_single_results(count, solvent):
    import xtb_amd
    from xtb_amd import workloads as w
    mols = [(w.water_cluster if m % 2 else w.alkane)(1 + 2 * m, m) for m in range(count)]
    b = xtb_amd.Batch([(z, x, 0.0, 0) for z, x in mols])
    if solvent:
        b.set_solvent(solvent, "p16", True)
    b.run()
    for m, r in enumerate(b.results()):
        s = b.result(m)
        assert list(r) == list(s)
        for k, v in s.items():
            assert type(r[k]) is type(v), k
            if isinstance(v, np.ndarray):
                assert r[k].shape == v.shape and r[k].dtype == v.dtype and np.array_equal(r[k], v), (m, k)
                assert r[k].flags.writeable
            else:
                assert r[k] == v, (m, k)
    b.close()
