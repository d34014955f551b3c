"""The SPH lists where their kernels change course: the wavefronts that share
a bucket's queries in the kNN (by the number of buckets, with all or few of
the particles searching).

Bars: neighbour sets equal a k-d tree's (random positions: no ties) and
fBall2 to 4 ulp (the tree forms the distance in another order); forces FP64
within 1e-12 of the oracle's or of the gathered balls' (sums in another
order); a repeated call bit for bit."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

pytestmark = pytest.mark.gpu


def put_gas(pk, d):
    pk.put("r", d["r"])
    pk.put("fMass", d["m"])
    pk.put("vPred", d["v"])
    pk.put("uPred", d["u"])


@pytest.mark.parametrize("part", [1.0, 0.05])
@pytest.mark.parametrize("n", [33, 4000, 9000, 20000, 45000, 120000, 420000])
def test_knn_wavefronts_per_bucket(gpu, n, part):
    K = 32
    rng = np.random.default_rng(n)
    r = rng.uniform(0, 1, (n, 3))
    on = rng.uniform(size=n) < part
    on[0] = True
    with gpu.Pkd(n, prec=gpu.PREC_FP64) as pk:
        put_gas(pk, dict(r=r, m=np.full(n, 1.0 / n), v=np.zeros((n, 3)), u=np.ones(n)))
        pk.put("iActive", np.where(on, 4, 0).astype(np.uint32) | gpu.TYPE_GAS | 3)
        pk.build_local()
        ns = pk.smooth(gpu.Smf.default(), K, False)
        nbr, fb2 = pk.smooth_lists(K), pk.get("fBall2")
    assert ns == on.sum()
    d, j = cKDTree(r).query(r[on], k=K)
    assert np.array_equal(np.sort(nbr[on], axis=1), np.sort(j, axis=1))
    assert np.allclose(fb2[on], d[:, -1] ** 2, rtol=4 * 2.3e-16, atol=0)
