"""What the elementwise updates hand back (counts, the largest rung, the
smallest step), at store sizes around a block, around the grid's limit and
beyond it, over repeated calls: whole numbers and minima, so exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 511, 512, 513, 262143, 262145, 700001])
def test_counts_and_reductions(gpu, n):
    rng = np.random.default_rng(n)
    bits = rng.choice(np.array([gpu.TYPE_GAS | 1, gpu.TYPE_DARK | 1], np.uint32), n)
    rung = rng.integers(0, 4, n).astype(np.int32)
    gas = (bits & gpu.TYPE_GAS) != 0
    pk = gpu.Pkd(n, prec=gpu.PREC_FP64)
    r = rng.uniform(-0.5, 0.5, (n, 3))
    pk.put("r", r)
    pk.put("iActive", bits)
    pk.put("iRung", rung)
    for k in (2, 0, 3, 2):
        assert pk.active_rung(k, True) == int((rung >= k).sum())
        assert pk.active_type(gpu.TYPE_GAS, gpu.TYPE_SMOOTHACTIVE) == int(gas.sum())
        assert np.array_equal((pk.get("iActive") & 1) != 0, rung >= k)
    dt = rng.uniform(0.11, 0.9, n)
    pk.put("iActive", bits)
    pk.put("dt", dt)
    pk.put("dtNew", np.full(n, 9.0))
    pk.put("fSoft", np.ones(n))
    dmin = pk.sph_step(1.0, 0.4)
    assert dmin == (dt[gas].min() if gas.any() else np.finfo(np.float64).max)
    top, nmax, ideal = pk.dt_to_rung(0, 1.0, 3)
    want = np.floor(1 / dt).astype(int)
    want = np.where(want == 0, 0, np.floor(np.log2(np.maximum(want, 1))).astype(int) + 1)
    assert ideal == want.max() + 1 and top == min(2, want.max())
    assert nmax == int((np.minimum(want, 2) == top).sum())
    # a drift that leaves the box counts the coordinates, one that stays none
    v = np.zeros((n, 3))
    pk.put("v", v)
    pk.drift(1.0, period=(1.0, 1.0, 1.0))
    v[n // 2, 1] = 7.0
    pk.put("v", v)
    with pytest.raises(gpu.GGError, match="1 coordinates"):
        pk.drift(1.0, period=(1.0, 1.0, 1.0))
    v[:] = 0.25
    pk.put("v", v)
    pk.put("r", r)
    pk.drift(1.0, period=(1.0, 1.0, 1.0))
    w = r + 0.25
    assert np.array_equal(pk.get("r"), np.where(w >= 0.5, w - 1.0, w))
    pk.close()


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 524287, 524289, 1100001])
def test_grav_step_over_its_blocks(gpu, n):
    rng = np.random.default_rng(n)
    on = rng.uniform(size=n) < 0.7
    on[-1] = True
    dtg, dt = rng.uniform(0.5, 2.0, n), rng.uniform(0.05, 0.2, n)
    with gpu.Pkd(n, prec=gpu.PREC_FP64) as pk:
        pk.put("r", np.zeros((n, 3)))
        pk.put("iActive", on.astype(np.uint32))
        pk.put("dtGrav", dtg)
        for _ in range(2):
            pk.put("dt", dt)
            pk.grav_step(0.1)
            assert np.array_equal(pk.get("dt"), np.where(on, np.minimum(dt, 0.1 / np.sqrt(dtg)), dt))
        bad = on & (rng.uniform(size=n) < 0.1)
        bad[-1] = True
        pk.put("dtGrav", np.where(bad, 0.0, dtg))
        with pytest.raises(gpu.GGError, match=f" {bad.sum()} active particles"):
            pk.grav_step(0.1)
        pk.put("dtGrav", dtg)
        pk.grav_step(0.1)
