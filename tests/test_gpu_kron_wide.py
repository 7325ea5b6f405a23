"""Chains of lattices with a direction of 17 to 32 sites: the factored E_K products against the dense
ones on the same fields and Philox streams -- the same decisions, G to rounding (1e-9 after two
stabilised sweeps, the bound of the narrower lattices' comparison)."""
import numpy as np
import pytest

from gpu_cases import spec_from
from latticeqmc_amd.engine import SweepEngine
from latticeqmc_amd.hubbard import HubbardModel
from oracle import model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(17, 2), (3, 32), (20, 8), (19, 21)])
def test_wide_factored_equals_dense(w, h):
    print(f"[kron wide] {w}x{h}", flush=True)
    m = HubbardModel(u=4.0, t=1.0, mu=0.3)
    m.build(w, h, cycling=(0, 1))
    k = m.ham_kinetic()
    spec = spec_from(k, 2.0, 20, 4.0, model.random_field(w * h, 20, 3), seed=5)
    kw = dict(mode="dqmc", delay=16, n_stab=6, rng="philox")
    a, b = SweepEngine([spec], **kw), SweepEngine([spec], dense_ek=True, **kw)
    try:
        n1, n2 = a.ek_split(0)
        assert n1 * n2 == w * h and max(n1, n2) > 16
        for e in (a, b):
            e.sweep(2, measure=True)
            e.sync()
        assert np.array_equal(a.field(0), b.field(0))
        for which in (0, 1):
            assert float(np.abs(a.green(0, which=which) - b.green(0, which=which)).max()) < 1e-9
    finally:
        a.close()
        b.close()
