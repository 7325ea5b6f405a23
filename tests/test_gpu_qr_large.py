"""The stable G of chains above 256 sites (QR over several workgroups up to 640 sites, one workgroup
above) against the oracle's, at the edges of that range, batched with a small chain; then a sweep,
whose recomputes have to meet the propagated G."""
import numpy as np
import pytest

from gpu_cases import spec_from
from latticeqmc_amd.engine import SweepEngine
from oracle import dqmc, model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(13, 20), (17, 16), (20, 32), (23, 28)])
def test_large_chain_recompute_matches_oracle(w, h):
    print(f"[qr large] {w}x{h} with 3x5", flush=True)
    cases = [(model.square_k(w, h), model.random_field(w * h, 16, 1)), (model.square_k(3, 5), model.random_field(15, 16, 2))]
    eng = SweepEngine([spec_from(k, 1.6, 16, 4.0, f) for k, f in cases], mode="dqmc", delay=16, n_stab=4, rng="philox")
    for i, (k, f) in enumerate(cases):
        o = dqmc.DQMCOracle(k, 1.6, 16, 4.0, f, n_stab=4)
        g = eng.green(i, which=0)
        assert max(np.abs(g[s] - o.g[s]).max() for s in range(2)) < 1e-10
    eng.sweep(1, measure=True)
    eng.sync()
    for i in range(2):
        assert eng.recompute_errors(i).max() < 1e-9
        assert eng.stats(i)["flags"] == 0
    eng.close()
