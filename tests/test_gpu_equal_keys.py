"""Boxes of equal monomers, where every pick falls among equal keys: the steps are
the oracle's, and those of a small box still share launches."""
import numpy as np
import pytest

import oracle_lib as O
from mcac_amd import ensemble

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,fv,steps", [(300, 1e-4, 900), (500, 2e-3, 600), (700, 1e-4, 500), (2500, 1e-3, 300)])
def test_steps_of_equal_monomers_share_launches(n, fv, steps):
    import mcac_amd
    print(f"case: {n} equal monomers, volume fraction {fv}", flush=True)
    ini = ensemble.box_ini(n, fv, 1500.0, 11, sd_d=0.0)
    sim = mcac_amd.Simulation(ini, trace_steps=True)
    ora = O.OracleSim(ini, fast_init=True)
    assert sim.run(steps) == ora.run(steps) == steps
    assert sim.steps().tobytes() == ora.steps().tobytes()
    ties, runs = sim.scalar("ties"), sim.scalar("step_runs")
    print(f"  {ties} ties, {runs} launches of steps", flush=True)
    assert ties > 0.8 * steps
    if n <= 500:  # a pick takes less than a step
        assert runs < 0.5 * steps
    sim.close()
