"""The count of hydraulic RHS evaluations that a run reports, against the
oracle's: hydraulic and Strang steps, with attempts refused by the CFL
re-checks and by the morphodynamic checks, in a run, a batch and a profiled
run, in both sub-block shapes."""
import numpy as np
import pytest

from kestrel_amd import workloads
from kestrel_amd.runtime import Batch
from tests.helpers import oracle_for, stepper_for

pytestmark = pytest.mark.gpu

# algebraic closures: the same step control as the oracle's, bit for bit
ALGEBRAIC = dict(erosion="fluid", deposition="simple", transition="none", damping="none")


def _hydraulic():
    wl = workloads.plain_cap(128, 0, tile=16, cap_x=0.0, cap_radius=12.0)
    wl.cfg.max_dt = 10.0
    return wl


def _wide():
    wl = workloads.morpho_cap(256, 0, tile=16, radius=392.0, dx=4.0, erosion="simple", deposition="simple",
                              transition="step", damping="rat3")
    wl.cfg.max_dt = 10.0
    return wl


CASES = {
    "hydraulic": _hydraulic,
    "morpho": lambda: workloads.morpho_cap(64, 0, tile=16, **ALGEBRAIC),
    "morpho_refused": lambda: workloads.morpho_cap(64, 0, tile=16, ero_rate=0.2, ero_critical_height=1e-4, **ALGEBRAIC),
    "morpho_recheck": lambda: workloads.morpho_cap(64, 0, tile=16, ero_rate=0.5, height=3.0, **ALGEBRAIC),
    "morpho_wide": _wide,
}


@pytest.mark.parametrize("how", ["run", "profiled", "batch"])
@pytest.mark.parametrize("name", CASES)
def test_rhs_evaluations(gpu, name, how):
    n = 12
    wl = CASES[name]()
    so = oracle_for(wl).step_n(n)
    g = stepper_for(wl)
    if how == "batch":
        b = Batch(2)
        s = b.attach(g)
        b.start(s, nsteps=n)
        b.run()
        sg = b.stats(s)
    else:
        g.profile(how == "profiled")
        sg = g.step_n(n)
    assert (sg["steps"], sg["rejected"]) == (so["steps"], so["rejected"])
    assert sg["rhs_evals"] == so["rhs_evals"]
    if name.startswith("morpho_"):
        assert so["rejected"] > 0, "attempts must be refused"
