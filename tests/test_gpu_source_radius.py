"""A flux source acts within |radius| of its place (only the radius' square is
compared), also where the radius is given with a minus sign: the state after a
few steps, bit for bit, on a 2D and a 1D grid."""
import copy

import numpy as np
import pytest

from kestrel_amd import config as C
from kestrel_amd import scenario as S
from kestrel_amd.runtime import Stepper
from tests.helpers import FIELDS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [(5, 5, 16, 16), (7, 1, 20, 1)], ids=["2d", "1d"])
def test_sign_of_the_radius(gpu, tiles):
    cfg = C.default_config(*tiles, dx=1.0)
    C.hydraulic_only(cfg)
    C.derive(cfg)
    b0v = S.topo_xslope(cfg, 0.1)
    src = C.FluxSource(0.5, 0.5, 3.0, [0.0, 100.0], [5.0, 5.0], [0.0, 0.0])
    init = S.initial_state(cfg, b0v, [], [src])
    states = []
    for sign in (1.0, -1.0):
        s = copy.copy(src)
        s.radius = sign * src.radius
        C.set_sources(cfg, [s])
        g = Stepper(cfg)
        g.set_topography(b0v)
        g.set_state(init)
        g.step_n(10)
        states.append(g.state())
        g.close()
    assert states[0]["Hn"].max() > 0.0, "the source must emit"
    for f in FIELDS:
        assert np.array_equal(states[0][f], states[1][f]), f
