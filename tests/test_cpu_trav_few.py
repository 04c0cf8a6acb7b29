"""The step traversal's form for trees of a few levels (kTravFew: the identity form with
the triangle phase repeated) against the general form, on the host: same hits,
occlusion and fetch counts."""
import pytest

import raygen
from cpu_harness import harness
from test_cpu_trav_modes import GENERAL, IDENTITIES, _rays, _trace, lib  # noqa: F401

FEW = 3


@pytest.mark.parametrize("any_hit", [False, True])
@pytest.mark.parametrize("flags", [0, 1], ids=["morton", "sah"])
@pytest.mark.parametrize("name", sorted(IDENTITIES))
def test_few_levels_form(lib, name, flags, any_hit):  # noqa: F811
    sd = IDENTITIES[name]()
    hs = harness.HostScene(sd, flags)
    rays = _rays(sd, 2.0) if name != "empty" else raygen.random_rays(50, (0, 0, 0), 1.0)
    assert _trace(lib, hs, rays, FEW, any_hit) == _trace(lib, hs, rays, GENERAL, any_hit)
