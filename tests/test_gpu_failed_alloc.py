"""A device allocation that fails is reported once: the solves after it run.
HIP keeps a failed call's error for hipGetLastError past calls that succeed,
and every launch is checked with that; GCR on the general stencil goes on with
a launch per phase where the directions of a resident launch find no room."""
import numpy as np
import pytest

from helpers import lattice_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("on", [True, False], ids=["resident", "launches"])
@pytest.mark.parametrize("what", ["cg", "gcr"])
def test_solve_after_a_failed_allocation(glx, orc, resident, what, on):
    resident(on)
    if what == "cg":
        links, b, _ = lattice_inputs(orc, 32, 16, seed=3)
        lat = glx.Lattice(links, 32, 16)
    else:
        o = orc.CStencil.random(np.random.default_rng(1), 4, 4, 2, False)
        o.hopping *= 0.1
        o.clover = (0.1 * o.clover.reshape(-1, 2, 2) + np.eye(2)).reshape(-1)
        h = glx.CStencilDev(glx.StencilNc(4, 4, 2, o.clover, o.hopping, None, o.shift, o.eo_shift, o.dof_shift, 0))
        b = np.ones(o.n, complex)
    db, dx = glx.DeviceArray(b), glx.DeviceArray(np.zeros_like(b))
    with pytest.raises(glx.GlxError, match="memory"):
        glx.DeviceArray(nbytes=1 << 50)
    if what == "cg":
        assert glx.dev_solve("cg", lat, "staggered_normal", 0.1, dx, db).success
        r = b - orc.apply("staggered_normal", dx.download(), links, 0.1, 32, 16)
    else:
        assert h.solve("gcr", dx, db, max_iter=200, eps=1e-10).success
        r = b - orc.cstencil_apply(o, dx.download())
    assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b)
