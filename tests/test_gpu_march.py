"""The gradient kernel's march: its default length where the box leaves CUs idle,
by the workgroups that share a CU (two with FP32 fluxes, one in FP64), and the
RHS bit for bit the same at every length."""
import numpy as np
import pytest

import nuc3d_amd as G
import oracle as O
from test_gpu_sweep_forms import _state

pytestmark = pytest.mark.gpu

# box, precision, planes
DEFAULTS = [((205, 210, 64), G.FP64, 32), ((205, 210, 64), G.FP32, 16), ((256, 256, 64), G.MIXED, 16),
            ((128, 128, 128), G.FP64, 16), ((128, 128, 128), G.FP32, 8), ((192, 192, 64), G.FP32, 4)]


@pytest.mark.parametrize("n,precision,planes", DEFAULTS, ids=str)
def test_default_march(n, precision, planes):
    with G.Context(G.make_config(n=n, precision=precision)) as ctx:
        assert ctx.tile_shape() == planes


@pytest.mark.parametrize("precision", [G.FP64, G.MIXED, G.FP32], ids=["fp64", "mixed", "fp32"])
@pytest.mark.parametrize("n", [(33, 17, 20), (70, 50, 37), (96, 40, 64)], ids=str)
def test_rhs_does_not_depend_on_it(n, precision):
    cfg = G.make_config(n=n, precision=precision, scheme=G.WENO5JS, vis=G.CD8)
    q = _state(O.make_config(n=n), 4)
    with G.Context(cfg) as ctx:
        ctx.upload(q)
        want, dt = ctx.rhs()
        for planes in (1, 3, 8, n[2]):
            ctx.set_tile_shape(planes)
            got, dt2 = ctx.rhs()
            assert np.array_equal(got, want) and dt2 == dt, planes
