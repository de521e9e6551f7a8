"""Alternative kernel paths give the same results, at the sizes where a path's
chunks, tiles and remainders end (needs a GPU)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from gpuattract_amd import hip
    c = hip.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("nl, mr, ml, n", [(1, 0, 0, 3), (65, 3, 0, 70), (400, 5, 5, 90)])
def test_energy_octets_same_bits(ctx, W, nl, mr, ml, n):
    """The adjoint from the energy octets and from the full octets: the same
    values are read and the same operations done, so the same bits."""
    # some poses inside the inner grid, some in the outer, some outside both
    wl = W.make_workload("octets", 300 + nl, 300, nl, n, mr, ml, shell=(5.0, 70.0),
                         with_lig_grid=False)
    hs = ctx.upload_workload(wl)
    got = ctx.adjoint(hs, wl.dofs)
    ctx.set_energy_octets(False)
    try:
        full = ctx.adjoint(ctx.upload_workload(wl), wl.dofs)
    finally:
        ctx.set_energy_octets(True)
    assert np.array_equal(got.view(np.uint32), full.view(np.uint32))
