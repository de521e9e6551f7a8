"""Optional copies never take memory that a required buffer needs (needs a GPU).

The energy octets of a grid (a second copy of its energy channel) are such a
copy.  One allocation and a row of small ones fill the device's memory for the
time of these tests; each test frees as much of it as it needs."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20
CHUNK = 64 * MB


class Card:
    """A context with one pair on it and the rest of the device's memory taken."""

    def __init__(self, W):
        from gpuattract_amd import hip
        self.hip, self.ctx = hip, hip.Context(0)
        # a body of 40 beads in grids of about 1.5 GB of octets per level
        self.wl = W.make_workload("memory", 700, 40, 30, 200, with_lig_grid=False)
        self.geoms = [W.cube_geom((0.0, 0.0, 0.0), 24.0, 0.5), W.cube_geom((0.0, 0.0, 0.0), 48.0, 1.0)]
        self.points = [16 * 13 * g.nx * g.ny * g.nz for g in self.geoms]
        self.octets = sum(128 * 13 * (g.nx - 1) * (g.ny - 1) * (g.nz - 1) for g in self.geoms)
        c, wl = self.ctx, self.wl
        self.hs = dict(rec=c.upload_protein(wl.rec), lig=c.upload_protein(wl.lig),
                       grid=c.build_grid(wl.rec, wl.params, *self.geoms), params=c.upload_params(wl.params))
        self.ref = c.adjoint(self.hs, wl.dofs)
        self.capture()
        self.big = c.dev_alloc(self.free() - 6144 * MB)
        self.chunks = []

    def capture(self):
        """A graph of one call on a grid of its own."""
        c, n = self.ctx, self.wl.dofs.shape[0]
        hs = dict(self.hs, grid=c.build_grid(self.wl.rec, self.wl.params, *self.geoms))
        self.rt, self.stream = c.L, C.c_void_p(c.new_stream())  # the runtime the library is bound to
        self.d_in, self.d_out = c.to_device(self.wl.dofs), c.dev_alloc(n * 28)
        graph, self.graph = C.c_void_p(), C.c_void_p()
        assert self.rt.hipStreamBeginCapture(self.stream, 2) == 0  # relaxed
        c.adjoint_dev_noalloc(hs, self.d_in.ptr, False, n, None, self.d_out.ptr, None, self.stream)
        assert self.rt.hipStreamEndCapture(self.stream, C.byref(graph)) == 0
        assert self.rt.hipGraphInstantiate(C.byref(self.graph), graph, None, None, C.c_size_t(0)) == 0

    def free(self):
        fr, total = C.c_size_t(), C.c_size_t()
        assert self.ctx.L.att_device_memory(self.ctx.h, C.byref(fr), C.byref(total)) == 0
        return fr.value

    def leave(self, nbytes):
        """Takes all memory (another context's allocations take no grid's), then
        frees nbytes of it (rounded up to 64 MB)."""
        other = self.hip.Context(0)
        while True:
            try:
                self.chunks.append(other.dev_alloc(CHUNK))
            except self.hip.AttError:
                break
        for _ in range(-(-nbytes // CHUNK)):
            self.chunks.pop().release()

    def open(self):
        while self.chunks:
            self.chunks.pop().release()

    def close(self):
        self.open()
        self.big.release()
        self.ctx.close()

    def scores(self, hs):
        got = self.ctx.adjoint(hs, self.wl.dofs)
        return np.array_equal(got.view(np.uint32), self.ref.view(np.uint32))


@pytest.fixture(scope="module")
def card(W):
    c = Card(W)
    yield c
    c.close()


def test_energy_octets_that_a_plan_reads_stay(card):
    """A batch plan keeps the pointers of its grids' octets: their memory is
    not taken while it lives, and the plan runs on."""
    ctx, n = card.ctx, card.wl.dofs.shape[0]
    d_in, d_out = ctx.to_device(card.wl.dofs), ctx.dev_alloc(n * 28)
    plan = ctx.batch([dict(hs=card.hs, d_dofs=d_in.ptr, d_out=d_out.ptr, n=n, modes=False)])
    plan.run()
    ctx.sync()
    try:
        card.leave(128 * MB)
        with pytest.raises(card.hip.AttError) as e:
            ctx.dev_alloc(card.octets // 5)
        assert e.value.status == 3
    finally:
        card.open()
    plan.run()
    ctx.sync()
    assert np.array_equal(ctx.to_host(d_out, (n, 7)).view(np.uint32), card.ref.view(np.uint32))
    plan.close()


def test_energy_octets_give_way_to_a_required_buffer(card):
    """A later allocation of the context that does not fit beside a grid's
    energy octets takes their memory; the grid then scores the same bits."""
    try:
        card.leave(128 * MB)
        card.ctx.dev_alloc(card.octets // 5).release()  # a little less than they take
    finally:
        card.open()
    assert card.scores(card.hs)


@pytest.mark.parametrize("uploaded", [False, True])
def test_a_grid_that_fits_without_energy_octets(card, uploaded):
    """Room for the grid's octets and the points they are made from, not for
    the energy octets of either level: the grid is there, nothing else stays
    allocated, and it scores as one with energy octets does."""
    from gpuattract_amd.workload import IGrid, NLGrid
    ctx, wl = card.ctx, card.wl
    card.open()
    if uploaded:
        grids = [IGrid(g, 13, ctx.generate_grid(wl.rec, wl.params, g)) for g in card.geoms]
        nl = NLGrid(card.geoms[0], 10.0, *ctx.generate_nl(wl.rec, card.geoms[0]))
    try:
        card.leave(card.octets + max(card.points) + 64 * MB)
        before = card.free()
        if uploaded:
            grid = ctx.upload_grid(*grids, nl)
        else:
            grid = ctx.build_grid(wl.rec, wl.params, *card.geoms)
        held = before - card.free()
    finally:
        card.open()
    assert card.octets <= held <= card.octets + 100 * MB
    assert card.scores(dict(card.hs, grid=grid))
    ctx.release(grid)


def test_energy_octets_that_a_captured_call_reads_stay(card):
    """A captured call keeps the pointers of its grid's octets: their memory
    (all that the tests above leave of it) is not taken, and the graph replays
    the same bits."""
    ctx, n = card.ctx, card.wl.dofs.shape[0]
    try:
        card.leave(128 * MB)
        with pytest.raises(card.hip.AttError) as e:
            ctx.dev_alloc(card.octets // 5)
        assert e.value.status == 3
    finally:
        card.open()
    for _ in range(2):
        ctx.write(card.d_out, np.zeros((n, 7), np.float32))
        assert card.rt.hipGraphLaunch(card.graph, card.stream) == 0
        ctx.sync(card.stream)
        got = ctx.to_host(card.d_out, (n, 7))
        assert np.array_equal(got.view(np.uint32), card.ref.view(np.uint32))
