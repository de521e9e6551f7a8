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


def test_energy_octets_dropped(ctx, W):
    """32 B per cell and grid of both levels; dropped, the same bits."""
    wl = W.make_workload("octets dropped", 310, 300, 65, 40, 2, 3, with_lig_grid=False)
    hs = ctx.upload_workload(wl)
    cells = sum((g.geom.nx - 1) * (g.geom.ny - 1) * (g.geom.nz - 1) for g in (wl.rec_inner, wl.rec_outer))
    assert ctx.grid_energy_bytes(hs["grid"]) == 32 * 13 * cells
    ref = ctx.adjoint(hs, wl.dofs)
    ctx.drop_energy_octets(hs["grid"])
    ctx.drop_energy_octets(hs["grid"])
    assert ctx.grid_energy_bytes(hs["grid"]) == 0
    assert np.array_equal(ctx.adjoint(hs, wl.dofs).view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("nl, mr, ml", [(1, 0, 0), (64, 0, 0), (257, 0, 0), (384, 0, 0), (67, 0, 7),
                                        (130, 1, 0), (300, 5, 5), (383, 10, 4), (513, 4, 9),
                                        (520, 10, 10)])
def test_list_walk_by_quads_is_the_kernel_order(ctx, W, O, nl, mr, ml):
    """Lists of every length (poses from contact to out of reach), queues that
    are no multiple of the 16 beads a wave walks at once, one to three
    super-chunks, every mode capacity: the oracle's kernel-order bits."""
    wl = W.make_workload("quads", 400 + nl, 250, nl, 24, mr, ml, shell=(8.0, 45.0),
                         with_lig_grid=False)
    hs = ctx.upload_workload(wl)
    w = np.linspace(-1.0, 2.0, 24).astype(np.float32)
    got = ctx.adjoint(hs, wl.dofs, w=w)
    ref = O.adjoint_kernel_order(wl, w=w)[:, :got.shape[1]].astype(np.float32)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


def test_receptor_bead_with_a_non_finite_mode_is_skipped(ctx, W, O):
    """Its pairs have no finite distance: they add nothing to any sum."""
    wl = W.make_workload("nan mode", 420, 250, 90, 30, 3, 2, shell=(8.0, 30.0), with_lig_grid=False)
    m = wl.rec.modes.reshape(3, wl.rec.n, 3)
    m[0, ::7, 1] = np.nan
    m[2, ::11, 2] = np.inf
    got = ctx.adjoint(ctx.upload_workload(wl), wl.dofs)
    ref = O.adjoint_kernel_order(wl)[:, :got.shape[1]].astype(np.float32)
    assert np.isfinite(got).all()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("nl, mr, ml", [(1, 1, 0), (67, 0, 7), (257, 5, 2), (384, 3, 5), (1030, 10, 10)])
def test_forward_walk_by_quads_is_the_reference_order(ctx, W, O, nl, mr, ml):
    """The forward kernels over lists of every length, one to four waves per
    pose, one to two super-chunks: the oracle's (the reference's) bits; the
    receptor mode gradients, projected per pair, to 1e-5 of their norm."""
    wl = W.make_workload("quads forward", 430 + nl, 250, nl, 20, mr, ml, shell=(8.0, 45.0))
    hs = ctx.upload_workload(wl)
    g, o = ctx.score_modes(hs, wl.dofs), O.score_modes(wl, nthreads=8)
    keep = list(range(7)) + list(range(17, 27))
    assert np.array_equal(g[:, keep].view(np.uint32), o[:, keep].view(np.uint32))
    r, q = g[:, 7:7 + mr].astype(np.float64), o[:, 7:7 + mr].astype(np.float64)
    fin = np.isfinite(q).all(axis=1)
    assert np.array_equal(fin, np.isfinite(r).all(axis=1))
    off = np.linalg.norm(r[fin] - q[fin], axis=1)
    assert np.all(off <= 1e-5 * np.linalg.norm(q[fin], axis=1) + 1e-30)
    d6 = np.ascontiguousarray(wl.dofs[:, :6])
    rigid = ctx.score_rigid(hs, d6)
    assert np.array_equal(rigid.view(np.uint32), O.score_rigid(wl, d6, nthreads=8).view(np.uint32))


@pytest.mark.parametrize("nl, mr, ml", [(80, 0, 0), (300, 0, 0), (400, 0, 0), (70, 2, 3), (300, 5, 5),
                                        (400, 4, 0), (600, 8, 10)])
def test_call_size_changes_no_bit(ctx, W, nl, mr, ml):
    """Few poses per call get more waves per pose: every pose scores the same
    bits in one large call and in calls of every width (the widths change
    between 512 and 2048 poses on 256 CUs, and with the ligand's size)."""
    n = 4300
    wl = W.make_workload("call size", 440 + nl + mr, 250, nl, n, mr, ml)
    hs = ctx.upload_workload(wl)
    whole = ctx.adjoint(hs, wl.dofs)
    rigid = np.ascontiguousarray(wl.dofs[:, :6])
    score = ctx.score_rigid(hs, rigid)
    for a, b in ((0, 1), (1, 513), (513, 513 + 1024), (1537, 1537 + 2049)):
        part = ctx.adjoint(hs, wl.dofs[a:b])
        assert np.array_equal(part.view(np.uint32), whole[a:b].view(np.uint32)), (a, b)
        part = ctx.score_rigid(hs, rigid[a:b])
        assert np.array_equal(part.view(np.uint32), score[a:b].view(np.uint32)), (a, b)


@pytest.mark.parametrize("n, mr, ml", [(1, 0, 0), (17, 10, 10), (33, 10, 8), (15, 2, 1)])
def test_minimizer_steps_in_lds(ctx, W, O, n, mr, ml):
    """Pose counts around the 16 (or, with 25 variables or more, 8) poses whose
    minimizers a workgroup advances: the oracle's trajectories."""
    wl = W.make_workload("lds steps", 460 + n, 200, 60, n, mr, ml, with_lig_grid=False)
    d, el, eb, nf = ctx.minimize(ctx.upload_workload(wl), wl.dofs, 25)
    od, oel, oeb, onf = O.minimize_kernel_order(wl, ivmax=25)
    assert np.array_equal(nf, onf)
    assert np.array_equal(d.view(np.uint32), od.astype(np.float32).view(np.uint32)[:, :d.shape[1]])
    assert np.array_equal(el.view(np.uint32), oel.astype(np.float32).view(np.uint32))
    assert np.array_equal(eb.view(np.uint32), oeb.astype(np.float32).view(np.uint32))


@pytest.mark.parametrize("types, n, weights", [(1, 40, False), (2, 1, True), (12, 700, True),
                                               (16, 90, False), (17, 90, True), (32, 90, False),
                                               (33, 60, True), (40, 60, False)])
def test_parameter_gradient_cell_pass(ctx, W, O, types, n, weights):
    """One and two matrix tiles of types, full and not, and the run pass above
    them; one workgroup's share from nothing to many buckets.  FP64 oracle to
    1e-4 of the largest entry, the per-bead basis path (16 types at most) to
    FP32 rounding (1e-5), and the same bits in a second call."""
    wl = W.make_workload("cells", 500 + types, 300, 130, n, 0, 0, num_types=types,
                         with_basis=True, shell=(8.0, 45.0), type0_frac=0.05)
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    w = np.linspace(-1.0, 2.0, n).astype(np.float32) if weights else None
    T = wl.params.T
    _, pg = ctx.adjoint(hs, wl.dofs, w=w, pgrad=True, T=T)
    _, again = ctx.adjoint(hs, wl.dofs, w=w, pgrad=True, T=T)
    assert np.array_equal(pg.view(np.uint32), again.view(np.uint32))
    ref = O.adjoint(wl, w=None if w is None else w.astype(np.float64), pgrad=True)[1].reshape(-1)
    assert np.abs(pg.reshape(-1) - ref).max() <= 1e-4 * np.abs(ref).max()
    if T > 16:
        return
    d_in, d_w = ctx.to_device(wl.dofs), None if w is None else ctx.to_device(w)
    d_out, d_pg = ctx.dev_alloc(n * 7 * 4), ctx.dev_alloc(3 * T * T * 4)
    ctx.adjoint_dev_noalloc(hs, d_in.ptr, False, n, d_w and d_w.ptr, d_out.ptr, d_pg.ptr)
    ctx.sync()
    beads = ctx.to_host(d_pg, (3 * T * T,))
    assert np.abs(pg.reshape(-1) - beads).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("types", [12, 20])
def test_parameter_gradient_basis_value_not_finite(ctx, W, types):
    """It reaches the types of the beads beside it and no others: everything
    that stays finite is what the finite basis gives (and, with 16 types or
    fewer, finite in the per-bead basis path too)."""
    wl = W.make_workload("cells inf", 540 + types, 300, 130, 12, 0, 0, num_types=types,
                         with_basis=True, shell=(8.0, 30.0))
    n, T = wl.dofs.shape[0], wl.params.T
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    clean = ctx.adjoint(hs, wl.dofs, pgrad=True, T=T)[1]
    # receptor type 1: some points of both grids; infinite in the inner, NaN in the outer
    nv = wl.rec_inner_basis.size // (2 * types)
    wl.rec_inner_basis[0:nv:97] = np.inf
    nv = wl.rec_outer_basis.size // (2 * types)
    wl.rec_outer_basis[nv:2 * nv:151] = np.nan
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    pg = ctx.adjoint(hs, wl.dofs, pgrad=True, T=T)[1]
    ok = np.isfinite(pg)
    assert ok[T:].all() and ok[:, 2].all()
    assert not ok[:T, :2].all() and ok[:T, :2].any()
    assert np.abs(pg - clean)[ok].max() <= 1e-5 * np.abs(clean).max()
    if T > 16:
        return
    d_in, d_out, d_pg = ctx.to_device(wl.dofs), ctx.dev_alloc(n * 28), ctx.dev_alloc(12 * T * T)
    ctx.adjoint_dev_noalloc(hs, d_in.ptr, False, n, None, d_out.ptr, d_pg.ptr)
    ctx.sync()
    assert np.array_equal(np.isfinite(ctx.to_host(d_pg, (T * T, 3))), ok)


@pytest.mark.parametrize("nl, mr, ml, n", [(20, 0, 0, 16391), (20, 0, 0, 33001), (400, 0, 0, 8501),
                                           (70, 5, 3, 16385), (40, 10, 10, 12300), (390, 2, 9, 6203)])
def test_poses_drawn_from_queues(ctx, W, nl, mr, ml, n):
    """Calls of a few rounds of poses, no multiple of the eight ranges: every
    pose is scored, with the bits of the input order."""
    wl = W.make_workload("queues", 600 + nl, 120, nl, n, mr, ml, shell=(5.0, 60.0),
                         with_lig_grid=False)
    hs = ctx.upload_workload(wl)
    w = np.linspace(0.5, 1.5, n).astype(np.float32)
    got = ctx.adjoint(hs, wl.dofs, w=w)
    again = ctx.adjoint(hs, wl.dofs, w=w)
    ctx.set_pose_order(False)
    try:
        ref = ctx.adjoint(hs, wl.dofs, w=w)
    finally:
        ctx.set_pose_order(True)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
    assert np.array_equal(again.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("kind, width, waves, n", [("rigid", 7, 4, (1 << 24) + 4096),
                                                   ("modes", 27, 8, (1 << 23) + 4096)])
def test_call_of_more_poses_than_one_launch_holds(ctx, W, kind, width, waves, n):
    """A launch has fewer than 2^32 threads: with a ligand of over 384 beads
    and four waves per pose, fewer than 2^24 poses (and with eight, which
    flexible calls can ask for, 2^23).  Every pose of a larger call is scored,
    with the bits of a small call."""
    wl = W.make_workload("many poses", 620, 30, 385, 64, 1, 1, spacing=2.0)
    hs = ctx.upload_workload(wl)
    dofs = wl.dofs if kind == "modes" else np.ascontiguousarray(wl.dofs[:, :6])
    ctx.set_modes_waves(waves if kind == "modes" else 0)
    try:
        ref = (ctx.score_modes if kind == "modes" else ctx.score_rigid)(hs, dofs)
        d_in, d_out = ctx.to_device(np.tile(dofs, (n // 64, 1))), ctx.dev_alloc(n * width * 4)
        (ctx.score_modes_dev if kind == "modes" else ctx.score_rigid_dev)(hs, d_in.ptr, n, d_out.ptr)
        ctx.sync()
    finally:
        ctx.set_modes_waves(0)
    got = ctx.to_host(d_out, (n // 64, 64 * width)).view(np.uint32)
    assert (got == ref.reshape(-1).view(np.uint32)).all()


@pytest.mark.parametrize("nl, mr", [(390, 0), (390, 2), (300, 0)])
def test_parameter_gradient_of_the_widest_tables(ctx, W, O, nl, mr):
    """The parameter sums of 79 types and a ligand of two waves nearly fill a
    workgroup's LDS: accepted with and without modes, and with one wave."""
    wl = W.make_workload("wide table", 579 + nl, 40, nl, 6, mr, 0, num_types=79, with_basis=True,
                         shell=(8.0, 30.0), with_lig_grid=False)
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    out, pg = ctx.adjoint(hs, wl.dofs, pgrad=True, T=79)
    plain = ctx.adjoint(hs, wl.dofs)
    assert np.array_equal(out.view(np.uint32), plain.view(np.uint32))
    ref = O.adjoint(wl, pgrad=True)[1].reshape(-1)
    assert np.abs(pg.reshape(-1) - ref).max() <= 1e-4 * np.abs(ref).max()


@pytest.mark.parametrize("types, n, places, weights", [(12, 8192, 0, True), (12, 8192, 1, False),
                                                       (16, 8200, 3, True), (32, 8192, 0, False),
                                                       (32, 8300, 2, True)])
def test_parameter_gradient_cell_pass_over_many_steps(ctx, W, O, types, n, places, weights):
    """Several steps of 64 records per workgroup, buckets that go on from one
    to the next, and poses at a few places only (whole steps of one cell and
    type): FP64 oracle to 1e-4 of the largest entry, the per-bead basis path
    (16 types at most) to FP32 rounding, and the same bits in a second call."""
    wl = W.make_workload("cell steps", 560 + types + places, 300, 130, n, 0, 0, num_types=types,
                         with_basis=True, shell=(8.0, 45.0), type0_frac=0.05)
    if places:
        wl.dofs = np.ascontiguousarray(wl.dofs[np.arange(n) % places])
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    w = np.linspace(-1.0, 2.0, n).astype(np.float32) if weights else None
    T = wl.params.T
    _, pg = ctx.adjoint(hs, wl.dofs, w=w, pgrad=True, T=T)
    _, again = ctx.adjoint(hs, wl.dofs, w=w, pgrad=True, T=T)
    assert np.array_equal(pg.view(np.uint32), again.view(np.uint32))
    ref = O.adjoint(wl, w=None if w is None else w.astype(np.float64), pgrad=True)[1].reshape(-1)
    assert np.abs(pg.reshape(-1) - ref).max() <= 1e-4 * np.abs(ref).max()
    if T > 16:
        return
    d_in, d_w = ctx.to_device(wl.dofs), None if w is None else ctx.to_device(w)
    d_out, d_pg = ctx.dev_alloc(n * 7 * 4), ctx.dev_alloc(3 * T * T * 4)
    ctx.adjoint_dev_noalloc(hs, d_in.ptr, False, n, d_w and d_w.ptr, d_out.ptr, d_pg.ptr)
    ctx.sync()
    beads = ctx.to_host(d_pg, (3 * T * T,))
    assert np.abs(pg.reshape(-1) - beads).max() <= 1e-5 * np.abs(ref).max()


def test_parameter_gradient_of_equal_poses_is_their_number_of_one(ctx, W):
    """400,000 equal poses out of reach of the receptor's beads (the grid part
    alone): 2000 records of one cell and type per workgroup.  A sum of at most
    32 steps' trees (6 levels), the 8 corners and the products: 50 roundings of
    2^-24 against one pose's gradient, times the number."""
    n = 400000
    wl = W.make_workload("equal poses", 590, 300, 20, 400, 0, 0, with_basis=True, shell=(8.0, 45.0))
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    far = wl.dofs[np.argmax(np.linalg.norm(wl.dofs[:, :3], axis=1))][None]
    assert ctx.pair_counts(lambda: ctx.adjoint(hs, far), 1)[0, 1] == 0
    one = ctx.adjoint(hs, far, pgrad=True, T=12)[1].astype(np.float64) * n
    assert (one[:, 2] == 0).all() and one[:, :2].any()
    many = ctx.adjoint(hs, np.repeat(far, n, axis=0), pgrad=True, T=12)[1].astype(np.float64)
    assert np.all(np.abs(many - one) <= 50 * 2.0 ** -24 * np.abs(one))


def test_parameter_gradient_buckets_of_64_cells(ctx, W, O):
    """2.4 million cells: 64 to a bucket, with 16 types the largest LDS.  3000
    poses 90 times over are two records per cell."""
    wl = W.make_workload("fine grid", 701, 30, 20, 3000, 0, 0, num_types=16, with_basis=True,
                         shell=(8.0, 20.0), outer_spacing=0.42, with_lig_grid=False)
    g = wl.rec_outer.geom
    assert (g.nx - 1) * (g.ny - 1) * (g.nz - 1) > 32 * 65536
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    pg = ctx.adjoint(hs, np.tile(wl.dofs, (90, 1)), pgrad=True, T=16)[1].reshape(-1)
    ref = 90 * O.adjoint(wl, pgrad=True)[1].reshape(-1)
    assert np.abs(pg - ref).max() <= 1e-4 * np.abs(ref).max()


def coarse(W, name, seed, types, n, **kw):
    """A pair on grids of some 30,000 cells: calls of a few hundred poses have
    more than two records per cell (the bucket pass)."""
    wl = W.make_workload(name, seed, 300, 130, n, 0, 0, num_types=types, with_basis=True, spacing=2.0,
                         outer_spacing=6.0, with_lig_grid=False, **kw)
    cells = sum((g.geom.nx - 1) * (g.geom.ny - 1) * (g.geom.nz - 1) for g in (wl.rec_inner, wl.rec_outer))
    return wl, cells


@pytest.mark.parametrize("types, weights", [(5, False), (6, True), (12, False), (16, True), (17, False),
                                            (31, True), (32, False), (33, False)])
@pytest.mark.parametrize("side", [-1, 0])
def test_parameter_gradient_passes_on_either_side_of_their_line(ctx, W, O, types, weights, side):
    """One pose under the bucket pass's records per cell (1.1 or 2), and the first
    number of poses from there on, by tables around its limits: FP64 oracle to 1e-4 of
    the largest entry, the per-bead basis path (16 types at most) to 1e-5."""
    _, cells = coarse(W, "line", 800 + types, types, 1)
    line = cells + cells // 10 if 10 <= types <= 16 else 2 * cells
    n = -(-line // 130) + side
    wl, _ = coarse(W, "line", 800 + types, types, n, shell=(8.0, 45.0), type0_frac=0.05)
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    w = np.linspace(-1.0, 2.0, n).astype(np.float32) if weights else None
    T = wl.params.T
    pg = ctx.adjoint(hs, wl.dofs, w=w, pgrad=True, T=T)[1].reshape(-1)
    ref = O.adjoint(wl, w=None if w is None else w.astype(np.float64), pgrad=True)[1].reshape(-1)
    assert np.abs(pg - ref).max() <= 1e-4 * np.abs(ref).max()
    if T > 16:
        return
    d_in, d_w = ctx.to_device(wl.dofs), None if w is None else ctx.to_device(w)
    d_out, d_pg = ctx.dev_alloc(n * 7 * 4), ctx.dev_alloc(3 * T * T * 4)
    ctx.adjoint_dev_noalloc(hs, d_in.ptr, False, n, d_w and d_w.ptr, d_out.ptr, d_pg.ptr)
    ctx.sync()
    beads = ctx.to_host(d_pg, (3 * T * T,))
    assert np.abs(pg - beads).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("types", [12, 20])
def test_parameter_gradient_bucket_basis_value_not_finite(ctx, W, types):
    """As test_parameter_gradient_basis_value_not_finite, with records enough
    for the bucket pass: the values reach the types of the beads beside them
    and no others."""
    wl, cells = coarse(W, "buckets inf", 840 + types, types, 600, shell=(8.0, 30.0))
    n, T = wl.dofs.shape[0], wl.params.T
    assert n * 130 >= 2 * cells
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    clean = ctx.adjoint(hs, wl.dofs, pgrad=True, T=T)[1]
    # receptor type 1: some points of both grids; infinite in the inner, NaN in the outer
    nv = wl.rec_inner_basis.size // (2 * types)
    wl.rec_inner_basis[0:nv:997] = np.inf
    nv = wl.rec_outer_basis.size // (2 * types)
    wl.rec_outer_basis[nv:2 * nv:499] = np.nan
    hs = ctx.upload_workload(wl)
    ctx.upload_basis(hs["grid"], wl)
    pg = ctx.adjoint(hs, wl.dofs, pgrad=True, T=T)[1]
    ok = np.isfinite(pg)
    assert ok[T:].all() and ok[:, 2].all() and not ok[:T, :2].all()
    assert np.abs(pg - clean)[ok].max() <= 1e-5 * np.abs(clean).max()
