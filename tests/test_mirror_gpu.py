"""Mirrored tiles of the near-field plan (needs a GPU).

A plan over one index array whose blocks come in mirrored pairs evaluates
each pair of triangles once for both entries; the persistent schedule does
not, and evaluates every tile for itself.  Constant basis: the same bits;
linear basis: the same up to the order of the sums (1e-14 of the largest
entry, a few thousand terms).  Both against the oracle to 1e-12.  The blocks
have sides of 1, 2, 63, 64 and 65 DOFs (diagonal tiles of odd and even
size, tile edges and remainders).
"""
import numpy as np
import pytest

from conftest import rel_block_err
from oracle_ffi import OracleBem

pytestmark = pytest.mark.gpu

SIDES = (1, 2, 63, 64, 65)


def mirrored_blocks(sides=SIDES):
    off = np.concatenate([[0], np.cumsum(sides)])
    return [(int(off[i]), sides[i], int(off[j]), sides[j])
            for i in range(len(sides)) for j in range(len(sides))]


def run(h, plan, op, schedule):
    plan.set_schedule(*schedule)
    out = h.DeviceArray(plan.entries, op.dtype)
    out.fill_nan()
    stream = h.Stream()
    plan.execute(op, out.ptr, stream.handle)
    stream.sync()
    return out.download()


# wave numbers below the tiny-phase bound 2 |k| h <= 1/4 (k = 0.41 on this mesh,
# h = 0.3015) and on both sides of the small-phase bound pi/4 (k = 1.3
# and 1.31), and a damped one
@pytest.mark.parametrize("kern,k", [(0, 0.0), (1, 0.41), (1, 1.3), (1, 1.31),
                                    (1, 1.3 + 0.5j)])
@pytest.mark.parametrize("layer", [0, 1, 2])
@pytest.mark.parametrize("basis", [0, 1])
def test_mirrored_tiles_match_single_tiles(kern, k, layer, basis, sphere8):
    import h2lib_amd as h
    gr = h.Surface3d(sphere8["x"], sphere8["t"])
    n = gr.vertices if basis else gr.triangles
    idx = np.random.default_rng(3).permutation(n).astype(np.uint32)
    blocks = mirrored_blocks()
    plan = h.NearfieldPlan(gr, basis, basis, idx, idx.copy(), blocks)
    alpha = 0.5 if layer else 0.0
    op = h.Bem3d(gr, kern, layer, 2, 4, basis, basis, alpha=alpha, k=k)
    orc = OracleBem(kern, layer, basis, basis, sphere8["x"], sphere8["t"],
                    q=2, q2=4, alpha=alpha, k=k)
    for mode in (0, 1, 2):
        op.set_precision(mode)
        got = run(h, plan, op, (0, 0, 0))
        want = run(h, plan, op, (0, 1, 0))
        if basis == 0:
            assert np.array_equal(got, want), mode
        else:
            err = np.abs(got - want).max() / np.abs(want).max()
            # mixed precision sums FP32 values formed from the other
            # triangle's anchor point: FP32 rounding of the entries
            assert err < (1e-14 if mode == 0 else 2e-6), (mode, err)
        if mode == 0:
            for b in (0, 1, 6, 12, 14, 18, 22, 24):
                ro, r, co, c = blocks[b]
                ref = orc.nearfield(idx[ro:ro + r], idx[co:co + c])
                assert rel_block_err(plan.block(got, b), ref) < 1e-12, b


@pytest.mark.parametrize("basis", [0, 1])
def test_unpaired_and_repeated_blocks_keep_single_tiles(basis, sphere8):
    """A block without its mirror, a block listed twice and index arrays that
    repeat DOFs take the general path or give its entries."""
    import h2lib_amd as h
    gr = h.Surface3d(sphere8["x"], sphere8["t"])
    n = gr.vertices if basis else gr.triangles
    rng = np.random.default_rng(4)
    idx = rng.permutation(n).astype(np.uint32)
    rep = idx.copy()
    rep[10] = rep[70]
    rep[71] = rep[72]
    op = h.Bem3d(gr, 0, 1, 2, 4, basis, basis, alpha=0.5)
    orc = OracleBem(0, 1, basis, basis, sphere8["x"], sphere8["t"], q=2,
                    q2=4, alpha=0.5)
    full = mirrored_blocks()
    for ix, blocks in ((idx, full[:-1]), (idx, full + full[1:2]),
                       (rep, full)):
        plan = h.NearfieldPlan(gr, basis, basis, ix, ix, blocks)
        got = run(h, plan, op, (0, 0, 0))
        want = run(h, plan, op, (0, 1, 0))
        scale = np.abs(want).max()
        assert np.abs(got - want).max() <= (1e-14 * scale if basis else 0.0)
        for b, (ro, r, co, c) in enumerate(blocks):
            ref = orc.nearfield(ix[ro:ro + r], ix[co:co + c])
            assert rel_block_err(plan.block(got, b), ref) < 1e-12, b


@pytest.mark.parametrize("kern,k", [(0, 0.0), (1, 2.0)])
@pytest.mark.parametrize("layer", [1, 2])
@pytest.mark.parametrize("basis", [0, 1])
def test_given_normals_that_are_not_perpendicular(kern, k, layer, basis,
                                                  sphere8):
    """A surface may be given any normals; the double layers' kernels take
    them as they are: <x - y, n> of every point."""
    import h2lib_amd as h
    x, t = sphere8["x"], sphere8["t"]
    plain = h.Surface3d(x, t)
    tilt = plain.n + 0.1 * np.roll(plain.n, 1, axis=1)
    dofs = plain.vertices if basis else plain.triangles
    rng = np.random.default_rng(8)
    ridx = rng.permutation(dofs).astype(np.uint32)
    blocks = mirrored_blocks((64, 9))
    vals = []
    # <d, n> is linear in n: the entries of the tilted normals are those of
    # the true ones plus a tenth of those of the rolled ones (which are not
    # perpendicular either)
    for nn in (plain.n, np.roll(plain.n, 1, axis=1), tilt):
        gr = h.Surface3d(x, t, nn, plain.g)
        op = h.Bem3d(gr, kern, layer, 2, 4, basis, basis, alpha=0.0, k=k)
        plan = h.NearfieldPlan(gr, basis, basis, ridx, ridx, blocks)
        vals.append([run(h, plan, op, s) for s in ((0, 0, 0), (0, 1, 0),
                                                   (0, 0, 1))])
    for a, b, c in zip(*vals):
        # (cancellation in the rolled entries: their scale bounds the error)
        scale = max(np.abs(b).max(), np.abs(a).max())
        assert np.abs(c - (a + 0.1 * b)).max() < 1e-13 * scale


@pytest.mark.parametrize("kern,k", [(0, 0.0), (1, 2.0)])
@pytest.mark.parametrize("layer", [1, 2])
@pytest.mark.parametrize("basis", [0, 1])
@pytest.mark.parametrize("perm", [(0, 2, 1), (2, 1, 0), (1, 0, 2)])
def test_folded_sheets_take_differences(kern, k, layer, basis, perm):
    """Two coplanar sheets folded at an edge, 1e-6 apart within their plane:
    quadrature points nearly coincide (for one of the orders of the vertices)
    and the double layers are rounding noise.  Formed from x - y, <x - y, n>
    stays linear in n to the rounding of one product of vectors, a few 1e-16
    of the values with normals in the plane; from a triangle's plane it is
    off by 1e-16 h / r of them, 1e-10."""
    import h2lib_amd as h
    m = 6
    q, _ = np.linalg.qr(np.random.default_rng(2).normal(size=(3, 3)))
    grid = np.array([(i / m, j / m, 0.0) for i in range(m + 1)
                     for j in range(m + 1)])
    x = np.concatenate([grid, grid + [0.0, 1e-6, 0.0]]) @ q.T
    nv = len(grid)
    t = []
    for i in range(m):
        for j in range(m):
            a = i * (m + 1) + j
            b, c, d = a + m + 1, a + m + 2, a + 1
            t += [(a, b, c), (a, c, d)]
    # the second sheet's vertices on the fold i = m are the first's
    back = np.where(np.arange(nv) >= m * (m + 1), np.arange(nv),
                    np.arange(nv) + nv)
    t = np.array(t, dtype=np.uint32)
    t = np.concatenate([t, back[t][:, perm]]).astype(np.uint32)
    used = np.unique(t)
    t = np.searchsorted(used, t).astype(np.uint32)
    x = np.ascontiguousarray(x[used])
    plain = h.Surface3d(x, t)
    assert np.allclose(plain.n[0], -plain.n[len(t) // 2])
    roll = np.roll(plain.n, 1, axis=1)
    dofs = plain.vertices if basis else plain.triangles
    idx = np.random.default_rng(8).permutation(dofs).astype(np.uint32)
    blocks = mirrored_blocks((64, 13))
    vals = []
    for nn in (plain.n, roll, plain.n + 0.1 * roll):
        gr = h.Surface3d(x, t, nn, plain.g)
        op = h.Bem3d(gr, kern, layer, 2, 4, basis, basis, alpha=0.0, k=k)
        plan = h.NearfieldPlan(gr, basis, basis, idx, idx, blocks)
        vals.append([run(h, plan, op, s) for s in ((0, 0, 0), (0, 1, 0),
                                                   (0, 0, 1))])
    for a, b, c in zip(*vals):
        assert np.abs(c - (a + 0.1 * b)).max() < 1e-13 * np.abs(b).max()


@pytest.mark.parametrize("kern,k", [(0, 0.0), (1, 0.05), (1, 6.0),
                                    (1, 2.0 + 0.5j)])
@pytest.mark.parametrize("layer", [1, 2])
@pytest.mark.parametrize("surface", ["folded", "tilted"])
def test_constant_basis_bits_in_every_schedule(kern, k, layer, surface,
                                               sphere8):
    """Surfaces whose double layers take <x - y, n> per value: the entries of
    the constant basis have the same bits in every schedule there too."""
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    if surface == "folded":
        mesh = G.cylinder(10)
        gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    else:
        plain = h.Surface3d(sphere8["x"], sphere8["t"])
        gr = h.Surface3d(sphere8["x"], sphere8["t"],
                         plain.n + 0.1 * np.roll(plain.n, 1, axis=1),
                         plain.g)
    idx = np.random.default_rng(5).permutation(gr.triangles).astype(np.uint32)
    blocks = mirrored_blocks((64, 63, 130))
    plan = h.NearfieldPlan(gr, 0, 0, idx, idx, blocks)
    op = h.Bem3d(gr, kern, layer, 2, 4, 0, 0, alpha=0.5, k=k)
    want = run(h, plan, op, (0, 0, 0))
    for schedule in ((1, 0, 0), (0, 1, 0), (1, 1, 0), (0, 0, 1), (0, 1, 1)):
        assert np.array_equal(run(h, plan, op, schedule), want), schedule


@pytest.mark.parametrize("q,q2,far", [(2, 4, True), (1, 3, False),
                                      (3, 5, False), (3, 4, True)])
@pytest.mark.parametrize("layer", [1, 2])
def test_laplace_bits_at_other_orders_and_far(q, q2, far, layer, sphere8):
    """The Laplace double layers take <x - y, n> per value in the far rule and
    (adjoint) at orders other than 2, in every schedule."""
    import h2lib_amd as h
    gr = h.Surface3d(sphere8["x"], sphere8["t"])
    idx = np.random.default_rng(6).permutation(gr.triangles).astype(np.uint32)
    blocks = mirrored_blocks((64, 65, 130))
    plan = h.NearfieldPlan(gr, 0, 0, idx, idx, blocks)
    op = h.Bem3d(gr, 0, layer, q, q2, 0, 0, alpha=0.5)
    orc = OracleBem(0, layer, 0, 0, sphere8["x"], sphere8["t"], q=q, q2=q2,
                    alpha=0.5)
    stream = h.Stream()
    outs = []
    for schedule in ((0, 0, 0), (0, 1, 0), (1, 0, 1)):
        plan.set_schedule(*schedule)
        out = h.DeviceArray(plan.entries, op.dtype)
        out.fill_nan()
        plan.execute(op, out.ptr, stream.handle, far)
        stream.sync()
        outs.append(out.download())
        # (the far rule of a triangle with itself is not a number)
        assert np.array_equal(outs[0], outs[-1], equal_nan=far), schedule
    for b, (ro, r, co, c) in enumerate(blocks):
        if far and ro == co:
            continue
        ref = orc.nearfield(idx[ro:ro + r], idx[co:co + c], far=far)
        assert rel_block_err(plan.block(outs[0], b), ref) < 1e-12, b


@pytest.mark.parametrize("kern,k", [(0, 0.0), (1, 0.1), (1, 5.0),
                                    (1, 2.0 + 0.5j)])
@pytest.mark.parametrize("layer", [1, 2])
@pytest.mark.parametrize("basis", [0, 1])
def test_fine_folded_cylinder_one_launch_per_class(kern, k, layer, basis):
    """More than 32768 touching pairs on a folded surface: a launch per rule
    class of the kernels with <x - y, n> per value.  A plan of a few of the
    blocks takes the launch of all classes: the same entries (constant basis:
    the same bits).  Where folded sheets lie in one plane the entries are
    rounding noise, so the oracle's are compared on the scale of all."""
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    mesh = G.cylinder(22)
    gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    rt = G.ClusterTree(mesh, basis, 64)
    bt = G.BlockTree(rt, rt, 2.0, 0)
    blocks = bt.near_block_list()
    plan = h.NearfieldPlan(gr, basis, basis, rt.idx, rt.idx, blocks)
    op = h.Bem3d(gr, kern, layer, 2, 4, basis, basis, alpha=0.5, k=k)
    assert plan.work(op)[1][1:].sum() > 32768
    got = run(h, plan, op, (0, 0, 0))
    scale = np.abs(got).max()
    sel = np.random.default_rng(1).choice(len(blocks), 10, replace=False)
    few = h.NearfieldPlan(gr, basis, basis, rt.idx, rt.idx, blocks[sel])
    assert few.work(op)[1][1:].sum() <= 32768
    part = run(h, few, op, (0, 0, 0))
    orc = OracleBem(kern, layer, basis, basis, mesh.x, mesh.t, q=2, q2=4,
                    alpha=0.5, k=k)
    for i, b in enumerate(sel):
        ro, r, co, c = (int(v) for v in blocks[b])
        a = plan.block(got, b)
        if basis == 0:
            assert np.array_equal(few.block(part, i), a), b
        else:
            assert np.abs(few.block(part, i) - a).max() < 1e-14 * scale, b
        ref = orc.nearfield(rt.idx[ro:ro + r], rt.idx[co:co + c])
        assert np.abs(a - ref).max() < 1e-12 * scale, b


@pytest.mark.parametrize("tilt", [3e-13, 1e-14])
@pytest.mark.parametrize("kern,k", [(0, 0.0), (1, 2.0)])
@pytest.mark.parametrize("layer", [1, 2])
@pytest.mark.parametrize("basis", [0, 1])
def test_given_normals_are_exact(tilt, kern, k, layer, basis, sphere8):
    """Normals off the perpendicular by a little more than rounding are taken
    as they are: <x - y, n> is linear in n.  Entries are sums of <d, n> / r^3
    with a few roundings of |d| / r^3 each, which the in-plane normals' entries
    have the size of: 16 * 2^-52 of their largest."""
    import h2lib_amd as h
    x, t = sphere8["x"], sphere8["t"]
    plain = h.Surface3d(x, t)
    roll = np.roll(plain.n, 1, axis=1)
    dofs = plain.vertices if basis else plain.triangles
    idx = np.random.default_rng(8).permutation(dofs).astype(np.uint32)
    vals = []
    for nn in (plain.n, roll, plain.n + tilt * roll):
        gr = h.Surface3d(x, t, nn, plain.g)
        op = h.Bem3d(gr, kern, layer, 2, 4, basis, basis, alpha=0.0, k=k)
        plan = h.NearfieldPlan(gr, basis, basis, idx, idx,
                               mirrored_blocks((64, 9)))
        vals.append(run(h, plan, op, (0, 0, 0)))
    a, b, c = vals
    assert np.abs(c - (a + tilt * b)).max() < 16 * 2.0 ** -52 * np.abs(b).max()


@pytest.mark.parametrize("layer", [1, 2])
@pytest.mark.parametrize("k", [0.0, 2.0])
def test_double_layer_entries_lose_no_digits(layer, k):
    """Entries of touching clusters against long double: no further off than a
    product <x - y, n> per value in FP64 (the regular rule of triangles
    without common vertices; the kernels take <x - y, n> as a factor of one
    triangle's point)."""
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    mesh = G.sphere(32)
    gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    op = h.Bem3d(gr, int(k != 0.0), layer, 2, 4, 0, 0, alpha=0.0, k=k)
    rt = G.ClusterTree(mesh, 0, 64)
    blocks = [b for b in G.BlockTree(rt, rt, 2.0, 0).near_block_list()
              if b[0] != b[2]][::9]
    gauss, wg = np.polynomial.legendre.leggauss(2)
    gauss, wg = 0.5 * (gauss + 1.0), 0.5 * wg
    u = np.repeat(gauss, 2)
    v = np.outer(gauss, gauss).ravel()
    w = (np.outer(wg, wg) * gauss[:, None]).ravel()
    x, t = np.asarray(mesh.x), np.asarray(mesh.t).astype(np.int64)

    def entries(ri, ci, real):
        X = x.astype(real)
        uu, vv, ww = u.astype(real), v.astype(real), w.astype(real)

        def points(tri):
            a, b, c = (X[t[tri, i]][:, None, :] for i in range(3))
            return (a * (1 - uu)[None, :, None] + b * (uu - vv)[None, :, None]
                    + c * vv[None, :, None])
        p, q = points(ri), points(ci)
        n = np.asarray(mesh.n).astype(real)
        g = np.asarray(mesh.g).astype(real)
        re = np.zeros((len(ri), len(ci)), real)
        im = np.zeros_like(re)
        for i in range(4):
            for j in range(4):
                d = p[:, None, i] - q[None, :, j]
                r2 = (d * d).sum(-1)
                r = np.sqrt(r2)
                dn = (d * n[ci][None]).sum(-1) if layer == 1 else \
                    -(d * n[ri][:, None]).sum(-1)
                val = ww[i] * ww[j] * dn / (r * r2)
                ph = real(k) * r
                re += val * (np.cos(ph) + ph * np.sin(ph))
                im += val * (np.sin(ph) - ph * np.cos(ph))
        f = g[ri][:, None] * g[ci][None] / (4 * real(np.pi))
        return (re * f, im * f) if k else (re * f,)

    err = np.zeros(2)
    for ro, r, co, c in blocks:
        ri, ci = rt.idx[ro:ro + r], rt.idx[co:co + c]
        got = op.nearfield(ri, ci)
        apart = ~(t[ri][:, None, :, None] == t[ci][None, :, None, :]).any(
            axis=(2, 3))
        want = entries(ri, ci, np.longdouble)
        plain = entries(ri, ci, np.float64)
        for part, a, b in zip((got.real, got.imag), want, plain):
            # (pi rounded in both references, the same factor)
            err += [float((((z - a) ** 2)[apart]).sum()) for z in (part, b)]
    print("error against a product per value: %.3f" % np.sqrt(
        err[0] / err[1]))
    assert err[0] <= 1.1 * err[1]
