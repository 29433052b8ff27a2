"""Mirrored coupling pairs and the one-wave adjoint near blocks of the H2
product (needs a GPU).

The default products evaluate each coupling value of an order-4 matrix once
for a block and its mirror, read or computed, forward and adjoint, and the
adjoint reads each near block once.  The reproducible products use neither
and are the reference here: the same values summed in another order, a few
thousand terms, 1e-13 of the largest entry.  With the pairs switched off the
general kernels run.  Leaves of 100 DOFs make blocks larger than the wave's
64 x 64, leaves of 3 small ones.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("clf", [64, 100, 3])
@pytest.mark.parametrize("kern,layer,basis,k", [
    (0, 0, 1, 0.0), (0, 1, 1, 0.0), (0, 2, 0, 0.0), (1, 0, 0, 3.0),
    (1, 1, 0, 2.0 + 0.5j), (1, 2, 1, 2.0)])
def test_pairs_and_adjoint_match_general_kernels(kern, layer, basis, k, clf):
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    from h2lib_amd.h2matrix import H2Matrix
    if clf == 3 and (kern, layer) not in ((0, 1), (1, 1)):
        pytest.skip("small leaves: one real and one complex case")
    mesh = G.sphere({3: 6, 64: 14, 100: 26}[clf])
    gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    op = h.Bem3d(gr, kern, layer, 2, 4, basis, basis,
                 alpha=0.5 if layer else 0.0, k=k)
    rt = G.ClusterTree(mesh, basis, clf)
    bt = G.BlockTree(rt, rt, 2.0, 0)
    H = H2Matrix(op, mesh, rt, rt, bt, 4)
    H.set_schedule(2)
    assert H.coupling_pairs() > 0
    rng = np.random.default_rng(2)
    x = rng.standard_normal(H.n)
    if kern:
        x = x + 1j * rng.standard_normal(H.n)
    d_x = h.DeviceArray.from_host(x.astype(H.dtype))
    d_y = h.DeviceArray(H.n, H.dtype)
    alpha = 0.75 - 0.5j if kern else 0.75

    def product(trans):
        d_y.zero()
        H.addeval(alpha, d_x, d_y, trans=trans)
        return d_y.download()

    try:
        for mode in (0, 1):
            H.set_coupling_mode(mode)
            for trans in (False, True):
                h.set_reproducible(True)
                want = product(trans)
                h.set_reproducible(False)
                for pairs in (1, 0):
                    H.set_coupling_pairs(pairs)
                    for _ in range(2):  # coefficients cleared in between
                        got = product(trans)
                        err = np.abs(got - want).max() / np.abs(want).max()
                        assert err < 1e-13, (mode, trans, pairs, err)
                H.set_coupling_pairs(1)
    finally:
        h.set_reproducible(True)


@pytest.mark.parametrize("kern,layer,basis,k", [
    (0, 0, 1, 0.0), (0, 1, 1, 0.0), (1, 0, 0, 3.0), (1, 1, 0, 2.0 + 0.5j)])
@pytest.mark.parametrize("nvec", [2, 3, 8])
def test_batched_pairs_match_general_kernels(kern, layer, basis, k, nvec):
    """Several vectors: the pairs' values used for all of them, and the
    vectors' layout in the other kernels."""
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    from h2lib_amd.h2matrix import H2Matrix
    mesh = G.sphere(13)
    gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    op = h.Bem3d(gr, kern, layer, 2, 4, basis, basis,
                 alpha=0.5 if layer else 0.0, k=k)
    rt = G.ClusterTree(mesh, basis, 60)
    bt = G.BlockTree(rt, rt, 2.0, 0)
    H = H2Matrix(op, mesh, rt, rt, bt, 4)
    H.set_schedule(2)
    assert H.coupling_pairs() > 0
    rng = np.random.default_rng(5)
    d_x = [h.DeviceArray.from_host((rng.standard_normal(H.n) + (
        1j * rng.standard_normal(H.n) if kern else 0.0)).astype(H.dtype))
        for _ in range(nvec)]
    d_y = [h.DeviceArray(H.n, H.dtype) for _ in range(nvec)]
    alphas = [0.5 + 0.25 * v for v in range(nvec)]

    def product(trans):
        for y in d_y:
            y.zero()
        H.addeval_batch(alphas, d_x, d_y, trans=trans)
        return np.array([y.download() for y in d_y])

    try:
        for mode in (0, 1):
            H.set_coupling_mode(mode)
            for trans in (False, True):
                h.set_reproducible(True)
                want = product(trans)
                h.set_reproducible(False)
                for pairs in (1, 0):
                    H.set_coupling_pairs(pairs)
                    for _ in range(2):
                        err = np.abs(product(trans) - want).max(1)
                        assert (err < 1e-13 * np.abs(want).max(1)).all(), (
                            mode, trans, pairs, err)
                H.set_coupling_pairs(1)
    finally:
        h.set_reproducible(True)


def test_large_helmholtz_product_runs_near_blocks_with_the_pairs():
    """At 131072 triangles the near blocks share the launch of the computed
    couplings."""
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    from h2lib_amd.h2matrix import H2Matrix
    mesh = G.sphere(128)
    gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    op = h.new_slp_helmholtz_bem3d(3.0, gr, 2, 4, 0, 0)
    rt = G.ClusterTree(mesh, 0, 64)
    bt = G.BlockTree(rt, rt, 2.0, 0)
    H = H2Matrix(op, mesh, rt, rt, bt, 4)
    H.set_schedule(2)
    H.set_coupling_mode(1)
    assert H.coupling_pairs() >= 8 * 768 * 4
    rng = np.random.default_rng(6)
    d_x = h.DeviceArray.from_host(rng.standard_normal(H.n) +
                                  1j * rng.standard_normal(H.n))
    d_y = h.DeviceArray(H.n, H.dtype)
    out = []
    try:
        for rep in (True, False, False):
            h.set_reproducible(rep)
            d_y.zero()
            H.addeval(0.5 + 0.25j, d_x, d_y)
            out.append(d_y.download())
    finally:
        h.set_reproducible(True)
    for got in out[1:]:
        assert np.abs(got - out[0]).max() < 1e-13 * np.abs(out[0]).max()


def test_large_damped_product_runs_near_blocks_with_the_pairs():
    """The same with a complex wave number and a double layer."""
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    from h2lib_amd.h2matrix import H2Matrix
    mesh = G.sphere(128)
    gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    op = h.new_dlp_helmholtz_bem3d(2.0 + 0.3j, gr, 2, 4, 0, 0, 0.5)
    rt = G.ClusterTree(mesh, 0, 64)
    bt = G.BlockTree(rt, rt, 2.0, 0)
    H = H2Matrix(op, mesh, rt, rt, bt, 4)
    H.set_schedule(2)
    H.set_coupling_mode(1)
    assert H.coupling_pairs() >= 8 * 768 * 4
    rng = np.random.default_rng(6)
    d_x = h.DeviceArray.from_host(rng.standard_normal(H.n) +
                                  1j * rng.standard_normal(H.n))
    d_y = h.DeviceArray(H.n, H.dtype)
    out = []
    try:
        for rep in (True, False, False):
            h.set_reproducible(rep)
            d_y.zero()
            H.addeval(0.5 + 0.25j, d_x, d_y)
            out.append(d_y.download())
    finally:
        h.set_reproducible(True)
    for got in out[1:]:
        assert np.abs(got - out[0]).max() < 1e-13 * np.abs(out[0]).max()


@pytest.mark.parametrize("schedule", [2, 0])
@pytest.mark.parametrize("kern,layer,basis,k", [
    (0, 0, 1, 0.0), (0, 1, 1, 0.0), (1, 0, 0, 3.0), (1, 1, 0, 2.0 + 0.5j)])
def test_many_pairs_match_general_kernels(kern, layer, basis, k, schedule):
    """Enough pairs for the pairs' kernels at every number of vectors, read
    and computed, forward and adjoint (fewer keep the general kernels: the
    tests above)."""
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    from h2lib_amd.h2matrix import H2Matrix
    mesh = G.sphere(20)
    gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    op = h.Bem3d(gr, kern, layer, 2, 4, basis, basis,
                 alpha=0.5 if layer else 0.0, k=k)
    rt = G.ClusterTree(mesh, basis, 12)
    bt = G.BlockTree(rt, rt, 2.0, 0)
    H = H2Matrix(op, mesh, rt, rt, bt, 4)
    H.set_schedule(schedule)
    assert H.coupling_pairs() >= 2048
    rng = np.random.default_rng(9)
    d_x = [h.DeviceArray.from_host((rng.standard_normal(H.n) + (
        1j * rng.standard_normal(H.n) if kern else 0.0)).astype(H.dtype))
        for _ in range(8)]
    d_y = [h.DeviceArray(H.n, H.dtype) for _ in range(8)]
    alphas = [0.5 + 0.25 * v for v in range(8)]

    def product(nv, trans):
        for y in d_y[:nv]:
            y.zero()
        if nv == 1:
            H.addeval(alphas[0], d_x[0], d_y[0], trans=trans)
        else:
            H.addeval_batch(alphas[:nv], d_x[:nv], d_y[:nv], trans=trans)
        return np.array([y.download() for y in d_y[:nv]])

    try:
        for mode in (0, 1):
            H.set_coupling_mode(mode)
            for trans in (False, True):
                h.set_reproducible(True)
                want = product(8, trans)
                h.set_reproducible(False)
                for nv in (1, 2, 4, 8):
                    for _ in range(2):
                        err = np.abs(product(nv, trans) - want[:nv]).max(1)
                        assert (err < 1e-13 * np.abs(want[:nv]).max(1)
                                ).all(), (mode, trans, nv, err)
    finally:
        h.set_reproducible(True)


@pytest.mark.parametrize("m", [4, 3])
def test_nan_wave_number_reaches_every_coupling(m):
    """A damping that is not a number gives couplings that are not (with the
    near field zero, so that they alone decide)."""
    import ctypes as C
    import h2lib_amd as h
    from h2lib_amd import geometry as G
    from h2lib_amd.h2matrix import H2Matrix
    mesh = G.sphere(12)
    gr = h.Surface3d(mesh.x, mesh.t, mesh.n, mesh.g)
    op = h.Bem3d(gr, 1, 0, 2, 4, 0, 0, k=complex(2.0, np.nan))
    rt = G.ClusterTree(mesh, 0, 16)
    bt = G.BlockTree(rt, rt, 2.0, 0)
    H = H2Matrix(op, mesh, rt, rt, bt, m)
    nb = bt.near_block_list().astype(np.int64)
    near = np.zeros(int((nb[:, 1] * nb[:, 3]).sum()), dtype=H.dtype)
    assert h.hip().h2hip_h2matrix_set_nearfield(
        H._h, near.ctypes.data_as(C.c_void_p)) == 0
    d_x = [h.DeviceArray.from_host(np.ones(H.n, dtype=H.dtype))] * 2
    d_y = [h.DeviceArray(H.n, H.dtype) for _ in range(2)]
    H.set_schedule(2)
    try:
        for mode in (0, 1):
            H.set_coupling_mode(mode)
            for rep in (False, True):
                h.set_reproducible(rep)
                for trans in (False, True):
                    for y in d_y:
                        y.zero()
                    H.addeval_batch([1.0, 1.0], d_x, d_y, trans=trans)
                    two = d_y[1].download()
                    d_y[0].zero()
                    H.addeval(1.0, d_x[0], d_y[0], trans=trans)
                    for y in (two, d_y[0].download()):
                        assert np.isnan(y).all(), (mode, rep, trans)
    finally:
        h.set_reproducible(True)
