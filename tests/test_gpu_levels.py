"""GPU tests of the coarse-level kernels at the sizes where their work split can go wrong, against the oracle.

Tolerances: a level's rows are sums of 81 products in FP64, so two orders of the sum agree to a few 1e-15 of the
row's largest term; 1e-12 (products) and 1e-11 (after a sweep's 3 x 3 solves) leave room for the cancellation in
the rows, as in test_gpu_parity."""
import numpy as np
import pytest

from oracle import oracle as orc
from voxelfem_amd import workloads as wl

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.abs(np.asarray(a) - np.asarray(b)).max() / max(np.abs(np.asarray(b)).max(), 1e-300)


def pair(ne, levels, layer=None, seed=0):
    """A solver and the oracle's on the same cantilever."""
    import voxelfem_amd

    rho = wl.noise_density(ne, seed)
    tps = wl.configure(voxelfem_amd.pyVoxelFEM, ne, wl.CANTILEVER_BC, rho)
    mg = tps.multigridSolver(levels)
    s = orc.Sim(ne)
    s.set_etensor(1.0, 0.3)
    s.set_law(0, 1.0, 1e-9, 3.0, 3.0)
    s.set_densities(rho)
    s.set_dirichlet(wl.cantilever_mask(ne))
    om = orc.MG(s, levels)
    if layer is not None:
        mg.setFabricationMaskHeightByLayer(layer)
        om.set_mask_layer(layer)
    mg.updateStiffnessMatrices()
    om.update_stiffness()
    return mg, om


# level 1 has (ne / 2 + 1) nodes per axis: colour classes of 1 to 45 nodes, with every remainder modulo the four nodes
# that the block rows interleave and the sixteen that a workgroup holds; with layers masked, rows end inside a class.
# Tiles of the two-launch sweep are 4 x 12 nodes of a plane: one and several, and a level (5 x 353 x 3) of too many for it
@pytest.mark.parametrize("ne,levels,layer", [((4, 8, 52), 2, None), ((4, 20, 52), 2, 9), ((8, 704, 4), 2, None),
                                             ((4, 4, 4), 2, None), ((8, 4, 4), 2, None), ((8, 12, 4), 2, None),
                                             ((16, 8, 12), 2, None), ((4, 12, 20), 2, 5), ((16, 16, 8), 3, 9)])
def test_block_rows(ne, levels, layer):
    mg, om = pair(ne, levels, layer)
    rng = np.random.default_rng(5)
    for l in range(1, levels):
        nn = om.num_nodes(l)
        u, b = rng.normal(size=(nn, 3)), rng.normal(size=(nn, 3))
        ny = (ne[1] >> l) + 1
        iy = (np.arange(nn) // ((ne[2] >> l) + 1)) % ny
        act = np.ones(nn, bool) if layer is None else iy < -(-layer >> l) + 1
        u[~act] = 0
        assert rel(mg.applyK(l, u)[act], om.apply_K(l, u)[act]) < 1e-12, l
        assert rel(mg.computeResidual(l, u, b)[act], om.residual(l, u, b)[act]) < 1e-12, l
        for fwd in (True, False):
            assert rel(mg._smooth(l, u, b, fwd)[act], om.smooth(l, u, b, fwd)[act]) < 1e-11, (l, fwd)


# single precision takes two nodes of a z-row at a time: rows of one to fourteen nodes per colour, even and odd, ending inside
# a pair, with colour launches (5 x 353 nodes per plane) and with the two-launch sweep; the sums are the same, rounded to
# single precision: 1e-5, as the V-cycles of test_gpu_tiled
@pytest.mark.parametrize("ne,levels,layer", [((8, 704, 4), 2, None), ((8, 704, 12), 2, None), ((8, 704, 16), 2, 353),
                                             ((4, 20, 52), 2, 9), ((4, 4, 4), 2, None), ((96, 48, 56), 3, None)])
def test_block_rows_fp32(ne, levels, layer):
    from voxelfem_amd import capi

    capi.set_kernel_variant(3)  # block rows on level 1
    try:
        mg, om = pair(ne, levels, layer)
        r = np.random.default_rng(5).normal(size=(om.num_nodes(0), 3))
        n = np.arange(len(r))
        r[n // ((ne[1] + 1) * (ne[2] + 1)) == 0] = 0
        if layer is not None:
            r[n // (ne[2] + 1) % (ne[1] + 1) > layer] = 0
        for fmg, nu in ((False, 1), (True, 2)):
            assert rel(mg._precondition(r, 1, nu, fmg, "fp32"), mg._precondition(r, 1, nu, fmg, "fp64")) < 1e-5
    finally:
        capi.set_kernel_variant(0)


# the marching smoothing filter: tiles of 8 or 16 rows by 64 columns, reaches 1 to 4, sides below the reach (repeated
# reflection), real radii, constant weights; thin grids (the last two) sum tap by tap; sums of up to 729 positive terms in
# another order: 1e-13
@pytest.mark.parametrize("dims", [(1, 1, 1), (2, 3, 1), (5, 8, 64), (7, 9, 65), (3, 17, 130), (40, 16, 63), (700, 300, 1),
                                  (60000, 1, 1)])
@pytest.mark.parametrize("rmin,linear", [(2.0, True), (3.0, True), (4.0, True), (5.0, True), (2.5, True), (3.7, True),
                                         (3.0, False), (4.0, False), (6.0, True)])
def test_smoothing_march(dims, rmin, linear):
    import voxelfem_amd

    pv = voxelfem_amd.pyVoxelFEM
    x = np.random.default_rng(9).uniform(size=int(np.prod(dims)))
    sf = pv.SmoothingFilter(1, pv.SmoothingFilter.Type.Linear if linear else pv.SmoothingFilter.Type.Const)
    sf.setInputDimensions(list(dims))
    sf.rmin = rmin
    assert rel(sf.apply(x), orc.smoothing_filter(x, dims, rmin, linear)) < 1e-13


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_smoothing_march_non_finite(bad):
    """A value that is not finite reaches the voxels within the kernel and no others."""
    import voxelfem_amd

    pv = voxelfem_amd.pyVoxelFEM
    dims = (11, 12, 13)
    for rmin, linear in ((4.0, True), (3.7, True), (3.0, False)):
        x = np.random.default_rng(9).uniform(size=int(np.prod(dims)))
        x[np.ravel_multi_index((5, 6, 6), dims)] = bad
        sf = pv.SmoothingFilter(1, pv.SmoothingFilter.Type.Linear if linear else pv.SmoothingFilter.Type.Const)
        sf.setInputDimensions(list(dims))
        sf.rmin = rmin
        assert np.array_equal(np.isfinite(sf.apply(x)), np.isfinite(orc.smoothing_filter(x, dims, rmin, linear)))


# the factorization's launches: one block and a padded remainder, no block below the diagonal, a band of several blocks;
# the coarse solve multiplies the relative rounding by the operator's condition number, as in test_gpu_parity: 1e-9
@pytest.mark.parametrize("ne,levels", [((2, 2, 2), 1), ((4, 4, 2), 1), ((16, 2, 2), 1), ((32, 4, 4), 1), ((8, 16, 16), 1),
                                       ((48, 16, 16), 1)])
@pytest.mark.parametrize("graphs", [False, True])
def test_coarse_factor(ne, levels, graphs):
    mg, om = pair(ne, levels)
    mg.useGraphs = graphs
    rng = np.random.default_rng(6)
    for _ in range(3):  # with graphs: captured, then replayed
        mg.updateStiffnessMatrices()
        b = rng.normal(size=(om.num_nodes(levels), 3))
        assert rel(mg._coarseSolve(b), om.coarse_solve(b)) < 1e-9


# wide bands (more than 512 pairs of panel blocks: the panel gets a launch of its own), long ones (more than 128 block
# columns: wide strips of the inverse) and both, against the operator itself: the solution's error, u kappa at most, is seen
# through A as u kappa of b, with the 1e-9 of test_coarse_factor
@pytest.mark.parametrize("ne", [(4, 52, 52), (40, 24, 24), (12, 60, 60)])
def test_coarse_factor_wide(ne):
    import voxelfem_amd

    tps = wl.configure(voxelfem_amd.pyVoxelFEM, ne, wl.CANTILEVER_BC, wl.noise_density(ne, 0))
    mg = tps.multigridSolver(1)
    mg.updateStiffnessMatrices()
    n = [e // 2 + 1 for e in ne]
    free = np.arange(int(np.prod(n))) >= n[1] * n[2]  # x = 0 is clamped
    b = np.random.default_rng(6).normal(size=(len(free), 3))
    b[~free] = 0
    x = mg._coarseSolve(b)
    assert not x[~free].any()
    assert rel(mg.applyK(1, x)[free], b[free]) < 1e-9


# stiff voxels floating in void: diagonal blocks of the coarsest matrix are nearly singular. Cholesky's error does not
# exceed a modest multiple of u kappa, kappa the condition number of the matrix scaled to a unit diagonal (van der Sluis);
# the stable orders of elimination reach a third of u kappa here, so u kappa itself is the bound. Reference: refined in long
# double
@pytest.mark.parametrize("ne,Emin", [((8, 4, 4), 1e-9), ((6, 5, 4), 1e-9), ((8, 4, 4), 1e-12)])
def test_direct_solve_stiff_pieces(ne, Emin):
    import scipy.linalg as sl

    import voxelfem_amd
    from tests import fem_reference as fr

    K0 = np.asarray(orc.element_stiffness(1.0, 0.3, (1.0, 1.0, 1.0))).reshape(24, 24)
    free = np.repeat(wl.cantilever_mask(ne) == 0, 3)
    for seed in range(16):
        rho = (np.random.default_rng(seed).uniform(size=int(np.prod(ne))) < 0.15).astype(float)
        K = fr.assemble_K(ne, K0, Emin + (1 - Emin) * rho).toarray()[np.ix_(free, free)]
        d = 1 / np.sqrt(np.diag(K))
        w = np.linalg.eigvalsh(K * d[:, None] * d)
        f = np.zeros(len(free))
        f[free] = np.random.default_rng(seed + 100).normal(size=len(K))
        c, KL = sl.cho_factor(K * d[:, None] * d), K.astype(np.longdouble)
        x = np.zeros(len(K), np.longdouble)
        for _ in range(20):
            x += d * sl.cho_solve(c, d * (f[free] - KL @ x).astype(float))
        tps = wl.configure(voxelfem_amd.pyVoxelFEM, ne, wl.CANTILEVER_BC, rho, Emin=Emin)
        u = tps.solve(f.reshape(-1, 3)).reshape(-1)[free]
        assert np.linalg.norm(u - x) <= 2.0 ** -53 * w[-1] / w[0] * np.linalg.norm(x), seed


# level 1 on the fly: every side of the grid within reach of every node, sides of different length and element size,
# masked layers, a partially filled workgroup; variant 1 keeps level 1 on the fly
@pytest.mark.parametrize("ne,levels,layer", [((4, 4, 4), 2, None), ((8, 4, 12), 2, None), ((12, 20, 8), 2, None),
                                             ((8, 24, 16), 3, 13), ((40, 8, 8), 3, None)])
@pytest.mark.parametrize("size", [(1.0, 1.0, 1.0), (0.5, 1.5, 2.0)])
def test_level1_on_the_fly(ne, levels, layer, size):
    import voxelfem_amd
    from voxelfem_amd import capi

    pv = voxelfem_amd.pyVoxelFEM
    rng = np.random.default_rng(8)
    rho = rng.uniform(0.1, 1.0, int(np.prod(ne)))
    hi = [n * h for n, h in zip(ne, size)]
    tps = pv.TensorProductSimulator([1, 1, 1], [[0.0, 0.0, 0.0], hi], list(ne))
    tps.readMaterial(wl.write_json(wl.MATERIAL, name="material.json"))
    tps.E_0, tps.E_min, tps.gamma = 1.0, 1e-9, 3.0
    tps.applyDisplacementsAndLoadsFromFile(wl.write_json(wl.CANTILEVER_BC))
    tps.setDensities(rho)
    s = orc.Sim(ne, [0.0, 0.0, 0.0], hi)
    s.set_etensor(1.0, 0.3)
    s.set_law(0, 1.0, 1e-9, 3.0, 3.0)
    s.set_densities(rho)
    s.set_dirichlet(wl.cantilever_mask(ne))
    capi.set_kernel_variant(1)
    try:
        mg, om = tps.multigridSolver(levels), orc.MG(s, levels)
        if layer is not None:
            mg.setFabricationMaskHeightByLayer(layer)
            om.set_mask_layer(layer)
        mg.updateStiffnessMatrices()
        om.update_stiffness()
        nn = om.num_nodes(1)
        u, b = rng.normal(size=(nn, 3)), rng.normal(size=(nn, 3))
        iy = (np.arange(nn) // (ne[2] // 2 + 1)) % (ne[1] // 2 + 1)
        act = np.ones(nn, bool) if layer is None else iy < -(-layer >> 1) + 1
        u[~act] = 0
        assert rel(mg.applyK(1, u)[act], om.apply_K(1, u)[act]) < 1e-12
        assert rel(mg.computeResidual(1, u, b)[act], om.residual(1, u, b)[act]) < 1e-12
        for fwd in (True, False):
            assert rel(mg._smooth(1, u, b, fwd)[act], om.smooth(1, u, b, fwd)[act]) < 1e-11, fwd
        if layer is None:  # single precision rounds the same sums: 1e-5, as the V-cycles of test_gpu_tiled
            r = rng.normal(size=(om.num_nodes(0), 3))
            r[np.arange(len(r)) // ((ne[1] + 1) * (ne[2] + 1)) == 0] = 0
            assert rel(mg._precondition(r, 1, 1, False, "fp32"), mg._precondition(r, 1, 1, False, "fp64")) < 1e-5
    finally:
        capi.set_kernel_variant(0)


# the planar sweep: tiles of 8 x 12 nodes (one, several, with remainders), both directions, layers masked so that rows end
# inside a tile, one and two sweeps per visit (residual with the only sweep or the second, correction before the first);
# an element row has 8 products, a node four elements: 1e-12 for a sweep, 1e-11 through a cycle's coarse solve
@pytest.mark.parametrize("ne,levels,layer,fmg,nu,sym", [((4, 4), 1, None, False, 1, True), ((8, 12), 2, None, True, 2, True),
                                                        ((36, 24), 2, 17, False, 2, True), ((20, 52), 2, 30, True, 1, True),
                                                        ((64, 48), 3, 40, True, 2, False), ((40, 24), 1, None, False, 3, True),
                                                        ((16, 32), 2, None, False, 0, True)])
def test_planar_sweep(ne, levels, layer, fmg, nu, sym):
    import voxelfem_amd
    from oracle import oracle2d as o2

    rho = wl.noise_density(ne, 3, base=0.5, amp=0.4)
    mg = wl.configure2d(voxelfem_amd.pyVoxelFEM, ne, wl.MBB2D_BC, rho).multigridSolver(levels)
    s = o2.Sim(ne)
    s.set_etensor(1.0, 0.3)
    s.set_law(0, 1.0, 1e-9, 3.0, 3.0)
    s.set_densities(rho)
    mask = wl.mbb2d_mask(ne)
    s.set_dirichlet(mask)
    om = o2.MG(s, levels)
    if layer is not None:
        mg.setFabricationMaskHeightByLayer(layer)
        om.set_mask_layer(layer)
    mg.setSymmetricGaussSeidel(sym)
    om.set_symmetric(sym)
    mg.updateStiffnessMatrices()
    om.update_stiffness()
    rng = np.random.default_rng(7)
    for l in range(levels):
        nn = om.num_nodes(l)
        u, b = rng.normal(size=(nn, 2)), rng.normal(size=(nn, 2))
        iy = np.arange(nn) % ((ne[1] >> l) + 1)
        act = np.ones(nn, bool) if layer is None else iy < -(-layer >> l) + 1
        u[~act] = 0
        for fwd in (True, False):
            assert rel(mg._smooth(l, u, b, fwd)[act], om.smooth(l, u, b, fwd)[act]) < 1e-12, (l, fwd)
    r = rng.normal(size=(om.num_nodes(0), 2))
    r[np.arange(len(r)) % (ne[1] + 1) >= (ne[1] if layer is None else layer) + 1] = 0
    assert rel(mg._precondition(r, 2, nu, fmg), om.precondition(r, 2, nu, fmg)) < 1e-11


# one and two levels of more than six workgroups per compute unit, whose colours are launches of their own. The second
# cycle's residual is rounded at u |K| |x|, which the inverse amplifies to u kappa of x: kappa of the finest level is
# taken as 4^levels times that of the coarsest
@pytest.mark.parametrize("ne,levels,layer,fmg,nu,sym", [((640, 320), 4, None, False, 2, False),
                                                        ((1536, 384), 5, 201, True, 1, True)])
def test_planar_colour_launches(ne, levels, layer, fmg, nu, sym):
    import voxelfem_amd
    from oracle import oracle2d as o2

    rho = wl.noise_density(ne, 3, base=0.5, amp=0.4)
    mg = wl.configure2d(voxelfem_amd.pyVoxelFEM, ne, wl.MBB2D_BC, rho).multigridSolver(levels)
    s = o2.Sim(ne)
    s.set_etensor(1.0, 0.3)
    s.set_law(0, 1.0, 1e-9, 3.0, 3.0)
    s.set_densities(rho)
    s.set_dirichlet(wl.mbb2d_mask(ne))
    om = o2.MG(s, levels)
    if layer is not None:
        mg.setFabricationMaskHeightByLayer(layer)
        om.set_mask_layer(layer)
    mg.setSymmetricGaussSeidel(sym)
    om.set_symmetric(sym)
    mg.updateStiffnessMatrices()
    om.update_stiffness()
    rng = np.random.default_rng(7)
    for l in range(levels):
        nn = om.num_nodes(l)
        u, b = rng.normal(size=(nn, 2)), rng.normal(size=(nn, 2))
        iy = np.arange(nn) % ((ne[1] >> l) + 1)
        act = np.ones(nn, bool) if layer is None else iy < -(-layer >> l) + 1
        u[~act] = 0
        for fwd in (True, False):
            assert rel(mg._smooth(l, u, b, fwd)[act], om.smooth(l, u, b, fwd)[act]) < 1e-12, (l, fwd)
    nn = om.num_nodes(levels)
    A = np.stack([om.apply_K(levels, e.reshape(nn, 2)).ravel() for e in np.eye(2 * nn)])
    free = (np.diag(A) > 0) & ((np.repeat(om.dirichlet_mask(levels), 2) >> np.tile([0, 1], nn)) & 1 == 0)
    A = A[np.ix_(free, free)]
    d = 1 / np.sqrt(np.diag(A))
    w = np.linalg.eigvalsh(A * d[:, None] * d)
    r = rng.normal(size=(om.num_nodes(0), 2))
    r[np.arange(len(r)) % (ne[1] + 1) >= (ne[1] if layer is None else layer) + 1] = 0
    tol = 2.0 ** -53 * 4 ** levels * w[-1] / w[0]
    assert rel(mg._precondition(r, 2, nu, fmg), om.precondition(r, 2, nu, fmg)) < tol
