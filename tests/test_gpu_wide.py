"""The four-wide BVH walk against the CPU oracle, bit for bit, where it can
go wrong: trees of a few facets (a root that is a leaf, nodes with empty
slots), meshes without extent along an axis, coordinates of very different
size, rays along an axis, and walks that need more deferred children than
the stack holds."""
import numpy as np
import pytest

from fluxpy_amd import meshes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    torch.cuda.set_device(0)
    return torch


def _soup(nf, seed, scale=1.0, offset=0.0, flat=False):
    """Random triangles, many of them large enough to overlap each other."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, (nf, 1, 3))
    s = np.exp(rng.uniform(np.log(0.01), np.log(1.5), (nf, 1, 1)))
    V = (c + s * rng.uniform(-1, 1, (nf, 3, 3))) * scale + offset
    if flat:
        V[..., 2] = offset
    return V.reshape(-1, 3), np.arange(3 * nf).reshape(nf, 3)


def deep_mesh():
    """16,000 large triangles whose centroids halve their distance to a
    corner again and again and then coincide, so the Morton tree is a chain
    of clusters over a deep balanced part; every box is as wide as the mesh
    and the planes are parallel, so a walk defers nearly all it meets."""
    rng = np.random.default_rng(3)
    t = np.concatenate([np.full(16, 0.9 * 0.5 ** k) for k in range(11)]
                       + [np.full(1 << 14, 2e-4)])
    n = t.size
    c = t[:, None] * np.array([1.0, 1.0, 0.3])
    a = rng.uniform(-2, 2, (n, 2, 2))
    e = np.stack([a[..., 0], a[..., 1], a[..., 0]], -1)     # in the planes z = x + const
    V = np.stack([c + e[:, 0], c + e[:, 1], c - e[:, 0] - e[:, 1]], 1)
    return V.reshape(-1, 3), np.arange(3 * n).reshape(n, 3)


def lost_blocker_mesh(n):
    """Two rows of n small facets that face each other, all centroids in the
    plane z = x + 0.5, and 560 sheets in other planes z = x + const whose
    boxes hold every ray between the rows.  The sheets' centroids close in on
    a corner one Morton bit at a time and the last 512 share a cell, so a ray
    from the first row to the second defers more children than the stack
    holds and drops some of those 512.  Eight of these are turned across the
    rays, each over a sixteenth of the rows' width: the only facets in
    between.  Returns V, F and the two rows' facets."""
    tri = []
    y = 0.05 + 0.9 * (np.arange(n) + 0.5) / n
    for x, s in ((0.35, 1.0), (0.65, -1.0)):        # normals towards each other
        c = np.stack([np.full(n, x), y, np.full(n, x + 0.5)], 1)
        a, b = np.array([1.0, 0.0, -1.0]) * 1e-4, np.array([0.0, 1.0, 0.0]) * 1e-4
        tri.append(np.stack([c + s * a, c + b, c - s * a - b], 1))
    axis = np.repeat(np.eye(3), 10, axis=0).reshape(3, 10, 3).swapaxes(0, 1).reshape(-1, 3)
    chain = axis * (0.5 ** np.repeat(np.arange(10), 3))[:, None] * 0.98
    ends = np.array([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]])
    flat = np.concatenate([ends, np.repeat(chain, 2, axis=0)[:46],
                           np.random.default_rng(2).uniform(1e-4, 4e-4, (512, 3))])
    e = 3.0 * np.array([[1.0, -1.0, 1.0], [-1.0, -1.0, -1.0], [0.0, 2.0, 0.0]])
    sheets = flat[:, None] + e
    for k in range(8):
        q = flat.shape[0] - 512 + 32 + 60 * k
        p1 = np.array([0.55, 0.06 + 0.115 * k, 1.10])
        p2 = p1 + [0.0, 0.06, 0.0]
        sheets[q] = np.stack([p1, p2, 3.0 * flat[q] - p1 - p2])
    tri.append(sheets)
    V = np.concatenate(tri)
    return (V.reshape(-1, 3), np.arange(3 * len(V)).reshape(-1, 3),
            np.arange(n), np.arange(n, 2 * n))


@pytest.mark.parametrize("cls", ["cgal", "embree"])
@pytest.mark.parametrize("nf,kw", [
    (1, {}), (2, {}), (3, {}), (4, {}), (5, {}), (17, {}), (200, {}),
    (60, {"flat": True}), (60, {"scale": 1e6, "offset": 3e7}), (60, {"scale": 1e-4})])
def test_soup_matches_oracle(torch_dev, oracle_mod, nf, kw, cls):
    from fluxpy_amd.shape import CgalTrimeshShapeModel, EmbreeTrimeshShapeModel
    V, F = _soup(nf, 100 + nf, **kw)
    sm = (CgalTrimeshShapeModel if cls == "cgal" else EmbreeTrimeshShapeModel)(V, F)
    S = oracle_mod.OracleScene(V, F)
    I = np.arange(nf)
    if cls == "cgal":
        assert np.array_equal(sm.get_visibility_matrix(), S.vis_mn(I, I))
    else:
        assert np.array_equal(sm.get_visibility_matrix(), S.vis_mn(I, I, mode=oracle_mod.MODE_EMBREE, P=sm.P))
    D = np.concatenate([np.eye(3), -np.eye(3), [[1.0, 0, 1e-9], [0, 1e-300, 1.0]],
                        meshes.sun_directions(5, seed=nf)])
    for d in D:
        if cls == "cgal":
            want = S.occluded(I, d)[:, 0]
        else:
            want = S.occluded(I, d, mode=oracle_mod.MODE_EMBREE, P=sm.P, N=sm.N)[:, 0]
        assert np.array_equal(sm.is_occluded(I, d), want)


def test_stack_overflow_matches_oracle(torch_dev, oracle_mod):
    from fluxpy_amd.shape import CgalTrimeshShapeModel
    V, F = deep_mesh()
    sm = CgalTrimeshShapeModel(V, F)
    S = oracle_mod.OracleScene(V, F)
    I = np.concatenate([np.arange(0, 176, 5), np.arange(176, len(F), 401)])
    for d in ([1.0, 0.13, 1.0], [-1.0, 0.4, -1.0], [0.02, 1.0, 0.02], [0.3, -0.2, 1.0]):
        d = np.array(d) / np.linalg.norm(d)
        assert np.array_equal(sm.is_occluded(I, d), S.occluded(I, d)[:, 0])
    assert np.array_equal(sm.get_visibility(I, I), S.vis_mn(I, I))


@pytest.mark.parametrize("query", ["visibility", "shared", "block", "list", "occlusion", "insolation"])
def test_stack_overflow_with_rays_under_way(torch_dev, oracle_mod, query):
    """Walks that drop children while their wave takes new rays for other
    lanes (several batches a wave): form factors of a block and of one list,
    1.44 M pairs, and queries of as many and of 473,600 rays; `shared`: a
    query small enough that lanes without work take parts of such walks."""
    from fluxpy_amd.form_factors import get_form_factor_matrix
    from fluxpy_amd.shape import CgalTrimeshShapeModel
    V, F, A, B = lost_blocker_mesh(1200)
    sm = CgalTrimeshShapeModel(V, F)
    S = oracle_mod.OracleScene(V, F)
    if query == "visibility":
        want = S.vis_mn(A, B)
        assert 0.2 < want.mean() < 0.8
        assert np.array_equal(sm.get_visibility(A, B), want)
    elif query == "shared":
        assert np.array_equal(sm.get_visibility(A[::4], B[::3]), S.vis_mn(A[::4], B[::3]))
    elif query in ("block", "list"):
        I, J = (A, B) if query == "block" else (np.concatenate([A, B]),) * 2
        want = S.form_factor_matrix(sm.P, sm.N, sm.A, I, J)
        got = get_form_factor_matrix(sm, I, J)
        assert got.nnz == want.nnz and (got != want).nnz == 0
    else:
        I, a = np.arange(len(F)), np.linspace(-1.0, 1.0, 160)
        D = np.stack([np.cos(a), np.sin(a), np.cos(a)], 1)
        D /= np.sqrt(1 + np.cos(a) ** 2)[:, None]
        want = S.occluded(I, D)
        assert want.size > 400000 and 0.1 < want[A].mean() < 0.9
        if query == "occlusion":
            assert np.array_equal(sm.is_occluded(I, D), want)
        else:
            E = sm.get_direct_irradiance_multi(1.0, D)
            assert np.array_equal(E, np.stack([
                oracle_mod.direct_irradiance(sm.N, want[:, k], 1.0, D[k])
                for k in range(D.shape[0])], 1))


@pytest.mark.parametrize("cls", ["cgal", "embree"])
def test_directions_of_any_length(torch_dev, oracle_mod, cls):
    """Sun directions that FP32 does not hold, finite and infinite ones,
    against every triangle of the mesh: a direction at a time, and all of
    them in many batches."""
    from fluxpy_amd.shape import CgalTrimeshShapeModel, EmbreeTrimeshShapeModel
    V, F = _soup(300, 21)
    sm = (CgalTrimeshShapeModel if cls == "cgal" else EmbreeTrimeshShapeModel)(V, F)
    S = oracle_mod.OracleScene(V, F, use_bvh=False)
    kw = {} if cls == "cgal" else {"mode": oracle_mod.MODE_EMBREE, "P": sm.P, "N": sm.N}
    I, inf = np.arange(300), np.inf
    D = np.concatenate([meshes.sun_directions(4, seed=3) * s
                        for s in (1.0, 1e-300, 1e-40, 1e-30, 1e30, 1e38, 1e39, 1e300)]
                       + [[[inf, 0, 0], [-inf, 0, 0], [0, inf, 1.0], [0, -1.0, -inf],
                           [inf, inf, 0], [np.nan, 0, 1.0]]])
    if cls == "embree":     # rays are FP32 there: no direction is left of these
        D = np.delete(D, np.s_[4:16], axis=0)
    want = S.occluded(I, D, **kw)
    assert 0.05 < want[:, :4].mean() < 0.95
    for k, d in enumerate(D):
        assert np.array_equal(sm.is_occluded(I, d), want[:, k]), d
    many = np.tile(np.arange(len(D)), 100)
    E = sm.get_direct_irradiance_multi(1.0, D[many])
    with np.errstate(invalid="ignore"):
        for k in range(len(D)):
            cosi = sm.N[:, 0] * D[k, 0] + sm.N[:, 1] * D[k, 1] + sm.N[:, 2] * D[k, 2]
            lit = np.where((cosi > 0) & ~want[:, k], cosi, 0.0)
            assert (E[:, k::len(D)] == lit[:, None]).all(), D[k]


@pytest.mark.parametrize("mesh", ["soup", "deep", "terrain"])
def test_small_queries_equal_large_ones(torch_dev, mesh):
    """Lanes without work take parts of other lanes' walks in queries of up
    to 131,072 rays only: the same rays in one larger query."""
    from fluxpy_amd.shape import CgalTrimeshShapeModel
    if mesh == "soup":
        V, F = _soup(400, 11)
    elif mesh == "deep":
        V, F = deep_mesh()
    else:
        V, F = meshes.fractal_terrain(grid=80, levels=6, n_craters=12, seed=4)
    sm = CgalTrimeshShapeModel(V, F)
    nf = sm.num_faces
    I, J = np.arange(nf), np.linspace(0, nf - 1, -(-140000 // nf)).astype(np.int64)
    assert nf * J.size > 131072 and nf * (J.size // 2) <= 131072
    full = sm.get_visibility(I, J)
    for a in np.array_split(np.arange(J.size), 3) + [np.array([J.size - 1])]:
        assert np.array_equal(sm.get_visibility(I, J[a]), full[:, a])
    few = I[:: max(1, nf // 50)]
    assert np.array_equal(sm.get_visibility(few, J), full[few])
    D = meshes.sun_directions(-(-140000 // nf), seed=2)
    E = sm.get_direct_irradiance_multi(1.0, D)
    for k in range(0, D.shape[0], max(1, D.shape[0] // 12)):
        assert np.array_equal(sm.get_direct_irradiance_multi(1.0, D[k:k + 1])[:, 0], E[:, k])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("mesh", ["soup", "crater", "terrain", "far", "sheet"])
def test_square_mask_equals_general_mask(torch_dev, oracle_mod, mesh, dtype):
    """All pairs of one list from one walk per pair against one walk per
    direction (the same list as rows and columns, the columns permuted so
    that the general path takes them) and against the oracle.  `sheet` has
    facets in common planes and rays through edges and vertices, where
    rounding decides and the two directions may differ."""
    from fluxpy_amd.form_factors import get_form_factor_matrix
    from fluxpy_amd.shape import CgalTrimeshShapeModel
    if mesh == "soup":
        V, F = _soup(150, 7)
    elif mesh == "crater":
        V, F = meshes.spherical_crater(npts=18, seed=5, depth=0.3)
    elif mesh == "terrain":
        V, F = meshes.fractal_terrain(grid=24, levels=5, n_craters=6, seed=8)
    elif mesh == "far":
        V, F = meshes.fractal_terrain(grid=16, levels=4, n_craters=4, seed=9)
        V = V * 3.0 + np.array([4e3, -9e3, 2e3])
    else:
        # a regular corrugated sheet: equal facets, symmetric rays
        x = np.arange(17.0)
        Z = np.abs((x % 8) - 4.0)[:, None] + 0 * x[None, :]
        V, F = meshes.grid_mesh(x, x, Z)
    V = V.astype(dtype)
    sm = CgalTrimeshShapeModel(V, F)
    nf = sm.num_faces
    I = np.arange(nf)
    full = get_form_factor_matrix(sm)
    S = oracle_mod.OracleScene(V, F)
    want = S.form_factor_matrix(sm.P, sm.N, sm.A)
    assert full.nnz == want.nnz and (full != want).nnz == 0
    rev = get_form_factor_matrix(sm, I, I[::-1].copy())       # general path
    assert (full.toarray()[:, ::-1] == rev.toarray()).all()
    rng = np.random.default_rng(1)
    sub = rng.integers(0, nf, max(1, nf // 3))                # a list with repeats
    assert (get_form_factor_matrix(sm, sub, sub).toarray()
            == full.toarray()[np.ix_(sub, sub)]).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("cls", ["cgal", "embree"])
def test_one_sun_by_value(torch_dev, cls, dtype):
    """The direction as an argument of the launch and as a device array."""
    from fluxpy_amd import _lib
    from fluxpy_amd.shape import CgalTrimeshShapeModel, EmbreeTrimeshShapeModel
    V, F = meshes.fractal_terrain(grid=20, levels=5, n_craters=6, seed=8)
    sm = (CgalTrimeshShapeModel if cls == "cgal" else EmbreeTrimeshShapeModel)(V.astype(dtype), F)
    for d in np.concatenate([meshes.sun_directions(3, seed=5), -np.eye(3)[2:]]):
        want = sm.get_direct_irradiance_multi(1365.0, d[None])[:, 0]
        P, N = _lib.to_dev(sm.P), _lib.to_dev(sm.N)
        E = torch_dev.empty(sm.num_faces, dtype=_lib.torch_dtype(sm.dtype), device="cuda")
        d = np.ascontiguousarray(d)
        _lib.call("flux_direct_irradiance_sun", sm._scene.handle, P.data_ptr(), N.data_ptr(),
                  _lib.dtype_code(sm.dtype), d.ctypes.data, 1365.0, sm._mode, E.data_ptr(),
                  _lib.stream())
        assert np.array_equal(E.cpu().numpy(), want)
