"""GPU parity of the exact FP64 winding number (igl::winding_number) against
the oracle: the reference's hierarchy (caps for boxes that do not contain the
query) and the FP64 brute force over every face.  Tolerance: max |dW| <= 1e-6
(stated by the workload definition); observed differences are ~1e-13
(summation order and the device atan2)."""
import numpy as np
import pytest

import oracle_py as O
from libigl_amd import datagen as D
from libigl_amd import gwn

pytestmark = pytest.mark.gpu
TOL = 1e-6


def test_exact_full_workload_vs_oracle_subset():
    V, F, Q = D.exact_workload()  # 20,480 tris, 100k queries
    W = gwn.winding_number(V, F, Q)
    assert W.shape == (Q.shape[0],) and np.all(np.isfinite(W))
    sub = np.arange(0, Q.shape[0], 20)  # 5,000 queries through the oracle
    Wo = O.winding_number_bf(V, F, Q[sub])
    err = np.abs(W[sub] - Wo)
    print(f"exact: max|dW| {err.max():.3e} over {sub.size} queries")
    assert err.max() <= TOL
    assert np.array_equal(W[sub] > 0.5, Wo > 0.5)
    # whole batch: a closed, outward surface gives w in {0, 1} away from it
    r = np.linalg.norm(Q, axis=1)
    assert np.all(np.abs(W[r < 0.9] - 1.0) < 1e-9)
    assert np.all(np.abs(W[r > 1.1]) < 1e-9)


def test_exact_hierarchy_matches_oracle_tree():
    """The GPU hierarchy is the oracle's node for node (same rand() state),
    and its sums equal the oracle's hierarchical sums and the brute force."""
    V, F, Q = D.exact_workload()
    Q = Q[:20000]
    O.libc_srand(4242)
    tree = gwn.WindingNumberAABB(V, F)
    O.libc_srand(4242)
    otree = O.WNTree(V, F)
    assert np.array_equal(tree.nodes(), otree.nodes())
    W = tree.winding_number(Q)
    assert np.abs(W - otree.query(Q)).max() < 1e-12
    assert np.abs(W - gwn.winding_number_bruteforce(V, F, Q)).max() < 1e-12


def test_exact_hierarchy_result_independent_of_batch():
    """One wavefront per query: large batches (from 6e6 over the root of the
    number of records on, here about 265,000) take them in Hilbert order, smaller
    ones in input order, and a query's lanes add the same terms in the same order
    either way, so its result does not depend on the batch it is in: bit for bit."""
    V, F, Q = D.exact_workload()
    rng = np.random.default_rng(7)
    tree = gwn.WindingNumberAABB(V, F)
    n = int(np.ceil(6e6 / np.sqrt(tree.nodes().shape[0])))
    Q = np.concatenate([Q, D.near_surface_queries(V, F, 4000, 1e-4, rng), V[:50]])
    Q = np.concatenate([Q, rng.uniform(-1.5, 1.5, (n - Q.shape[0], 3))])
    W = tree.winding_number(Q)  # sorted
    Wl = np.concatenate([tree.winding_number(Q[k:k + 40_000]) for k in range(0, Q.shape[0], 40_000)])
    assert np.array_equal(W, Wl)
    assert np.array_equal(tree.winding_number(Q[::-1][:3000]), W[::-1][:3000])
    assert np.array_equal(tree.winding_number(Q[:-1]), W[:-1])
    assert np.array_equal(tree.winding_number(Q[99_000:105_000]), W[99_000:105_000])


def test_exact_hierarchy_1310720_tris_vs_brute_force():
    """The 1,310,720-triangle mesh: exact queries through the hierarchy within
    1e-6 of the sum over every face (observed ~1e-12), 80% uniform, 20% within
    1e-4 of the surface."""
    V, F = D.bumpy_sphere(8, 64, 44)
    assert F.shape[0] == 1_310_720
    rng = np.random.default_rng(45)
    Q = np.concatenate([D.uniform_queries(V.min(0), V.max(0), 16000, rng), D.near_surface_queries(V, F, 4000, 1e-4, rng)])
    tree = gwn.WindingNumberAABB(V, F)
    W = tree.winding_number(Q)
    Wb = gwn.winding_number_bruteforce(V, F, Q)
    err = np.abs(W - Wb)
    print(f"1.31M tris, {tree.nodes().shape[0]} nodes: max|W_tree - W_brute| {err.max():.3e}")
    assert err.max() <= TOL and err.max() < 1e-9
    assert np.array_equal(W > 0.5, Wb > 0.5)
    chk = np.arange(0, Q.shape[0], 400)
    assert np.abs(W[chk] - O.winding_number_bf(V, F, Q[chk])).max() < 1e-9


def test_exact_small_cases():
    # single tet (tests/include/igl/signed_distance.cpp:4-44)
    V = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], float)
    F = np.array([[0, 1, 3], [0, 2, 1], [0, 3, 2], [1, 2, 3]], np.int32)
    Q = np.array([[0.5, 0.5, 0.5], [0.1, 0.1, 0.1], [0, 0, 0], [0.2, 0.2, 0.0]])
    W = gwn.winding_number(V, F, Q)
    Wo = O.winding_number_bf(V, F, Q)
    assert np.abs(W - Wo).max() <= 1e-14
    assert abs(W[0]) < 1e-15 and abs(W[1] - 1) < 1e-15
    # empty mesh and empty query set
    assert np.all(gwn.winding_number(np.zeros((0, 3)), np.zeros((0, 3), np.int32), Q) == 0)
    assert gwn.winding_number(V, F, np.zeros((0, 3))).shape == (0,)


def test_exact_ragged_sizes():
    # query counts and face counts that are not multiples of the tile sizes
    V, F = D.noisy_sphere(2, 0.01, 3)
    for nf in (1, 7, 255, 257, 320):
        for nq in (1, 3, 511, 513):
            Q = np.random.default_rng(nf * 1000 + nq).uniform(-1.3, 1.3, (nq, 3))
            Wo = O.winding_number_bf(V, F[:nf], Q)
            for W in (gwn.winding_number(V, F[:nf], Q), gwn.winding_number_bruteforce(V, F[:nf], Q)):
                assert np.abs(W - Wo).max() <= 1e-12, (nf, nq)


def test_exact_split_over_triangle_chunks():
    # few queries against thousands of triangles: the kernel splits the
    # triangles into chunks (1,025 -> 2, 3,001 -> 3 of 1,001, 5,120 -> 5) and
    # adds the partial sums afterwards
    V, F = D.noisy_sphere(4, 0.01, 5)
    for nf in (1025, 3001, 5120):
        for nq in (1, 300, 4097):
            Q = np.random.default_rng(nf + 7 * nq).uniform(-1.3, 1.3, (nq, 3))
            W = gwn.winding_number_bruteforce(V, F[:nf], Q)
            Wo = O.winding_number_bf(V, F[:nf], Q)
            assert np.abs(W - Wo).max() <= 1e-12, (nf, nq)
            assert np.abs(gwn.winding_number(V, F[:nf], Q) - Wo).max() <= 1e-12, (nf, nq)


def test_exact_rejects_bad_index():
    V, F = D.noisy_sphere(1, 0.01, 3)
    F = F.copy()
    F[0, 0] = -1
    with pytest.raises(gwn.GWNError):
        gwn.winding_number(V, F, np.zeros((1, 3)))


def test_exact_2d_curves_vs_oracle():
    """2D curves (igl::winding_number with F.cols() == 2): GPU FP64 against the
    oracle's restatement of signed_angle summed over edges (pinned by closed
    forms), on a noisy closed star polygon and an open arc, plus the square's
    closed forms through the C ABI."""
    import oracle_py as Op
    rng = np.random.default_rng(3)
    n = 3000
    t = np.sort(rng.uniform(0, 2 * np.pi, n))
    r = 1 + 0.3 * np.sin(7 * t) + 0.01 * rng.normal(size=n)
    V = np.stack([r * np.cos(t), r * np.sin(t)], 1)
    E = np.stack([np.arange(n), (np.arange(n) + 1) % n], 1).astype(np.int32)
    O = rng.uniform(-1.6, 1.6, (20000, 2))
    W = gwn.winding_number(V, E, O)
    Wo = Op.winding_number_2d(V, E, O)
    assert np.abs(W - Wo).max() < 1e-12
    inside = np.abs(Wo - 1) < 1e-9
    outside = np.abs(Wo) < 1e-9
    assert inside.sum() > 1000 and outside.sum() > 1000 and np.all(np.abs(W[outside]) < 1e-9)
    Wa = gwn.winding_number(V, E[: n // 3], O[:500])
    assert np.abs(Wa - Op.winding_number_2d(V, E[: n // 3], O[:500])).max() < 1e-12
    Vs = np.array([[0, 0], [1, 0], [1, 1], [0, 1]], float)
    Es = np.array([[0, 1], [1, 2], [2, 3], [3, 0]], np.int32)
    assert np.allclose(gwn.winding_number(Vs, Es, np.array([[0.5, 0.5], [3.0, 3.0]])), [1, 0], atol=1e-15)


def test_exact_2d_few_queries_many_edges():
    """A few queries against thousands of edges: the edges are split into
    chunks whose partial sums are added in chunk order."""
    import oracle_py as Op
    n = 12_000
    t = np.linspace(0, 2 * np.pi, n, endpoint=False)
    V = np.stack([np.cos(t) * (1 + 0.2 * np.cos(5 * t)), np.sin(t) * (1 + 0.2 * np.cos(5 * t))], 1)
    E = np.stack([np.arange(n), (np.arange(n) + 1) % n], 1).astype(np.int32)
    for nq in (1, 300):
        Q = np.random.default_rng(nq).uniform(-1.4, 1.4, (nq, 2))
        W = gwn.winding_number(V, E, Q)
        assert np.abs(W - Op.winding_number_2d(V, E, Q)).max() < 1e-12, nq



def _cube(scale=1.0):
    """An axis-aligned cube, two triangles a side, outward."""
    V = np.array([[x, y, z] for x in (-1, 1) for y in (-1, 1) for z in (-1, 1)], np.float64) * 0.5 * scale
    quads = [(0, 1, 3, 2), (4, 6, 7, 5), (0, 4, 5, 1), (2, 3, 7, 6), (0, 2, 6, 4), (1, 5, 7, 3)]
    F = np.array([t for a, b, c, d in quads for t in ((a, b, c), (a, c, d))], np.int32)
    return V, F


@pytest.mark.parametrize("nq", [125, 65_541])
def test_queries_on_vertices_edges_and_faces(nq):
    """Queries at a cube's corners, on its edges, face diagonals and faces: the
    terms there hang on the sign of a zero and on last bits (a half turn each
    way), and the angle product leaves them to the per-triangle form, so the
    sums equal the oracle's term by term sum."""
    V, F = _cube()
    g = np.linspace(-1.0, 1.0, 5)  # -1 -0.5 0 0.5 1: corners, edge and face midpoints, diagonals
    Q = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    Q = np.tile(Q, (-(-nq // Q.shape[0]), 1))[:nq]
    Wo = O.winding_number_bf(V, F, Q[:125])
    assert len(np.unique(np.round(Wo * 8))) > 3  # corners, edges and faces do differ
    W = gwn.winding_number_bruteforce(V, F, Q)
    np.testing.assert_allclose(W, np.tile(Wo, -(-nq // 125))[:nq], rtol=0, atol=1e-12)
    P = np.array([[-0.5, -0.5], [0.5, -0.5], [0.5, 0.5], [-0.5, 0.5]])
    E = np.array([[0, 1], [1, 2], [2, 3], [3, 0]], np.int32)
    W2 = gwn.winding_number(P, E, Q[:, :2])
    np.testing.assert_allclose(W2[:125], O.winding_number_2d(P, E, Q[:125, :2]), rtol=0, atol=1e-12)


@pytest.mark.parametrize("tris,nq", [(5_000, 20_000), (32_000, 10_000), (89_000, 70_000)])
def test_hierarchy_sums_are_those_of_its_terms(tris, nq):
    """Some queries of any batch lie near an edge of a face or a cap, where the
    angle turns by the roundings of its vector over that vector's length: the
    product leaves those terms to the per-triangle form, and the sums equal the
    oracle's hierarchy, term by term.  Bounds: a term in the product differs by
    less than 1e-13 rad (1.6e-14 in w), and two such may meet in a query; the
    2-norm is twice what the forms differ by on the host with the same lists,
    9e-16.  With every term in the product they differ by 2.5e-15 to 5.5e-14
    (2-norm) and 1.7e-13 to 4e-12 (largest, in root mean squares)."""
    V, F = D.uv_sphere(tris, 0, 3)
    rng = np.random.default_rng(tris)
    V = V * (1.0 + rng.normal(0.0, 0.01, (V.shape[0], 1)))
    Q = rng.uniform(-1.5, 1.5, (nq, 3))
    O.libc_srand(tris)
    tree = gwn.WindingNumberAABB(V, F)
    O.libc_srand(tris)
    Wo = O.WNTree(V, F).query(Q)
    d = tree.winding_number(Q) - Wo
    rms = np.sqrt(np.mean(Wo * Wo))
    print(f"{F.shape[0]} faces: rel {np.linalg.norm(d) / np.linalg.norm(Wo):.2e} max {np.abs(d).max() / rms:.2e}")
    assert np.linalg.norm(d) <= 2e-15 * np.linalg.norm(Wo)
    assert np.abs(d).max() <= 1e-13 * rms


@pytest.mark.parametrize("nq", [1, 63, 65, 4097, 65_535, 65_536, 540_001])
def test_hierarchy_lanes_and_order_by_batch_size(nq):
    """Input order, and the Hilbert order from 532,414 queries on (a tree of 127
    records), 64 lanes a query: the reference's lists (leaves of up to 100 faces, caps of any
    length) agree with the sum over every face to rounding."""
    V, F = D.noisy_sphere(4, 0.01, 5)
    Q = np.random.default_rng(nq).uniform(-1.3, 1.3, (nq, 3))
    W = gwn.WindingNumberAABB(V, F).winding_number(Q)
    np.testing.assert_allclose(W, gwn.winding_number_bruteforce(V, F, Q), rtol=0, atol=1e-11)


@pytest.mark.parametrize("nq", [125, 65_541])
def test_fp64_soup_exact_terms_on_edges_and_faces(nq):
    """The FP64 walk with every triangle exact (accuracy_scale 1e3), queries on
    a cube's corners, edges, diagonals and faces: UTsignedSolidAngleTri in FP64
    (6070-6110) term by term, zero where the numerator or a length is zero."""
    V, F = _cube()
    g = np.linspace(-1.0, 1.0, 5)
    Q = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    ref = np.zeros(125)
    for t in F:
        d = V[t][None] - Q[:, None]  # 125 x 3 x 3
        l = np.sqrt(d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1] + d[..., 2] * d[..., 2])
        ok = (l != 0).all(1)
        d = d / np.where(l == 0, 1.0, l)[..., None]
        a, b, c = d[:, 0], d[:, 1], d[:, 2]
        u, w = b - a, c - a
        num = (a[:, 0] * (u[:, 1] * w[:, 2] - u[:, 2] * w[:, 1]) + a[:, 1] * (u[:, 2] * w[:, 0] - u[:, 0] * w[:, 2])
               + a[:, 2] * (u[:, 0] * w[:, 1] - u[:, 1] * w[:, 0]))

        def dot(p, q):
            return p[:, 0] * q[:, 0] + p[:, 1] * q[:, 1] + p[:, 2] * q[:, 2]
        den = 1.0 + dot(a, b) + dot(a, c) + dot(b, c)
        ref += np.where(ok & (num != 0), 2.0 * np.arctan2(num, den), 0.0)
    Qn = np.tile(Q, (-(-nq // 125), 1))[:nq]
    bvh = gwn.FastWindingNumberBVH().build(V, F, 2)
    W = bvh.query(Qn, 1e3, gwn.PREC_FP64)
    np.testing.assert_allclose(W, np.tile(ref / (4 * np.pi), -(-nq // 125))[:nq], rtol=0, atol=1e-12)


@pytest.mark.parametrize("nq", [2_000, 65_541])
@pytest.mark.parametrize("where", ["near edges", "on the surface"])
def test_fp64_soup_terms_at_the_surface(where, nq):
    """The FP64 walk with every triangle exact (accuracy_scale 1e3), queries
    1e-6 to 1e-3 from the edges of 1,280 triangles, or at their corners, the
    middles of their edges and their centroids: a triangle's vector (den, num)
    may be short there and turns by its roundings over its length, and in a
    triangle's plane the sign of num decides a half turn.  Such terms are
    UTsignedSolidAngleTri's own (6070-6110), so W equals their sum.  Bound: the
    other terms' vectors are 1e-2 or longer and round by a few 1.1e-16 (a few
    1e-14 rad, a fourth of it in w, for the two triangles at the edge), and
    1,280 products of 1.1e-16.  The mixed form takes these terms in FP64 too and
    the others in FP32."""
    V, F = D.bumpy_sphere(3, 8, 12)
    rng = np.random.default_rng(12)
    T = V.astype(np.float32).astype(np.float64)[F]
    f, s = rng.integers(0, F.shape[0], 2000), rng.random((2000, 1))
    if where == "near edges":
        r = 10.0 ** rng.uniform(-6, -3, (2000, 1))
        Q = (1 - s) * T[f, 0] + s * T[f, 1] + r * rng.normal(size=(2000, 3))
    else:
        Q = np.concatenate([T[f[:200], 0], 0.5 * (T[f[200:1200], 0] + T[f[200:1200], 1]), T[f[1200:]].mean(1)])
    Q = Q.astype(np.float32).astype(np.float64)
    ref = np.empty(2000)
    for i, q in enumerate(Q):
        d = T - q
        l = np.sqrt(d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1] + d[..., 2] * d[..., 2])
        d = d * (1.0 / np.where(l == 0, 1.0, l))[..., None]
        (a0, a1, a2), (b0, b1, b2), (c0, c1, c2) = (d[:, k].T for k in range(3))
        u0, u1, u2, w0, w1, w2 = b0 - a0, b1 - a1, b2 - a2, c0 - a0, c1 - a1, c2 - a2
        num = a0 * (u1 * w2 - u2 * w1) + a1 * (u2 * w0 - u0 * w2) + a2 * (u0 * w1 - u1 * w0)
        den = (1.0 + (a0 * b0 + a1 * b1 + a2 * b2) + (a0 * c0 + a1 * c1 + a2 * c2) + (b0 * c0 + b1 * c1 + b2 * c2))
        t = np.where((num != 0) & (l != 0).all(1), 2.0 * np.arctan2(num, den), 0.0)
        ref[i] = t.astype(np.longdouble).sum() / (4 * np.pi)
    bvh = gwn.FastWindingNumberBVH().build(V, F, 2)
    for prec, tol in ((gwn.PREC_FP64, 1e-13), (gwn.PREC_MIXED, 1e-5)):
        W = bvh.query(np.tile(Q, (-(-nq // 2000), 1))[:nq], 1e3, prec)
        err = np.abs(W - np.tile(ref, -(-nq // 2000))[:nq])
        print(f"{where}: max |W - sum of terms| {err.max():.2e}")
        assert err.max() <= tol


@pytest.mark.parametrize("power", [-525, -300, 300])
@pytest.mark.parametrize("nq", [300, 20_000])
def test_exact_2d_at_any_scale(power, nq):
    """A curve and its queries scaled by a power of two have the same angles, also
    where the products of two lengths are denormal (2^-525: 1e-316): the angle
    product takes no vector that the denormals have rounded."""
    n = 1500
    t = np.linspace(0, 2 * np.pi, n, endpoint=False)
    r = 1 + 0.3 * np.sin(7 * t)
    V = np.stack([r * np.cos(t), r * np.sin(t)], 1)
    E = np.stack([np.arange(n), (np.arange(n) + 1) % n], 1).astype(np.int32)
    Q = np.random.default_rng(9).uniform(-1.6, 1.6, (nq, 2))
    Wo = O.winding_number_2d(V, E, Q)
    err = np.abs(gwn.winding_number(np.ldexp(V, power), E, np.ldexp(Q, power)) - Wo).max()
    print(f"2^{power}: max |dW| {err:.2e}")
    assert err < 1e-12
