"""GPU parity of the point-cloud path (igl::octree + fast_winding_number(P,N,A,...)).

Against the FP32 instantiation of the oracle restatement (itself pinned to the
reference's golden values and brute force):
  * octree: CH, cell centres, widths and the point set of every cell identical;
  * CM and R bit-identical (FP32 sums in ascending point order, as the
    reference), EC within 2e-5 relative (accumulated in FP64 on the GPU);
  * W within 1e-4 at beta = 2 and identical 0.5 classification outside a 1e-4
    band (the fast path's winding-number tolerance);
  * beta <= 0 brute force within 1e-5.
"""
import numpy as np
import pytest

import oracle_py as O
from libigl_amd import datagen as D
from libigl_amd import gwn

pytestmark = pytest.mark.gpu


def _cloud(n, seed=1, level=3):
    V, F = D.noisy_sphere(level, 0.01, 11)
    rng = np.random.default_rng(seed)
    P, N, _ = D.sample_surface(V, F, n, rng)
    _, area = D.face_normals(V, F)
    A = np.full(n, area.sum() / n)
    return P.astype(np.float32), N.astype(np.float32), A.astype(np.float32)


def test_one_point_golden_fp32():
    # tests/include/igl/fast_winding_number.cpp:17-53 (double there; FP32 here)
    P = np.array([[0.1, 0.2, 0.3]])
    N = np.array([[4.0, 5.0, 6.0]])
    N /= np.linalg.norm(N)
    A = np.array([0.7])
    Q = np.array([[0, 0, 0], [4, -3, 2], [-1, 1, 3], [0, 5, -2]], float)
    gold = np.array([0.38779369004261133, -0.00041235296362485, -0.00362978253577090, -0.00041235296362485])
    W = gwn.fast_winding_number(P, N, A, Q)
    assert np.abs(W - gold).max() < 1e-6 * np.abs(gold).max()


@pytest.mark.parametrize("n", [2, 3, 17, 500, 20000])
def test_octree_identical_to_reference_rules(n):
    P, N, A = _cloud(n, seed=n)
    c = gwn.PointCloudFWN(P, N, A, 2)
    CH, CN, W, cs, cc, pl = c.octree()
    o = O.Octree(P, np.float32)
    assert np.array_equal(CH, o.CH)
    assert np.array_equal(CN, o.CN) and np.array_equal(W, o.W)
    assert np.array_equal(cc, o.cell_count)
    for cell in range(CH.shape[0]):
        assert np.array_equal(np.sort(pl[cs[cell]:cs[cell] + cc[cell]]), o.point_indices(cell))


@pytest.mark.parametrize("order", [0, 1, 2])
def test_expansion_coefficients(order):
    P, N, A = _cloud(5000, seed=7)
    c = gwn.PointCloudFWN(P, N, A, order)
    CM, R, EC = c.expansion()
    oc = O.Cloud(P, N, A, order, np.float32)
    ne = oc.oct.cell_count > 0
    assert np.array_equal(np.isnan(CM[:, 0]), ~ne)
    scale = np.abs(oc.EC[ne]).max()
    # CM is summed as the reference sums it (FP32, ascending point index), so
    # CM and R match bit for bit and every near/far decision is the same
    assert np.array_equal(CM[ne], oc.CM[ne])
    assert np.array_equal(R[ne], oc.R[ne])
    assert np.abs(EC[ne] - oc.EC[ne]).max() < 2e-5 * scale
    assert np.all(EC[~ne] == 0) and np.all(R[~ne] == 0)


@pytest.mark.parametrize("beta", [1.0, 2.0, 4.0])
def test_eval_vs_oracle(beta):
    P, N, A = _cloud(20000, seed=3)
    rng = np.random.default_rng(4)
    V, F = D.noisy_sphere(3, 0.01, 11)
    Q = np.concatenate([rng.uniform(-1.3, 1.3, (4000, 3)), D.near_surface_queries(V, F, 2000, 1e-2, rng)])
    Q = Q.astype(np.float32)
    W = gwn.PointCloudFWN(P, N, A, 2).query(Q, beta)
    Wo = O.Cloud(P, N, A, 2, np.float32).eval(Q, beta)
    err = np.abs(W.astype(np.float64) - Wo)
    print(f"cloud beta {beta}: max {err.max():.3e}")
    assert err.max() <= 1e-4
    m = np.abs(Wo - 0.5) > 1e-4
    assert np.array_equal(W[m] > 0.5, Wo[m] > 0.5)


def test_brute_force_branch_and_large_beta():
    P, N, A = _cloud(3000, seed=5)
    Q = np.random.default_rng(6).uniform(-1.3, 1.3, (1000, 3)).astype(np.float32)
    c = gwn.PointCloudFWN(P, N, A, 2)
    Wb = c.query(Q, 0.0)
    Wo = O.Cloud(P, N, A, 2, np.float32).eval(Q, 0.0)
    assert np.abs(Wb - Wo).max() < 1e-5
    # very large beta: every cell is near, the walk ends at leaves -> brute force
    assert np.abs(c.query(Q, 1e9) - Wb).max() < 1e-4


def test_cloud_edge_cases():
    Q = np.random.default_rng(1).uniform(-1, 1, (100, 3)).astype(np.float32)
    # empty cloud
    c0 = gwn.PointCloudFWN(np.zeros((0, 3)), np.zeros((0, 3)), np.zeros(0), 2)
    assert np.all(c0.query(Q) == 0)
    # one point (root leaf) and a query on the point (0.5, fast_winding_number.cpp:163-166)
    P = np.array([[0.1, 0.2, 0.3]], np.float32)
    N = np.array([[0.0, 0.0, 1.0]], np.float32)
    A = np.array([0.5], np.float32)
    c1 = gwn.PointCloudFWN(P, N, A, 2)
    assert c1.query(P)[0] == 0.5
    # duplicate points: their cell cannot be split; values stay finite
    P2, N2, A2 = _cloud(200, seed=9)
    P2 = np.concatenate([P2, P2[:5]])
    N2 = np.concatenate([N2, N2[:5]])
    A2 = np.concatenate([A2, A2[:5]])
    c2 = gwn.PointCloudFWN(P2, N2, A2, 2)
    W2 = c2.query(Q, 2.0)
    assert np.all(np.isfinite(W2))
    assert np.abs(W2 - c2.query(Q, 0.0)).max() < 0.05
    with pytest.raises(ValueError):
        gwn.PointCloudFWN(P, N, A, 3)


def test_cloud_workload_full_size():
    P, N, A, Q = D.cloud_workload()  # 2M points, 160^3 grid
    c = gwn.PointCloudFWN(P, N, A, 2)
    W = c.query(Q, 2.0)
    assert W.shape == (Q.shape[0],) and np.all(np.isfinite(W))
    sub = np.arange(0, Q.shape[0], 4096)
    oc = O.Cloud(P.astype(np.float32), N.astype(np.float32), A.astype(np.float32), 2, np.float32)
    Wo = oc.eval(Q[sub].astype(np.float32), 2.0)
    err = np.abs(W[sub] - Wo)
    print(f"cloud 2M: cells {c.ncells()}, max|dW| on {sub.size} grid queries {err.max():.3e}")
    assert err.max() <= 1e-4
    r = np.linalg.norm(Q, axis=1)
    assert np.all(np.abs(W[r < 0.8] - 1) < 0.05) and np.all(np.abs(W[r > 1.2]) < 0.05)


# ---- precompute / evaluation over a caller's octree (fast_winding_number.h:44-53, 88-99) ----

def _lists(o):
    return [o.point_indices(c).tolist() for c in range(o.CH.shape[0])]


def test_from_octree_reference_lists():
    """The reference's own octree and lists: CM, R bit-identical to the
    oracle's precompute, EC within 2e-5 relative, W within 1e-4."""
    P, N, A = _cloud(20000, seed=21)
    o = O.Octree(P, np.float32)
    lists = _lists(o)
    c = gwn.PointCloudFWN.from_octree(P, N, A, lists, o.CH, 2)
    CM, R, EC = c.expansion()
    ot = O.Octree.from_lists(o.CH, lists, np.float32)
    CMo, Ro, ECo, ev = O.cloud_over(P, N, A, ot, 2)
    ne = o.cell_count > 0
    assert np.array_equal(CM[ne], CMo[ne]) and np.array_equal(R[ne], Ro[ne])
    scale = np.abs(ECo[ne]).max(axis=1, keepdims=True) + 1e-30
    assert (np.abs(EC[ne] - ECo[ne]) / scale).max() < 2e-5
    Q = np.random.default_rng(3).uniform(-1.3, 1.3, (4000, 3)).astype(np.float32)
    W = c.query(Q, 2.0)
    assert np.abs(W - ev(Q, 2.0)).max() <= 1e-4
    # same tree and lists as the library's own octree: same answers
    W_own = gwn.PointCloudFWN(P, N, A, 2).query(Q, 2.0)
    assert np.abs(W - W_own).max() <= 1e-5


def test_from_octree_list_order_is_summation_order():
    """Centres are summed over each cell's list in list order (FP32, as
    fast_winding_number.cpp:60-73): shuffled lists give the oracle's shuffled
    centres bit for bit."""
    P, N, A = _cloud(20000, seed=22)
    o = O.Octree(P, np.float32)
    rng = np.random.default_rng(5)
    lists = [rng.permutation(o.point_indices(c)).tolist() for c in range(o.CH.shape[0])]
    c = gwn.PointCloudFWN.from_octree(P, N, A, lists, o.CH, 1)
    CM, R, EC = c.expansion()
    CMo, Ro, ECo, ev = O.cloud_over(P, N, A, O.Octree.from_lists(o.CH, lists, np.float32), 1)
    CMa, _, _, _ = O.cloud_over(P, N, A, O.Octree.from_lists(o.CH, _lists(o), np.float32), 1)
    ne = o.cell_count > 0
    assert np.array_equal(CM[ne], CMo[ne]) and np.array_equal(R[ne], Ro[ne])
    assert not np.array_equal(CMo[ne], CMa[ne])  # the order is visible in the last bits
    Q = np.random.default_rng(6).uniform(-1.3, 1.3, (2000, 3)).astype(np.float32)
    assert np.abs(c.query(Q, 2.0) - ev(Q, 2.0)).max() <= 1e-4


def test_from_octree_given_expansion_is_used():
    """CM, R, EC passed to the evaluation overload are used as given (here
    scaled so they differ from any precompute)."""
    P, N, A = _cloud(5000, seed=23)
    o = O.Octree(P, np.float32)
    lists = _lists(o)
    ot = O.Octree.from_lists(o.CH, lists, np.float32)
    CMo, Ro, ECo, _ = O.cloud_over(P, N, A, ot, 2)
    CMg, Rg, ECg = CMo.copy(), (Ro * 0.75).astype(np.float32), (ECo * 1.5).astype(np.float32)
    *_, ev = O.cloud_over(P, N, A, ot, 2, CM=CMg, R=Rg, EC=ECg)
    Q = np.random.default_rng(7).uniform(-1.5, 1.5, (3000, 3)).astype(np.float32)
    W = gwn.fast_winding_number(P, N, A, lists, o.CH, CMg, Rg, ECg, Q, 2.0)
    Wo = ev(Q, 2.0)
    assert np.abs(W - Wo).max() <= 1.5e-4
    assert np.abs(W - gwn.PointCloudFWN(P, N, A, 2).query(Q, 2.0)).max() > 1e-3  # the scaling shows
    # precompute overload returns the same CM/R as the oracle's over these lists
    CM, R, EC = gwn.fast_winding_number(P, N, A, lists, o.CH, 2)
    ne = o.cell_count > 0
    assert np.array_equal(CM[ne], CMo[ne]) and np.array_equal(R[ne], Ro[ne])


def test_from_octree_root_leaf_and_custom_tree():
    P, N, A = _cloud(300, seed=24)
    Q = np.random.default_rng(8).uniform(-1.5, 1.5, (500, 3)).astype(np.float32)
    # a single leaf holding every point: brute force over its list
    CH = -np.ones((1, 8), np.int32)
    lists = [list(range(300))]
    W = gwn.PointCloudFWN.from_octree(P, N, A, lists, CH, 2).query(Q, 2.0)
    *_, ev = O.cloud_over(P, N, A, O.Octree.from_lists(CH, lists, np.float32), 2)
    assert np.abs(W - ev(Q, 2.0)).max() <= 1e-5
    # a hand-made two-level tree that is no geometric octree (points dealt
    # round-robin to the 8 children), with one empty child
    CH = -np.ones((9, 8), np.int32)
    CH[0] = np.arange(1, 9)
    lists = [list(range(300))] + [list(range(k, 300, 7)) for k in range(7)] + [[]]
    c = gwn.PointCloudFWN.from_octree(P, N, A, lists, CH, 2)
    *_, ev = O.cloud_over(P, N, A, O.Octree.from_lists(CH, lists, np.float32), 2)
    for beta in (0.5, 2.0, 8.0):
        assert np.abs(c.query(Q, beta) - ev(Q, beta)).max() <= 1e-4


def test_from_octree_rejects_bad_trees():
    P, N, A = _cloud(50, seed=25)
    lists = [list(range(50))] + [[]] * 8
    CH = -np.ones((9, 8), np.int32)
    CH[0] = np.arange(1, 9)
    CH[1] = [0, 2, 3, 4, 5, 6, 7, 8]  # cycle back to the root
    with pytest.raises(gwn.GWNError):
        gwn.PointCloudFWN.from_octree(P, N, A, lists, CH, 2)
    CH[1] = -1
    CH[0, 3] = -1  # split cell with a missing child
    with pytest.raises(gwn.GWNError):
        gwn.PointCloudFWN.from_octree(P, N, A, lists, CH, 2)
    CH[0, 3] = 4
    CH[0] = np.arange(1, 9)
    bad = [list(range(50)) + [50]] + [[]] * 8  # point index out of range
    with pytest.raises(gwn.GWNError):
        gwn.PointCloudFWN.from_octree(P, N, A, bad, CH, 2)
    # an octree built without normals/areas holds no expansion
    c = gwn.PointCloudFWN(P)
    with pytest.raises(gwn.GWNError):
        c.query(P[:3])
    pi, CH2, CN2, W2 = gwn.octree(P)
    o = O.Octree(P, np.float32)
    assert np.array_equal(CH2, o.CH) and np.array_equal(CN2, o.CN) and np.array_equal(W2, o.W)
    assert all(pi[k] == o.point_indices(k).tolist() for k in range(len(pi)))


@pytest.mark.parametrize("radius", [1.0, 0.0, -1.0, 1e-20, 1e25])
@pytest.mark.parametrize("beta", [1e-4, 2.0, 1e7])
def test_far_test_by_squares(radius, beta):
    """The far test compares squares where FP32 holds them and takes the root
    otherwise.  A caller's radii times `radius`: as they are, zero, negative,
    and with squares outside FP32's range; beta inside and outside the plain
    range; queries at cell centres and at the threshold to a last bit either
    way.  The decisions are the oracle's, which takes the root and the double
    product everywhere: a wrong one would show as a whole cell's error."""
    P, N, A = _cloud(5000, seed=29)
    o = O.Octree(P, np.float32)
    lists = _lists(o)
    CM, R, EC, _ = O.cloud_over(P, N, A, O.Octree.from_lists(o.CH, lists, np.float32), 2)
    R = (R * np.float32(radius)).astype(np.float32)
    *_, ev = O.cloud_over(P, N, A, O.Octree.from_lists(o.CH, lists, np.float32), 2, CM=CM, R=R, EC=EC)
    rng = np.random.default_rng(29)
    k = rng.integers(0, CM.shape[0], 400)
    k = k[o.cell_count[k] > 0]
    with np.errstate(over="ignore", invalid="ignore"):
        edge = CM[k] + np.stack([np.float64(beta) * R[k]] + [np.zeros(k.size)] * 2, 1).astype(np.float32)
    edge = edge[np.isfinite(edge).all(1) & (np.abs(edge) < 1e6).all(1)]
    Q = np.concatenate([edge, np.nextafter(edge, np.float32(9)), np.nextafter(edge, np.float32(-9)), CM[k],
                        rng.uniform(-1.3, 1.3, (500, 3))]).astype(np.float32)
    W, Wo = gwn.fast_winding_number(P, N, A, lists, o.CH, CM, R, EC, Q, beta), ev(Q, beta)
    ok = np.isfinite(Wo) & (np.abs(Wo) < 1e3)  # not at a centre taken for far
    assert ok.sum() > 500
    d = np.abs(W - Wo)[ok] / np.maximum(1.0, np.abs(Wo[ok]))
    assert (d <= 2e-4).all(), (d.max(), int((d > 2e-4).sum()))


def _clusters(sizes, copies):
    rng = np.random.default_rng(len(sizes) + copies)
    parts = [rng.uniform(-1, 1, (n, 3)) * 40.0 ** -k + [0.3, -0.2, 0.1] for k, n in enumerate(sizes)]
    parts.append(np.repeat([[0.25, 0.5, -0.75]], copies, axis=0))
    P = np.concatenate(parts)
    P = P[rng.permutation(len(P))].astype(np.float32)
    return P, rng.normal(size=P.shape).astype(np.float32), rng.uniform(0.5, 2.0, len(P)).astype(np.float32)


@pytest.mark.parametrize("sizes", [(2,), (64, 3), (513, 130, 40, 9, 4), (5000, 2000, 700, 129, 2, 2), (66000, 512)])
def test_levels_of_few_points(sizes):
    # clusters inside clusters: most points leave the split cells from one
    # level to the next, in rows of 64 and 512 terms and past them; octree, CM
    # and R are bit-identical
    P, N, A = _clusters(sizes, 0)
    c = gwn.PointCloudFWN(P, N, A, 2)
    oc = O.Cloud(P, N, A, 2, np.float32)
    CH, CN, W, _, cc, _ = c.octree()
    assert np.array_equal(CH, oc.oct.CH) and np.array_equal(CN, oc.oct.CN) and np.array_equal(W, oc.oct.W)
    assert np.array_equal(cc, oc.oct.cell_count)
    CM, R, EC = c.expansion()
    ne = cc > 0
    assert np.array_equal(CM[ne], oc.CM[ne]) and np.array_equal(R[ne], oc.R[ne])
    assert np.isnan(CM[~ne]).all() and np.all(EC[~ne] == 0) and np.all(R[~ne] == 0)


@pytest.mark.parametrize("copies", [2, 33, 70, 600])
def test_centres_with_points_that_no_level_tells_apart(copies):
    # every centre is the FP32 sum over its cell's points in index order
    P, N, A = _clusters((513, 130, 9), copies)
    c = gwn.PointCloudFWN(P, N, A, 0)
    _, _, _, cs, cc, pl = c.octree()
    CM, _, _ = c.expansion()
    for cell in np.flatnonzero(cc):
        i = np.sort(pl[cs[cell]:cs[cell] + cc[cell]])
        m = np.cumsum(A[i, None] * P[i], axis=0, dtype=np.float32)[-1] / np.cumsum(A[i], dtype=np.float32)[-1]
        assert np.array_equal(CM[cell], m)


@pytest.mark.parametrize("first", [0.0, -0.0])
def test_flat_cloud_keeps_its_signs(first):
    # a cloud in the plane z = 0: the root's centre is what minima and maxima
    # that start from the first point give
    P = np.random.default_rng(5).uniform(-1, 1, (1000, 3)).astype(np.float32)
    P[:, 2] = -first
    P[0, 2] = first
    _, CN, _, _, _, _ = gwn.PointCloudFWN(P, np.ones_like(P), np.ones(1000, np.float32), 0).octree()
    o = O.Octree(P, np.float32)
    assert np.array_equal(CN, o.CN) and np.array_equal(np.signbit(CN[0]), np.signbit(o.CN[0]))
