"""What a program that uses this library has it compute, as cases to be timed.

Each case is one pass through the library's public entry points (include/gwn.h,
libigl_amd/gwn.py): the resident meshes, clouds and curves are what a program
keeps, the queries are what it asks.  The device entry points take torch
tensors by address; the one-shot calls take and return numpy arrays, as igl's
functions take matrices.

Kinds:
  soup       fast winding number of a triangle mesh (igl::fast_winding_number)
  oneshot    the same from host arrays, tree built for the call
  cloud      fast winding number of an oriented point cloud
  estimated  the same for a cloud without areas: knn, point areas, octree,
             precompute and query, from host arrays
  exact      exact FP64 winding number through the cap hierarchy
  distance   signed distance with the fast winding number's sign
  antipodal  winding number by boundary term and ray crossings
  curve      2D fast winding number (UT_SubtendedAngle)
"""
import ctypes
import functools
import math

import numpy as np
import torch

from libigl_amd import datagen, gwn
from libigl_amd._native import check, lib

DEVICE = "cuda"
PREC = {"fp32": gwn.PREC_FP32, "mixed": gwn.PREC_MIXED, "fp64": gwn.PREC_FP64}
TREE = {"sah4": gwn.TREE_SAH4, "lbvh": gwn.TREE_LBVH}
# Brute-force pairs that exact() takes on: about 20 s of FP64 torch.
MOST_PAIRS = 9e10
MOST_DISTANCE_PAIRS = 2e9


def listed():
    return [
        # one point against a resident mesh: the single-point overload
        # (fast_winding_number.h:203-206), called in a loop by interactive tools
        dict(name="soup_point", kind="soup", tris=81920, queries=1, beta=2.0, precision="fp32", tree="sah4", order=2),
        # a small request of a serving trace (batches of 1k to 1M), ragged, at
        # the accuracy scale that keeps |dw| near 1e-4, in the mixed form
        dict(name="soup_request", kind="soup", tris=119025, queries=5003, beta=4.9, precision="mixed", tree="sah4",
             order=2),
        # the benchmark's headline: 81,920 triangles, 1M queries, |dw| <= 1e-4
        dict(name="soup_batch", kind="soup", tris=81920, queries=1000000, beta=4.9, precision="fp32", tree="sah4",
             order=2),
        # the FP64 form at the reference's default accuracy scale, ragged
        dict(name="soup_fp64", kind="soup", tris=81920, queries=200003, beta=2.0, precision="fp64", tree="sah4",
             order=2),
        # the largest: 1.31M triangles, 10M queries, mixed form
        dict(name="soup_large", kind="soup", tris=1310720, queries=10000000, beta=5.25, precision="mixed", tree="sah4",
             order=2),
        # igl::fast_winding_number(V,F,Q,W): a user with a new mesh, host arrays
        dict(name="soup_oneshot", kind="oneshot", tris=20480, queries=100000, tree="sah4"),
        # point cloud: 2M points, a 160^3 grid of queries (surface reconstruction)
        dict(name="cloud_grid", kind="cloud", points=2000000, queries=4096000, beta=2.0, order=2),
        # a scanned cloud with normals and no areas, host arrays in and out
        dict(name="cloud_estimated", kind="estimated", points=500000, queries=262144, beta=2.0, order=2),
        # exact winding number of a resident hierarchy, 100k queries
        dict(name="exact_tree", kind="exact", tris=20480, queries=100000),
        # signed distance of 1M points, sign by fast winding number
        dict(name="signed_distance", kind="distance", tris=81920, queries=1000000),
        # antipodal method on a closed mesh, 1M queries
        dict(name="antipodal", kind="antipodal", tris=81920, queries=1000000),
        # 2D curve, 1M queries at the reference's default accuracy scale
        dict(name="curve", kind="curve", segments=262144, queries=1000000, beta=2.0, order=2),
    ]


def _log_int(rng, lo, hi):
    """An integer whose logarithm is uniform; odd ones as often as even ones."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["soup"] * 5 + ["oneshot", "cloud", "estimated", "exact", "distance", "antipodal", "curve"])
    if kind == "soup":
        # meshes of 1k to 500k triangles, batches of one to 2M queries
        return dict(kind=kind, tris=_log_int(rng, 1000, 500000), queries=_log_int(rng, 1, 2000000),
                    beta=round(rng.uniform(2.0, 5.25), 2), precision=rng.choice(["fp32", "fp32", "mixed", "fp64"]),
                    tree=rng.choice(["sah4", "sah4", "lbvh"]), order=rng.choice([2, 2, 1, 0]))
    if kind == "oneshot":
        return dict(kind=kind, tris=_log_int(rng, 1000, 80000), queries=_log_int(rng, 1000, 300000),
                    tree=rng.choice(["sah4", "lbvh"]))
    if kind == "cloud":
        return dict(kind=kind, points=_log_int(rng, 10000, 2000000), queries=_log_int(rng, 1000, 4000000),
                    beta=round(rng.uniform(1.5, 3.0), 2), order=rng.choice([2, 2, 1, 0]))
    if kind == "estimated":
        return dict(kind=kind, points=_log_int(rng, 10000, 500000), queries=_log_int(rng, 1000, 300000), beta=2.0,
                    order=2)
    if kind == "curve":
        return dict(kind=kind, segments=_log_int(rng, 1000, 300000), queries=_log_int(rng, 1000, 2000000),
                    beta=round(rng.uniform(2.0, 5.0), 2), order=rng.choice([2, 2, 1, 0]))
    return dict(kind=kind, tris=_log_int(rng, 1000, 100000), queries=_log_int(rng, 1000, 1000000))


# ---------------------------------------------------------------------------
# inputs: bumpy and noisy spheres, queries half (a fifth for the largest mesh)
# next to the surface, as in libigl_amd/datagen.py, made on the GPU

@functools.lru_cache(maxsize=8)
def _sphere(tris):
    """A unit sphere's vertices and faces: an icosphere where the count is
    20 * 4^level, a latitude/longitude sphere of about `tris` otherwise."""
    for level in range(10):
        if tris == 20 * 4 ** level:
            return datagen.icosphere(level)
    return datagen.uv_sphere(tris, nbumps=0)


def _mesh(tris, seed, bumps=None):
    """A closed mesh: the sphere displaced by Gaussian bumps (or, with
    bumps=0, by 1% radial noise).  V float64, F int32 numpy arrays."""
    U, F = _sphere(tris)
    rng = np.random.default_rng(seed)
    if bumps == 0:
        return U * (1.0 + rng.normal(0.0, 0.01, size=(U.shape[0], 1))), F
    n = bumps or (64 if tris > 1000000 else 16)
    c = rng.normal(size=(n, 3))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    a, w = rng.uniform(-0.3, 0.3, size=n), rng.uniform(0.1, 0.4, size=n)
    u, ct = torch.from_numpy(U).to(DEVICE), torch.from_numpy(c).to(DEVICE)
    d2 = ((u * u).sum(1, keepdim=True) + 1.0) - 2.0 * (u @ ct.T)
    r = 1.0 + torch.exp(-d2 / torch.from_numpy(w * w).to(DEVICE)) @ torch.from_numpy(a).to(DEVICE)
    return (u * r[:, None]).cpu().numpy(), F


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) + 1000)
    return g


def _surface(V, F, n, g):
    """n points area-uniform on the mesh and their unit face normals (FP64, GPU)."""
    v, f = torch.from_numpy(V).to(DEVICE), torch.from_numpy(F).to(DEVICE).long()
    a, b, c = v[f[:, 0]], v[f[:, 1]], v[f[:, 2]]
    nrm = torch.linalg.cross(b - a, c - a)
    dbl = nrm.norm(dim=1)
    cum = torch.cumsum(dbl, 0)
    k = torch.searchsorted(cum, torch.rand(n, generator=g, device=DEVICE, dtype=torch.float64) * cum[-1])
    k.clamp_(max=f.shape[0] - 1)
    r1 = torch.rand(n, 1, generator=g, device=DEVICE, dtype=torch.float64).sqrt()
    r2 = torch.rand(n, 1, generator=g, device=DEVICE, dtype=torch.float64)
    pts = (1 - r1) * a[k] + (r1 * (1 - r2)) * b[k] + (r1 * r2) * c[k]
    return pts, nrm[k] / dbl[k].clamp(min=1e-300)[:, None], float(dbl.sum()) / 2


def _queries(V, F, n, seed, near=0.5, dist=1e-3):
    """n queries, a share `near` of them at +-dist from the surface, the others
    uniform in the mesh's box (FP64, GPU).  The first is a point inside, so
    that the results of the smallest batches are not all near zero."""
    g = _generator(seed)
    lo, hi = torch.from_numpy(V.min(0)).to(DEVICE), torch.from_numpy(V.max(0)).to(DEVICE)
    nn = int(n * near)
    q = lo + (hi - lo) * torch.rand(n - nn, 3, generator=g, device=DEVICE, dtype=torch.float64)
    q[0] = _surface(V, F, 1, g)[0][0] * torch.rand(1, generator=g, device=DEVICE, dtype=torch.float64) * 0.9
    if nn == 0:
        return q
    p, nrm, _ = _surface(V, F, nn, g)
    s = torch.rand(nn, 1, generator=g, device=DEVICE, dtype=torch.float64) < 0.5
    return torch.cat([q, p + torch.where(s, -dist, dist) * nrm])


def _grid(P, n):
    """About n^(1/3) queries a side over the cloud's box padded by 10% (the
    first n of the grid's points), FP32 on the GPU."""
    res = int(math.ceil(n ** (1.0 / 3.0) - 1e-9))
    lo, hi = P.amin(0), P.amax(0)
    ext = hi - lo
    t = torch.linspace(0.0, 1.0, res, device=DEVICE, dtype=torch.float64)
    ax = [(lo[d] - 0.1 * ext[d]) + t * (1.2 * ext[d]) for d in range(3)]
    g = torch.stack(torch.meshgrid(*ax, indexing="ij"), -1).reshape(-1, 3)
    return g[:n].float().contiguous()


def _curve(segments, queries, seed):
    """A closed bumpy curve and queries half uniform, half within 1e-3 of it."""
    P, E = datagen.bumpy_curve(segments, 16, seed)
    p, g = torch.from_numpy(P).to(DEVICE), _generator(seed)
    lo, hi = p.amin(0), p.amax(0)
    nn = queries // 2
    q = lo + (hi - lo) * torch.rand(queries - nn, 2, generator=g, device=DEVICE, dtype=torch.float64)
    k = torch.randint(segments, (nn,), generator=g, device=DEVICE)
    a, b = p[k], p[(k + 1) % segments]
    d = b - a
    n = torch.stack([d[:, 1], -d[:, 0]], 1) / d.norm(dim=1, keepdim=True).clamp(min=1e-300)
    s, r = (torch.rand(nn, 1, generator=g, device=DEVICE, dtype=torch.float64) for _ in range(2))
    return P.astype(np.float32), E, torch.cat([q, a + s * d + n * (2e-3 * r - 1e-3)]).float().contiguous()


class Handle:
    """A resident object made through the C interface, freed with this one."""

    def __init__(self, build, free, *args):
        h = ctypes.c_void_p()
        check(getattr(lib(), build)(*args, ctypes.byref(h)))
        self.h, self.free = h.value, getattr(lib(), free)

    def __del__(self):
        if getattr(self, "h", None):
            self.free(self.h)


def _inputs(case, seed):
    """The arrays of the case, from the seed alone."""
    kind = case["kind"]
    if kind == "curve":
        return _curve(case["segments"], case["queries"], seed)
    if kind in ("cloud", "estimated"):
        V, F = _mesh(20480, seed, bumps=0)
        P, N, area = _surface(V, F, case["points"], _generator(seed))
        return P, N, area / case["points"], _grid(P, case["queries"])
    V, F = _mesh(case["tris"], seed, bumps=0 if kind == "exact" else None)
    if kind == "exact":  # queries uniform in [-1.5, 1.5]^3
        return V, F, torch.rand(case["queries"], 3, generator=_generator(seed), device=DEVICE,
                                dtype=torch.float64) * 3.0 - 1.5
    near, dist = (0.2, 1e-4) if case["tris"] > 1000000 else (0.5, 1e-3)
    return V, F, _queries(V, F, case["queries"], seed, near, dist)


def prepare(case, seed):
    kind, n = case["kind"], case["queries"]
    a = _inputs(case, seed)
    if kind == "soup":
        V, F, Q = a
        bvh = gwn.FastWindingNumberBVH().build(V, F, case["order"], TREE[case["tree"]])
        return dict(kind=kind, bvh=bvh, Q=Q.float().contiguous(), beta=case["beta"], precision=PREC[case["precision"]],
                    W=torch.empty(n, dtype=torch.float64, device=DEVICE))
    if kind == "oneshot":
        V, F, Q = a
        return dict(kind=kind, V=V, F=F, Q=Q.cpu().numpy(), tree=TREE[case["tree"]])
    if kind == "cloud":
        P, N, area, Q = a
        Ph, Nh = P.float().cpu().numpy(), N.float().cpu().numpy()
        A = np.full(P.shape[0], area, np.float32)
        h = Handle("gwn_cloud_build", "gwn_cloud_free", Ph, Nh.ctypes.data, A.ctypes.data, P.shape[0], case["order"])
        return dict(kind=kind, h=h, Q=Q, beta=case["beta"], W=torch.empty(n, dtype=torch.float32, device=DEVICE))
    if kind == "estimated":
        P, N, _, Q = a
        return dict(kind=kind, P=P.cpu().numpy(), N=N.cpu().numpy(), Q=Q.cpu().numpy(), beta=case["beta"],
                    order=case["order"])
    if kind == "exact":
        V, F, Q = a
        ctypes.CDLL(None).srand(int(seed) & 0x7FFFFFFF)  # the hierarchy's caps draw rand()
        h = Handle("gwn_exact_tree_build", "gwn_exact_tree_free", V, V.shape[0], F, F.shape[0])
        return dict(kind=kind, h=h, Q=Q, W=torch.empty(n, dtype=torch.float64, device=DEVICE))
    if kind == "distance":
        V, F, Q = a
        bvh = gwn.FastWindingNumberBVH().build(V, F, 2)
        return dict(kind=kind, bvh=bvh, Q=Q, S=torch.empty(n, dtype=torch.float64, device=DEVICE),
                    I=torch.empty(n, dtype=torch.int32, device=DEVICE),
                    C=torch.empty(n, 3, dtype=torch.float64, device=DEVICE))
    if kind == "antipodal":
        V, F, Q = a
        h = Handle("gwn_antipodal_build", "gwn_antipodal_free", V, V.shape[0], F, F.shape[0], None)
        return dict(kind=kind, h=h, Q=Q, W=torch.empty(n, dtype=torch.float64, device=DEVICE))
    P, E, Q = a
    c = gwn.SubtendedAngle(P, E, case["order"])
    return dict(kind=kind, c=c, Q=Q, beta=case["beta"], W=torch.empty(n, dtype=torch.float32, device=DEVICE))


def run(s):
    kind = s["kind"]
    if kind == "oneshot":
        return gwn.fast_winding_number(s["V"], s["F"], s["Q"], tree=s["tree"])
    if kind == "estimated":
        return gwn.fast_winding_number_estimated_areas(s["P"], s["N"], s["Q"], s["order"], s["beta"])
    Q, n, st = s["Q"], s["Q"].shape[0], torch.cuda.current_stream().cuda_stream
    if kind == "soup":
        s["bvh"].query_device(Q.data_ptr(), n, s["W"].data_ptr(), s["beta"], s["precision"], st)
    elif kind == "curve":
        s["c"].query_device(Q.data_ptr(), n, s["W"].data_ptr(), s["beta"], st)
    elif kind == "cloud":
        check(lib().gwn_cloud_query_device(s["h"].h, Q.data_ptr(), n, s["beta"], s["W"].data_ptr(), st))
    elif kind == "exact":
        check(lib().gwn_exact_tree_query_device(s["h"].h, Q.data_ptr(), n, s["W"].data_ptr(), st))
    elif kind == "antipodal":
        check(lib().gwn_antipodal_query_device(s["h"].h, Q.data_ptr(), n, s["W"].data_ptr(), st))
    else:
        check(lib().gwn_signed_distance_device(s["bvh"].handle, Q.data_ptr(), n, gwn.SIGN_FAST_WINDING_NUMBER,
                                               gwn.DBL_MIN, gwn.DBL_MAX, s["S"].data_ptr(), s["I"].data_ptr(),
                                               s["C"].data_ptr(), st))
        return s["S"], s["I"], s["C"]
    return s["W"]


# ---------------------------------------------------------------------------

def work(case):
    """Bytes: queries in, results out, and the resident object's geometry read
    once.  Operations: a fast winding number needs about 2,750 beta^2 per query
    on a mesh (child tests, expansions and exact triangles counted on meshes
    of 320 to 1.3M triangles, uniform queries), at most every triangle; the
    other kinds' counts per query are those of their algorithms."""
    kind, n = case["kind"], case["queries"]
    if kind == "curve":
        return {"bytes": 8 * n + 4 * n + 16 * case["segments"], "flops": 890.0 * case["beta"] * n}
    if kind == "cloud":
        return {"bytes": 12 * n + 4 * n + 28 * case["points"], "flops": 5700.0 * case["beta"] ** 2 * n}
    if kind == "estimated":
        return {"bytes": 12 * n + 4 * n + 48 * case["points"], "flops": 22800.0 * n + 4000.0 * case["points"]}
    mesh = 12 * case["tris"] + 12 * case["tris"]  # faces, and half as many vertices of 24 bytes
    if kind == "soup":
        return {"bytes": 12 * n + 8 * n + mesh, "flops": min(2750.0 * case["beta"] ** 2, 85.0 * case["tris"]) * n}
    if kind == "oneshot":
        return {"bytes": 24 * n + 8 * n + mesh, "flops": 11000.0 * n + 1000.0 * case["tris"]}
    if kind == "exact":
        return {"bytes": 24 * n + 8 * n + mesh, "flops": 89.0 * 267.0 * n}
    if kind == "distance":
        return {"bytes": 24 * n + 36 * n + mesh, "flops": 12000.0 * n}
    return {"bytes": 24 * n + 8 * n + mesh, "flops": 1000.0 * n}


def tolerance(case):
    """About four times what two correct orders of the same sums were seen to
    differ by: the one-wavefront and the wave-coherent mesh walks (rel 4.9e-7,
    max 3.0e-6 of the root mean square in FP32 and mixed; 9e-16 and 7e-15 in
    FP64), the cap hierarchy and the sum over every face (1.3e-15, 5.8e-14),
    the cloud and the curve against their restatements on the host (2.6e-7 and
    5.3e-6; 1.1e-7 and 6.9e-7)."""
    kind = case["kind"]
    if kind in ("exact", "antipodal") or (kind == "soup" and case["precision"] == "fp64"):
        return {"rel": 1e-14, "max": 1e-12}
    if kind == "distance":
        # S carries the FP32 winding number; a point as close to two faces may take either
        return {"rel": 2e-6, "max": 5e-5, "differ": 1e-4}
    if kind == "curve":
        return {"rel": 5e-7, "max": 5e-6}
    if kind in ("cloud", "estimated"):
        return {"rel": 1.5e-6, "max": 5e-5}
    return {"rel": 2e-6, "max": 5e-5}


# ---------------------------------------------------------------------------
# 64-bit values of what the cases compute, by plain sums over every pair

def _winding(V, F, Q):
    """Winding number of every query (FP64 tensors): the solid angles of
    Van Oosterom and Strackee, det and dot products by matrix products."""
    f = F.long()
    a, b, c = V[f[:, 0]], V[f[:, 1]], V[f[:, 2]]
    det = (a * torch.linalg.cross(b, c)).sum(1)
    nrm = (torch.linalg.cross(a, b) + torch.linalg.cross(b, c) + torch.linalg.cross(c, a)).T.contiguous()
    pairs = [((u * v).sum(1), (u + v).T.contiguous()) for u, v in ((b, c), (c, a), (a, b))]
    out = torch.empty(Q.shape[0], dtype=torch.float64, device=Q.device)
    step = max(1, int(1.5e8 // max(1, F.shape[0])))
    for i in range(0, Q.shape[0], step):
        q = Q[i:i + step]
        q2 = (q * q).sum(1, keepdim=True)
        L = sum((q[:, k:k + 1] - V[None, :, k]).square_() for k in range(3)).sqrt_()
        la, lb, lc = L[:, f[:, 0]], L[:, f[:, 1]], L[:, f[:, 2]]
        den = la * lb
        den.mul_(lc)
        for (uv, s), l in zip(pairs, (la, lb, lc)):
            d = torch.mm(q, s)
            d.neg_().add_(uv).add_(q2)
            den.addcmul_(d, l)
        num = torch.mm(q, nrm).neg_().add_(det)
        out[i:i + step] = torch.atan2(num, den).sum(1)
    return out / (2.0 * math.pi)


def _closest(V, F, Q):
    """Closest point of the mesh to every query, over every face (FP64)."""
    f = F.long()
    A, B, C = V[f[:, 0]], V[f[:, 1]], V[f[:, 2]]
    out = torch.empty_like(Q)
    step = max(1, int(4e6 // max(1, F.shape[0])))

    def on_segment(p, a, d):
        t = (((p - a) * d).sum(-1) / (d * d).sum(-1).clamp(min=1e-300)).clamp(0.0, 1.0)
        return a + t[..., None] * d

    n = torch.linalg.cross(B - A, C - A)
    n2 = (n * n).sum(1).clamp(min=1e-300)
    for i in range(0, Q.shape[0], step):
        p = Q[i:i + step, None, :]
        h = p - (((p - A) * n).sum(-1) / n2)[..., None] * n
        inside = torch.ones(h.shape[:2], dtype=torch.bool, device=Q.device)
        for a, b in ((A, B), (B, C), (C, A)):
            inside &= (torch.linalg.cross((b - a).expand_as(h), h - a) * n).sum(-1) >= 0.0
        best = torch.where(inside, ((p - h) ** 2).sum(-1), math.inf)
        at = h
        for a, b in ((A, B), (B, C), (C, A)):
            e = on_segment(p, a, b - a)
            d2 = ((p - e) ** 2).sum(-1)
            nearer = d2 < best
            best = torch.where(nearer, d2, best)
            at = torch.where(nearer[..., None], e, at)
        k = best.argmin(1)
        out[i:i + step] = at[torch.arange(at.shape[0], device=Q.device), k]
    return out


def exact(case, seed):
    kind, n = case["kind"], case["queries"]
    size = case.get("tris", case.get("segments", case.get("points", 0)))
    if kind == "estimated" or float(n) * size > (MOST_DISTANCE_PAIRS if kind == "distance" else MOST_PAIRS):
        return None
    a = _inputs(case, seed)
    if kind == "curve":
        P, E, Q = torch.from_numpy(a[0]).to(DEVICE).double(), torch.from_numpy(a[1]).to(DEVICE).long(), a[2].double()
        out = torch.empty(n, dtype=torch.float64, device=DEVICE)
        step = max(1, int(1e8 // P.shape[0]))
        for i in range(0, n, step):
            x, y = (P[None, :, k] - Q[i:i + step, k:k + 1] for k in (0, 1))
            xa, ya, xb, yb = x[:, E[:, 0]], y[:, E[:, 0]], x[:, E[:, 1]], y[:, E[:, 1]]
            out[i:i + step] = torch.atan2(xa * yb - ya * xb, xa * xb + ya * yb).sum(1)
        return out
    if kind == "cloud":
        P, N, area, Q = a
        P, N, Q = P.float().double(), N.float().double() * float(np.float32(area)), Q.double()
        PN, Nt, Pt = (P * N).sum(1), N.T.contiguous(), P.T.contiguous()
        out = torch.empty(n, dtype=torch.float64, device=DEVICE)
        step = max(1, int(1e8 // P.shape[0]))
        p2 = (P * P).sum(1)
        for i in range(0, n, step):
            q = Q[i:i + step]
            r2 = torch.mm(q, Pt).mul_(-2.0).add_(p2).add_((q * q).sum(1, keepdim=True))
            out[i:i + step] = ((PN - torch.mm(q, Nt)) / (r2 * r2.sqrt())).sum(1)
        return out / (4.0 * math.pi)
    V, F, Q = torch.from_numpy(a[0]).to(DEVICE), torch.from_numpy(a[1]).to(DEVICE), a[2]
    if kind == "distance":
        C = _closest(V, F, Q)
        w = _winding(V.float().double(), F, Q.float().double())
        return (1.0 - 2.0 * w.abs()) * (Q - C).norm(dim=1), None, C
    if kind in ("soup", "oneshot"):  # the fast winding number takes mesh and queries as floats
        V, Q = V.float().double(), Q.float().double()
    return _winding(V, F, Q)
