"""GPU index-build and evaluation tools (cora_tool_*): rotation, nearest-centroid
assignment, k-means and the exhaustive top-k that produces the benchmarks' ground truth.

Distances on the GPU are FP32 GEMM results, so near-ties may order differently from an
FP64 brute force; the checks compare what is fixed regardless of rounding: the FP64
distances of the returned neighbours against the FP64 optimum, to FP32 accuracy.
"""
import ctypes
import sys
import threading
import time

import numpy as np
import pytest

import cora_oracle as orc
import coraanns_amd as ca

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def fp64_scores(base, queries, metric):
    b = base.astype(np.float64)
    q = queries.astype(np.float64)
    if metric == 1:
        return -(q @ b.T)
    return (q * q).sum(1)[:, None] + (b * b).sum(1)[None, :] - 2.0 * (q @ b.T)


def check_topk(base, queries, k, metric, ids):
    assert ids.shape == (queries.shape[0], k)
    assert ids.max() < base.shape[0]
    for r in ids:  # no id twice
        assert len(np.unique(r)) == k
    s = fp64_scores(base, queries, metric)
    got = np.sort(np.take_along_axis(s, ids.astype(np.int64), axis=1), axis=1)
    best = np.sort(s, axis=1)[:, :k]
    scale = np.abs(s).max(axis=1, keepdims=True) + 1e-30
    assert np.all(np.abs(got - best) <= 1e-5 * scale), np.abs(got - best).max()
    # the returned order is ascending in distance up to FP32 rounding
    own = np.take_along_axis(s, ids.astype(np.int64), axis=1)
    assert np.all(np.diff(own, axis=1) >= -1e-5 * scale)


@pytest.mark.parametrize("metric", [0, 1])
def test_topk_single_block(metric):
    rng = np.random.default_rng(11 + metric)
    base = rng.standard_normal((5000, 72)).astype(np.float32)
    q = rng.standard_normal((70, 72)).astype(np.float32)
    say(f"[tools] topk single block metric={metric}")
    check_topk(base, q, 26, metric, ca.gpu_topk(base, q, 26, metric))


@pytest.mark.parametrize("metric", [0, 1])
def test_topk_two_level_blocks(metric):
    """A base of several blocks, selected separately and merged: the true neighbours are planted
    on both sides of every block boundary and at both ends, so a merge that drops a block or a
    block's edge fails."""
    rng = np.random.default_rng(5 + metric)
    nb, dim, nq, k = (1 << 21) + 777, 16, 24, 26
    base = rng.standard_normal((nb, dim)).astype(np.float32)
    q = rng.standard_normal((nq, dim)).astype(np.float32)
    # the tool's split: blocks of about 2^18 rows where their candidates number 4,096 at most
    nblk = -(-nb >> 18)
    assert nblk * k <= 4096
    blk = -(-nb // nblk)
    assert nblk == 9 and nb - (nblk - 1) * blk > nq  # the last block is a little shorter
    where = [0, nb - 1] + [j * blk + e for j in range(1, nblk) for e in (-1, 0)]
    where += [j * blk + 1 for j in range(1, 1 + nq - len(where))]
    assert len(set(where)) == nq
    for w, v in zip(where, q):
        base[w] = v * (1.5 if metric == 1 else 1.0)
    say(f"[tools] topk two-level metric={metric} nb={nb}")
    ids = ca.gpu_topk(base, q, k, metric)
    check_topk(base, q, k, metric, ids)
    for i in range(nq):
        assert where[i] in ids[i]


def test_topk_k_equals_nb():
    rng = np.random.default_rng(3)
    base = rng.standard_normal((40, 64)).astype(np.float32)
    q = rng.standard_normal((5, 64)).astype(np.float32)
    ids = ca.gpu_topk(base, q, 40, 0)
    assert np.all(np.sort(ids, axis=1) == np.arange(40))
    check_topk(base, q, 40, 0, ids)


def test_assign_and_rotate():
    rng = np.random.default_rng(21)
    x = rng.standard_normal((20000, 96)).astype(np.float32)
    c = rng.standard_normal((300, 96)).astype(np.float32)
    say("[tools] assign + rotate")
    a = ca.gpu_assign(x, c)
    s = fp64_scores(c, x, 0)
    got = s[np.arange(x.shape[0]), a.astype(np.int64)]
    scale = np.abs(s).max(axis=1)
    assert np.all(got - s.min(axis=1) <= 1e-5 * scale)
    R = np.linalg.qr(rng.standard_normal((128, 128)))[0][:96].astype(np.float32)
    xr = ca.gpu_rotate(x, R)
    ref = x.astype(np.float64) @ R.astype(np.float64)
    assert np.allclose(xr, ref, rtol=0, atol=1e-4)


def test_kmeans_reduces_inertia():
    rng = np.random.default_rng(8)
    centers = rng.standard_normal((32, 48)).astype(np.float32) * 4
    lab = rng.integers(0, 32, 30000)
    x = (centers[lab] + rng.standard_normal((30000, 48)).astype(np.float32)).astype(np.float32)
    say("[tools] kmeans")
    c1 = ca.gpu_kmeans(x, 32, 1, seed=4)
    c20 = ca.gpu_kmeans(x, 32, 20, seed=4)

    def inertia(c):
        return fp64_scores(c, x, 0).min(axis=1).sum()

    assert np.isfinite(c20).all()
    assert inertia(c20) <= inertia(c1) * (1 + 1e-6)


def test_kmeans_reseeds_empty_clusters():
    """Well-separated unit-norm clusters (the 20M x 768 configuration's shape, scaled down)
    with twice as many centroids as true clusters: random initialisation leaves some true
    clusters without a centroid and the absorbing centroids drift to the origin, emptying
    others. Empty clusters are re-seeded by splitting populated ones, so at the end every
    centroid owns training rows and none sits near the origin."""
    rng = np.random.default_rng(9)
    ntrue, k, dim, n = 64, 128, 256, 32768
    centers = rng.standard_normal((ntrue, dim)).astype(np.float32)
    x = centers[rng.integers(0, ntrue, n)] + 0.5 * rng.standard_normal((n, dim)).astype(np.float32)
    x /= np.linalg.norm(x, axis=1, keepdims=True)
    say("[tools] kmeans re-seeds empty clusters")
    c = ca.gpu_kmeans(x, k, 20, seed=5)
    a = ca.gpu_assign(x, c)
    sizes = np.bincount(a, minlength=k)
    assert sizes.min() >= 1, np.sort(sizes)[:8]
    # a populated centroid is the mean of one true cluster's unit vectors (norm ~0.9)
    assert np.linalg.norm(c, axis=1).min() > 0.5


@pytest.mark.parametrize("dim,P,metric", [(128, 128, 0), (128, 128, 1), (250, 256, 0), (768, 768, 1)])
def test_gpu_builder_matches_host_builder(dim, P, metric, tmp_path):
    """The GPU quantiser (cora_build_ivf_gpu) writes the same index file, byte for byte (no row here
    has its best t below the GPU sweep's start), as the host builder (cora_build_ivf, itself pinned to the reference builder's codes) on the
    GPU-rotated rows: sign codes, all factors, ex-codes, ids."""
    rng = np.random.default_rng(dim + metric)
    n, nl = 3000, 12
    centers = rng.standard_normal((nl, dim)).astype(np.float32)
    x = (centers[rng.integers(0, nl, n)] + 0.6 * rng.standard_normal((n, dim))).astype(np.float32)
    if metric == 1:
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    x[7] = centers[0]  # a row equal to its centre's neighbourhood, ties in |o|
    R = np.linalg.qr(rng.standard_normal((P, P)))[0][:dim].astype(np.float32)
    cent = ca.gpu_kmeans(x, nl, 5, seed=3)
    assign = ca.gpu_assign(x, cent)
    cr = (cent.astype(np.float64) @ R.astype(np.float64)).astype(np.float32)
    say(f"[tools] GPU builder vs host builder, dim {dim} P {P} metric {metric}")
    ca.build_ivf(tmp_path / "host.index", ca.gpu_rotate(x, R), cr, assign, R, metric=metric)
    ca.build_ivf_gpu(tmp_path / "gpu.index", x, cr, assign, R, metric=metric)
    a, b = (tmp_path / "host.index").read_bytes(), (tmp_path / "gpu.index").read_bytes()
    assert len(a) == len(b)
    if a != b:
        ha, hb = ca.IvfIndex(tmp_path / "host.index"), ca.IvfIndex(tmp_path / "gpu.index")
        for name in ("short_data", "short_factors", "long_codes", "ex_factors", "ids"):
            u, v = getattr(ha, name), getattr(hb, name)
            bad = np.nonzero((u != v).reshape(u.shape[0], -1).any(1))[0]
            assert bad.size == 0, (name, bad[:8], bad.size)
        assert a == b


def test_topk_l2_beyond_2_32_work_items():
    """More than 2^32 / 64 base rows (70M x 4, L2): every row's norm takes part (a launch of
    one 64-lane workgroup per row would exceed the dispatch's 32-bit work-item count and
    leave the last rows without norms, which then look nearest)."""
    rng = np.random.default_rng(70)
    nb, dim, nq, k = 70_000_000, 4, 4, 10
    base = rng.standard_normal((nb, dim), dtype=np.float32)
    q = rng.standard_normal((nq, dim), dtype=np.float32)
    plant = [3, 20_000_001, 45_000_007, nb - 2]
    for i, w in enumerate(plant):
        base[w] = q[i]
    say(f"[tools] topk L2 over {nb:,} rows")
    ids = ca.gpu_topk(base, q, k, 0)
    for i, w in enumerate(plant):
        assert ids[i, 0] == w, (i, ids[i, :3])
        d = ((base.astype(np.float64) - q[i]) ** 2).sum(1) if i == 0 else None
        if d is not None:
            want = np.argsort(d, kind="stable")[:k]
            assert set(want.tolist()) == set(ids[i].tolist())


def test_kmeans_beyond_2_32_work_items():
    """More than 2^32 / 64 rows (67.2M x 8): one 64-lane wave per row in one launch would exceed the
    dispatch's 32-bit work-item count. Rows of zeros and ones, of 256 kinds, so that the sums are
    whole numbers below 2^24: after one iteration every centroid is the mean of its rows."""
    n, dim, k = 67_200_000, 8, 16
    kinds = ((np.arange(256)[:, None] >> np.arange(8)) & 1).astype(np.float32)
    kind = np.random.default_rng(67).integers(0, 256, n, dtype=np.uint8)
    x = kinds[kind]
    count = np.bincount(kind, minlength=256).astype(np.float64)
    say(f"[tools] k-means over {n:,} rows")
    for seed in range(20):
        c = ca.gpu_kmeans(x, k, 0, seed=seed)
        a = fp64_scores(c, kinds, 0).argmin(1)  # whole numbers: ties exact, to the lower id
        rows = np.bincount(a, weights=count, minlength=k)
        if len(np.unique(c, axis=0)) == k and rows.max() < 2 ** 24:
            break
    else:
        raise AssertionError("no seed with distinct first rows")
    want = np.stack([np.bincount(a, weights=count * kinds[:, d], minlength=k) for d in range(dim)], 1) / rows[:, None]
    assert np.abs(ca.gpu_kmeans(x, k, 1, seed=seed) - want).max() < 1e-6


@pytest.mark.parametrize("P", [64, 192, 384, 768, 960, 1024])
@pytest.mark.parametrize("metric", [0, 1])
def test_quantiser_on_unusual_rows(P, metric):
    """The GPU quantiser against the host's (quantize_rows) byte for byte, at every register
    width, on rows whose rescale search is unlike a Gaussian row's: no residual, one non-zero
    coordinate, equal magnitudes (every increment at the same t), small whole numbers (many
    ties and zeros), magnitudes over many powers of two (sums that round), tiny values. The
    rotation is the identity, so the rows reach the quantiser as they are. The GPU's sweep
    begins at 0.81 t_end and the host's at 0.77: rows whose best t lies between are left out."""
    rng = np.random.default_rng(P + metric)
    n = 260
    cen = (np.round(4 * rng.standard_normal((1, P))) / 4).astype(np.float32)  # exact residuals of rows 0-3
    x = rng.standard_normal((n, P)).astype(np.float32)
    x[0] = 0
    x[1] = 0
    x[1, 3] = 1
    x[2] = np.where(rng.random(P) < 0.5, 1, -1)
    x[3] = 0
    x[3, ::2] = 2
    x[4] = 1e-6
    x[4, 0] = 1
    x[5] = 1e-20
    x[6] *= 1e15
    for r in range(7, 60):
        x[r] = rng.integers(-5, 6, P) * 2.0 ** rng.integers(-20, 3)
    for r in range(60, 160):
        x[r] = rng.standard_normal(P) * np.exp(rng.uniform(0, 8) * rng.standard_normal(P))
    x = x.astype(np.float32)
    x[:130] += cen  # residuals about the centroid, rounded; the others as they are
    x = np.ascontiguousarray(x)
    say(f"[tools] quantiser on unusual rows, P {P} metric {metric}")
    bits, f1, code, f2 = ca.quantize_rows(x, cen[0], metric)
    gpu = ca.libs()[0]
    R = np.eye(P, dtype=np.float32)
    asg = np.zeros(n, np.uint32)
    gb, g1 = np.empty((n, P // 8), np.uint8), np.empty((n, 3), np.float32)
    gc, g2 = np.empty((n, P), np.uint8), np.empty((n, 2), np.float32)
    p = [a.ctypes.data_as(ctypes.c_void_p) for a in (x, R, cen, asg, gb, g1, gc, g2)]
    assert gpu.cora_tool_quantize(p[0], n, P, p[1], P, p[2], 1, p[3], metric, p[4], p[5], p[6], p[7], 0) == 0
    assert np.array_equal(np.unpackbits(gb, axis=1), bits)
    assert np.array_equal(g1.view(np.uint32), f1.view(np.uint32))
    late = np.zeros(n, bool)
    for r in range(1, n):
        oa = orc.excode_residual_abs(x[r], cen[0])[1]
        late[r] = orc.best_rescale_factor(oa, 7) >= 0.81 * 137 / float(oa.max())
    late[0] = True
    assert late.mean() > 0.9, late.mean()
    assert np.array_equal(gc[late], code[late])
    assert np.array_equal(g2[late].view(np.uint32), f2[late].view(np.uint32))


@pytest.mark.parametrize("n,dim,k", [(1, 1, 1), (5, 33, 2), (127, 64, 127), (129, 96, 129), (300, 100, 1000),
                                     (1000, 768, 257), (4097, 31, 640), (513, 300, 4100)])
def test_assign_is_the_fp64_nearest(n, dim, k):
    """gpu_assign at the edges of the GEMM's 128 x 128 tiles and of its K step: the nearest
    centroid in FP64, ties to the lower id, also where centroids repeat (within one tile of 128
    and across tiles), rows lie half-way between two, and a row or a centroid is huge."""
    rng = np.random.default_rng(n + dim + k)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    c = rng.standard_normal((k, dim)).astype(np.float32)
    if k > 4:
        c[k // 2] = c[1]
        c[k - 1] = c[3]
        c[2] = c[1]
        x[: n // 4] = c[1] + 0.01 * x[: n // 4]
        x[n // 4: n // 2] = (c[3] + c[0]) / 2
        x[n // 2] *= 1e4
        c[4] *= 1e3
    say(f"[tools] assign n={n} dim={dim} k={k}")
    d = ((x.astype(np.float64)[:, None, :] - c.astype(np.float64)[None]) ** 2).sum(2) if n * k * dim < 1 << 28 else \
        np.stack([((r.astype(np.float64) - c.astype(np.float64)) ** 2).sum(1) for r in x])
    a = ca.gpu_assign(x, c).astype(np.int64)
    got, best = d[np.arange(n), a], d.min(1)
    # the two FP64 sums may order differently below their own rounding
    assert np.all(got <= best * (1 + dim * 2.0 ** -50))
    first = (d <= best[:, None]).argmax(1)
    assert np.array_equal(a[got == best], first[got == best])


def call_seconds(f, n=15):
    f()
    best = float("inf")
    for _ in range(n):
        t = time.perf_counter()
        f()
        best = min(best, time.perf_counter() - t)
    return best


def test_settling_one_row_costs_little():
    """A row half-way between two centroids is evaluated again in FP64, over the 128 centroids of
    their tile: a call that holds one takes about as long as one that holds none."""
    rng = np.random.default_rng(77)
    n, dim, k = 1024, 1024, 128
    c = rng.standard_normal((k, dim)).astype(np.float32)
    x = (c[rng.integers(0, k, n)] + 0.1 * rng.standard_normal((n, dim))).astype(np.float32)
    y = x.copy()
    y[5] = (c[0] + c[1]) / 2
    none, one = (call_seconds(lambda v=v: ca.gpu_assign(v, c)) for v in (x, y))
    say(f"[tools] assign {n} x {dim}, k {k}: no row settled {none * 1e3:.3f} ms, one {one * 1e3:.3f} ms")
    assert one <= 1.3 * none


def fp64_nearest(x, c):
    """Nearest centroid of each row in FP64, and the distance to the second nearest less that."""
    d = fp64_scores(c, x, 0)
    two = np.partition(d, 1, axis=1)[:, :2]
    return d.argmin(1), two[:, 1] - two[:, 0]


def test_assign_rows_in_several_chunks():
    """84 MB of rows: two chunks of the staged upload, the first assigned while the second is on its
    way (their split operands and tile minima share arrays). Every row's FP64 nearest."""
    rng = np.random.default_rng(31)
    n, dim, k = 70_001, 300, 200
    c = rng.standard_normal((k, dim)).astype(np.float32)
    x = (c[rng.integers(0, k, n)] + rng.standard_normal((n, dim))).astype(np.float32)
    say(f"[tools] assign {n} x {dim} in chunks")
    want, gap = fp64_nearest(x, c)
    assert gap.min() > 1e-9
    assert np.array_equal(ca.gpu_assign(x, c), want)


def test_kmeans_rows_in_several_chunks():
    """The rows of some clusters lie in the second chunk of the upload alone: after one iteration
    every centroid is the mean of the rows nearest to its first row (which no iteration returns)."""
    rng = np.random.default_rng(32)
    n, dim, k = 70_001, 300, 24
    centers = 3 * rng.standard_normal((k, dim)).astype(np.float32)
    lab = np.where(np.arange(n) < 56_000, rng.integers(0, k // 2, n), rng.integers(k // 2, k, n))
    x = (centers[lab] + rng.standard_normal((n, dim))).astype(np.float32)
    say(f"[tools] k-means {n} x {dim} in chunks")
    first, c = ca.gpu_kmeans(x, k, 0, seed=1), ca.gpu_kmeans(x, k, 1, seed=1)
    a, gap = fp64_nearest(x, first)
    assert gap.min() > 1e-9
    for j in range(k):
        rows = x[a == j].astype(np.float64)
        # m additions in any order, each rounded within 2^-24 of a partial sum of at most sum |x|
        tol = 2.0 ** -24 * (len(rows) + 2) * np.abs(rows).mean(0).max()
        assert np.abs(c[j] - rows.mean(0)).max() <= tol, j


def test_rotate_rows_in_several_chunks():
    """An upload of two chunks and a download longer than the page-locked buffers (each reused),
    neither a whole number of 4 MiB pieces."""
    rng = np.random.default_rng(33)
    n, dim, P = 70_001, 300, 320
    x = rng.standard_normal((n, dim)).astype(np.float32)
    R = np.linalg.qr(rng.standard_normal((P, P)))[0][:dim].astype(np.float32)
    say(f"[tools] rotate {n} x {dim} in chunks")
    ref = x.astype(np.float64) @ R.astype(np.float64)
    # a sum of dim products: its roundings are within dim 2^-24 of the row norms' product
    tol = dim * 2.0 ** -24 * np.linalg.norm(x, axis=1).max()
    assert np.abs(ca.gpu_rotate(x, R) - ref).max() < tol


def test_quantise_rows_in_several_chunks():
    """More than three rounds of the resident waves, with a ragged last one, uploaded and
    downloaded through the page-locked buffers: the host's codes and factors at every row (but for
    rows whose best t lies below the GPU sweep's start)."""
    rng = np.random.default_rng(34)
    n, P = 40_001, 256
    x = rng.standard_normal((n, P)).astype(np.float32)
    cen = 0.1 * rng.standard_normal((1, P)).astype(np.float32)
    say(f"[tools] quantise {n} x {P} in chunks")
    bits, f1, code, f2 = ca.quantize_rows(x, cen[0], 0)
    R, asg = np.eye(P, dtype=np.float32), np.zeros(n, np.uint32)
    gb, g1 = np.empty((n, P // 8), np.uint8), np.empty((n, 3), np.float32)
    gc, g2 = np.empty((n, P), np.uint8), np.empty((n, 2), np.float32)
    p = [a.ctypes.data_as(ctypes.c_void_p) for a in (x, R, cen, asg, gb, g1, gc, g2)]
    assert ca.libs()[0].cora_tool_quantize(p[0], n, P, p[1], P, p[2], 1, p[3], 0, p[4], p[5], p[6], p[7], 0) == 0
    assert np.array_equal(np.unpackbits(gb, axis=1), bits)
    assert np.array_equal(g1.view(np.uint32), f1.view(np.uint32))
    for r in np.nonzero((gc != code).any(1) | (g2.view(np.uint32) != f2.view(np.uint32)).any(1))[0]:
        oa = orc.excode_residual_abs(x[r], cen[0])[1]
        assert orc.best_rescale_factor(oa, 7) < 0.81 * 137 / float(oa.max()), r


def test_tools_from_several_threads():
    """Calls on different data at once, from more threads than staging sets are kept: each gets its
    own answer."""
    rng = np.random.default_rng(35)
    n, dim, k = 40_000, 256, 100
    jobs = []
    for _ in range(4):
        c = rng.standard_normal((k, dim)).astype(np.float32)
        x = (c[rng.integers(0, k, n)] + rng.standard_normal((n, dim))).astype(np.float32)
        jobs.append((x, c, fp64_nearest(x, c)[0]))
    say("[tools] assign from four threads")
    got = [[None] * 3 for _ in jobs]

    def work(i):
        for r in range(3):
            got[i][r] = ca.gpu_assign(jobs[i][0], jobs[i][1])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, job in enumerate(jobs):
        for r in range(3):
            assert np.array_equal(got[i][r], job[2]), (i, r)


@pytest.mark.parametrize("kind", ["offset", "repeated", "far rows"])
def test_settling_many_rows_is_bounded(kind):
    """Data on which the bound of a row's distances spans many centroids: a common offset of 100
    times the spread (shifted away: the FP64 answer at every row), every centroid 64 times (the
    first of equals), rows far away from all centroids. A call takes at most a few times the
    time that it takes on centred data."""
    rng = np.random.default_rng(91)
    n, dim, k = 60_000, 128, 2048
    c = rng.standard_normal((k, dim)).astype(np.float32)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    centred = call_seconds(lambda: ca.gpu_assign(x, c), 5)
    if kind == "offset":
        x, c = x + np.float32(100), c + np.float32(100)
    elif kind == "repeated":
        c = np.ascontiguousarray(np.tile(c[:32], (64, 1)))
    else:
        x *= np.float32(3e3)
    a = ca.gpu_assign(x, c).astype(np.int64)
    m = c.astype(np.float64).mean(0)
    d = fp64_scores(c.astype(np.float64) - m, x.astype(np.float64) - m, 0)
    got, best = np.take_along_axis(d, a[:, None], 1)[:, 0], d.min(1)
    scale = (np.sqrt((x.astype(np.float64) ** 2).sum(1)) + np.sqrt(best)) ** 2
    if kind == "offset":
        assert np.array_equal(a, d.argmin(1))
    elif kind == "repeated":
        assert a.max() < 32 and np.array_equal(a, d[:, :32].argmin(1))
    # at worst the GEMM's answer: two of its error bounds
    assert np.all(got - best <= 2.2 * (dim + 34) * 2.0 ** -24 * scale)
    t = call_seconds(lambda: ca.gpu_assign(x, c), 5)
    say(f"[tools] assign {n} x {dim}, k {k}: centred {centred * 1e3:.2f} ms, {kind} {t * 1e3:.2f} ms")
    assert t <= 3 * centred


def test_fp32_path_where_the_split_operands_do_not_fit():
    """What the tools do where the device has no room for the split-FP16 operands: assign still
    gives the FP64 nearest (near ties and repeated centroids among the rows), k-means the means
    of the rows nearest to its first ones, top-k the neighbours to FP32 accuracy."""
    rng = np.random.default_rng(41)
    n, dim, k = 9001, 100, 333
    x = rng.standard_normal((n, dim)).astype(np.float32)
    c = rng.standard_normal((k, dim)).astype(np.float32)
    c[200] = c[7]
    x[:100] = c[7] + 0.01 * x[:100]
    x[100:200] = (c[5] + c[9]) / 2
    q = rng.standard_normal((50, dim)).astype(np.float32)
    say("[tools] the FP32 path")
    gpu = ca.libs()[0]
    was = gpu.cora_tool_debug_no_split(1)
    try:
        a = ca.gpu_assign(x, c).astype(np.int64)
        first, mean = ca.gpu_kmeans(x, 40, 0, seed=1), ca.gpu_kmeans(x, 40, 1, seed=1)
        tops = [ca.gpu_topk(x, q, 20, m) for m in (0, 1)]
    finally:
        gpu.cora_tool_debug_no_split(was)
    d = np.stack([((r.astype(np.float64) - c.astype(np.float64)) ** 2).sum(1) for r in x])
    got, best = d[np.arange(n), a], d.min(1)
    assert np.all(got <= best * (1 + dim * 2.0 ** -50))
    assert not np.any(a == 200)
    near = fp64_nearest(x, first)[0]
    for j in range(40):
        rows = x[near == j].astype(np.float64)
        tol = 2.0 ** -24 * (len(rows) + 2) * np.abs(rows).mean(0).max()
        assert np.abs(mean[j] - rows.mean(0)).max() <= tol, j
    for m in (0, 1):
        check_topk(x, q, 20, m, tops[m])


def test_calls_of_changing_sizes():
    """Calls take their device arrays from blocks that earlier calls of other sizes left: whatever
    these hold, every call gives its own answer."""
    rng = np.random.default_rng(51)
    say("[tools] calls of changing sizes")
    for n, dim, k in [(9000, 100, 40), (200, 33, 7), (30_000, 64, 300), (5, 3, 2), (700, 384, 129), (30_000, 31, 5)]:
        c = rng.standard_normal((k, dim)).astype(np.float32)
        x = (c[rng.integers(0, k, n)] + rng.standard_normal((n, dim))).astype(np.float32)
        want, gap = fp64_nearest(x, c)
        assert gap.min() > 1e-9
        assert np.array_equal(ca.gpu_assign(x, c), want)
        q = rng.standard_normal((9, dim)).astype(np.float32)
        for metric in (0, 1):
            check_topk(x, q, 5, metric, ca.gpu_topk(x, q, 5, metric))
        R = np.linalg.qr(rng.standard_normal((dim, dim)))[0].astype(np.float32)
        tol = dim * 2.0 ** -24 * np.linalg.norm(x, axis=1).max()
        assert np.abs(ca.gpu_rotate(x, R) - x.astype(np.float64) @ R.astype(np.float64)).max() < tol
