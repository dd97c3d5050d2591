"""GPU parity of the backward kernels (dL/dX) and the fused MDS stress.

The FP64 oracle (oracle_dist_backward / oracle_mds_stress, itself pinned
against central differences in test_oracle.py) is the reference.  The GPU
computes in FP32 and sums n terms per output, so gradients are compared by
relative Frobenius error (<= 1e-5) plus an elementwise check scaled by the
largest gradient entry (<= 1e-4); the stress by relative error <= 1e-6.
"""
import numpy as np
import pytest

from oracle import oracle as orc

torch = pytest.importorskip("torch")

import gputools_amd as gt  # noqa: E402
from gputools_amd import workloads as wl  # noqa: E402

pytestmark = pytest.mark.gpu


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda()


def assert_grad_close(got, want, frob=1e-5, elem=1e-4):
    got = got.astype(np.float64)
    scale = np.max(np.abs(want))
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert rel <= frob, "relative Frobenius error %.3g" % rel
    assert np.max(np.abs(got - want)) <= elem * scale


@pytest.mark.parametrize("method,p", [("euclidean", 2.0), ("minkowski", 3.0), ("minkowski", 1.5),
                                      ("minkowski", 2.0), ("minkowski", 4.5)])
@pytest.mark.parametrize("n,k", [(300, 37), (129, 5), (256, 128), (70, 200)])
def test_backward_vs_oracle(method, p, n, k):
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal((n, k)).astype(np.float32)
    g = rng.standard_normal(n * (n - 1) // 2).astype(np.float32)
    got = gt.dist_backward(dev(x), dev(g), method, p).cpu().numpy()
    want = orc.dist_backward(x, g.astype(np.float64), method, p)
    assert_grad_close(got, want)


def test_backward_duplicate_rows_are_zero_subgradient():
    rng = np.random.default_rng(40)
    x = rng.standard_normal((50, 8)).astype(np.float32)
    x[10] = x[3]
    g = np.ones(50 * 49 // 2, np.float32)
    got = gt.dist_backward(dev(x), dev(g), "euclidean").cpu().numpy()
    want = orc.dist_backward(x, g.astype(np.float64), "euclidean")
    assert np.all(np.isfinite(got))
    assert_grad_close(got, want)


def test_autograd_function_matches_backward():
    rng = np.random.default_rng(41)
    x = dev(rng.standard_normal((200, 30)))
    w = dev(rng.standard_normal(200 * 199 // 2))
    xr = x.clone().requires_grad_(True)
    loss = (gt.pdist(xr, "euclidean") * w).sum()
    loss.backward()
    direct = gt.dist_backward(x, w, "euclidean")
    np.testing.assert_array_equal(xr.grad.cpu().numpy(), direct.cpu().numpy())
    # forward value of pdist equals gt.dist
    np.testing.assert_array_equal(gt.pdist(x).detach().cpu().numpy(), gt.dist(x).cpu().numpy())


def test_gradcheck_n256_against_fp64_finite_differences():
    """n = 256: the FP32 kernel gradient against central differences of the
    FP64 oracle loss L(X) = sum_q w_q d_q(X), on a random subset of entries."""
    rng = np.random.default_rng(42)
    n, k = 256, 6
    x = rng.standard_normal((n, k)).astype(np.float32)
    w = rng.standard_normal(n * (n - 1) // 2)
    got = gt.dist_backward(dev(x), dev(w), "euclidean").cpu().numpy()
    h = 1e-3
    for idx in [tuple(v) for v in rng.integers(0, [n, k], size=(20, 2))]:
        xp = x.copy(); xm = x.copy()
        xp[idx] = np.float32(x[idx] + h)
        xm[idx] = np.float32(x[idx] - h)
        fd = (np.dot(w, orc.dist(xp)) - np.dot(w, orc.dist(xm))) / (float(xp[idx]) - float(xm[idx]))
        assert abs(got[idx] - fd) <= 2e-3 * max(1.0, abs(fd)), (idx, got[idx], fd)


@pytest.mark.parametrize("q", [2, 32])
def test_mds_stress_n256_vs_oracle_and_autograd(q):
    rng = np.random.default_rng(43 + q)
    n = 256
    xs = rng.standard_normal((n, 16)).astype(np.float32)
    delta = orc.dist(xs).astype(np.float32)
    y = rng.standard_normal((n, q)).astype(np.float32)
    yt = dev(y).requires_grad_(True)
    s = gt.mds_stress(yt, dev(delta))
    s.backward()
    s_ref, dy_ref = orc.mds_stress(y, delta.astype(np.float64))
    assert s.dtype == torch.float64
    assert abs(s.item() - s_ref) <= 1e-6 * s_ref
    assert_grad_close(yt.grad.cpu().numpy(), dy_ref)


@pytest.mark.parametrize("q", [2, 32])
def test_mds_stress_16384(q):
    """The differentiation workload: delta from 16384 x 128 N(0,1) points,
    embedding Y 16384 x q, forward stress plus dY with tile recompute."""
    n = 16384
    print("case mds 16384 q=%d" % q, flush=True)
    x = wl.normal(n, 128, seed=4)
    delta = gt.dist(dev(x))
    y = wl.normal(n, q, seed=44)
    yt = dev(y).requires_grad_(True)
    s = gt.mds_stress(yt, delta)
    s.backward()
    torch.cuda.synchronize()
    s_ref, dy_ref = orc.mds_stress(y, delta.cpu().numpy().astype(np.float64))
    assert abs(s.item() - s_ref) <= 1e-6 * s_ref
    assert_grad_close(yt.grad.cpu().numpy(), dy_ref)


def test_backward_rejects_other_methods():
    x = dev(np.ones((4, 3)))
    g = dev(np.ones(6))
    with pytest.raises(gt.GputoolsError, match="UNSUPPORTED"):
        gt.dist_backward(x, g, "manhattan")
    with pytest.raises(gt.GputoolsError, match="INVALID"):
        gt.dist_backward(x, g, "minkowski", 0.5)


@pytest.mark.parametrize("n,k,data", [(1500, 33, "normal"), (1537, 64, "offset"), (1793, 97, "mixture"),
                                      (2049, 128, "normal"), (3000, 16, "uniform"), (3009, 31, "clusters"),
                                      (1600, 128, "clusters"), (1700, 50, "duplicates"),
                                      (1700, 96, "upstream")])
def test_matrix_core_gradient(n, k, data):
    """The matrix-core form (euclidean, up to 128 features) at the edges of its
    blocks, on strided rows that start anywhere, where the Gram form needs its
    near pairs recomputed (mixture, duplicates: subgradient 0), where most
    pairs are near (two clusters: rows left to the sweep), and with upstream
    gradients that three BF16 terms cannot hold (1e-36: rows left).  Centred
    data far from the origin: the reference is the oracle on the FP32 values;
    its gradient cancels, so the bound is relative to the terms there."""
    rng = np.random.default_rng(n + k)
    base = rng.standard_normal((n, k + 3)).astype(np.float32)
    x = base[:, 1:k + 1]
    if data == "uniform":
        x[:] = rng.random((n, k))
    elif data == "offset":
        x += np.float32(100.0)
    elif data == "mixture":
        x[:] = x * np.float32(1e-3) + rng.standard_normal((64, k)).astype(np.float32)[np.arange(n) % 64]
    elif data == "clusters":
        x[:] = x * np.float32(1e-2) + rng.standard_normal((2, k)).astype(np.float32)[rng.integers(0, 2, n)]
    elif data == "duplicates":
        x[n // 2:n // 2 + 90] = x[:90]
        x[33] = x[32]
    g = rng.standard_normal(n * (n - 1) // 2).astype(np.float32)
    if data == "upstream":
        g[::1001] = 1e-36
        g[5::977] = 0.0
    print("case matrix-core gradient n=%d k=%d %s" % (n, k, data), flush=True)
    xd = dev(base)[:, 1:k + 1]
    got = gt.dist_backward(xd, dev(g), "euclidean").cpu().numpy()
    again = gt.dist_backward(xd, dev(g), "euclidean").cpu().numpy()
    np.testing.assert_array_equal(got, again)          # deterministic
    want = orc.dist_backward(np.ascontiguousarray(x), g.astype(np.float64), "euclidean")
    # near pairs have large weights whose sum cancels against w x_j: FP32 sums
    # of terms |w| |x| 1e-2 or 1e-3 apart carry that factor (the sweep's error
    # there is 1e-5 to 8e-5)
    close = {"mixture": 2e-4, "clusters": 5e-5}.get(data, 1e-5)
    assert_grad_close(got, want, frob=close, elem=max(1e-4, 2 * close))


def test_matrix_core_gradient_non_finite_upstream():
    """An infinite and a NaN entry of dL/dD reach the rows of their pairs and no
    other: the other rows equal those without the entries."""
    n, k = 1600, 40
    rng = np.random.default_rng(7)
    x = dev(rng.standard_normal((n, k)))
    g = rng.standard_normal(n * (n - 1) // 2).astype(np.float32)

    def at(i, j):   # i > j
        return j * n - j * (j + 1) // 2 + i - j - 1

    clean = g.copy()
    clean[at(700, 3)] = clean[at(1300, 900)] = 0.0
    g[at(700, 3)] = np.inf
    g[at(1300, 900)] = np.nan
    print("case matrix-core gradient non-finite", flush=True)
    got = gt.dist_backward(x, dev(g)).cpu().numpy()
    want = gt.dist_backward(x, dev(clean)).cpu().numpy()
    hit = np.zeros(n, bool)
    hit[[700, 3, 1300, 900]] = True
    assert not np.isfinite(got[hit]).all(1).any()
    assert np.isfinite(got[~hit]).all()
    rel = np.linalg.norm(got[~hit].astype(np.float64) - want[~hit]) / np.linalg.norm(want[~hit])
    assert rel <= 1e-5


@pytest.mark.parametrize("n,q", [(2, 1), (64, 2), (255, 3), (256, 4), (257, 5), (300, 6), (2500, 2), (2501, 3),
                                 (3073, 8), (3100, 7), (6001, 1)])
def test_mds_few_features(n, q):
    """The form that visits each pair once (few features) at the edges of its
    blocks (256 rows; 16, 32 or 64 columns a wave), on strided rows, with
    coincident points (distance 0: no gradient, full residual), with and
    without the gradient."""
    rng = np.random.default_rng(n * 10 + q)
    base = rng.standard_normal((n, q + 2)).astype(np.float32)
    if n > 10:
        base[n - 1] = base[0]
        base[n // 2] = base[n // 2 - 1]
    y = np.ascontiguousarray(base[:, 1:q + 1])
    delta = (rng.random(n * (n - 1) // 2) * 3.0).astype(np.float32)
    print("case mds few features n=%d q=%d" % (n, q), flush=True)
    s_ref, dy_ref = orc.mds_stress(y, delta.astype(np.float64))
    yd = dev(base)[:, 1:q + 1]
    dd = dev(delta)
    from gputools_amd.autograd import _mds
    for grad in (True, False):
        s, dy = _mds(yd, dd, grad)
        assert abs(s.item() - s_ref) <= 1e-6 * s_ref
        if grad:
            assert_grad_close(dy.cpu().numpy(), dy_ref)
            s2, dy2 = _mds(yd, dd, True)
            assert s2.item() == s.item()                              # deterministic
            np.testing.assert_array_equal(dy.cpu().numpy(), dy2.cpu().numpy())


def _mds_reference(y, delta):
    """Stress and gradient in FP64 on the GPU, some rows at a time."""
    n = y.shape[0]
    yd = y.double()
    stress, dy = 0.0, torch.zeros_like(yd)
    cols = torch.arange(n, device="cuda")
    for i in range(0, n, 1024):
        rows = cols[i:i + 1024]
        diff2 = sum((yd[i:i + 1024, c, None] - yd[None, :, c]).square_() for c in range(y.shape[1]))
        d = diff2.sqrt_()
        hi, lo = torch.maximum(rows[:, None], cols), torch.minimum(rows[:, None], cols)
        at = lo * n - lo * (lo + 1) // 2 + hi - lo - 1
        off = hi != lo
        dl = torch.where(off, delta[at.clamp_(0, delta.numel() - 1)].double(), torch.zeros((), dtype=torch.float64, device="cuda"))
        r = torch.where(off, d - dl, torch.zeros_like(d))
        stress += 0.5 * r.square().sum().item()
        w = torch.where(d > 0, 2.0 * r / d, torch.zeros_like(d))
        dy[i:i + 1024] = yd[i:i + 1024] * w.sum(1, keepdim=True) - w @ yd
    return stress, dy


@pytest.mark.parametrize("n,q", [(33025, 8), (50001, 8), (65793, 2)])
def test_mds_scratch_is_bounded(n, q):
    """The partial slices of the few-feature form grow with n^2; beyond 256 MiB
    the rows are taken in several passes (two or three here, with a ragged
    last block)."""
    import os
    g = torch.Generator(device="cuda").manual_seed(n)
    y = torch.randn((n, q), generator=g, device="cuda")
    y[n - 1] = y[3]
    delta = torch.rand(n * (n - 1) // 2, generator=g, device="cuda") * 3.0
    from gputools_amd.autograd import _mds
    print("case mds bounded scratch n=%d q=%d" % (n, q), flush=True)
    os.environ["GT_FAIL_ALLOC_ABOVE"] = str((256 << 20) + (4 << 20))   # and the stress partials
    try:
        s, dy = _mds(y, delta, True)
        s2, dy2 = _mds(y, delta, True)
        s3, _ = _mds(y, delta, False)
    finally:
        del os.environ["GT_FAIL_ALLOC_ABOVE"]
    assert s2.item() == s.item() == s3.item() and torch.equal(dy, dy2)
    want_s, want = _mds_reference(y, delta)
    assert abs(s.item() - want_s) <= 1e-6 * want_s
    assert_grad_close(dy.cpu().numpy(), want.cpu().numpy())


@pytest.mark.parametrize("data", ["dominant", "ordered", "tiny"])
def test_gradient_of_many_near_pairs_costs_the_sweep(data):
    """Data whose pairs are mostly near by the rule of the matrix-core form (one
    dominant direction; clusters that lie in order; values whose squares are
    denormal) is left to the sweep as a whole, before work is done on it: the
    same values as the sweep's, in about its time."""
    import os
    n, k = 6000, 64
    gen = torch.Generator(device="cuda").manual_seed(8)
    x = torch.randn((n, k), generator=gen, device="cuda")
    if data == "dominant":
        x[:, 0] *= 40.0
    elif data == "ordered":
        x = x * 1e-2 + torch.randn((8, k), generator=gen, device="cuda")[torch.arange(n, device="cuda") * 8 // n]
    else:
        x *= 1e-17
    g = torch.randn(n * (n - 1) // 2, generator=gen, device="cuda")
    print("case gradient of near pairs %s" % data, flush=True)

    def timed():
        times = []
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(4):
                dx = gt.dist_backward(x, g)
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1))
        return dx, min(times)

    dx, usual = timed()
    os.environ["GT_FAIL_ALLOC_ABOVE"] = "26000000"   # the sweep's 25 MB, not the operands beside it
    try:
        want, sweep = timed()
    finally:
        del os.environ["GT_FAIL_ALLOC_ABOVE"]
    assert torch.equal(dx, want)
    assert usual <= 1.4 * sweep, (usual, sweep)      # 1.05; 1.6 to 1.8 without the samples


@pytest.mark.parametrize("n,k,data", [(4000, 16, "uniform"), (4009, 31, "clusters"), (4001, 32, "duplicates")])
def test_matrix_core_gradient_of_few_features(n, k, data):
    """The same up to 32 features, where the form begins at 4000 points."""
    test_matrix_core_gradient(n, k, data)


def test_gradient_error_with_dominant_directions():
    """Three features of five times the others' spread, and upstream gradients at
    the nearest pairs alone: a distance is then up to half the size of the norms
    it comes from in the matrix-core form, and few terms make up a row.  Rows of
    dX are not much further from FP64 than the sweep's, which takes differences."""
    import os
    n, k = 4000, 128
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = torch.randn((n, k), generator=gen, device="cuda")
    x[:, :3] *= 5.0
    g = torch.randn(n * (n - 1) // 2, generator=gen, device="cuda")
    d = gt.dist(x)
    g *= d <= torch.quantile(d[torch.randint(d.numel(), (1000000,), generator=gen, device="cuda")], 0.01)
    print("case gradient of near pairs alone", flush=True)
    dx = gt.dist_backward(x, g)
    os.environ["GT_FAIL_ALLOC_ABOVE"] = "33000000"   # the sweep's 32.8 MB, not the operands beside it
    try:
        sweep = gt.dist_backward(x, g)
    finally:
        del os.environ["GT_FAIL_ALLOC_ABOVE"]
    assert not torch.equal(dx, sweep)
    xd = x.double()
    w = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    w[torch.ones((n, n), dtype=torch.bool, device="cuda").triu_(1)] = g.double()
    w += w.T.clone()
    d2 = torch.zeros_like(w)
    for f in range(k):
        d2 += (xd[:, f, None] - xd[None, :, f]).square_()
    w /= d2.sqrt_().fill_diagonal_(1.0)
    want = torch.empty_like(xd)
    for f in range(k):
        want[:, f] = (w * (xd[:, f, None] - xd[None, :, f])).sum(1)

    def worst_row(got):
        some = want.norm(dim=1) > 0          # (rows without a near pair are zero)
        return ((got.double() - want).norm(dim=1) / want.norm(dim=1))[some].max().item()

    ours, theirs = worst_row(dx), worst_row(sweep)
    assert ours <= 1.8 * theirs, (ours, theirs)


@pytest.mark.parametrize("rows", [16, 32, 64])
def test_gradient_of_near_points_in_order_costs_the_sweep(rows):
    """Groups of near points next to each other (only the blocks on the diagonal
    hold near pairs, up to all of theirs): left to the sweep as a whole."""
    import os
    n, k = 3000, 64
    gen = torch.Generator(device="cuda").manual_seed(9)
    at = torch.arange(n, device="cuda") // rows
    x = 1e-2 * torch.randn((n, k), generator=gen, device="cuda") + torch.randn((n // rows + 1, k), generator=gen, device="cuda")[at]
    g = torch.randn(n * (n - 1) // 2, generator=gen, device="cuda")
    print("case gradient of groups of %d in order" % rows, flush=True)

    def timed():
        times = []
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(8):
                dx = gt.dist_backward(x, g)
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1))
        return dx, min(times)

    dx, usual = timed()
    os.environ["GT_FAIL_ALLOC_ABOVE"] = "13000000"   # the sweep's 12.3 MB, not the operands beside it
    try:
        want, sweep = timed()
    finally:
        del os.environ["GT_FAIL_ALLOC_ABOVE"]
    assert torch.equal(dx, want)
    assert usual <= 1.5 * sweep, (usual, sweep)      # 1.15; 1.3 (16 rows) and 2.3 (32) with samples beside the diagonal
