"""Failure paths: every device allocation of an entry point made to fail in
turn (GT_FAIL_ALLOC=N fails the Nth allocation after the variable is set).

The reference raises an R error from inside distance() and friends with
longjmp, so a failed cudaMalloc leaks the buffers allocated before it
(src/distance.cpp:277-311, src/cuseful.cpp:95-102).  Here each failure must
come back as GT_ERR_ALLOC (or the message of one for the void .C exports),
with every buffer the call held released: the device's free memory after the
failed call equals what it was before.
"""
import ctypes
import os

import numpy as np
import pytest

from oracle import oracle as orc

torch = pytest.importorskip("torch")

import gputools_amd as gt  # noqa: E402
from gputools_amd import _lib  # noqa: E402
from gputools_amd import workloads as wl  # noqa: E402

pytestmark = pytest.mark.gpu

FP = ctypes.POINTER(ctypes.c_float)
IP = ctypes.POINTER(ctypes.c_int)
SLACK = 1 << 20          # every buffer below is several MB


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def fail_each_allocation(call):
    """call() -> (ok, message).  Returns the number of device allocations the
    call makes, having failed each of them once."""
    ok, msg = call()                      # warm-up: kernels loaded, pools settled
    assert ok, msg
    base = free_bytes()
    n = 1
    while True:
        os.environ["GT_FAIL_ALLOC"] = str(n)
        try:
            ok, msg = call()
        finally:
            del os.environ["GT_FAIL_ALLOC"]
        if ok:
            break
        assert "out of memory" in msg, msg
        after = free_bytes()
        # a leak lowers the free memory; more free memory than before is the
        # stream-ordered pool returning blocks it had cached
        assert base - after <= SLACK, "allocation %d: %d bytes not released" % (n, base - after)
        n += 1
        assert n < 20
    assert base - free_bytes() <= SLACK
    return n - 1


def c_call(fn, *args):
    fn(*args)
    msg = _lib.last_error()
    return msg == "", msg


def test_Rdistances_releases_on_allocation_failure():
    x = np.ascontiguousarray(wl.normal(1500, 700, seed=41))     # 4.2 MB of points, 9 MB out
    n, k = x.shape
    d = np.zeros(n * n, np.float32)
    cn, ck, cp = ctypes.c_int(n), ctypes.c_int(k), ctypes.c_float(2.0)
    for method in (b"euclidean", b"binary"):
        cm = (ctypes.c_char_p * 1)(method)
        count = fail_each_allocation(lambda: c_call(
            _lib.lib().Rdistances, x.ctypes.data_as(FP), ctypes.byref(cn), ctypes.byref(ck),
            d.ctypes.data_as(FP), cm, ctypes.byref(cp)))
        # points and distances; binary also its bit rows
        assert count == (3 if method == b"binary" else 2)
    want = orc.dist(x[:200], "binary")
    d2 = d.reshape(n, n)[:200, :200]
    ii, jj = np.tril_indices(200, -1)
    order = np.lexsort((ii, jj))
    np.testing.assert_array_equal(d2[ii[order], jj[order]], want.astype(np.float32))


def test_gt_dist_workspace_failure_returns_alloc():
    x = torch.from_numpy(wl.normal(2000, 512, seed=42)).cuda()
    out = torch.empty(2000 * 1999 // 2, device="cuda")
    L = _lib.lib()

    def call():
        s = L.gt_dist(x.data_ptr(), 2000, 512, 512, _lib.EUCLIDEAN, 2.0, _lib.PREC_BF16X3,
                      _lib.LAYOUT_PACKED, out.data_ptr(), 2000, None)
        if s != _lib.GT_OK:
            assert s == _lib.GT_ERR_ALLOC, (s, _lib.last_error())
        return s == _lib.GT_OK, _lib.last_error() if s else ""

    assert fail_each_allocation(call) == 1      # the split-precision workspace
    torch.cuda.synchronize()
    idx = np.arange(0, out.numel(), 997)
    want = orc.dist(x.cpu().numpy(), "euclidean")[idx]
    got = out.cpu().numpy()[idx].astype(np.float64)
    assert np.max(np.abs(got - want) / want) <= 1e-5


def test_Rdistclust_releases_on_allocation_failure():
    rng = np.random.default_rng(43)
    n, k = 1200, 900
    x = np.ascontiguousarray(rng.standard_normal((n, k)), dtype=np.float32)
    merge = np.zeros(2 * (n - 1), np.int32)
    order = np.zeros(n, np.int32)
    val = np.zeros(n - 1, np.float32)
    cn, ck = ctypes.c_int(n), ctypes.c_int(k)
    dm = (ctypes.c_char_p * 1)(b"euclidean")
    cm = (ctypes.c_char_p * 1)(b"average")
    count = fail_each_allocation(lambda: c_call(
        _lib.lib().Rdistclust, dm, cm, x.ctypes.data_as(FP), ctypes.byref(cn), ctypes.byref(ck),
        merge.ctypes.data_as(IP), order.ctypes.data_as(IP), val.ctypes.data_as(FP)))
    # points, the pitched matrix, the clustering workspace and its results
    assert count == 4
    sub, sup, h = orc.hclust(gt.dist(torch.from_numpy(x).cuda(), layout="full").cpu().numpy(),
                             "average")
    np.testing.assert_array_equal(val, h)


def test_rpmcc_releases_on_allocation_failure():
    a = np.ascontiguousarray(wl.normal(700, 1500, seed=44))
    b = np.ascontiguousarray(wl.normal(600, 1500, seed=45))
    na, nb, size = 700, 600, 1500
    pairs = np.zeros(na * nb, np.float32)
    corr = np.zeros(na * nb, np.float32)
    ts = np.zeros(na * nb, np.float32)
    for use in (0, 1):
        cu, cna, cnb, cs = ctypes.c_int(use), ctypes.c_int(na), ctypes.c_int(nb), ctypes.c_int(size)
        count = fail_each_allocation(lambda: c_call(
            _lib.lib().rpmcc, ctypes.byref(cu), a.ctypes.data_as(FP), ctypes.byref(cna),
            b.ctypes.data_as(FP), ctypes.byref(cnb), ctypes.byref(cs), pairs.ctypes.data_as(FP),
            corr.ctypes.data_as(FP), ts.ctypes.data_as(FP)))
        # both variable sets and the outputs; "everything" also its split terms
        assert count == (4 if use == 0 else 3)
    want = orc.pmcc(a, b, "pairwise.complete.obs")[1]
    assert np.max(np.abs(corr.reshape(na, nb) - want)) <= 1e-5


def test_gt_dist_device_full_and_kendall_release():
    x = np.ascontiguousarray(wl.normal(1400, 800, seed=46))
    L = _lib.lib()

    def full():
        ptr, pitch = ctypes.c_void_p(), ctypes.c_size_t()
        s = L.gt_dist_device_full(x.ctypes.data, 1400, 800, _lib.MANHATTAN, 2.0,
                                  ctypes.byref(ptr), ctypes.byref(pitch))
        if s == _lib.GT_OK:
            assert L.gt_free(ptr) == 0
        else:
            assert s == _lib.GT_ERR_ALLOC and not ptr.value
        return s == _lib.GT_OK, _lib.last_error() if s else ""

    assert fail_each_allocation(full) == 2
    v = np.ascontiguousarray(wl.normal(300, 2500, seed=47))
    tau = np.zeros(300 * 300, np.float64)

    def kendall():
        s = L.gt_kendall_host(v.ctypes.data, 300, None, 300, 2500, tau.ctypes.data)
        if s != _lib.GT_OK:
            assert s == _lib.GT_ERR_ALLOC
        return s == _lib.GT_OK, _lib.last_error() if s else ""

    assert fail_each_allocation(kendall) == 3


def _cluster_matrix(n, seed):
    x = torch.from_numpy(wl.normal(n, 5, seed=seed)).cuda()
    return gt.dist(x, layout="full")


def _hclust_chosen(d, method):
    """hclust on the device through the C ABI: its results and the XCD choice in
    the workspace's meeting point (0: none, 1 + XCD, or 0xffff: given up)."""
    n = d.shape[0]
    size = ctypes.c_size_t()
    L = _lib.lib()
    assert L.gt_hclust_workspace_size(n, ctypes.byref(size)) == 0
    ws = torch.full((size.value,), 0xA5, dtype=torch.uint8, device="cuda")
    out = [torch.empty(n - 1, dtype=t, device="cuda") for t in (torch.int32, torch.int32, torch.float32)]
    assert L.gt_hclust(d.data_ptr(), n, d.stride(0), L.gt_hclust_method_from_name(method.encode()), 0.5, 0.5,
                       *(t.data_ptr() for t in out), ws.data_ptr(), size.value, None) == 0
    torch.cuda.synchronize()
    at = ws.data_ptr() + size.value - 4096
    at = (at + 255) // 256 * 256 + 64 - ws.data_ptr()
    return [t.cpu().numpy() for t in out], int(ws[at:at + 4].cpu().numpy().view(np.uint32)[0])


@pytest.mark.parametrize("n", [257, 1000, 9300])
def test_hclust_without_room_for_the_workgroups(n):
    """The clustering workgroups do not come together: one workgroup does the
    rounds, with the same merges; without the failure an XCD is chosen."""
    d = _cluster_matrix(n, 47)
    print("case hclust without room n=%d" % n, flush=True)
    want, chosen = _hclust_chosen(d.clone(), "average")
    assert 1 <= chosen <= 16
    os.environ["GT_FAIL_MEETING"] = "join"
    try:
        got, chosen = _hclust_chosen(d.clone(), "average")
    finally:
        del os.environ["GT_FAIL_MEETING"]
    assert chosen == 0xFFFF
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g.view(np.uint32), w.view(np.uint32))


def test_hclust_lost_workgroup_is_an_error():
    """A workgroup that gives another one up ends the kernel; host callers get
    an error, device callers merges with sub == sup."""
    n = 700
    d = _cluster_matrix(n, 48)
    host = np.ascontiguousarray(d.cpu().numpy())
    sub, sup = np.zeros(n - 1, np.int32), np.zeros(n - 1, np.int32)
    height = np.zeros(n - 1, np.float32)
    L = _lib.lib()

    def call():
        return L.gt_hclust_host(host.ctypes.data, n, n, L.gt_hclust_method_from_name(b"average"), 0.5, 0.5,
                                sub.ctypes.data, sup.ctypes.data, height.ctypes.data)

    print("case hclust lost workgroup", flush=True)
    os.environ["GT_FAIL_MEETING"] = "partner"
    try:
        assert call() == _lib.GT_ERR_HIP
        assert "stopped early" in _lib.last_error()
        got, chosen = _hclust_chosen(d.clone(), "average")
    finally:
        del os.environ["GT_FAIL_MEETING"]
    assert got[0][-1] == got[1][-1] == 0 and np.isnan(got[2][-1])
    assert call() == 0
    want = orc.hclust(host, "average")
    for g, w in zip((sub, sup, height), want):
        np.testing.assert_array_equal(g, w)


@pytest.mark.parametrize("n", [257, 600])
def test_hclust_short_wait_for_room(n):
    """Where the workgroups find no room together (masked CUs, other work) the
    wait before one workgroup takes over follows the work it could save: small
    calls don't wait for tens of milliseconds."""
    import time
    d = _cluster_matrix(n, 49)

    def best(state):
        times = []
        for _ in range(5):
            c = d.clone()
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            gt.hclust(c, "average", state=state)
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t0)
        return min(times)

    alone = best("lds")
    os.environ["GT_FAIL_MEETING"] = "join"
    try:
        handed_over = best("auto")
    finally:
        del os.environ["GT_FAIL_MEETING"]
    print("case hclust wait n=%d: %.2f ms alone, %.2f ms handed over" % (n, alone * 1e3, handed_over * 1e3), flush=True)
    # one microsecond per point, and as much again for the launches
    assert handed_over - alone <= 2e-6 * n + 1e-3


def _table(n, dim, seed):
    x = np.ascontiguousarray(wl.normal(n, dim, seed=seed))
    x[np.random.default_rng(seed).random(x.shape) < 0.05] = np.nan
    return x


def test_pairwise_without_room_for_its_workspace(monkeypatch):
    """pairwise.complete.obs needs no workspace: where it finds none, the call
    runs without (host entry point and package function)."""
    n, dim = 400, 3000
    a, b = _table(n, dim, 50), _table(n, dim, 51)
    outs = [np.zeros(n * n, np.float32) for _ in range(3)]
    cu, cn, cs = ctypes.c_int(1), ctypes.c_int(n), ctypes.c_int(dim)
    # variables 4.8 MB, results 1.9 MB, workspace 35 MB
    os.environ["GT_FAIL_ALLOC_ABOVE"] = str(8 << 20)
    try:
        ok, msg = c_call(_lib.lib().rpmcc, ctypes.byref(cu), a.ctypes.data_as(FP), ctypes.byref(cn),
                         b.ctypes.data_as(FP), ctypes.byref(cn), ctypes.byref(cs),
                         *(o.ctypes.data_as(FP) for o in outs))
    finally:
        del os.environ["GT_FAIL_ALLOC_ABOVE"]
    assert ok, msg
    pairs, corr = orc.pmcc(a, b, "pairwise.complete.obs")
    np.testing.assert_array_equal(outs[0].reshape(n, n), pairs)
    assert np.max(np.abs(outs[1].reshape(n, n) - corr)) <= 1e-5

    ad, bd = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    res = tuple(torch.empty((n, n), device="cuda") for _ in range(3))
    real = torch.empty

    def no_room(*args, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.cuda.OutOfMemoryError("no room for a workspace")
        return real(*args, **kw)

    monkeypatch.setattr(torch, "empty", no_room)
    gt.pmcc(ad, bd, use="pairwise.complete.obs", precision="fp32", out=res)
    got = res[1].cpu().numpy()
    with pytest.raises(torch.cuda.OutOfMemoryError):
        gt.pmcc(ad.nan_to_num_(), bd.nan_to_num_(), precision="bf16x3", out=res)   # needs its workspace
    assert np.max(np.abs(got - corr)) <= 1e-5


def test_gradient_and_mds_without_room_for_the_faster_form():
    """The matrix-core gradient and the MDS form that visits each pair once take
    more scratch than the sweep over both owners of a pair: where there is no
    room for it, the sweep runs."""
    from gputools_amd.autograd import _mds
    rng = np.random.default_rng(60)
    n, k = 2000, 64
    x = rng.standard_normal((n, k)).astype(np.float32)
    g = rng.standard_normal(n * (n - 1) // 2).astype(np.float32)
    xd, gd = torch.from_numpy(x).cuda(), torch.from_numpy(g).cuda()
    m = 4000
    y = rng.standard_normal((m, 2)).astype(np.float32)
    delta = (rng.random(m * (m - 1) // 2) * 3.0).astype(np.float32)
    yd, dd = torch.from_numpy(y).cuda(), torch.from_numpy(delta).cuda()
    usual, (s_usual, dy_usual) = gt.dist_backward(xd, gd), _mds(yd, dd, True)

    def limited(limit, call):
        os.environ["GT_FAIL_ALLOC_ABOVE"] = str(limit)
        try:
            return call()
        finally:
            del os.environ["GT_FAIL_ALLOC_ABOVE"]

    dx = limited(9000000, lambda: gt.dist_backward(xd, gd))        # 9.8 MB, sweep 8.2
    s, dy = limited(1000000, lambda: _mds(yd, dd, True))           # 1.5 MB, sweep 0.5
    assert not torch.equal(dx, usual) and not torch.equal(dy, dy_usual)
    for got, want in ((dx, orc.dist_backward(x, g.astype(np.float64), "euclidean")),
                      (dy, orc.mds_stress(y, delta.astype(np.float64))[1])):
        got = got.cpu().numpy().astype(np.float64)
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    assert abs(s.item() - s_usual.item()) <= 1e-6 * s_usual.item()
    with pytest.raises(gt.GputoolsError, match="ALLOC"):           # nor for the sweep
        limited(1000, lambda: gt.dist_backward(xd, gd))
