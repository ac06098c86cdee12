"""Triangular solves of the stored factor over the paths a group of four
256-blocks can take: whole groups (k_solve_pair), partial groups and odd
leading dimensions (k_solve_group), more than 1024 right-hand sides (FP64:
diagonal blocks in place and GEMMs, the same under capture and beside other
threads' solves); FP32 split products and their scale cache."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

from conftest import Launches

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def om():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import openmeeg_amd
    return openmeeg_amd


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,r,pad", [(256, 1, 0), (255, 3, 1), (1024, 2, 0), (1024, 5, 3), (1025, 7, 3), (1536, 64, 0),
                                     (2048, 33, 4), (2300, 130, 4), (1280, 1030, 0), (1300, 1100, 1)])
def test_solve_residual(om, n, r, pad, dtype):
    import torch
    from openmeeg_amd import _lib
    lib = _lib.lib()
    rng = np.random.default_rng(n + r)
    t = torch.float64 if dtype == np.float64 else torch.float32
    size = np.dtype(dtype).itemsize
    # quasi-definite: +/- diagonal blocks, well conditioned
    A = rng.standard_normal((n, n)) / np.sqrt(n)
    A = 0.25 * (A + A.T) + np.diag(np.where(np.arange(n) < n // 2, 2.0, -2.0))
    ld, ldb = n + pad, n + pad
    dA = torch.zeros((n, ld), dtype=t, device="cuda")
    dA[:, :n] = torch.from_numpy(A.astype(dtype))
    Ad = dA[:, :n].double().clone()
    B = rng.standard_normal((r, ldb))
    dB = torch.from_numpy(B.astype(dtype)).cuda()
    B0 = dB.double().clone()
    work = torch.zeros(int(lib.omh_factor_workspace_bytes(n, size)), dtype=torch.uint8, device="cuda")
    info = C.c_int32()
    f = lib.omh_sym_factor_f64 if size == 8 else lib.omh_sym_factor_f32
    s = lib.omh_sym_solve_f64 if size == 8 else lib.omh_sym_solve_f32
    p = lambda x: C.c_void_p(x.data_ptr())
    _lib.check(f(p(dA), n, ld, p(work), C.byref(info), C.c_void_p(0)))
    assert info.value == 0
    _lib.check(s(p(dA), n, ld, p(work), p(dB), ldb, r, C.c_void_p(0)))
    torch.cuda.synchronize()
    X = dB[:, :n].double()
    res = (X @ Ad - B0[:, :n]).norm(dim=1) / (Ad.abs().sum(1).max() * X.norm(dim=1))
    # ||b - A x|| <= c n eps ||A|| ||x|| (backward stability of the factor and
    # both substitutions, explicit 256-block inverses of condition < 10)
    assert float(res.max()) < 10 * np.sqrt(n) * np.finfo(dtype).eps
    if pad:
        assert torch.equal(dB[:, n:].double(), B0[:, n:])


def _system(n, r, seed, pad=0):
    """A factored quasi-definite FP64 matrix and its right-hand sides."""
    import torch
    from openmeeg_amd import _lib
    lib = _lib.lib()
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((n, n)) / np.sqrt(n)
    A = 0.25 * (A + A.T) + np.diag(np.where(np.arange(n) < n // 2, 2.0, -2.0))
    dA = torch.zeros((n, n + pad), dtype=torch.float64, device="cuda")
    dA[:, :n] = torch.from_numpy(A)
    work = torch.zeros(int(lib.omh_factor_workspace_bytes(n, 8)), dtype=torch.uint8, device="cuda")
    info = C.c_int32()
    _lib.check(lib.omh_sym_factor_f64(C.c_void_p(dA.data_ptr()), n, n + pad, C.c_void_p(work.data_ptr()),
                                      C.byref(info), C.c_void_p(0)))
    assert info.value == 0
    B = torch.from_numpy(rng.standard_normal((r, n))).cuda()

    def solve(X, stream):
        _lib.check(lib.omh_sym_solve_f64(C.c_void_p(dA.data_ptr()), n, n + pad, C.c_void_p(work.data_ptr()),
                                         C.c_void_p(X.data_ptr()), n, r, C.c_void_p(stream.cuda_stream)))

    torch.cuda.synchronize()
    return B, solve


@pytest.mark.parametrize("n,r,pad", [(1024, 1025, 0), (1300, 1100, 1), (2309, 2000, 3)])
def test_many_rhs_same_under_capture(om, n, r, pad):
    """A captured FP64 solve of more than 1024 right-hand sides takes the
    eager call's kernels: the same bits on every replay."""
    import torch
    B, solve = _system(n, r, n, pad)
    X, Y = B.clone(), B.clone()
    solve(X, torch.cuda.current_stream())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        solve(Y, torch.cuda.current_stream())
    for _ in range(3):
        Y.copy_(B)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(X, Y)


def test_many_rhs_on_two_streams(om):
    """FP64 solves of more than 1024 right-hand sides on two streams share
    nothing: the second one runs while the first stream is still busy."""
    import torch
    n, r = 1300, 1100
    B, solve = _system(n, r, 5)
    streams = [torch.cuda.Stream() for _ in range(8)]
    X = [B.clone() for _ in streams]
    torch.cuda.synchronize()
    for x, s in zip(X, streams):
        solve(x, s)
        s.synchronize()
    busy, done = streams[0], torch.cuda.Event()
    solve(X[0], busy)
    with torch.cuda.stream(busy):
        torch.cuda._sleep(int(1e9))
        done.record()
    # a stream that does not share the first one's hardware queue
    for x, s in zip(X[1:], streams[1:]):
        mark = torch.cuda.Event()
        with torch.cuda.stream(s):
            x.copy_(B)
            mark.record()
        t = time.time()
        while not mark.query() and time.time() - t < 0.02:
            pass
        if mark.query():
            break
    assert mark.query() and not done.query(), "no stream runs beside the busy one"
    solve(x, s)
    s.synchronize()
    assert not done.query()
    torch.cuda.synchronize()


def test_many_rhs_from_several_threads(om):
    """FP64 solves of more than 1024 right-hand sides hold no buffer that
    calls share: three host threads with factors and streams of their own
    get the bits of the solves one after the other."""
    import torch
    systems = [_system(n, r, n + r) for n, r in ((1536, 1500), (1300, 1100), (2048, 1030))]
    want = []
    for B, solve in systems:
        X = B.clone()
        solve(X, torch.cuda.current_stream())
        want.append(X)
    torch.cuda.synchronize()
    bad = []

    def work(k):
        B, solve = systems[k]
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                X = B.clone()
                solve(X, stream)
                if not torch.equal(X, want[k]):
                    bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(systems))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_refinement_beside_a_split_gemm(om):
    """The chunked residual of a small head's refinement and the split-K
    products of omh_gemm_f64 on another thread use buffers of their own: the
    bits of each alone."""
    import torch
    from openmeeg_amd import _lib, spheres as S
    from openmeeg_amd.api import _head_mat_device, factor
    g = om.make_nested_geometry(S.nested_sphere_meshes(8, (0.87, 0.92, 1.0)), (1.0, 0.0125, 1.0))
    n, r = g.size, 37
    H = _head_mat_device(g, far_field=True)
    F = factor(H, n, "mixed", structure=g.factor_segments(), order=g.factor_order())
    rng = np.random.default_rng(1)
    B = torch.from_numpy(rng.standard_normal(n * r)).cuda()
    m, q, k = 96, 320, 20000
    P = torch.from_numpy(rng.standard_normal(m * k)).cuda()
    Q = torch.from_numpy(rng.standard_normal(q * k)).cuda()

    def refine(stream):
        X = B.clone()
        F.solve(X, r, tol=1e-12)
        return X

    def gemm(stream):
        Z = torch.empty(m * q, dtype=torch.float64, device="cuda")
        _lib.check(_lib.lib().omh_gemm_f64(1, 0, m, q, k, 1.0, C.c_void_p(P.data_ptr()), k, C.c_void_p(Q.data_ptr()), k,
                                           0.0, C.c_void_p(Z.data_ptr()), m, C.c_void_p(stream.cuda_stream)))
        return Z

    calls = (refine, gemm)
    want = [f(torch.cuda.current_stream()) for f in calls]
    assert F.iterations >= 2
    torch.cuda.synchronize()
    bad = []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(30):
                if not torch.equal(calls[i](stream), want[i]):
                    bad.append(calls[i].__name__)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(calls))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_split_products_scale_cache_many_rhs(om, monkeypatch):
    """Enough right-hand sides that the split products run (1024 tiles of
    64 x 64 and more): cached scales against scales formed by every solve,
    bitwise, on a factor whose order is not a multiple of 4."""
    import torch
    from openmeeg_amd.api import _head_mat_device, factor
    from openmeeg_amd import spheres as S
    g = om.make_nested_geometry(S.nested_sphere_meshes(12, (0.87, 0.92, 1.0)), (1.0, 0.0125, 1.0))
    n, r = g.size, 700
    assert n % 4 == 2
    H = _head_mat_device(g, far_field=True)
    F = factor(H, n, "mixed16", structure=g.factor_segments(), n_positive=n - g.n_vertex_unknowns,
               order=g.factor_order())
    assert F.ld % 4 == 0
    B = torch.from_numpy(np.random.default_rng(4).standard_normal(n * r)).cuda()
    X = {}
    for mode in ("cache", "none"):
        if mode == "none":
            monkeypatch.setenv("OMH_SOLVE_SCALE_CACHE", "0")
        X[mode] = B.clone()
        with Launches() as ran:
            F.solve(X[mode], r, max_iter=10, tol=1e-12)
            torch.cuda.synchronize()
            split = ran("solve_update_f32s")
        assert split >= 2 * F.iterations
        monkeypatch.delenv("OMH_SOLVE_SCALE_CACHE", raising=False)
    assert F.iterations >= 2
    assert torch.equal(X["cache"], X["none"])
    res = torch.linalg.norm(B.view(r, n) - X["cache"].view(r, n) @ H.view(n, n)) / torch.linalg.norm(B)
    assert float(res) < 1e-12


@pytest.mark.parametrize("order", [False, True])
@pytest.mark.parametrize("freqs,r", [((9, 8, 6), 37), ((10, 9, 8), 1), ((14, 12, 11), 129), ((9, 9, 9), 200)])
def test_chunked_residual(om, freqs, r, order):
    """The FP64 residual of small heads runs in chunks of the inner dimension
    (uneven segments, odd right-hand sides, a ragged last chunk): the refined
    solution's own residual, formed by torch, is that of a backward stable
    FP64 solve."""
    import torch
    from openmeeg_amd.api import _head_mat_device, factor
    from openmeeg_amd import spheres as S
    meshes = [S.nested_sphere_meshes(f, (R,))[0] for f, R in zip(freqs, (0.87, 0.92, 1.0))]
    g = om.make_nested_geometry(meshes, (1.0, 0.0125, 1.0))
    n = g.size
    H = _head_mat_device(g, far_field=True)
    F = factor(H, n, "mixed", structure=g.factor_segments(), order=g.factor_order() if order else None)
    B = torch.from_numpy(np.random.default_rng(n + r).standard_normal((r, n))).cuda()
    X = B.clone().view(-1)
    with Launches() as ran:
        F.solve(X, r, max_iter=20, tol=1e-14)
        torch.cuda.synchronize()
        chunks = ran("residual_f64_split")
    assert chunks > 0 and F.iterations >= 2 and not F.fell_back
    X, Hm = X.view(r, n), H.view(n, n)
    res = (X @ Hm - B).norm(dim=1) / (Hm.abs().sum(1).max() * X.norm(dim=1))
    print("n=%d r=%d: %d chunked products, %d passes, residual %.3e" % (n, r, chunks, F.iterations, float(res.max())),
          flush=True)
    # the last correction is below 1e-14 |X|; X and the residual it came from
    # are rounded in FP64: a few eps |H| |X| a row, sqrt(n) over the rows
    assert float(res.max()) < 10 * np.sqrt(n) * np.finfo(float).eps
