"""Diagonal blocks of the pivot-free factorisation (k_diag_factor,
k_diag_inverse): sizes at the edges of the 16-wide tiles and of the 256-wide
blocks, both types, any sign pattern, an odd leading dimension; the index of
a vanishing pivot."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NB = 256


@pytest.fixture(scope="module")
def om():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    import openmeeg_amd
    return openmeeg_amd


def _factor(A, n, ld, dtype):
    import torch
    from openmeeg_amd import _lib
    t = torch.float64 if dtype == np.float64 else torch.float32
    dA = torch.full((n, ld), 7.0, dtype=t, device="cuda")   # column j in row j
    dA[:, :n] = torch.from_numpy(np.ascontiguousarray(A.T.astype(dtype)))
    size = np.dtype(dtype).itemsize
    work = torch.zeros(int(_lib.lib().omh_factor_workspace_bytes(n, size)), dtype=torch.uint8, device="cuda")
    info = C.c_int32()
    fn = _lib.lib().omh_sym_factor_f64 if size == 8 else _lib.lib().omh_sym_factor_f32
    _lib.check(fn(C.c_void_p(dA.data_ptr()), n, ld, C.c_void_p(work.data_ptr()), C.byref(info), C.c_void_p(0)))
    torch.cuda.synchronize()
    w = work.cpu().numpy().view(dtype)
    nblk = -(-n // NB)
    inv = w[n * NB:n * NB + nblk * NB * NB].reshape(nblk, NB, NB).transpose(0, 2, 1)
    sgn = w[n * NB + nblk * NB * NB:][:n]
    out = dA.cpu().numpy()
    assert np.all(out[:, n:] == 7.0)
    return out[:, :n].T.astype(np.float64), inv.astype(np.float64), sgn, info.value


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 33, 100, 127, 128, 129, 240, 241, 255, 256, 257, 300, 513, 700])
def test_factor_and_block_inverse(om, n, dtype):
    rng = np.random.default_rng(n)
    s = rng.choice([-1.0, 1.0], n)
    L0 = np.tril(rng.standard_normal((n, n)) / np.sqrt(n), -1) + np.diag(0.5 + rng.random(n))
    A = ((L0 * s) @ L0.T).astype(dtype).astype(np.float64)
    # the strictly upper half is not read
    L, inv, sgn, info = _factor(np.tril(A) + np.triu(np.full((n, n), np.nan), 1), n, n + 3, dtype)
    assert info == 0
    L = np.tril(L)
    eps = np.finfo(dtype).eps
    assert np.array_equal(np.sign(sgn), s)
    # |A - L S L^T| <= c n eps |L| |L|^T element by element (Higham, Accuracy
    # and Stability, th. 10.3); the products with explicit tile inverses add
    # their condition, below 30 here
    bound = 30 * (n + 1) * eps * (np.abs(L) @ np.abs(L).T)
    assert np.all(np.abs(np.tril(A - (L * s) @ L.T)) <= bound)
    for b in range(len(inv)):
        k, w = b * NB, min(NB, n - b * NB)
        M, Lb = inv[b][:w, :w], L[k:k + w, k:k + w]
        assert np.all(np.triu(M, 1) == 0)
        assert np.all(np.abs(M @ Lb - np.eye(w)) <= 30 * (w + 1) * eps * (np.abs(M) @ np.abs(Lb)))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n,k", [(1, 0), (16, 15), (40, 17), (256, 0), (256, 255), (300, 259), (300, 299)])
def test_first_vanishing_pivot(om, n, k, dtype):
    A = np.diag(np.where(np.arange(n) % 2, -2.0, 3.0))
    A[k, k] = 0.0
    if k + 1 < n:
        A[n - 1, n - 1] = 0.0   # a later one too
    assert _factor(A, n, n, dtype)[3] == k + 1
