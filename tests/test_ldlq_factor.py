"""The LDLQ factor of csrc/chol.cuh (gpuq_prepare_hessian_dev) at the sizes where its blocking can go wrong: 2 to 20
blocks of 128 columns, so that the doubling of the inverse ends in no pair, a whole pair or a ragged one, against a
float64 factor by the same mathematics (A = V V^T, U = V^-1) in numpy; and the inputs whose factorization fails."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    torch.cuda.init()
    import gpuq
    return torch, gpuq.load_gpuq(0)


def prepare(env, H, n, damp=0.01):
    torch, gq = env
    ne0 = H.shape[0]
    dH = torch.from_numpy(np.ascontiguousarray(H)).cuda()
    # (a factor in an 8-byte aligned place of a larger buffer, with values around it that must stay)
    buf = torch.full((ne0 * ne0 + 2,), 7.0, dtype=torch.float64, device="cuda")
    perm = np.empty(ne0, dtype=np.int64)
    rc = gq.gpuq_prepare_hessian_dev(dH.data_ptr(), ne0, float(n), damp, 0, buf.data_ptr() + 8, perm.ctypes.data, None,
                                     None, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    out = buf.cpu().numpy()
    assert out[0] == 7.0 and out[-1] == 7.0
    return rc, out[1:-1].reshape(ne0, ne0)


def factor(A):
    """U upper with U^T U = A^-1, and V = U^-1 (the Cholesky factor of A read backwards)"""
    V = np.linalg.cholesky(A[::-1, ::-1])[::-1, ::-1]
    return np.linalg.inv(V), V


@pytest.mark.parametrize("ne0", [256, 512, 768, 1280, 1792, 2560])
def test_factor(env, ne0):
    rng = np.random.default_rng(ne0)
    X = rng.standard_t(4, (ne0 + 512, ne0)) * (0.5 + rng.random(ne0))
    n = X.shape[0]
    H = X.T @ X
    A = H / n
    A[np.diag_indices(ne0)] += 0.01 * np.mean(np.diag(A))
    want, V = factor(A)
    print("case factor %d" % ne0, flush=True)
    rc, U = prepare(env, H, n)
    assert rc == 0
    assert np.array_equal(np.tril(U, -1), np.zeros_like(U))
    # first-order bound of both factorizations: each off by at most n u cond(V) relative
    rel = np.linalg.norm(U - want) / np.linalg.norm(want)
    assert rel <= 2 * ne0 * 2.0 ** -53 * np.linalg.cond(V)
    # and four times what these well-conditioned inputs (cond(V) 7 to 20) measure, n u / 90: 3.2e-16 to 2.4e-15
    assert rel <= ne0 * 2.0 ** -53 / 22


def singular(n, seed):
    """an exactly singular H: whole numbers, one column twice"""
    rng = np.random.default_rng(seed)
    X = rng.integers(-9, 10, (n + 64, n)).astype(np.float64)
    j, k = rng.integers(0, n, 2)
    X[:, j] = X[:, k]
    return X.T @ X


@pytest.mark.parametrize("ne0,seed", [(256, 6), (512, 0), (512, 5), (512, 8), (768, 8)])
def test_factor_refuses_singular(env, ne0, seed):
    """singular matrices that a factorization last column first lets pass (its last pivots are rounding errors above 0),
    while one first column first, or that of the inverse, does not (the reference's, tools/ldlq.py:57-68): refused"""
    print("case factor singular", ne0, seed, flush=True)
    assert prepare(env, singular(ne0, seed), 1, damp=0.0)[0] == 3


@pytest.mark.parametrize("ne0", [256, 768])
@pytest.mark.parametrize("back", [False, True])
def test_factor_of_a_graded_matrix(env, ne0, back):
    """a condition of 1e24 that is scaling alone is no reason to refuse, and costs no accuracy: with A = D B D,
    U D is B's factor's inverse"""
    d = np.logspace(0, -12, ne0)[::-1 if back else 1]
    i = np.arange(ne0)
    B = np.eye(ne0) + 0.3 * np.exp(-abs(i[:, None] - i[None]) / 3.0)
    print("case factor graded", ne0, back, flush=True)
    rc, U = prepare(env, d[:, None] * B * d[None], 1, damp=0.0)
    assert rc == 0
    want, V = factor(B)
    # (two factorizations as in test_factor, and the roundings of D B D)
    assert np.linalg.norm(U * d - want) <= 3 * ne0 * 2.0 ** -53 * np.linalg.cond(V) * np.linalg.norm(want)


def test_factor_retries_with_more_ridge_and_refuses(env):
    """Not positive definite with the ridge, but with ten times more: the retry's factor; with neither, or with a value
    that is not finite: 3"""
    ne0, n = 256, 4
    A = np.eye(ne0)
    A[3, 200] = A[200, 3] = 1.05                 # least eigenvalue -0.05: -0.04 with the ridge, 0.06 with the retry's
    print("case factor retry", flush=True)
    rc, U = prepare(env, A * n, n)
    assert rc == 0
    want, V = factor(A + (0.01 + 10 * 0.01) * np.eye(ne0))
    assert np.linalg.norm(U - want) <= 2 * ne0 * 2.0 ** -53 * np.linalg.cond(V) * np.linalg.norm(want)
    A[3, 200] = A[200, 3] = 2.0
    assert prepare(env, A * n, n)[0] == 3
    for i, j, v in ((5, 5, np.nan), (5, 200, np.nan), (130, 130, np.inf), (130, 7, np.inf)):
        B = np.eye(ne0)
        B[i, j] = B[j, i] = v
        print("case factor refuses", i, j, v, flush=True)
        assert prepare(env, B * n, n)[0] == 3
