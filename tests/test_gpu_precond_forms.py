"""GPU tests of the block-diagonal preconditioner's two forms (superblocks for symmetric channels,
block LU otherwise) at the edges of their sizes, against dense solves of the same matrices."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    from pyprop_amd import _native
    _native.load()
    return t


def _band(rng, n, b):
    S = np.diag(rng.uniform(1.0, 2.0, n))
    for d in range(1, b + 1):
        if d < n:
            v = rng.uniform(-0.4, 0.4, n - d) / b
            S += np.diag(v, d) + np.diag(v, -d)
    return S


def _pairs(n, b):
    return np.array([(i, j) for i in range(n) for j in range(max(0, i - b), min(n, i + b + 1))], dtype=np.int32)


def _growth(M):
    """The largest entry of the factors without pivoting over the largest of M: what the backward error of
    such an elimination is proportional to."""
    A = M.copy()
    for k in range(len(A)):
        A[k + 1:, k] /= A[k, k]
        A[k + 1:, k + 1:] -= np.outer(A[k + 1:, k], A[k, k + 1:])
    return np.abs(A).max() / np.abs(M).max()


def _check(torch, nchan, n1, n2, b, kind, sh, ss, seed=0, before_solve=None, indefinite=False):
    from pyprop_amd import _native as N, device as D
    rng = np.random.default_rng(seed)
    S1, S2 = _band(rng, n1, b), _band(rng, n2, b)
    p1, p2 = _pairs(n1, b), _pairs(n2, b)
    full = rng.standard_normal((nchan, n1, n2, n1, n2))
    if kind != "unsymmetric":
        full = full + full.transpose(0, 3, 4, 1, 2)  # symmetric under the exchange of (I, i) and (J, j)
    full = full / (2 * b + 1)
    P = full[:, p1[:, 0][:, None], p2[:, 0][None, :], p1[:, 1][:, None], p2[:, 1][None, :]].astype(complex)
    if kind == "complex":
        P = P * (1 + 0.2j)
    P = np.ascontiguousarray(P)
    h = C.c_void_p()
    N.check(N.load().pp_precond_create(nchan, n1, n2, b, D.hptr(S1), D.hptr(S2), D.hptr(P), len(p1), D.hptr(p1), len(p2),
                                       D.hptr(p2), N.cplx(sh), N.cplx(ss), C.byref(h)))
    if before_solve:
        before_solve()
    x = rng.standard_normal((nchan, n1, n2)) + 1j * rng.standard_normal((nchan, n1, n2))
    t = torch.from_numpy(x.copy()).to("cuda")
    guard = t.clone()
    N.check(N.load().pp_precond_solve(h, D.ptr(t), D.stream_handle()))
    got = t.cpu().numpy()
    N.check(N.load().pp_precond_solve(h, D.ptr(guard), D.stream_handle()))
    assert np.array_equal(guard.cpu().numpy(), got)  # nothing is kept from the first solve
    N.load().pp_precond_destroy(h)
    for c in range(nchan):
        M = np.zeros((n1, n2, n1, n2), complex)
        M[p1[:, 0][:, None], p2[:, 0][None, :], p1[:, 1][:, None], p2[:, 1][None, :]] = sh * P[c]
        M = (M + ss * np.einsum("ab,cd->acbd", S1, S2)).reshape(n1 * n2, n1 * n2)
        ref = np.linalg.solve(M, x[c].ravel())
        err = np.linalg.norm(got[c].ravel() - ref) / np.linalg.norm(ref)
        bound = 4e-14 if not indefinite else 16 * 2.0 ** -53 * _growth(M)
        assert err < bound * np.linalg.cond(M), (c, err)


# two to ten superblocks, a short last one, each band limit (4, 6, 8) with each of its counts of 64-column tiles
SIZES = [(2, 1, 1), (5, 3, 1), (13, 13, 4), (20, 33, 2), (7, 64, 3), (9, 49, 4), (7, 7, 6), (12, 10, 6), (19, 21, 5),
         (11, 29, 5), (24, 40, 6), (13, 64, 5), (13, 60, 6), (9, 9, 7), (16, 16, 8), (17, 24, 8), (15, 32, 8), (16, 40, 8),
         (15, 54, 7), (16, 64, 7), (9, 64, 8)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_symmetric_superblocks(torch, size):
    _check(torch, 3 if size[0] * size[1] < 700 else 1, *size, "symmetric", 0.3j, 1.0, seed=size[0])


def test_a_smaller_preconditioner_of_the_same_form_in_between(torch):
    """74 KB of LDS; the one that is created before the solve needs 73 KB."""
    _check(torch, 1, 12, 64, 6, "symmetric", 0.3j, 1.0,
           before_solve=lambda: _check(torch, 1, 12, 54, 6, "symmetric", 0.3j, 1.0))


@pytest.mark.parametrize("kind", ["unsymmetric", "complex"])
@pytest.mark.parametrize("size", [(7, 7, 6), (13, 13, 4)], ids=lambda s: "x".join(map(str, s)))
def test_general_block_lu(torch, kind, size):
    _check(torch, 2, *size, kind, 0.3j, 1.0)


def test_block_rows_beyond_the_superblock_kernel(torch):
    _check(torch, 1, 12, 66, 3, "symmetric", 0.3j, 1.0)


def test_real_scaling(torch):
    """H - sigma S with sigma below the spectrum, as the shift-invert solver asks for it."""
    _check(torch, 2, 13, 12, 4, "symmetric", 0.2, 1.5)


# sigma inside the spectrum: H - sigma S is indefinite, real or nearly so
@pytest.mark.parametrize("seed", range(4))
@pytest.mark.parametrize("ss", [-0.5, 0.3, -0.1 + 1e-6j])
@pytest.mark.parametrize("size", [(13, 13, 4), (20, 20, 5), (24, 24, 6)], ids=lambda s: "x".join(map(str, s)))
def test_shift_inside_the_spectrum(torch, size, ss, seed):
    """Elimination without pivoting loses digits to the growth of its factors, and explicit inverses of
    whole superblocks more than that: such matrices are factorized as a block LU."""
    _check(torch, 1, *size, "symmetric", 1.0, ss, seed=seed, indefinite=True)
