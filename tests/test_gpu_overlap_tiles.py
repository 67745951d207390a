"""GPU tests of the overlap operations along one rank at the edges of the tile kernel: row counts
around a wave and around each tile width, the last size with a dense inverse and the first without, few
and many fibres, first, middle and last ranks, against the factor in extended
precision."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MULTIPLY, SOLVE, SQRT_MULTIPLY, SQRT_SOLVE = 0, 1, 2, 3


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    from pyprop_amd import _native
    _native.load()
    return t


def _overlap(n, sd, seed=0, scale=1.0):
    """A banded positive definite S, its upper band, the device object and its factor U (extended)."""
    from pyprop_amd.propagator import OverlapMatrix
    rng = np.random.default_rng(seed)
    S = np.diag(rng.uniform(1.0, 2.0, n))
    for d in range(1, sd + 1):
        v = rng.uniform(-0.5, 0.5, n - d) / sd
        S += np.diag(v, d) + np.diag(v, -d)
    S *= scale
    ov = OverlapMatrix(S, sd)
    from pyprop_amd import _native as N, device as D
    band = np.zeros((n, sd + 1))
    N.check(N.load().pp_overlap_get_factor(ov.h, D.hptr(band)))
    U = np.zeros((n, n), dtype=np.longdouble)
    for j in range(n):
        for i in range(max(0, j - sd), j + 1):
            U[i, j] = band[j, sd + i - j]
    return ov, U


_BAND = 12  # more than any test's superdiagonals: the entries beyond are zero


def _solve_upper(U, b):
    x = b.copy()
    for i in range(U.shape[0] - 1, -1, -1):
        j = slice(i + 1, i + _BAND)
        x[i] = (x[i] - U[i, j] @ x[j]) / U[i, i]
    return x


def _solve_lower(L, b):
    x = b.copy()
    for i in range(L.shape[0]):
        j = slice(max(0, i - _BAND), i)
        x[i] = (x[i] - L[i, j] @ x[j]) / L[i, i]
    return x


def _multiply(U, b):
    return np.stack([U[i, max(0, i - _BAND):i + _BAND] @ b[max(0, i - _BAND):i + _BAND] for i in range(U.shape[0])])


def _reference(U, op, conj, x):
    """op applied to the columns of x (extended precision)."""
    if op == MULTIPLY:
        return _multiply(U.T, _multiply(U, x))
    if op == SOLVE:
        return _solve_upper(U, _solve_lower(U.T, x))
    if op == SQRT_MULTIPLY:
        return _multiply(U.T if conj else U, x)
    return _solve_lower(U.T, x) if conj else _solve_upper(U, x)


def _apply(torch, ov, op, conj, x):
    """x: (pre, n, post) complex128, along the middle rank."""
    from pyprop_amd import _native as N, device as D
    t = torch.from_numpy(x.copy()).to("cuda")
    ext = np.array(x.shape, dtype=np.int32)
    N.check(N.load().pp_overlap_apply(ov.h, op, int(conj), 3, D.hptr(ext), 1, D.ptr(t), D.stream_handle()))
    return t.cpu().numpy()


@pytest.mark.parametrize("n,sd", [(1, 0), (2, 1), (13, 4), (63, 6), (64, 6), (65, 6), (161, 6), (321, 3), (512, 8),
                                  (513, 8), (40, 11)])
@pytest.mark.parametrize("layout", [(1, 1), (5, 1), (520, 1), (3, 7), (2, 300)], ids=str)
def test_overlap_ops(torch, n, sd, layout):
    if n > 300 and layout[0] * layout[1] > 200:
        layout = (layout[0] % 7 + 1, layout[1] % 7 + 1)
    _check_ops(torch, n, sd, layout)


# more than 64 KB of LDS per multiply; pairs of fibres; fibre counts on both sides of the lines from
# which on a thread takes a fibre of a substitution
@pytest.mark.parametrize("n,sd,layout", [(512, 8, (3, 50)), (321, 3, (2, 131)), (160, 6, (300, 2)), (400, 5, (260, 2)),
                                         (15, 6, (600, 1)), (16, 6, (600, 1)), (17, 4, (32768, 1)), (17, 4, (32769, 1)),
                                         (321, 2, (5, 810)), (161, 1, (1, 4000)), (161, 1, (4001, 1)),
                                         (505, 3, (2, 1290))], ids=str)
def test_overlap_ops_at_the_lines_between_forms(torch, n, sd, layout):
    _check_ops(torch, n, sd, layout)


def _check_ops(torch, n, sd, layout):
    ov, U = _overlap(n, sd, seed=n)
    pre, post = layout
    rng = np.random.default_rng(pre + post)
    x = rng.standard_normal((pre, n, post)) + 1j * rng.standard_normal((pre, n, post))
    cols = np.moveaxis(x, 1, 0).reshape(n, -1).astype(np.clongdouble)
    for op in (MULTIPLY, SOLVE, SQRT_MULTIPLY, SQRT_SOLVE):
        for conj in ((False, True) if op >= SQRT_MULTIPLY else (False,)):
            ref = np.moveaxis(_reference(U, op, conj, cols).reshape(n, pre, post), 0, 1)
            got = _apply(torch, ov, op, conj, x)
            # sums of at most n terms with factors of condition below 10
            err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
            assert err < 2.0 ** -53 * 10 * (sd + 16), (op, conj, float(err))


def test_more_tiles_than_a_launch_holds(torch):
    """2^26 + 4 fibres of two rows: at four fibres to a workgroup of 256 threads, over 2^32 threads."""
    from pyprop_amd import _native as N, device as D
    fibres = 2 ** 26 + 4
    if torch.cuda.mem_get_info()[0] < 6 * 32 * fibres:
        pytest.skip("needs %d GB of device memory" % (6 * 32 * fibres >> 30))
    ov, U = _overlap(2, 1, seed=2)
    u00, u01, u11 = (float(U[i, j]) for i, j in ((0, 0), (0, 1), (1, 1)))
    x = torch.arange(2 * fibres, dtype=torch.float64, device="cuda").remainder_(8191.0).to(torch.complex128)
    x = x.reshape(fibres, 2)
    want0, want1 = u00 * x[:, 0] + u01 * x[:, 1], u11 * x[:, 1]
    ext = np.array([fibres, 2], dtype=np.int32)
    N.check(N.load().pp_overlap_apply(ov.h, SQRT_MULTIPLY, 0, 2, D.hptr(ext), 1, D.ptr(x), D.stream_handle()))
    # two products and a sum of values below 2^13
    assert (x[:, 0] - want0).abs().max().item() < 2.0 ** -38 and (x[:, 1] - want1).abs().max().item() < 2.0 ** -38


@pytest.mark.parametrize("n", [64, 100])
def test_overlap_solve_keeps_nan_where_substitution_does(torch, n):
    """Back substitution carries a NaN of row j to the rows before it, forward to those after."""
    ov, _ = _overlap(n, 6, seed=n)
    x = np.ones((1, n, 1), complex)
    j = n // 2 + 3
    x[0, j, 0] = np.nan
    back, fwd = _apply(torch, ov, SQRT_SOLVE, False, x), _apply(torch, ov, SQRT_SOLVE, True, x)
    assert np.all(np.isnan(back[0, :j + 1, 0])) and not np.any(np.isnan(back[0, j + 1:, 0]))
    assert np.all(np.isnan(fwd[0, j:, 0])) and not np.any(np.isnan(fwd[0, :j, 0]))


@pytest.mark.parametrize("n,sd", [(9, 8), (120, 6), (512, 3)])
def test_overlap_substitution_extreme_values(torch, n, sd):
    """Rows scaled over the exponent range, zeros and infinities: where the quotient is not formed
    by residual corrections it is the division."""
    ov, U = _overlap(n, sd, seed=n)
    rng = np.random.default_rng(n)
    for scale in (1e-300, 1e-260, 1e-240, 1e240, 1e260, 1e300):
        x = scale * (rng.standard_normal((1, n, 1)) + 1j * rng.standard_normal((1, n, 1)))
        got = _apply(torch, ov, SQRT_SOLVE, True, x)[0, :, 0]
        ref = _reference(U, SQRT_SOLVE, True, x[0].astype(np.clongdouble))[:, 0]
        # below 1e-292 the products of the sums are subnormal: one unit of 2^-1074 each
        assert np.max(np.abs(got - ref)) < 2.0 ** -53 * 10 * (sd + 16) * np.max(np.abs(ref)) + (sd + 2) * 20 * 5e-324
    x = np.zeros((1, n, 1), complex)
    assert np.all(_apply(torch, ov, SQRT_SOLVE, False, x) == 0)
    x[0, 0, 0] = np.inf
    assert np.isinf(_apply(torch, ov, SQRT_SOLVE, True, x)[0, 0, 0].real)


# factors of 1e-35 and 1e35 lie outside the range whose reciprocals are formed (2^+-100), the others inside
@pytest.mark.parametrize("scale", [1e-70, 1e-56, 1e56, 1e70])
@pytest.mark.parametrize("n,sd", [(9, 8), (120, 6), (512, 3)])
def test_overlap_substitution_of_zeros_with_extreme_factors(torch, n, sd, scale):
    """Zeros stay zeros and the rest is the quotient, whatever the scale of S."""
    ov, U = _overlap(n, sd, seed=n, scale=scale)
    x = np.zeros((3, n, 1), complex)
    x[1, n // 2] = 1.0 - 0.5j
    x[2, 0] = 2.0  # the imaginary part is zero throughout
    for conj in (False, True):
        got = _apply(torch, ov, SQRT_SOLVE, conj, x)
        ref = _reference(U, SQRT_SOLVE, conj, x[:, :, 0].T.astype(np.clongdouble)).T
        assert np.all(got[0] == 0) and np.all(got[2].imag == 0)
        assert np.max(np.abs(got[:, :, 0] - ref)) < 2.0 ** -53 * 10 * (sd + 16) * np.max(np.abs(ref))
