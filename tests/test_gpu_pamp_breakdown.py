"""GPU tests of pAMP steps whose Krylov space ends early (a state inside a small invariant subspace):
every coefficient of the last complete row belongs to the result, also those past the first 64, which
other waves of the workgroup store than the one that records the breakdown."""
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


class _Vector:
    def __init__(self, data):
        self.data = data


# (sites of the chain, elements of the state, basis size, time): the breakdown comes at step `sites`;
# one and several workgroups per vector, basis sizes on both sides of the exponential's LDS form (25)
@pytest.mark.parametrize("double_orth", [False, True])
@pytest.mark.parametrize("sites,n,m,dt", [(12, 12, 20, 6.0), (12, 17, 25, 6.0), (12, 700, 26, 6.0), (66, 66, 127, 60.0),
                                          (70, 1500, 80, 60.0), (100, 105, 127, 90.0), (127, 3000, 127, 110.0)])
def test_breakdown_keeps_every_coefficient(torch, sites, n, m, dt, double_orth):
    import oracle
    from pyprop_amd.propagator import PampWrapper
    # a chain of sites with hops of 1/2 and diagonal steps of 1/4, started at its end: every Krylov
    # vector is the next site, exactly, and the last residual is zero
    i = np.arange(sites)
    H = np.zeros((n, n))
    H[i, i] = 0.25 * ((7 * i) % 5 - 2)
    H[i[:-1], i[1:]] = H[i[1:], i[:-1]] = 0.5
    Hd = torch.from_numpy(H).to("cuda").to(torch.complex128)
    start = np.zeros(n, complex)
    start[0] = 1.0
    ref, _, _, broken = oracle.pamp_propagate(lambda x: H @ x, start, m, dt, order=12, dorth=double_orth)
    assert broken == (sites < m)
    pamp = PampWrapper(n, m, pade_order=12, krylov_double_orthogonalization=double_orth)
    for _ in range(3):
        psi, tmp = _Vector(torch.from_numpy(start.copy()).to("cuda")), _Vector(torch.zeros_like(Hd[0]))
        pamp.AdvanceStep(lambda s, d, dt_, t: d.data.copy_(Hd @ s.data), psi, tmp, dt, 0.0)
        # up to eight squarings of an m x m exponential, each doubling its rounding
        assert np.max(np.abs(psi.data.cpu().numpy() - ref)) < 2.0 ** 8 * m * 2.0 ** -53
