"""GPU tests of potentials generated term by term (project each term's grid function once, then
combine per angular pair) against the pair-by-pair projection and a float64 numpy sum, at the
edges of the rule that chooses between them and of the combining kernel's tiles."""
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


# one to more than twelve terms (one pass of the kernel), one pair to more than a range, radial
# counts around a workgroup of 256
@pytest.mark.parametrize("dims", [(1, 1, 1), (3, 5, 255), (11, 394, 257), (12, 7, 256), (13, 40, 300), (26, 3, 1000)],
                         ids=lambda d: "x".join(map(str, d)))
def test_expand_potential(torch, dims):
    from pyprop_amd import _native as N, device as D
    T, p0, rc = dims
    rng = np.random.default_rng(T)
    c, r = rng.standard_normal((T, p0)), rng.standard_normal((T, rc))
    dc, dr = D.to_device(c), D.to_device(r)
    out = torch.full((p0 + 1, rc), 5.0 - 1.0j, dtype=torch.complex128, device="cuda")
    N.check(N.load().pp_expand_potential(T, p0, rc, D.ptr(dc), D.ptr(dr), D.ptr(out), D.stream_handle()))
    got = out.cpu().numpy()
    assert np.all(got[p0] == 5.0 - 1.0j) and np.all(got[:p0].imag == 0)
    bound = T * 2.0 ** -53 * (np.abs(c).T @ np.abs(r))
    assert np.all(np.abs(got[:p0].real - c.T @ r) <= 2 * bound)


def test_expand_more_radial_values_than_a_launch_holds(torch):
    """2^32 + 300 radial values, a thread each: two launches."""
    from pyprop_amd import _native as N, device as D
    rc, slab = 2 ** 32 + 300, 2 ** 28
    if torch.cuda.mem_get_info()[0] < 30 * rc:
        pytest.skip("needs %d GB of device memory" % (30 * rc >> 30))
    radial = torch.empty(rc, dtype=torch.float64, device="cuda")
    for a in range(0, rc, slab):
        radial[a:a + slab] = torch.arange(a, min(rc, a + slab), dtype=torch.float64, device="cuda")
    coeffs = torch.full((1, 1), 0.5, dtype=torch.float64, device="cuda")
    out = torch.empty(rc, dtype=torch.complex128, device="cuda")
    N.check(N.load().pp_expand_potential(1, 1, rc, D.ptr(coeffs), D.ptr(radial), D.ptr(out), D.stream_handle()))
    for a in range(0, rc, slab):
        part = out[a:a + slab]
        assert torch.equal(part.real, 0.5 * radial[a:a + slab]) and not part.imag.any()


@pytest.mark.parametrize("kind", ["multipole", "separable"])
@pytest.mark.parametrize("pairs", [1, 2, 5, 6, 7, 40])  # two terms need six pairs (P1 < 2 Q1) to be combined
@pytest.mark.parametrize("accumulate", [False, True])
def test_terms_against_pairs(torch, kind, pairs, accumulate):
    """The generated potential against the staged path, which projects every pair's grid."""
    from pyprop_amd.potgen import generate_device_potential, generate_device_potential_staged
    from pyprop_amd.geometry import Geometry
    from pyprop_amd.systems import GridTerm, TensorPotentialData, helium_system
    s = helium_system(lmax=1, L=(0, 1), order=5, n_breakpoints=12, rmax=15.0, n_inner=6, gamma=2.5)
    basis = s.bases[1]
    g1, g2 = s.potentials[1].geometries[1:]
    rng = np.random.default_rng(pairs)
    g0 = Geometry("Simp", np.stack([np.arange(pairs), np.arange(pairs)], 1).astype(np.int32), False, pairs)
    coeffs = rng.standard_normal((2, pairs))
    Q = basis.grid.size

    def term():
        if kind == "multipole":
            return GridTerm("multipole", coeffs, (0, 0), lams=[0, 3])
        return GridTerm("separable", coeffs, (2, 0), [rng.standard_normal((2, Q)), rng.standard_normal((2, Q))])

    data = TensorPotentialData("v", [g0, g1, g2], None, None, None, None, [term(), term()] if accumulate else [term()])
    a = generate_device_potential(data).cpu().numpy()
    b = generate_device_potential_staged(data).cpu().numpy()
    assert np.all(a.imag == 0)
    # two orders of the same sum of 2 terms x 25 x 25 grid points
    assert np.linalg.norm(a - b) <= 1e-14 * np.linalg.norm(b)
