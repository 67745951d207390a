"""GPU tests of potentials that the multiply plan stores compactly (symmetric bands kept as half their
diagonals, equal fibres kept once) against a dense product: all, some or none of a Hamiltonian's terms
compact, real and complex, row counts below, at and above a wave, every band width the kernel has."""
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


def _potential(rng, nc, n1, b1, n2, b2, kind):
    """(TensorPotentialData, dense (nc n1 n2)^2 matrix); kind "symmetric" in every rank, "half" only in
    the innermost, "none", "complex"."""
    from pyprop_amd.geometry import Geometry
    from pyprop_amd.systems import TensorPotentialData
    p0 = np.array([(a, b) for a in range(nc) for b in range(nc)], dtype=np.int32)
    p1 = np.array([(a, b) for a in range(n1) for b in range(max(0, a - b1), min(n1, a + b1 + 1))], dtype=np.int32)
    w = 2 * b2 + 1
    full = rng.standard_normal((nc, nc, n1, n1, n2, n2))
    if kind == "complex":
        full = full + 1j * rng.standard_normal(full.shape)
    elif kind != "none":
        full = full + full.swapaxes(4, 5)
    if kind == "symmetric":
        full = full + full.swapaxes(0, 1)
        full = full + full.swapaxes(2, 3)
    keep1 = np.abs(np.subtract.outer(np.arange(n1), np.arange(n1))) <= b1
    keep2 = np.abs(np.subtract.outer(np.arange(n2), np.arange(n2))) <= b2
    full = full * keep1[None, None, :, :, None, None] * keep2
    data = np.zeros((len(p0), len(p1), n2 * w), complex)
    pairs2 = np.zeros((n2 * w, 2), dtype=np.int32)
    for j in range(n2):
        for i in range(max(0, j - b2), min(n2, j + b2 + 1)):
            k = j * w + b2 + i - j
            pairs2[k] = (i, j)
            data[:, :, k] = full[p0[:, 0][:, None], p0[:, 1][:, None], p1[:, 0][None], p1[:, 1][None], i, j]
    geo = [Geometry("Simp", p0, False, nc), Geometry("Simp", p1, True, n1), Geometry("BandNH", pairs2, True, n2)]
    dense = full.transpose(0, 2, 4, 1, 3, 5).reshape(nc * n1 * n2, nc * n1 * n2)
    return TensorPotentialData(kind, geo, data), dense


def _outer(n2, b2, least):
    """Channels, rows and band of the outer ranks that give a term at least `least` stored values."""
    for nc, n1, b1 in ((2, 3, 1), (3, 4, 2), (5, 5, 2), (6, 6, 2), (8, 8, 2), (16, 8, 2)):
        pairs = sum(min(n1, a + b1 + 1) - max(0, a - b1) for a in range(n1))
        if nc * nc * pairs * n2 * (2 * b2 + 1) >= least:
            break
    return nc, n1, b1


COMPACT_FROM = 2 ** 15  # values from which compact storage is looked for


@pytest.mark.parametrize("b2", range(11))
@pytest.mark.parametrize("kinds", [("symmetric",), ("none",), ("complex",), ("symmetric", "none")], ids="+".join)
@pytest.mark.parametrize("n2", [40, 100, 200, 260])
def test_band_widths(torch, kinds, n2, b2):
    _check_hamiltonian(torch, kinds, n2, b2)


@pytest.mark.parametrize("kinds", [("symmetric",), ("half",), ("none",), ("symmetric", "half"), ("symmetric", "none"),
                                   ("none", "half", "symmetric")], ids="+".join)
@pytest.mark.parametrize("n2,b2", [(3, 1), (13, 4), (63, 6), (64, 6), (65, 6), (130, 2), (300, 3)])
def test_hamiltonian_of_compact_terms(torch, kinds, n2, b2):
    _check_hamiltonian(torch, kinds, n2, b2)


def test_small_terms_are_kept_as_they_are(torch):
    _check_hamiltonian(torch, ("symmetric", "half"), 13, 4, least=0)


def _check_hamiltonian(torch, kinds, n2, b2, least=COMPACT_FROM):
    from pyprop_amd.propagator import BasisPropagator, CombinedRepresentation, Wavefunction
    rng = np.random.default_rng(n2 + len(kinds))
    nc, n1, b1 = _outer(n2, b2, least)
    made = [_potential(rng, nc, n1, b1, n2, b2, k) for k in kinds]
    repr_ = CombinedRepresentation((nc, n1, n2), [None, None, None])
    x = rng.standard_normal((nc, n1, n2)) + 1j * rng.standard_normal((nc, n1, n2))
    psi = Wavefunction(repr_, x)
    base = BasisPropagator(psi, [m[0] for m in made], consolidate=False)
    out = Wavefunction(repr_)
    base.MultiplyHamiltonianNoOverlap(psi, out, 0.0)
    M = sum(m[1] for m in made)
    ref = (M @ x.ravel()).reshape(x.shape)
    bound = 2.0 ** -53 * (nc * (2 * b1 + 1) * (2 * b2 + 1) * len(kinds) + 4) * (np.abs(M) @ np.abs(x.ravel()))
    assert np.all(np.abs(out.numpy().ravel() - ref.ravel()) <= 2 * bound)
    # stored bytes: half the diagonals of symmetric bands, and of equal fibres one
    for p, k in zip(base.PotentialList, kinds):
        full = 8 * nc * nc * p.GeometryList[1].pair_count * (2 * b2 + 1) * n2
        if k in ("none", "complex"):
            assert p.stream_bytes == (full if k == "none" else 2 * full)
        elif least == 0:
            assert p.stream_bytes == full
        elif b2 > 0:  # (a diagonal has no mirror image)
            assert p.stream_bytes < 0.76 * full
    # one potential at a time, added to what is there
    for (data, dense), p in zip(made, base.PotentialList):
        acc = torch.ones_like(psi.data)
        p.MultiplyPotential(psi, acc, 0.0)
        r = (dense @ x.ravel()).reshape(x.shape) + 1.0
        assert np.linalg.norm(acc.cpu().numpy() - r) < 1e-14 * np.linalg.norm(r)


@pytest.mark.parametrize("n2,b2", [(13, 4), (64, 6), (100, 3)])
def test_fp32_multiply_of_compact_terms(torch, n2, b2):
    import ctypes as C
    from pyprop_amd import _native as N, device as D
    from pyprop_amd.tensorpotential import TensorPotential
    rng = np.random.default_rng(n2)
    nc, n1, b1 = _outer(n2, b2, COMPACT_FROM)
    data, dense = _potential(rng, nc, n1, b1, n2, b2, "symmetric")
    p = TensorPotential(data, (nc, n1, n2))
    p.SetupStep()
    assert p.stream_bytes < 8 * 0.76 * data.data.size
    x = rng.standard_normal((nc, n1, n2)) + 1j * rng.standard_normal((nc, n1, n2))
    src = torch.from_numpy(x).to("cuda").to(torch.complex64)
    dst = torch.zeros_like(src)
    N.check(N.load().pp_tp_multiply_f32(p.plan, C.c_float(1.0), D.ptr(src), D.ptr(dst), D.stream_handle()))
    ref = dense @ x.ravel()
    assert np.linalg.norm(dst.cpu().numpy().ravel() - ref) < 1e-6 * np.linalg.norm(ref)


def test_nan_stays_in_the_rows_it_couples_to(torch):
    """A NaN of row j reaches rows j - b .. j + b of the innermost rank, as in the banded product."""
    from pyprop_amd.propagator import BasisPropagator, CombinedRepresentation, Wavefunction
    rng = np.random.default_rng(1)
    for n2 in (40, 90):
        nc, n1, b1 = _outer(n2, 3, COMPACT_FROM)
        data, _ = _potential(rng, nc, n1, b1, n2, 3, "symmetric")
        repr_ = CombinedRepresentation((nc, n1, n2), [None, None, None])
        x = np.ones((nc, n1, n2), complex)
        x[1, 0, 20] = np.nan
        psi, out = Wavefunction(repr_, x), Wavefunction(repr_)
        base = BasisPropagator(psi, [data], consolidate=False)
        base.MultiplyHamiltonianNoOverlap(psi, out, 0.0)
        assert base.PotentialList[0].stream_bytes < 8 * 0.76 * data.data.size
        bad = np.argwhere(np.isnan(out.numpy().real))
        expected = [(c, i, j) for c in range(nc) for i in range(b1 + 1) for j in range(17, 24)]
        assert np.array_equal(bad, expected)


def test_uneven_fibres(torch):
    """One destination fibre with nearly all tuples: the launch order by XCDs would be mostly empty."""
    from pyprop_amd.geometry import Geometry
    from pyprop_amd.propagator import BasisPropagator, CombinedRepresentation, Wavefunction
    from pyprop_amd.systems import TensorPotentialData
    rng = np.random.default_rng(5)
    nc, n, b, repeats = 300, 8, 2, 40
    pairs0 = np.array([(0, c) for c in range(nc)] * repeats + [(c, c) for c in range(1, nc)], dtype=np.int32)
    pairs1 = np.array([(i, j) for j in range(n) for i in range(j - b, j + b + 1)], dtype=np.int32)
    inside = (pairs1[:, 0] >= 0) & (pairs1[:, 0] < n)
    band = np.add.outer(np.arange(n), np.arange(n)) / 4.0
    row = np.where(inside, band[pairs1[:, 0] * inside, pairs1[:, 1]], 0.0)
    amp = rng.integers(1, 5, len(pairs0)) / 4.0
    data = TensorPotentialData("uneven", [Geometry("Simp", pairs0, False, nc),
                                          Geometry("BandNH", np.where(inside[:, None], pairs1, 0), True, n)],
                               (amp[:, None] * row).astype(complex))
    x = rng.standard_normal((nc, n)) + 1j * rng.standard_normal((nc, n))
    repr_ = CombinedRepresentation((nc, n), [None, None])
    psi, out = Wavefunction(repr_, x), Wavefunction(repr_)
    base = BasisPropagator(psi, [data], consolidate=False)
    assert base.PotentialList[0].stream_bytes < 8 * 0.1 * data.data.size  # four amplitudes
    base.MultiplyHamiltonianNoOverlap(psi, out, 0.0)
    M = band * (np.abs(np.subtract.outer(np.arange(n), np.arange(n))) <= b)
    A = np.zeros((nc, nc))
    np.add.at(A, (pairs0[:, 0], pairs0[:, 1]), amp)
    ref = A @ x @ M.T
    bound = 2.0 ** -53 * (len(pairs0) * (2 * b + 1) + 4) * (A @ np.abs(x) @ M.T)
    assert np.all(np.abs(out.numpy() - ref) <= bound)


def test_more_fibres_than_a_launch_has_waves(torch):
    """8195 x 8195 channels of one row, over 2^26 potential fibres: kept as they are."""
    from pyprop_amd.geometry import Geometry
    from pyprop_amd.systems import TensorPotentialData
    from pyprop_amd.tensorpotential import TensorPotential
    nc = 8195
    a = np.arange(nc, dtype=np.int32)
    pairs = np.stack(np.broadcast_arrays(a[:, None], a[None, :]), -1).reshape(-1, 2)
    u, w = 1.0 + a % 7, 2.0 + a % 5
    data = TensorPotentialData("one row", [Geometry("Simp", pairs, False, nc),
                                           Geometry("BandNH", np.zeros((1, 2), np.int32), True, 1)],
                               np.multiply.outer(u, w).astype(complex).reshape(-1, 1))
    p = TensorPotential(data, (nc, 1))
    p.SetupStep()
    assert p.stream_bytes == 8 * nc * nc
    x = torch.from_numpy(np.arange(nc) % 3 + 1j * (np.arange(nc) % 4)).to("cuda").reshape(nc, 1)
    out = torch.zeros_like(x)
    p.MultiplyPotential(x, out, 0.0)
    # whole numbers below 2^53: exact
    assert np.array_equal(out.cpu().numpy()[:, 0], u * (w @ x.cpu().numpy()[:, 0]))


def test_without_room_for_a_second_copy(torch):
    """A potential that fits the device once but not once and a half is kept as it is."""
    import ctypes as C
    from pyprop_amd import _native as N, device as D
    nc, n, b = 1600, 40, 2
    values = nc * nc * n * (2 * b + 1)  # 512 million, 4 GB stored
    a = np.arange(nc, dtype=np.int32)
    pairs = np.ascontiguousarray(np.stack(np.broadcast_arrays(a[:, None], a[None, :]), -1).reshape(-1, 2))
    pot = torch.zeros((nc * nc, n, 2 * b + 1), dtype=torch.complex128, device="cuda")
    pot.real[:, :, b] = torch.arange(nc * nc, dtype=torch.float64, device="cuda")[:, None]  # all different
    x = torch.ones((nc, n), dtype=torch.complex128, device="cuda")
    out = torch.zeros_like(x)
    want = pot.real[:, 0, b].reshape(nc, nc).sum(1)  # whole numbers: exact
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    hog = torch.empty(max(0, torch.cuda.mem_get_info()[0] - 8 * values - (1 << 30)), dtype=torch.uint8, device="cuda")
    h = C.c_void_p()
    ids = np.array([N.STORAGE["Simp"], N.STORAGE["BandNH"]], dtype=np.int32)
    ext, src = np.array([nc * nc, n * (2 * b + 1)], dtype=np.int32), np.array([nc, n], dtype=np.int32)
    lists, counts = (C.c_void_p * 2)(pairs.ctypes.data, None), np.array([nc * nc, 0], dtype=np.int32)
    lib = N.load()
    N.check(lib.pp_tp_create(2, D.hptr(ids), D.ptr(pot), D.hptr(ext), D.hptr(src), C.cast(lists, C.c_void_p),
                             D.hptr(counts), D.stream_handle(), C.byref(h)))
    del hog
    try:
        nbytes = C.c_int64()
        N.check(lib.pp_tp_info(h, C.byref(nbytes), None, None, None))
        assert nbytes.value == 8 * values
        N.check(lib.pp_tp_multiply(h, 1.0, D.ptr(x), D.ptr(out), D.stream_handle()))
        assert torch.equal(out.real, want[:, None].expand(nc, n)) and not out.imag.any()
    finally:
        lib.pp_tp_destroy(h)
        del pot
        torch.cuda.empty_cache()
