"""GPU tests of the training kernels of the learned preconditioner at the edges of their tiles
(rows, hidden width and channels that are no multiple of a wave) against the float64 oracle
with the device's BF16 rounding points."""
import numpy as np
import pytest

from oracle import mlp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch():
    import torch as t
    assert t.cuda.is_available(), "GPU tests need a HIP device"
    from pyprop_amd import _native
    _native.load()
    return t


class _Shape:
    def __init__(self, nchan, n):
        self.system = type("System", (), {"shape": (nchan, n, n)})

    def Setup(self):
        pass


def _rel(a, b):
    return np.linalg.norm(np.ravel(a) - np.ravel(b)) / max(np.linalg.norm(np.ravel(b)), 1e-300)


def _case(nchan, n, hidden, rows, seed):
    from pyprop_amd.mixed import LearnedPreconditioner
    rng = np.random.default_rng(seed)
    net = LearnedPreconditioner(_Shape(nchan, n), hidden)
    inp = 2 * n * n
    flat = net.get_params().astype(np.float64)
    lay, _ = mlp.layout(inp, hidden, nchan)
    for name, scale in (("W3", hidden ** -0.5), ("b1", 0.1), ("emb", 0.1), ("b2", 0.1), ("b3", 0.1)):
        o, shp = lay[name]
        k = int(np.prod(shp))
        flat[o:o + k] = scale * rng.standard_normal(k)
    flat = flat.astype(np.float32)
    net.set_params(flat)
    x = (rng.standard_normal((rows, inp)) / np.sqrt(inp)).astype(np.float32)
    t = (0.3 * rng.standard_normal((rows, inp))).astype(np.float32)
    chan = rng.integers(0, nchan, rows).astype(np.int32)
    return net, flat, x, t, chan


# rows below, at and above a ballot of 64 and the 16 waves of a column sum; widths below and
# above the 64 columns of a workgroup; channels without a row
@pytest.mark.parametrize("dims", [(1, 1, 8, 1), (5, 3, 72, 15), (70, 2, 64, 64), (9, 6, 136, 65), (2, 5, 64, 203)],
                         ids=lambda d: "x".join(map(str, d)))
def test_gradients_at_tile_edges(torch, dims):
    nchan, n, hidden, rows = dims
    net, flat, x, t, chan = _case(nchan, n, hidden, rows, 3)
    inp = 2 * n * n
    dev = [torch.from_numpy(a).to("cuda") for a in (x, chan, t)]
    loss = net.gradient(*dev)
    loss_ref, g_ref = mlp.loss_and_grad(mlp.unpack(flat.astype(np.float64), inp, hidden, nchan), x, chan, t, 1.0)
    assert abs(loss - loss_ref) < 1e-4 * loss_ref
    g = mlp.unpack(net.get_grads().astype(np.float64), inp, hidden, nchan)
    for name in mlp.NAMES:
        # FP32 sums; a backward signal whose FP32 value sits on a BF16 rounding boundary moves
        # by one BF16 ulp (2^-8), which few of a sum's terms do
        assert _rel(g[name], g_ref[name]) < 2e-3, name
    for c in set(range(nchan)) - set(chan.tolist()):
        assert np.all(g["emb"][c] == 0)


# around the 64 x 64 x 64 tile: below it, exact, one over, K steps 1 to 5 (two are loaded ahead),
# extents that forbid 16-byte loads in both operands, in one of them or in none; strides padded to a
# multiple of eight, so that rows are aligned but their last share is not whole
@pytest.mark.parametrize("pad", [False, True])
@pytest.mark.parametrize("a_k", [True, False])
@pytest.mark.parametrize("b_k", [True, False])
@pytest.mark.parametrize("dims", [(1, 1, 1), (64, 64, 64), (65, 63, 129), (128, 72, 192), (40, 200, 264), (66, 130, 320),
                                  (64, 66, 40), (130, 72, 100)],
                         ids=lambda d: "x".join(map(str, d)))
def test_gemm_at_tile_edges(torch, dims, a_k, b_k, pad):
    from pyprop_amd import _native as N, device as D
    M, N_, K = dims
    rng = np.random.default_rng(M * K)
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N_)).astype(np.float32)

    def operand(X):  # rows of X contiguous; the padding holds NaN, which no product may see
        ld = -(-X.shape[1] // 8) * 8 if pad else X.shape[1]
        wide = np.full((X.shape[0], ld), np.nan, np.float32)
        wide[:, :X.shape[1]] = mlp.bf16(X)
        return torch.from_numpy(wide).to("cuda").to(torch.bfloat16), ld

    da, lda = operand(A if a_k else A.T)
    db, ldb = operand(B.T if b_k else B)
    sam, sak = (lda, 1) if a_k else (1, lda)
    sbk, sbn = (1, ldb) if b_k else (ldb, 1)
    dc = torch.full((M + 1, N_), 7.0, dtype=torch.float32, device="cuda")
    N.check(N.load().pp_gemm_bf16(M, N_, K, D.ptr(da), sam, sak, D.ptr(db), sbk, sbn, D.ptr(dc), D.stream_handle()))
    got = dc.cpu().numpy().astype(np.float64)
    assert np.all(got[M] == 7.0)  # nothing past the result
    # exact products of BF16 values, K FP32 additions
    bound = K * 2.0 ** -24 * (np.abs(mlp.bf16(A)) @ np.abs(mlp.bf16(B)))
    assert np.all(np.abs(got[:M] - mlp.bf16(A) @ mlp.bf16(B)) <= bound + 1e-30)


def test_gemm_of_any_strides(torch):
    """A with its rows in descending order, B with every other column: read value by value."""
    from pyprop_amd import _native as N, device as D
    rng = np.random.default_rng(0)
    M, N_, K = 70, 66, 72
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, 2 * N_)).astype(np.float32)
    da, db = (torch.from_numpy(x).to("cuda").to(torch.bfloat16) for x in (A, B))
    dc = torch.empty((M, N_), dtype=torch.float32, device="cuda")
    N.check(N.load().pp_gemm_bf16(M, N_, K, da[M - 1].data_ptr(), -K, 1, D.ptr(db), 2 * N_, 2, D.ptr(dc),
                                  D.stream_handle()))
    a, b = mlp.bf16(A)[::-1], mlp.bf16(B)[:, ::2]
    assert np.all(np.abs(dc.cpu().numpy() - a @ b) <= K * 2.0 ** -24 * (np.abs(a) @ np.abs(b)))


# parameter counts with and without a remainder of two past the 16-byte groups, hidden widths whose
# matrices start at every offset the layout allows
@pytest.mark.parametrize("dims", [(1, 1, 8, 3), (5, 3, 72, 15), (3, 4, 64, 40)], ids=lambda d: "x".join(map(str, d)))
def test_adam_step_and_bf16_copies(torch, dims):
    nchan, n, hidden, rows = dims
    net, flat, x, t, chan = _case(nchan, n, hidden, rows, 4)
    inp = 2 * n * n
    dev = [torch.from_numpy(a).to("cuda") for a in (x, chan, t)]
    ref = flat.astype(np.float64)
    m, v = np.zeros_like(ref), np.zeros_like(ref)
    for step in (1, 2):
        net.train_step(*dev, 1e-2)
        mlp.adam_step(ref, net.get_grads().astype(np.float64), m, v, step, 1e-2)
        # a step of lr 1e-2 in FP32: a few ulp of the update and of the parameter
        assert np.max(np.abs(net.get_params() - ref)) < 4 * 2.0 ** -24 * (1.0 + np.max(np.abs(ref)))
        ref = net.get_params().astype(np.float64)
    # the next forward pass multiplies with the updated weights, rounded to BF16
    y = net.forward(dev[0], dev[1]).cpu().numpy().astype(np.float64)
    y_ref, _ = mlp.forward(mlp.unpack(ref, inp, hidden, nchan), x, chan)
    assert _rel(y, y_ref) < 1e-4  # one BF16 boundary case in thousands of activations
