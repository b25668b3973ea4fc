"""The GEMM kernels behind the dispatch's size rules: the small-product kernel (k
split over a block's waves), the 64 x 64 tile and the 4-byte loads of operands
that are not 16-byte granular, at tile edges, remainders and both ends of their
ranges, in every layout, against a float64 product twice: operands of small whole
numbers, where every order of the sums is exact and the results must be equal (a
lost or doubled term is at least 1), and normal ones under the worst case of a
sum of K products, K u |A||B| (u the unit roundoff, eps = 2 u: the other half
covers the float64 reference's own sum)."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

LAYOUTS = [(True, False), (True, True), (False, False), (False, True)]


def _draw(rng, shape, dt, whole):
    """Normal numbers, or whole ones of -8 to 8 without 0 (sums of up to 2^18
    products, and of as many terms, are exact in either type)."""
    if whole:
        return (rng.integers(1, 9, shape) * rng.choice([-1, 1], shape)).astype(dt)
    return rng.standard_normal(shape).astype(dt)


def _operands(dt, M, N, K, akc, bkc, seed, whole=False):
    rng = np.random.default_rng(seed)
    A = _draw(rng, (M, K) if akc else (K, M), dt, whole)
    B = _draw(rng, (N, K) if bkc else (K, N), dt, whole)
    a = (A if akc else A.T).astype(np.float64)
    b = (B.T if bkc else B).astype(a.dtype)
    return A, B, a, b


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("M,N,K", [
    (1, 1, 1), (33, 31, 7), (32, 64, 32), (512, 128, 128), (128, 384, 511), (201, 65, 385),  # small products
    (257, 259, 261), (320, 512, 300), (300, 700, 2050),  # 64 x 64 tiles, with and without splits and folds
    (1031, 1029, 515),  # odd in every dimension
])
def test_gemm_plans_against_reference(dev, dt, akc, bkc, M, N, K):
    from dtmi import device as D, kernels as K_
    for whole in (True, False):
        A, B, a, b = _operands(dt, M, N, K, akc, bkc, M * 7 + N * 3 + K, whole)
        bias = _draw(np.random.default_rng(1), N, dt, whole)
        got = K_.gemm(D.from_numpy(A), D.from_numpy(B), a_kcontig=akc, b_kcontig=bkc, bias=D.from_numpy(bias)).numpy()
        if whole:
            assert np.array_equal(got, a @ b + bias)
        else:
            bound = np.finfo(dt).eps * (K * (np.abs(a) @ np.abs(b)) + np.abs(bias))
            assert np.all(np.abs(got - (a @ b + bias)) <= bound)


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("M,N,K,splits", [(512, 128, 128, 1), (512, 128, 512, 2), (96, 65, 200, 1), (65, 2000, 777, 3),
                                          (1000, 130, 1920, 7), (250, 1030, 515, 2)])
def test_small_float32_products_keep_the_wide_tiles_bits(dev, akc, bkc, M, N, K, splits):
    """A float32 product with a dimension of at most 256 gives the bits of the
    128-wide tiles at their own split of k, whichever kernel takes it."""
    from dtmi import device as D, kernels as K_
    A, B, _, _ = _operands(np.float32, M, N, K, akc, bkc, K)
    da, db = D.from_numpy(A), D.from_numpy(B)
    got = K_.gemm(da, db, a_kcontig=akc, b_kcontig=bkc).numpy()
    assert bits_equal(got, K_.gemm(da, db, a_kcontig=akc, b_kcontig=bkc, splits=splits).numpy())


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("M,K,N", [(512, 128, 384), (77, 33, 65), (1000, 256, 768), (2495, 300, 513)])
def test_linear_backward_column_sums_and_epilogues(dev, dt, M, K, N):
    """dW, db and dX, and the fused forward epilogues, through the small plans."""
    from dtmi import device as D, kernels as K_
    rng = np.random.default_rng(M + N)
    x, w, g, b, r = (_draw(rng, s, dt, True) for s in ((M, K), (K, N), (M, N), (N,), (M, N)))
    dx, dw, db = K_.linear_bwd(D.from_numpy(x), D.from_numpy(w), D.from_numpy(g))
    assert np.array_equal(dx.numpy(), g @ w.T) and np.array_equal(dw.numpy(), x.T @ g)
    assert np.array_equal(db.numpy(), g.sum(axis=0))
    y, _ = K_.linear_fwd_fused(D.from_numpy(x), D.from_numpy(w), D.from_numpy(b), residual=D.from_numpy(r))
    assert np.array_equal(y.numpy(), x @ w + b + r)
    x, w, g = (rng.standard_normal(s).astype(dt) for s in ((M, K), (K, N), (M, N)))
    b, r = rng.standard_normal(N).astype(dt), rng.standard_normal((M, N)).astype(dt)
    X, W, G = (v.astype(np.float64) for v in (x, w, g))
    eps = np.finfo(dt).eps
    dx, dw, db = K_.linear_bwd(D.from_numpy(x), D.from_numpy(w), D.from_numpy(g))
    assert np.all(np.abs(dx.numpy() - G @ W.T) <= eps * N * (np.abs(G) @ np.abs(W.T)))
    assert np.all(np.abs(dw.numpy() - X.T @ G) <= eps * M * (np.abs(X.T) @ np.abs(G)))
    assert np.all(np.abs(db.numpy() - G.sum(0)) <= eps * M * np.abs(G).sum(0))
    y, _ = K_.linear_fwd_fused(D.from_numpy(x), D.from_numpy(w), D.from_numpy(b), residual=D.from_numpy(r))
    bound = eps * (K * (np.abs(X) @ np.abs(W)) + np.abs(b) + 2 * np.abs(r))
    assert np.all(np.abs(y.numpy() - (X @ W + b + r)) <= bound)
    h, act = K_.linear_fwd_fused(D.from_numpy(x), D.from_numpy(w), D.from_numpy(b), gelu=True)
    assert bits_equal(act.numpy(), K_.gelu_fwd(h).numpy())


def _strided(a, ld):
    """`a` in HBM with rows `ld` elements apart, NaN between them."""
    from dtmi import device as D
    buf = D.full(((a.shape[0] - 1) * ld + a.shape[1],), np.nan, a.dtype)
    v = D.DeviceArray(buf.block, a.shape, a.dtype, 0, (ld, 1))
    v.assign(a)
    return v


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("akc,bkc", LAYOUTS)
@pytest.mark.parametrize("pad_a,pad_b", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_leading_dimensions_of_2_24_bytes(dev, dt, akc, bkc, pad_a, pad_b):
    """Leading dimensions beyond the direct-to-LDS kernel's 32-bit offsets take the
    register-staged kernel: 16-byte granular operands as vectors, others element
    by element, with ragged M and N, a partial last k-tile and a split of k.
    Small whole numbers, so that every order of the sums gives the exact result."""
    from dtmi import _lib, device as D
    M, N, K = 132, 68, 76
    rng = np.random.default_rng(M + pad_a + 2 * pad_b)
    A = rng.integers(-8, 9, (M, K) if akc else (K, M)).astype(dt)
    B = rng.integers(-8, 9, (N, K) if bkc else (K, N)).astype(dt)
    bias = rng.integers(-8, 9, N).astype(dt)
    ld = (1 << 24) // np.dtype(dt).itemsize
    da, db, dbias = _strided(A, ld + pad_a), _strided(B, ld + pad_b), D.from_numpy(bias)
    ref = (A if akc else A.T) @ (B.T if bkc else B) + bias
    for splits in (0, 1, 2):
        C = D.full((M, N), 7.0, dt)
        _lib.call("dtmi_gemm", _lib.dtype_code(dt), int(akc), int(bkc), M, N, K, da.ptr, ld + pad_a, 0, db.ptr,
                  ld + pad_b, 0, C.ptr, N, 0, 1, dbias.ptr, 0, splits)
        assert np.array_equal(C.numpy(), ref)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("akc,bkc", LAYOUTS)
def test_register_staged_kernel_matches_the_direct_to_lds_kernel_bitwise(dev, dt, akc, bkc):
    """The same operands with rows 2^24 bytes apart (register-staged, as vectors)
    and contiguous (direct to LDS): both feed the MFMAs the same k order, so the
    products agree to the bit (one split, ragged M and N, a partial last k-tile)."""
    from dtmi import _lib, device as D, kernels as K_
    M, N, K = 132, 68, 200
    A, B, _, _ = _operands(dt, M, N, K, akc, bkc, 5)
    ld = (1 << 24) // np.dtype(dt).itemsize
    da, db, C = _strided(A, ld), _strided(B, ld), D.empty((M, N), dt)
    _lib.call("dtmi_gemm", _lib.dtype_code(dt), int(akc), int(bkc), M, N, K, da.ptr, ld, 0, db.ptr, ld, 0, C.ptr, N, 0,
              1, None, 0, 1)
    ref = K_.gemm(D.from_numpy(A), D.from_numpy(B), a_kcontig=akc, b_kcontig=bkc, splits=1)
    assert bits_equal(C.numpy(), ref.numpy())


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("pad", [0, 1])
def test_weight_gradient_and_column_sums_of_rows_of_2_24_bytes(dev, dt, pad):
    """dW and db where a row of dY is 2^24 bytes: the register-staged kernel's
    column sums, exact on small whole numbers."""
    from dtmi import _lib, device as D
    M, K, N = 37, 4, (1 << 24) // np.dtype(dt).itemsize + pad
    rng = np.random.default_rng(N)
    x, g = (rng.integers(-8, 9, s, dtype=np.int8).astype(dt) for s in ((M, K), (M, N)))
    dx, dg, dw, db = D.from_numpy(x), D.from_numpy(g), D.empty((K, N), dt), D.empty((N,), dt)
    _lib.call("dtmi_linear_bwd_dw", _lib.dtype_code(dt), dw.ptr, db.ptr, dx.ptr, dg.ptr, M, K, N, 0)
    assert np.array_equal(dw.numpy(), x.T @ g)
    assert np.array_equal(db.numpy(), g.sum(axis=0))
