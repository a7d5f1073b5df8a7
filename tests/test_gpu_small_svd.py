"""pq_decompose on the one-workgroup SVD (shorter side at most 64) against
numpy's SVD in complex128: the bond dimension, the split's product (the
truncated matrix), the factors' norms (sqrt of the singular values) and
orthogonality, over padded sizes (4, 8, 16, 32, 64 columns; 16 to 256 rows)
and their edges, tall and wide, graded and rank-deficient spectra, strided
tensors.

Tolerance: a column passes at most about 10 sweeps x 63 rotations, each
rounding at most 4 eps of the matrix norm: 2.8e-13 for complex128, 1.5e-4
for complex64 (both relative to the largest singular value)."""
import numpy as np
import pytest

from picoquant_hip import _lib

pytestmark = pytest.mark.gpu

TOL = {np.complex128: 2.8e-13, np.complex64: 1.5e-4}


@pytest.fixture(scope="module", params=[np.complex128, np.complex64], ids=["c128", "c64"])
def ctx(request):
    c = _lib.Context(request.param)
    yield c
    c.close()


def rnd(rng, m, n):
    return rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))


def graded(rng, m, n, digits):
    k = min(m, n)
    u, w = np.linalg.qr(rnd(rng, m, k))[0], np.linalg.qr(rnd(rng, n, k))[0]
    return (u * np.logspace(0, -digits, k)) @ w.conj().T


def check(ctx, A, B, C, chi, threshold=0.0, max_rank=0):
    tol = TOL[ctx.np_dtype.type]
    u, s, vh = np.linalg.svd(A)
    thr = max(threshold, np.sqrt(np.finfo(ctx.np_dtype).eps))
    rel = s / np.linalg.norm(s)
    want = int(np.sum(rel > thr))
    sure = int(np.sum(rel > thr + 4 * tol))          # values at the cut-off may fall either way
    maybe = int(np.sum(rel > thr - 4 * tol))
    if max_rank > 0:
        want, sure, maybe = (min(x, max_rank) for x in (want, sure, maybe))
    assert sure <= chi <= maybe, (chi, want)
    assert B.shape == (A.shape[0], chi) and C.shape == (chi, A.shape[1])
    trunc = (u[:, :chi] * s[:chi]) @ vh[:chi]
    gap = s[chi - 1] - s[chi] if chi < len(s) else s[chi - 1]
    # a truncated product is defined up to tol x norm / gap
    assert np.linalg.norm(B @ C - trunc) <= tol * s[0] * max(1.0, s[0] / max(gap, 1e-300) if chi < len(s) else 1.0)
    assert np.all(np.abs(np.sum(np.abs(B) ** 2, axis=0) - s[:chi]) <= tol * s[0])
    assert np.all(np.abs(np.sum(np.abs(C) ** 2, axis=1) - s[:chi]) <= tol * s[0])
    for g in (B.conj().T @ B, C @ C.conj().T):
        assert np.max(np.abs(g - np.diag(s[:chi]))) <= tol * s[0]


def split(ctx, A, threshold=0.0, max_rank=0):
    h = ctx.upload(A.astype(ctx.np_dtype))
    hb, hc, chi = ctx.decompose(h, [1], [2], threshold, max_rank)
    B, C = ctx.download(hb), ctx.download(hc)
    for x in (h, hb, hc):
        ctx.free(x)
    return B.astype(np.complex128), C.astype(np.complex128), chi


SHAPES = [(1, 1), (1, 7), (9, 1), (2, 2), (4, 4), (5, 4), (4, 16), (8, 8), (9, 8), (16, 16), (17, 16), (8, 32),
          (32, 8), (31, 33), (32, 32), (65, 32), (128, 16), (129, 16), (256, 4), (3, 256), (257, 4), (48, 48), (64, 33),
          (64, 64), (63, 64), (65, 64), (70, 66)]


@pytest.mark.parametrize("m,n", SHAPES)
def test_shapes(ctx, m, n):
    A = rnd(np.random.default_rng(1000 * m + n), m, n).astype(ctx.np_dtype).astype(np.complex128)
    check(ctx, A, *split(ctx, A))
    if min(m, n) > 2:
        r = min(m, n) // 2
        check(ctx, A, *split(ctx, A, max_rank=r), max_rank=r)


@pytest.mark.parametrize("m,n", [(4, 4), (8, 6), (24, 16), (20, 32), (64, 64), (100, 20)])
@pytest.mark.parametrize("digits", [3, 12, 20])
def test_graded_spectra(ctx, m, n, digits):
    """Singular values falling over `digits` decades, far below the cut-off."""
    A = graded(np.random.default_rng(m + n + digits), m, n, digits).astype(ctx.np_dtype).astype(np.complex128)
    check(ctx, A, *split(ctx, A))
    check(ctx, A, *split(ctx, A, threshold=1e-2), threshold=1e-2)


def test_rank_deficient_degenerate_and_scaled(ctx):
    rng = np.random.default_rng(5)
    low = rnd(rng, 40, 6) @ rnd(rng, 6, 30)
    unit = np.linalg.qr(rnd(rng, 32, 32))[0]            # every singular value 1
    sparse = np.zeros((16, 16), complex)
    sparse[3, 5], sparse[7, 5], sparse[3, 11] = 2, 1j, -1
    for A in (low, unit, sparse, np.eye(64), 1e-30 * rnd(rng, 12, 20), 1e30 * rnd(rng, 64, 40)):
        A = A.astype(ctx.np_dtype).astype(np.complex128)
        check(ctx, A, *split(ctx, A))
    with pytest.raises(_lib.PQError) as e:
        split(ctx, np.zeros((16, 8)))
    assert e.value.code == _lib.PQ_ERR_UNSUPPORTED


def test_strided_tensor(ctx):
    """A permuted, sliced rank-5 tensor split across its axes."""
    rng = np.random.default_rng(6)
    T = (rng.standard_normal((3, 4, 2, 5, 4)) + 1j * rng.standard_normal((3, 4, 2, 5, 4)))
    T = T.astype(ctx.np_dtype).astype(np.complex128)
    h = ctx.upload(T.astype(ctx.np_dtype))
    hp = ctx.permute(h, [4, 1, 5, 3, 2])
    hv = ctx.view(hp, 1, 2, 4)
    ref = np.transpose(T, (3, 0, 4, 2, 1))[1:4]
    hb, hc, chi = ctx.decompose(hv, [2, 5], [4, 1, 3])
    B, C = ctx.download(hb), ctx.download(hc)
    assert B.shape == (3, 4, chi) and C.shape == (chi, 2, 3, 4)
    A = np.transpose(ref, (1, 4, 3, 0, 2)).reshape(12, 24, order="F")
    check(ctx, A, B.reshape(12, chi, order="F"), C.reshape(chi, 24, order="F"), chi)
    assert np.array_equal(ctx.download(h), T.astype(ctx.np_dtype))       # not consumed
    for x in (h, hp, hv, hb, hc):
        ctx.free(x)


@pytest.mark.parametrize("wide", [False, True], ids=["tall", "wide"])
@pytest.mark.parametrize("m,n,col", [(4, 2, 0), (4, 3, 0), (4, 4, 1), (6, 5, 2), (33, 20, 7)])
def test_nearly_zero_columns(ctx, m, n, col, wide):
    """A column of the size of a rounding error (cos(pi/2) = 6e-17 in a gate)
    in front of columns of ordinary size, over the scales where its square
    leaves the type's range, its diagonal element as large as the rest,
    smaller or zero.  With `col` > 0 the columns before it only touch the
    rows above, so the reflections before it leave it as it is."""
    rng = np.random.default_rng(10 * m + n)
    lo, hi = (1e-21, 1e-7) if ctx.np_dtype == np.complex64 else (1e-146, 1e-125)
    for scale in np.geomspace(lo, hi, 57):
        for diag in (1.0, 0.3, 1e-2, 1e-6, 0.0):
            A = rnd(rng, m, n)
            A[col:, :col] = 0
            A[:, col] *= scale
            A[:col, col] = 0
            A[col, col] *= diag
            A = A.astype(ctx.np_dtype).astype(np.complex128)
            A = A.T if wide else A
            check(ctx, A, *split(ctx, A))


@pytest.mark.parametrize("g", [7.7e-20, 8.2e-20, 9e-20, 1e-19, 1.07e-19, 1.2e-19, 5e-19])
def test_columns_with_a_subnormal_inner_product(ctx, g):
    """Two columns far below the cut-off whose inner product's square is
    subnormal in complex64: one singular value is left, and the split stays
    on the kernel -- the library's path starts with a copy of the tensor,
    which the profile counts."""
    b = np.sqrt(g)
    A = np.array([[0.5, 0, 0], [0, b, b], [0, 0, b]], dtype=complex)
    ctx.profile_enable(True)
    B, C, chi = split(ctx, A)
    copies = ctx.profile_read(_lib.KC_COPY)["launches"]
    ctx.profile_enable(False)
    assert copies == 0
    assert chi == 1
    assert np.allclose(B @ C, np.diag([0.5, 0, 0]), rtol=0, atol=1e-7)


@pytest.mark.parametrize("wide", [False, True], ids=["tall", "wide"])
@pytest.mark.parametrize("m,n,zero", [(4, 4, [3]), (4, 4, [0]), (6, 4, [1, 2]), (16, 9, [0, 8]), (40, 33, [5, 32]),
                                      (5, 1, []), (1, 1, [])])
def test_zero_columns(ctx, m, n, zero, wide):
    """Columns that are zero, or zero below the diagonal: split by the
    kernel itself (the library's path starts with a copy)."""
    rng = np.random.default_rng(m + n)
    for tail in (False, True):
        A = rnd(rng, m, n)
        A[:, zero] = 0
        if tail:
            A = np.triu(A)
        A = A.astype(ctx.np_dtype).astype(np.complex128)
        A = A.T if wide else A
        ctx.profile_enable(True)
        got = split(ctx, A)
        copies = ctx.profile_read(_lib.KC_COPY)["launches"]
        ctx.profile_enable(False)
        assert copies == 0
        check(ctx, A, *got)


def rounding_bound(n):
    """Relative error of a split of n columns, in units of the roundoff u, if
    every rotation and every reflection rounds an element once: at most 8
    sweeps of n - 1 rotations on V Sigma and on U, 2 n reflections on U and R
    and four more operations (scaling both factors), independent errors
    uniform in +-u."""
    return np.sqrt((2 * 8 * (n - 1) + 2 * n + 4) / 3)


@pytest.mark.parametrize("m,n", [(8, 8), (16, 16), (20, 48), (64, 32), (32, 32), (64, 64)])
def test_errors_grow_as_one_rounding_per_rotation(ctx, m, n):
    """rms over matrices of |A - B C| / |A| in extended precision."""
    rng = np.random.default_rng(m + n)
    k, sq = min(m, n), []
    for _ in range(max(4, 8192 // (m * n))):
        u, w = np.linalg.qr(rnd(rng, m, k))[0], np.linalg.qr(rnd(rng, n, k))[0]
        A = ((u * np.linspace(1, 0.1, k)) @ w.conj().T).astype(ctx.np_dtype).astype(np.clongdouble)
        B, C, chi = split(ctx, A)
        assert chi == k
        d = (A - B.astype(np.clongdouble) @ C.astype(np.clongdouble)).astype(np.complex128)
        sq.append((np.linalg.norm(d) / np.linalg.norm(A.astype(np.complex128))) ** 2)
    assert np.sqrt(np.mean(sq)) <= rounding_bound(k) * np.finfo(ctx.np_dtype).eps / 2


@pytest.mark.parametrize("m,n", [(4, 4), (12, 16), (32, 32), (64, 40), (64, 64)])
def test_bond_dimension_beside_the_cutoff(ctx, m, n):
    """Half the singular values lie beside the cut-off, in turn above and
    below by twice four times the rounding error of a split: chi counts
    exactly those above."""
    rng = np.random.default_rng(7 * m + n)
    k, eps = min(m, n), np.finfo(ctx.np_dtype).eps
    cut = np.sqrt(eps)
    near = 4 * rounding_bound(k) * eps / 2 / cut             # relative to the cut-off
    s = np.linspace(1, 0.1, k)
    head = k // 2
    s[head:] = cut * np.linalg.norm(s[:head]) * (1 + 2 * near * np.where(np.arange(k - head) % 2, -1, 1))
    u, w = np.linalg.qr(rnd(rng, m, k))[0], np.linalg.qr(rnd(rng, n, k))[0]
    A = ((u * s) @ w.conj().T).astype(ctx.np_dtype).astype(np.complex128)
    rel = np.linalg.svd(A, compute_uv=False)
    rel /= np.linalg.norm(rel) * cut
    assert np.all(np.abs(rel - 1) > near)                    # the input's own rounding moved none across
    assert split(ctx, A)[2] == int(np.sum(rel > 1))


@pytest.mark.parametrize("shorter,longer", [(1, (255, 127)), (4, (252, 124)), (5, (256, 251)), (8, (256, 248)),
                                            (9, (256, 256)), (32, (256, 256)), (33, (128, 256)), (44, (128, 256)),
                                            (45, (64, 256)), (60, (64, 256)), (61, (64, 128)), (64, (64, 128))])
def test_size_rule(ctx, shorter, longer):
    """The longest matrix (complex128, complex64) that the kernel takes, and
    one row or column more, which the library takes (its path starts with a
    copy, which the profile counts)."""
    rng = np.random.default_rng(shorter)
    most = longer[0 if ctx.np_dtype == np.complex128 else 1]
    for m, n, copied in ((most, shorter, 0), (shorter, most, 0), (most + 1, shorter, 1), (shorter, most + 1, 1)):
        A = rnd(rng, m, n).astype(ctx.np_dtype).astype(np.complex128)
        ctx.profile_enable(True)
        got = split(ctx, A)
        copies = ctx.profile_read(_lib.KC_COPY)["launches"]
        ctx.profile_enable(False)
        assert copies == copied, (m, n)
        check(ctx, A, *got)
