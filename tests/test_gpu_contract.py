"""pq_contract / permute / view / reshape through the C ABI on the GPU versus
the oracle's contraction (numpy tensordot in complex128).

Tolerances: ComplexF64 -- 1e-12 relative to sum_k |a||b| (the natural scale of
each output element); ComplexF32 -- 2e-6 of the same scale."""
import numpy as np
import pytest

from oracle import pq_oracle as O
from picoquant_hip import _lib

pytestmark = pytest.mark.gpu

TOL = {np.complex128: 1e-12, np.complex64: 2e-6}


@pytest.fixture(scope="module", params=[np.complex128, np.complex64], ids=["c128", "c64"])
def ctx(request):
    c = _lib.Context(request.param)
    yield c
    c.close()


def rand(rng, shape, dtype=np.complex128):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(dtype)


def check(ctx, A, ia, B, ib, got):
    want = O.contract_tensors_data(A.astype(np.complex128), ia, B.astype(np.complex128), ib)
    scale = O.contract_tensors_data(np.abs(A).astype(np.complex128), ia,
                                    np.abs(B).astype(np.complex128), ib).real
    assert got.shape == want.shape
    err = np.abs(got - want) / np.maximum(scale, 1e-300)
    assert err.max() <= TOL[ctx.np_dtype.type], err.max()


def run(ctx, A, ia, B, ib, kc=-1):
    ha, hb = ctx.upload(A), ctx.upload(B)
    ctx.set_kernel_override(kc)
    try:
        hc = ctx.contract(ha, ia, hb, ib)
    finally:
        ctx.set_kernel_override(-1)
    got = ctx.download(hc)
    for h in (ha, hb, hc):
        ctx.free(h)
    return got


def random_case(rng, max_rank=6):
    ra = int(rng.integers(0, max_rank + 1))
    rb = int(rng.integers(0, max_rank + 1))
    nc = int(rng.integers(0, min(ra, rb) + 1))
    dims_c = [int(rng.integers(1, 5)) for _ in range(nc)]
    da = [int(rng.integers(1, 5)) for _ in range(ra - nc)]
    db = [int(rng.integers(1, 5)) for _ in range(rb - nc)]
    la = list(range(1, nc + 1)) + [-(i + 1) for i in range(ra - nc)]
    lb = list(range(1, nc + 1)) + [-(ra - nc + i + 1) for i in range(rb - nc)]
    dimsA = dims_c + da
    dimsB = dims_c + db
    pa = rng.permutation(ra)
    pb = rng.permutation(rb)
    ia = [la[i] for i in pa]
    ib = [lb[i] for i in pb]
    sa = [dimsA[i] for i in pa]
    sb = [dimsB[i] for i in pb]
    return rand(rng, sa), ia, rand(rng, sb), ib


def test_random_label_patterns(ctx):
    rng = np.random.default_rng(0)
    for _ in range(60):
        A, ia, B, ib = random_case(rng)
        check(ctx, A, ia, B, ib, run(ctx, A, ia, B, ib))


@pytest.mark.parametrize("kc", [_lib.KC_GENERIC, _lib.KC_STREAM])
def test_forced_kernel_classes(ctx, kc):
    rng = np.random.default_rng(1)
    n = 0
    while n < 25:
        A, ia, B, ib = random_case(rng, 5)
        try:
            got = run(ctx, A, ia, B, ib, kc)
        except _lib.PQError as e:
            assert e.code == _lib.PQ_ERR_UNSUPPORTED
            continue
        check(ctx, A, ia, B, ib, got)
        n += 1


@pytest.mark.parametrize("pos", [0, 3, 9, 16])
def test_gate_on_state(ctx, pos):
    """One- and two-qubit gates applied to a rank-17 state (2^17 elements)."""
    rng = np.random.default_rng(pos)
    n = 17
    psi = rand(rng, (2,) * n)
    ia = [-(i + 1) for i in range(n)]
    ia[pos] = 1
    G = rand(rng, (2, 2))
    check(ctx, psi, ia, G, [1, -(n + 1)], run(ctx, psi, ia, G, [1, -(n + 1)]))
    ia2 = list(ia)
    q2 = (pos + 5) % n
    ia2[q2] = 2
    G2 = rand(rng, (2, 2, 2, 2))
    ib2 = [1, 2, -(n + 1), -(n + 2)]
    check(ctx, psi, ia2, G2, ib2, run(ctx, psi, ia2, G2, ib2))
    # small operand first: C order starts with the gate's open index
    check(ctx, G, [-1, 1], psi, [1 if i == pos else -(i + 2) for i in range(n)],
          run(ctx, G, [-1, 1], psi, [1 if i == pos else -(i + 2) for i in range(n)]))


def test_reduce_to_scalar(ctx):
    rng = np.random.default_rng(5)
    A = rand(rng, (2,) * 18)
    B = rand(rng, (2,) * 18)
    ia = list(range(1, 19))
    ib = [int(p) + 1 for p in rng.permutation(18)]      # B's axes in another order
    check(ctx, A, ia, B, ib, run(ctx, A, ia, B, ib))
    check(ctx, A, ia, B, ib, run(ctx, A, ia, B, ib, _lib.KC_REDUCE))
    # A's first/last and B's matching axes stay open: 2x2x2x2 = 16 outputs
    ia2 = [-1] + ia[1:-1] + [-2]
    ib2 = [-3 if x == 1 else (-4 if x == 18 else x) for x in ib]
    check(ctx, A, ia2, B, ib2, run(ctx, A, ia2, B, ib2))
    check(ctx, A, ia2, B, ib2, run(ctx, A, ia2, B, ib2, _lib.KC_REDUCE))


def test_dense_pair(ctx):
    """Two rank-10 tensors sharing 5 indices (GEMM-like, M=N=K=32)."""
    rng = np.random.default_rng(7)
    A = rand(rng, (2,) * 10)
    B = rand(rng, (2,) * 10)
    ia = [1, -1, 2, -2, 3, -3, 4, -4, 5, -5]
    ib = [-6, 5, -7, 4, -8, 3, -9, 2, -10, 1]
    check(ctx, A, ia, B, ib, run(ctx, A, ia, B, ib))


def test_outer_product(ctx):
    rng = np.random.default_rng(8)
    A = rand(rng, (2, 3, 2))
    B = rand(rng, (4, 2))
    check(ctx, A, [-1, -2, -3], B, [-4, -5], run(ctx, A, [-1, -2, -3], B, [-4, -5]))
    s = rand(rng, ())
    check(ctx, s, [], B, [-1, -2], run(ctx, s, [], B, [-1, -2]))


def test_permute_view_reshape(ctx):
    rng = np.random.default_rng(9)
    T = rand(rng, (2, 3, 4, 5))
    h = ctx.upload(T)
    hp = ctx.permute(h, [3, 1, 4, 2])
    np.testing.assert_array_equal(ctx.download(hp), np.transpose(T, (2, 0, 3, 1)).astype(ctx.np_dtype))
    hv = ctx.view(hp, 3, 2, 4)
    want_v = np.transpose(T, (2, 0, 3, 1))[:, :, 1:4, :].astype(ctx.np_dtype)
    np.testing.assert_array_equal(ctx.download(hv), want_v)
    # contraction straight from the strided view
    G = rand(rng, (3, 2))
    got = run_handles(ctx, hv, [-1, -2, 1, -3], ctx.upload(G), [1, -4])
    check(ctx, want_v, [-1, -2, 1, -3], G, [1, -4], got)
    ctx.reshape(hv, [4 * 2, 3 * 3])
    np.testing.assert_array_equal(ctx.download(hv), np.reshape(want_v, (8, 9), order="F"))
    assert ctx.shape(hv) == (8, 9)
    for x in (h, hp, hv):
        ctx.free(x)


def run_handles(ctx, ha, ia, hb, ib):
    hc = ctx.contract(ha, ia, hb, ib)
    out = ctx.download(hc)
    ctx.free(hc)
    ctx.free(hb)
    return out


def test_error_paths(ctx):
    rng = np.random.default_rng(10)
    h = ctx.upload(rand(rng, (2, 2)))
    with pytest.raises(KeyError):
        ctx.download(987654321)
    with pytest.raises(_lib.PQError):
        ctx.contract(h, [1, 1], h, [-1, -2])          # repeated label
    with pytest.raises(_lib.PQError):
        ctx.contract(h, [1, -1], h, [2, -2])          # summed label missing from B
    with pytest.raises(_lib.PQError):
        ctx.contract(h, [1], h, [1, -1])              # rank mismatch
    with pytest.raises(_lib.PQError):
        ctx.permute(h, [1, 1])
    with pytest.raises(_lib.PQError):
        ctx.view(h, 3, 1, 1)
    with pytest.raises(_lib.PQError):
        ctx.reshape(h, [3])
    ctx.free(h)
    with pytest.raises(KeyError):
        ctx.free(h)


@pytest.mark.parametrize("M,N", [(1, 1), (2, 1), (1, 3), (4, 4), (5, 3), (3, 5), (16, 1), (1, 9), (2, 8), (7, 2)])
@pytest.mark.parametrize("K", [65, 255, 256, 511, 512, 1000, 4096, 3 * 2 ** 12, 2 ** 17, 100003])
def test_reduce_outputs_and_extents(ctx, M, N, K):
    """Every padded output shape of the split reduction, one workgroup and
    many, summed extents around its workgroup size and not powers of two;
    summed axes in another order in B."""
    rng = np.random.default_rng(M * 100 + N + K)
    if K & (K - 1) == 0:
        q = K.bit_length() - 1
        perm = rng.permutation(q)
        A = rand(rng, [2] * q + [M], ctx.np_dtype)
        B = rand(rng, [N] + [2] * q, ctx.np_dtype)
        ia, ib = list(range(1, q + 1)) + [-1], [-2] + [int(x) + 1 for x in perm]
    else:
        A, B = rand(rng, (M, K), ctx.np_dtype), rand(rng, (K, N), ctx.np_dtype)
        ia, ib = [-1, 1], [1, -2]
    check(ctx, A, ia, B, ib, run(ctx, A, ia, B, ib, _lib.KC_REDUCE))


@pytest.mark.parametrize("K,N,k_first", [(1, 2, False), (2, 2, True), (2, 2, False), (4, 3, False), (7, 5, True),
                                         (16, 4, False), (32, 8, False), (32, 1, True)])
def test_stream_past_the_caches(ctx, K, N, k_first):
    """Operand and result together over 384 MiB (loads and stores that pass
    the caches), every K table size, lanes along and across the operand's
    lines, an odd number of open elements."""
    es = ctx.np_dtype.itemsize
    M = (400 << 20) // es // (K + N) | 1
    rng = np.random.default_rng(K * 10 + N)

    def uniform(*shape):
        r = rng.random(shape + (2,), dtype=np.float64 if es == 16 else np.float32)
        r -= 0.5
        return r.view(ctx.np_dtype)[..., 0]

    # column-major tensors: numpy's row-major shapes reversed
    X, Y = uniform(*((M, K) if k_first else (K, M))), uniform(N, K)
    hx, hy = ctx.upload(X.T), ctx.upload(Y.T)
    ctx.set_kernel_override(_lib.KC_STREAM)
    try:
        hz = ctx.contract(hx, [1, -1] if k_first else [-1, 1], hy, [1, -2])
    finally:
        ctx.set_kernel_override(-1)
    got = ctx.download(hz).T                                   # [N, M]
    for h in (hx, hy, hz):
        ctx.free(h)
    eps = 2.0 ** -53 if es == 16 else 2.0 ** -24
    y = Y.astype(np.complex128)
    for m in range(0, M, 1 << 20):
        x = X[m:m + (1 << 20)].T if k_first else X[:, m:m + (1 << 20)]
        x = x.astype(np.complex128)
        bound = (np.abs(y) @ np.abs(x)) * (2 * K + 4) * eps
        assert np.all(np.abs(got[:, m:m + (1 << 20)] - y @ x) <= bound)


@pytest.mark.parametrize("run,K,N", [(1, 2, 2), (2, 4, 4), (4, 4, 2), (4, 8, 3), (7, 4, 1), (8, 2, 5), (8, 4, 4),
                                     (15, 3, 4), (16, 4, 4), (16, 5, 2)])
def test_stream_past_the_caches_runs(ctx, run, K, N):
    """As above with the summed mode inside the operand: its first open mode
    runs over less than a line, just a line or more."""
    es = ctx.np_dtype.itemsize
    rest = (400 << 20) // es // (K + N) // run | 1
    rng = np.random.default_rng(run * 100 + K * 10 + N)
    X = rng.random((rest, K, run, 2), dtype=np.float64 if es == 16 else np.float32)
    X -= 0.5
    X = X.view(ctx.np_dtype)[..., 0]                           # column-major [run, K, rest]
    Y = rand(rng, (K, N), ctx.np_dtype)
    hx, hy = ctx.upload(X.T), ctx.upload(Y)
    ctx.set_kernel_override(_lib.KC_STREAM)
    try:
        hz = ctx.contract(hx, [-1, 1, -2], hy, [1, -3])
    finally:
        ctx.set_kernel_override(-1)
    got = ctx.download(hz).T                                   # [N, rest, run]
    for h in (hx, hy, hz):
        ctx.free(h)
    eps = 2.0 ** -53 if es == 16 else 2.0 ** -24
    y = Y.T.astype(np.complex128)
    step = max(1, (1 << 20) // run)
    for m in range(0, rest, step):
        x = X[m:m + step].transpose(1, 0, 2).reshape(K, -1).astype(np.complex128)
        bound = (np.abs(y) @ np.abs(x)) * (2 * K + 4) * eps
        assert np.all(np.abs(got[:, m:m + step].reshape(N, -1) - y @ x) <= bound)


@pytest.mark.parametrize("M,N,K", [(7, 6, (301,)), (5, 3, ()), (9, 4, (1,)), (3, 17, (2, 3)), (4, 5, (5, 2, 7)),
                                   (13, 11, (2, 2, 2, 2, 2, 2)), (300, 2, (3, 4)), (2, 3, (4, 9, 3, 5))])
@pytest.mark.parametrize("flip", [False, True])
def test_generic_sums_along_runs(ctx, M, N, K, flip):
    """The serial kernel over summed modes of every number and run length,
    in the same order in both tensors (one run) and reversed (many)."""
    rng = np.random.default_rng(M + N + sum(K))
    q = len(K)
    A = rand(rng, (M,) + K, ctx.np_dtype)
    order = list(range(q))[::-1] if flip else list(range(q))
    B = rand(rng, tuple(K[i] for i in order) + (N,), ctx.np_dtype)
    ia, ib = [-1] + [i + 1 for i in range(q)], [i + 1 for i in order] + [-2]
    check(ctx, A, ia, B, ib, run(ctx, A, ia, B, ib, _lib.KC_GENERIC))
