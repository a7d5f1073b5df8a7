"""pq_materialize of permuted and sliced tensors: the LDS-tiled copy (2^15
elements or more with enough factors of two) and the element-wise one, bit
for bit against numpy's transpose."""
import numpy as np
import pytest

from picoquant_hip import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[np.complex128, np.complex64], ids=["c128", "c64"])
def ctx(request):
    c = _lib.Context(request.param)
    yield c
    c.close()


def check(ctx, dims, perm, view=None):
    """view: (axis, lo, hi) of the permuted tensor, 1-based."""
    rng = np.random.default_rng(len(dims) + sum(perm[:3]))
    T = (rng.standard_normal(dims) + 1j * rng.standard_normal(dims)).astype(ctx.np_dtype)
    hs = [ctx.upload(T)]
    hs.append(ctx.permute(hs[-1], [p + 1 for p in perm]))
    want = np.transpose(T, perm)
    if view:
        ax, lo, hi = view
        hs.append(ctx.view(hs[-1], ax, lo, hi))
        want = np.take(want, range(lo - 1, hi), axis=ax - 1)
    hs.append(ctx.materialize(hs[-1]))
    assert np.array_equal(ctx.download(hs[-1]), want)
    for h in hs:
        ctx.free(h)


@pytest.mark.parametrize("n", [11, 12, 14, 15, 16, 19, 21])
@pytest.mark.parametrize("seed", range(4))
def test_qubit_permutations(ctx, n, seed):
    perm = np.random.default_rng(100 * n + seed).permutation(n).tolist()
    check(ctx, [2] * n, perm)


@pytest.mark.parametrize("dims,perm", [
    ([2] * 17, list(range(16, -1, -1))),                      # full reversal
    ([2] * 17, [16] + list(range(16))),                       # one axis to the front
    ([2] * 17, list(range(1, 17)) + [0]),
    ([2] * 17, [1, 0] + list(range(2, 17))),                  # long common runs after the swap
    ([512, 512], [1, 0]), ([4096, 16], [1, 0]), ([16, 4096], [1, 0]), ([96, 64, 40], [2, 0, 1]),
    ([6, 20, 12, 28, 4], [4, 2, 0, 3, 1]),                    # odd parts in every mode
    ([3, 2 ** 14], [1, 0]), ([2 ** 14, 3], [1, 0]), ([5, 7, 2 ** 11], [2, 1, 0]),
    ([37, 45, 33], [2, 0, 1]), ([243, 243], [1, 0]),          # no factors of two
    ([32, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2], [0, 10, 9, 8, 7, 6, 5, 4, 3, 2, 1]),
    ([16, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2, 2], [0, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2, 1])])
def test_mixed_extents(ctx, dims, perm):
    check(ctx, dims, perm)


@pytest.mark.parametrize("axis", [1, 4, 9])
def test_sliced_views(ctx, axis):
    """A slice of a permuted tensor: strides with a hole, an odd offset."""
    dims = [3] + [2] * 16
    perm = np.random.default_rng(axis).permutation(17).tolist()
    where = perm.index(0) + 1
    check(ctx, dims, perm, (where, 2, 3))
    check(ctx, dims, perm, (where, 2, 2))
    other = axis if axis != where else axis + 1
    check(ctx, dims, perm, (other, 2, 2))


def test_past_the_caches(ctx):
    """Tensor and copy together over 384 MiB (stores that pass the caches),
    an odd factor among the extents."""
    dims = [2] * 22 + ([5] if ctx.np_dtype == np.complex128 else [2, 5])
    check(ctx, dims, np.random.default_rng(len(dims)).permutation(len(dims)).tolist())


@pytest.mark.parametrize("dims,perm", [
    ([31, 2048, 32], [0, 2, 1]), ([2048, 1025], [1, 0]), ([1025, 2048], [1, 0]),    # an odd extent fastest
    ([64, 64, 64, 7], [3, 0, 1, 2]), ([9, 512, 3, 128], [0, 2, 1, 3]),
    ([64, 3, 64, 3, 64], [1, 4, 3, 0, 2]), ([48, 48, 48, 20], [3, 2, 1, 0]), ([7, 64, 64, 64], [3, 2, 1, 0]),
    ([3, 1024, 512], [2, 1, 0]), ([12, 24, 36, 16, 8], [4, 2, 0, 3, 1]), ([16, 65536, 2], [1, 0, 2]),
    ([24, 2048, 32], [0, 2, 1]), ([2] * 9 + [3] + [2] * 11, [20, 3, 1, 19, 9, 0, 18, 2, 17, 4, 16, 5, 15, 6, 14, 7, 13, 8, 12, 10, 11]),
    ([2] * 21, [0, 1, 2, 3] + list(range(20, 3, -1))), ([128, 2, 31, 96, 3], [2, 1, 4, 3, 0])])
def test_odd_extents_beside_factors_of_two(ctx, dims, perm):
    """Copies over the size where tiles begin, whose odd extents keep them out
    of tiles or run beside them, and a slice of each."""
    check(ctx, dims, perm)
    n = dims[perm[0]]
    check(ctx, dims, perm, (1, n // 2 + 1, n))
