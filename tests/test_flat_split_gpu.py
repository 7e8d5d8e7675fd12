"""The flat search's f16 split candidate pass against the oracle, bit for bit
(the candidates are rescored exactly and certified, so no tolerance applies):
the edges of its tiles (32, 64 and 128 queries, 128 rows, 32 dimensions), its
smallest width, slots without a row, filters, and norms at both ends of what
its scales hold."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _check(px, idx, data, metric, q, k, live=None, accept=None):
    got_i, got_d, got_c = idx.search_batch(q, k, None if accept is None else lambda i, _m: bool(accept[i]))
    with np.errstate(all="ignore"):
        want_i, want_d, want_c = orc.flat_search(orc.prepare_rows(metric, data), np.arange(data.shape[0]), metric,
                                                 orc.prepare_rows(metric, q), k, live=live, accept=accept, threads=8)
    assert np.array_equal(got_c, want_c)
    for i in range(got_c.size):
        c = int(got_c[i])
        assert np.array_equal(got_i[i, :c], want_i[i, :c]), i
        assert np.array_equal(got_d[i, :c].view(np.uint32), want_d[i, :c].view(np.uint32)), i


def _index(px, data, metric):
    idx = px.FlatIndex(px.VectorSpace(data.shape[1], metric))  # grown, not sized in advance
    half = data.shape[0] // 2
    idx.insert_batch(np.arange(half, dtype=np.uint64), data[:half])
    idx.insert_batch(np.arange(half, data.shape[0], dtype=np.uint64), data[half:])
    idx.set_search_mode(1)
    return idx


def _clustered(rng, n, dim, nq):
    centres = rng.standard_normal((20, dim))
    data = (centres[rng.integers(0, 20, n)] + 0.2 * rng.standard_normal((n, dim))).astype(np.float32)
    q = (centres[rng.integers(0, 20, nq)] + 0.2 * rng.standard_normal((nq, dim))).astype(np.float32)
    return data, q


@pytest.mark.parametrize("metric", [0, 1, 2])
@pytest.mark.parametrize("n,dim,nq,k", [
    (128, 64, 1, 1), (129, 65, 32, 10), (127, 95, 33, 3), (5000, 96, 64, 10), (5003, 127, 65, 17),
    (9001, 128, 128, 10), (8191, 129, 129, 48), (6007, 300, 31, 49), (4100, 768, 200, 100), (20_011, 100, 257, 256),
])
def test_tile_edges(gpu, metric, n, dim, nq, k):
    rng = np.random.default_rng(dim * 7 + nq + metric)
    data, q = _clustered(rng, n, dim, nq)
    idx = _index(gpu, data, metric)
    _check(gpu, idx, data, metric, q, k)
    # removed rows (the first and last of a tile among them), then a filter on top
    live = np.ones(n, np.uint8)
    for i in {0, min(127, n - 1), n - 1, *rng.integers(0, n, 20).tolist()}:
        idx.remove(int(i))
        live[i] = 0
    _check(gpu, idx, data, metric, q, k, live=live)
    _check(gpu, idx, data, metric, q, k, live=live, accept=(rng.random(n) < 0.3).astype(np.uint8))


@pytest.mark.parametrize("metric", [0, 2])
@pytest.mark.parametrize("rows,queries", [(1e17, 1.0), (1e18, 1e18), (1e-17, 1.0), (1e-19, 1e-19), (1.0, 1e25), (1.0, 1e-25)])
def test_norm_range(gpu, metric, rows, queries):
    """Norms inside, at and beyond 2^-60 .. 2^60 (1e-18 .. 1e18): beyond, the
    f32 pass or the exact scan answers."""
    rng = np.random.default_rng(17)
    data, q = _clustered(rng, 6000, 80, 40)
    data, q = (data * np.float32(rows)).astype(np.float32), (q * np.float32(queries)).astype(np.float32)
    q[3] = 0.0
    _check(gpu, _index(gpu, data, metric), data, metric, q, 10)


@pytest.mark.parametrize("k", [1, 10])
@pytest.mark.parametrize("metric,rows,queries", [
    (0, 1e-16, 1e-16), (0, 3e-17, 1e-16), (2, 1e-16, 1e-16), (2, 5e16, 1e-24), (2, 8e16, 4e-24), (2, 8e16, 2e-23),
    (0, 8e16, 1e-24),
])
def test_norm_range_inside(gpu, metric, rows, queries, k):
    """Rows inside 2^-60 .. 2^60 with queries whose factor back from the scaled
    product is at the end of f32 (1e-16 on both sides), or whose squared norm
    underflows to zero, or nearly, though they are not zero."""
    rng = np.random.default_rng(18)
    data, q = _clustered(rng, 6000, 80, 400)
    data, q = (data * np.float32(rows)).astype(np.float32), (q * np.float32(queries)).astype(np.float32)
    q[3] = 0.0
    _check(gpu, _index(gpu, data, metric), data, metric, q, k)


@pytest.mark.parametrize("metric,queries", [(0, 1e-25), (2, 1e18)])
def test_far_queries_are_certified(gpu, metric, queries):
    """Queries far below or above 2^-60 .. 2^60 against ordinary rows stay with
    the candidate pass: for the small ones, what they lose is far inside the
    Euclidean certificate."""
    rng = np.random.default_rng(19)
    data, q = _clustered(rng, 6000, 80, 400)
    q = (q * np.float32(queries)).astype(np.float32)
    idx = _index(gpu, data, metric)
    _check(gpu, idx, data, metric, q, 10)
    assert gpu.FlatIndex.last_fallbacks() == 0


@pytest.mark.parametrize("metric", [0, 1, 2])
def test_mixed_norms_and_ties(gpu, metric):
    """Rows of very different norms under one scale, and repeated rows (ties by id)."""
    rng = np.random.default_rng(23)
    data, q = _clustered(rng, 6000, 72, 70)
    data *= np.exp(rng.uniform(-9, 9, (6000, 1))).astype(np.float32)
    data[1000:1040] = data[7]
    data[3000] = 0.0
    q[:5] = data[7]
    _check(gpu, _index(gpu, data, metric), data, metric, q, 30)


@pytest.mark.parametrize("metric", [0, 1, 2])
@pytest.mark.parametrize("n,dim,nq", [(5003, 95, 20), (9001, 130, 50), (12_001, 64, 70), (8000, 768, 200)])
def test_the_split_pass_answers(gpu, metric, n, dim, nq):
    """Well separated rows of ordinary norms are answered from the candidates:
    no query goes to the exact scan, whose results would hide a pass or a
    certificate that always fails."""
    rng = np.random.default_rng(dim + metric)
    data, q = _clustered(rng, n, dim, nq)
    idx = _index(gpu, data, metric)
    _check(gpu, idx, data, metric, q, 10)
    assert gpu.FlatIndex.last_fallbacks() == 0


@pytest.mark.parametrize("nq,k,near", [(8, 10, 100), (300, 64, 100), (300, 100, 300), (800, 10, 100), (800, 256, 200),
                                       (2000, 10, 100), (2000, 100, 300)])
def test_merge_gathers_more_than_its_lds_holds(gpu, nq, k, near):
    """20,000 rows are 32 splits of 640 (5 tiles) at every batch here. The first
    tile of each, which seeds the threshold, is far off and `near` rows of the
    rest are close, few enough that no list is compacted: every one of them is
    at or below the seed threshold, 3200 to 9600 keys a query for merges that
    hold 512 to 4096, so the merge gathers again, more than once for some."""
    rng = np.random.default_rng(nq + k)
    n, dim, split = 20_000, 64, 640
    data = rng.standard_normal((n, dim))
    data /= np.linalg.norm(data, axis=1, keepdims=True)
    at = np.arange(n) % split
    norm = np.where(at < 128, 2.0, 3.0) + rng.uniform(0.0, 0.2, n)
    for a in range(0, n, split):
        rows = a + 128 + rng.permutation(min(split, n - a) - 128)[:near] if n - a > 128 else []
        norm[rows] = rng.uniform(0.9, 1.1, len(rows))
    data = (data * norm[:, None]).astype(np.float32)
    q = (0.01 * rng.standard_normal((nq, dim)) / 8.0).astype(np.float32)
    idx = _index(gpu, data, 0)
    _check(gpu, idx, data, 0, q, k)
    assert gpu.FlatIndex.last_fallbacks() <= nq // 20
