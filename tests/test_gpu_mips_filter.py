"""The filtered search (one-digit bounds, then exact scores of the listed
vectors) returns the full scan's results bit for bit.  The full scan takes
every search of more than 64 neighbours, so a search of k <= 64 is compared
with the first k columns of one of 65 over the same index."""

import pytest
import torch

from quashkv_amd import _native as N
from quashkv_amd.nn_search import QuashIndex

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(autouse=True, scope="module")
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a HIP device")
    N.lib()


def _same(idx, q, k):
    full_s, full_i = idx.search(q, 65)
    s, i = idx.search(q, k)
    assert torch.equal(i, full_i[:, :k])
    assert torch.equal(s.view(torch.int32), full_s[:, :k].contiguous().view(torch.int32))


# one, two and four 16-query tiles per wave and their remainders; one, two and
# four tiles per workgroup; vector counts around the 16-vector group
@pytest.mark.parametrize("d,bits,n,m,k", [
    (128, 3, 65536, 16, 10), (128, 3, 65537, 17, 1), (128, 3, 70001, 33, 64),
    (128, 3, 100015, 300, 10), (128, 2, 40000, 65, 10), (128, 4, 50003, 130, 7),
    (64, 3, 50016, 200, 10), (64, 4, 65599, 40, 32), (64, 2, 40001, 31, 5),
    (128, 3, 256, 5, 10), (64, 3, 300, 70, 64), (128, 4, 8191, 20, 64), (96, 2, 8192, 20, 9),
    (96, 3, 49999, 64, 10), (96, 4, 33333, 129, 10), (96, 2, 34567, 257, 3),
    # either side of the line below which the scan runs
    (128, 3, 699, 1, 1), (128, 3, 700, 1, 1), (64, 3, 350, 2, 2), (64, 3, 349, 2, 2),
])
def test_filter_equals_full_scan(d, bits, n, m, k):
    g = torch.Generator(device=DEV).manual_seed(n + m)
    db = torch.randn(n, d, device=DEV, generator=g)
    db *= torch.rand(n, 1, device=DEV, generator=g) + 0.5   # norms differ
    idx = QuashIndex(dim=d, bits=bits, seed=3, device=DEV)
    idx.add(db)
    q = torch.randn(m, d, device=DEV, generator=g)
    q[: m // 2] *= torch.logspace(-6, 6, m // 2, device=DEV)[:, None]
    if m > 2:
        q[m // 3, 1:] = 0.0                                  # one coordinate only
    _same(idx, q, k)


def test_queries_left_to_the_full_scan():
    """Lists that overflow (2,000 equal best vectors), zero and non-finite
    queries, infinite and NaN norms, fewer finite scores than neighbours."""
    g = torch.Generator(device=DEV).manual_seed(5)
    n, d = 65536 + 9, 128
    db = torch.randn(n, d, device=DEV, generator=g)
    q = torch.randn(80, d, device=DEV, generator=g)
    at = torch.randperm(n, device=DEV, generator=g)[:2000]
    db[at] = 3.0 * q[7]
    idx = QuashIndex(dim=d, bits=3, seed=3, device=DEV)
    idx.add(db)
    q[20] = 0.0
    q[21, 5] = float("inf")
    q[22, 5] = float("nan")
    q[23] *= 1e-35
    _same(idx, q, 10)
    _, i = idx.search(q, 10)
    assert torch.equal(i[7], at.sort().values[:10])          # ties: lower index first
    idx._norms[100:200] = float("inf")
    idx._norms[300:400] = float("nan")
    _same(idx, q, 10)
    idx._norms[:] = float("nan")
    idx._norms[40:45] = 1.0
    _same(idx, q, 10)


def test_sorted_database_and_batches():
    """Vectors sorted by score against a query, ascending (every later group
    beats the earlier ones); more queries than one batch holds."""
    g = torch.Generator(device=DEV).manual_seed(6)
    n, d = 40000, 64
    db = torch.randn(n, d, device=DEV, generator=g)
    q = torch.randn(16384 + 70, d, device=DEV, generator=g)
    db = db[(db @ q[0]).argsort()].contiguous()
    idx = QuashIndex(dim=d, bits=3, seed=3, device=DEV)
    idx.add(db)
    _same(idx, q, 10)


@pytest.mark.parametrize("bits,cent", [(3, (-1, -20, 20, 1)), (4, (-1, -40, -30, -2, 2, 30, 40, 1))])
def test_codebooks_in_any_order(bits, cent):
    g = torch.Generator(device=DEV).manual_seed(7)
    idx = QuashIndex(dim=128, bits=bits, seed=3, device=DEV)
    idx.add(torch.randn(30000, 128, device=DEV, generator=g))
    own = idx._host_tables()
    idx._host_tables = lambda: (N.HostFloats([0.03 * c for c in cent]), *own[1:])
    _same(idx, torch.randn(40, 128, device=DEV, generator=g), 10)


@pytest.mark.parametrize("size", [1e4, 1e6, 1e9])
def test_large_signs(size):
    """QJL weights whose bounds are past int32 in units of a digit."""
    g = torch.Generator(device=DEV).manual_seed(8)
    idx = QuashIndex(dim=128, bits=3, seed=3, device=DEV)
    idx.add(torch.randn(30000, 128, device=DEV, generator=g))
    idx.quantizer.S = idx.quantizer.S * size
    _same(idx, torch.randn(40, 128, device=DEV, generator=g), 10)


@pytest.mark.parametrize("d,n,m,copies,k", [
    (128, 60000, 203, 2000, 10),   # predicted from the sampled groups: never listed
    (128, 60000, 37, 1100, 10),    # past the cap by little: found while listing
    (64, 60000, 301, 5000, 64), (128, 6000, 70, 1500, 3), (96, 40000, 1, 3000, 10),
    (128, 60000, 513, 30000, 10),  # half of the vectors equal
])
def test_some_queries_left_to_the_full_scan(d, n, m, copies, k):
    """Queries of duplicated vectors among others: the full scan takes their 4-query
    chunks alone and starts from the filter's bound."""
    g = torch.Generator(device=DEV).manual_seed(n + m)
    db = torch.randn(n, d, device=DEV, generator=g)
    q = torch.randn(m, d, device=DEV, generator=g)
    hit = torch.randperm(m, device=DEV, generator=g)[: max(1, m // 20)]
    for i, j in enumerate(hit[: max(1, n // (2 * copies))].tolist()):
        at = torch.randperm(n, device=DEV, generator=g)[:copies]
        db[at] = 2.0 * q[j]
    idx = QuashIndex(dim=d, bits=3, seed=3, device=DEV)
    idx.add(db)
    _same(idx, q, k)
    _same(idx, q[hit].contiguous(), k)
    _same(idx, -q, k)


def test_replays_of_a_captured_search():
    """The list of chunks left to the full scan is the replay's own: queries change
    between replays from ones that overflow to ones that do not, and back."""
    g = torch.Generator(device=DEV).manual_seed(9)
    db = torch.randn(30000, 128, device=DEV, generator=g)
    hot = torch.randn(3, 128, device=DEV, generator=g)
    db[:4000] = hot[0]
    idx = QuashIndex(dim=128, bits=3, seed=3, device=DEV)
    idx.add(db)
    plain = torch.randn(50, 128, device=DEV, generator=g)
    mixed = plain.clone()
    mixed[[0, 17, 49]] = hot[0]
    q = mixed.clone()
    idx.search(q, 10)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        s, i = idx.search(q, 10)
    for new in (mixed, plain, mixed, plain):
        q.copy_(new)
        graph.replay()
        torch.cuda.synchronize()
        got_s, got_i = s.clone(), i.clone()
        es, ei = idx.search(q, 10)
        assert torch.equal(got_i, ei) and torch.equal(got_s, es)
