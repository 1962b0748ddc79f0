"""Two-stage exact top-k over the 16-bit fixed-point index (csrc/ops/similarity_q16.hip) on
the GPU against the CPU reference (ops.reference.q16_topk: exact int64 dot products, the same
float64 -> float32 step): identical rows and bit-identical scores, on random and planted sets,
with the priority / tag / expiry filters, one and many slices, and the exact-scan fallback."""
import pytest
import torch

from pilottai_amd import ops
from pilottai_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _index(N, D, gpu, seed=0, planted=None):
    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.randn(N, D, device=gpu, generator=g)
    if planted is not None:
        for row, q in planted:
            x[row] = q + 0.05 * torch.randn(D, device=gpu, generator=g)
    x = torch.nn.functional.normalize(x, dim=1)
    pad = (-N) % 16
    hi, lo, sc, bd = ops.q16_quantize(torch.cat([x, torch.zeros(pad, D, device=gpu)]) if pad else x)
    rmeta = torch.stack([sc, bd], 1).contiguous()
    return ops.q16_pack(hi).contiguous(), ops.q16_pack(lo).contiguous(), rmeta


def _filters(N, Q, gpu, on):
    prio = (torch.arange(N, device=gpu) % 4).to(torch.int32)
    tags = torch.where(torch.arange(N, device=gpu) % 2 == 0, 1, 2).to(torch.int64)
    exp = torch.zeros(N, device=gpu)
    if on:
        exp[torch.arange(N, device=gpu) % 10 == 5] = 1.0  # expired at now = 2
    minp = torch.tensor([(i % 3) if on else 0 for i in range(Q)], dtype=torch.int32, device=gpu)
    qtags = torch.tensor([(1 if i % 4 == 1 else 2 if i % 4 == 3 else 0) if on else 0 for i in range(Q)],
                         dtype=torch.int64, device=gpu)
    return prio, tags, exp, minp, qtags


def _check(gpu, N, D, Q, K, filters, exact=False, seed=0, planted=False):
    g = torch.Generator(device=gpu).manual_seed(seed + 1)
    q = torch.nn.functional.normalize(torch.randn(Q, D, device=gpu, generator=g), dim=1)
    pl = [(int((i * 7919 + 13) % N), q[i]) for i in range(Q)] if planted else None
    hi, lo, rmeta = _index(N, D, gpu, seed, pl)
    prio, tags, exp, minp, qtags = _filters(N, Q, gpu, filters)
    stats = {}
    s, r = ops.q16_topk(q, hi, lo, rmeta, N, K, prio, tags, exp, minp, qtags, 2.0, exact=exact, stats=stats)
    torch.cuda.synchronize()
    qv, qm = ops.q16_queries(q)
    rs, rr = ref.q16_topk(qv.cpu(), qm.cpu(), hi.cpu(), lo.cpu(), rmeta.cpu(), N, K, prio.cpu(), tags.cpu(),
                          exp.cpu(), minp.cpu(), qtags.cpu(), 2.0)
    assert torch.equal(r.cpu(), rr), (r.cpu()[:2], rr[:2])
    assert torch.equal(s.cpu(), rs)
    if planted and not filters:
        assert all(int(r[i, 0]) == pl[i][0] for i in range(Q))
    return stats


@pytest.mark.parametrize("N,D,Q,K,filters", [
    (500, 1024, 1, 1, False), (3000, 1024, 13, 5, True), (50_000, 1024, 64, 64, True),
    (300_000, 1024, 64, 5, False), (300_000, 256, 7, 20, True), (70_001, 512, 33, 3, True)])
def test_q16_two_stage_matches_exact_reference(gpu, N, D, Q, K, filters):
    st = _check(gpu, N, D, Q, K, filters)
    assert st.get("q16_fallbacks", 0) == 0  # random unit vectors: the drop check never fires


@pytest.mark.parametrize("K", [1, 5, 32, 64])
@pytest.mark.parametrize("N", [40, 64, 65, 250, 1000, 2000, 4100, 16_000, 16_500, 20_011])  # lists of 64 in slices of 256 rows
def test_q16_lists_of_any_length(gpu, N, K):
    """Around the lines between the selections of the second stage: up to 64, 256, 1,024 and 4,096 listed entries, and 64 re-ranked."""
    _check(gpu, N, 256, 3, K, N % 2 == 1, seed=K)


@pytest.mark.parametrize("N,Q,K", [(20_000, 16, 5), (200_000, 64, 10)])
def test_q16_exact_scan_matches_reference(gpu, N, Q, K):
    _check(gpu, N, 1024, Q, K, True, exact=True, seed=5)


@pytest.mark.parametrize("N,D,Q,K,filters", [
    (255, 64, 3, 64, False), (257, 192, 2, 7, True),  # one slice, two slices
    (65_536 + 31, 256, 64, 33, True), (2 * 65_536, 256, 64, 64, False),  # slices of two rounds, which share bounds
    (2 * 65_536 + 1, 256, 64, 1, True), (600_011, 256, 5, 64, True)])
def test_q16_slices_and_shared_bounds(gpu, N, D, Q, K, filters):
    _check(gpu, N, D, Q, K, filters, seed=11)


@pytest.mark.parametrize("N,D,Q,K", [  # one tile of queries and two, whole steps of dimensions and padded ones, slices of one round
    (65_536, 512, 32, 64), (65_537, 448, 33, 1), (66_000, 1024, 1, 16), (131_073, 960, 64, 8), (400_000, 192, 32, 17),
    (300_000, 128, 33, 64)])  # (whose first round fills buffers)
def test_q16_tiles_of_queries(gpu, N, D, Q, K):
    _check(gpu, N, D, Q, K, True, seed=3)


@pytest.mark.parametrize("N,D,Q,K", [(3_000, 128, 64, 5), (70_000, 64, 40, 64), (140_000, 128, 3, 20)])
def test_q16_rows_in_rising_order(gpu, N, D, Q, K):
    """Every row is nearer to the queries than the one before: each round admits all of its rows, and the waves ask for
    compactions all the time."""
    g = torch.Generator(device=gpu).manual_seed(N)
    q = torch.nn.functional.normalize(torch.randn(1, D, device=gpu, generator=g), dim=1)
    x = torch.nn.functional.normalize(torch.randn(N, D, device=gpu, generator=g), dim=1) + torch.linspace(0, 2, N, device=gpu)[:, None] * q
    pad = (-N) % 16
    x = torch.cat([torch.nn.functional.normalize(x, dim=1), torch.zeros(pad, D, device=gpu)])
    hi, lo, sc, bd = ops.q16_quantize(x)
    hi, lo, rmeta = ops.q16_pack(hi).contiguous(), ops.q16_pack(lo).contiguous(), torch.stack([sc, bd], 1).contiguous()
    qs = torch.nn.functional.normalize(q + 0.02 * torch.randn(Q, D, device=gpu, generator=g), dim=1)
    filters = _filters(N, Q, gpu, True)
    s, r = ops.q16_topk(qs, hi, lo, rmeta, N, K, *filters, 2.0)
    qv, qm = ops.q16_queries(qs)
    rs, rr = ref.q16_topk(qv.cpu(), qm.cpu(), hi.cpu(), lo.cpu(), rmeta.cpu(), N, K, *(f.cpu() for f in filters), 2.0)
    assert torch.equal(r.cpu(), rr) and torch.equal(s.cpu(), rs)


def test_q16_fewer_hits_than_k(gpu):
    """Rows that pass the filters are fewer than K, and lie in few slices."""
    N, D, Q, K = 200_000, 256, 3, 9
    hi, lo, rmeta = _index(N, D, gpu, 4)
    prio = torch.zeros(N, dtype=torch.int32, device=gpu)
    prio[[5, 70_000, 199_999]] = 7
    tags, exp = torch.zeros(N, dtype=torch.int64, device=gpu), torch.zeros(N, device=gpu)
    minp = torch.full((Q,), 7, dtype=torch.int32, device=gpu)
    q = torch.randn(Q, D, device=gpu)
    s, r = ops.q16_topk(q, hi, lo, rmeta, N, K, prio, tags, exp, minp, torch.zeros_like(minp, dtype=torch.int64), 0.0)
    assert (r[:, 3:] == -1).all() and bool((s[:, 3:] == -float("inf")).all())
    assert all(sorted(x[:3]) == [5, 70_000, 199_999] for x in r.tolist())


@pytest.mark.parametrize("Q,D", [(1, 64), (64, 1024), (5, 320)])
def test_query_preparation_matches_torch(gpu, Q, D):
    """The kernel's queries against the CPU's at several shapes, and against torch's normalised rows: bf16's rounding."""
    q = torch.randn(Q, D, device=gpu) * 3.0
    q[0, 1:] = 0.0
    if Q > 2:
        q[2] = 0.0
    qv, qm = ops.q16_queries(q)
    rv, rm = ops.q16_queries(q.cpu())
    assert torch.equal(qv.cpu(), rv) and torch.equal(qm.cpu(), rm)
    qv, qm = ops.q16_queries(q, normalize=True)
    rv, rm = ops.q16_queries(q.cpu(), normalize=True)
    whole = lambda v: 256 * v[:, 0].int() + v[:, 1].int()  # noqa: E731
    assert int((whole(qv.cpu()) - whole(rv)).abs().max()) <= 1
    assert torch.allclose(qm.cpu(), rm, rtol=4 * 2.0 ** -24, atol=0)
    u = torch.nn.functional.normalize(q.cpu(), dim=1)
    assert (ops.unit_queries(q).cpu().float() - u).abs().max() <= 2.0 ** -8 * u.abs().max()


@pytest.mark.parametrize("normalize", [False, True])
def test_query_preparation_has_the_bits_of_the_cpu(gpu, normalize):
    """Both forms of a query, bit for bit; zeros, tiny and huge values, NaN and infinities among them."""
    q = torch.randn(40, 512, generator=torch.Generator().manual_seed(2)) * torch.logspace(-18, 17, 40)[:, None]
    q[3], q[5, 7], q[6, 100], q[8, 5:9], q[9] = 0.0, float("nan"), float("inf"), -float("inf"), float("nan")
    bits = lambda t: t.contiguous().cpu().view(torch.int32)  # noqa: E731
    nan = lambda t: torch.where(torch.isnan(t), torch.full_like(t, 7.0), t)  # noqa: E731  (whichever NaN)
    qv, qm = ops.q16_queries(q.to(gpu), normalize=normalize)
    rv, rm = ops.q16_queries(q, normalize=normalize)
    assert torch.equal(qv.cpu(), rv) and torch.equal(bits(nan(qm)), bits(nan(rm)))
    if normalize:
        assert torch.equal(bits(nan(ops.unit_queries(q.to(gpu)).cpu().float())), bits(nan(ops.unit_queries(q).float())))


def test_q16_planted_neighbours_found(gpu):
    _check(gpu, 400_000, 1024, 32, 5, False, seed=7, planted=True)


def test_q16_fallback_on_ties(gpu):
    """Every row the same vector: every slice's list is full of equal upper bounds, the drop
    check fires, and the exact scan answers (same scores as the reference; rows are ties)."""
    N, D, Q, K = 40_000, 1024, 4, 5
    base = torch.nn.functional.normalize(torch.randn(1, D, device=gpu), dim=1).expand(N, D).contiguous()
    hi, lo, sc, bd = ops.q16_quantize(base)
    hi, lo, rmeta = ops.q16_pack(hi), ops.q16_pack(lo), torch.stack([sc, bd], 1).contiguous()
    prio, tags, exp, minp, qtags = _filters(N, Q, gpu, False)
    q = torch.nn.functional.normalize(base[:Q] + 0.01 * torch.randn(Q, D, device=gpu), dim=1)
    stats = {}
    s, r = ops.q16_topk(q, hi, lo, rmeta, N, K, prio, tags, exp, minp, qtags, 2.0, stats=stats)
    qv, qm = ops.q16_queries(q)
    rs, _ = ref.q16_topk(qv.cpu(), qm.cpu(), hi.cpu(), lo.cpu(), rmeta.cpu(), N, K, prio.cpu(), tags.cpu(),
                         exp.cpu(), minp.cpu(), qtags.cpu(), 2.0)
    assert stats.get("q16_fallbacks", 0) == 1
    assert torch.equal(s.cpu(), rs) and bool((r >= 0).all())


def test_q16_semantic_index_on_gpu(gpu):
    """The index front end (storage="q16") on the GPU equals the same index on the CPU."""
    import numpy as np

    from pilottai_amd.memory.semantic_index import SemanticIndex

    g = np.random.default_rng(3)
    v = g.standard_normal((5000, 1024)).astype(np.float32)
    prio = [i % 3 for i in range(5000)]
    tags = [{"a"} if i % 2 else {"b"} for i in range(5000)]
    q = g.standard_normal((9, 1024)).astype(np.float32)
    res = []
    for dev in (gpu, "cpu"):
        idx = SemanticIndex(dim=1024, capacity=1024, device=dev, storage="q16")
        idx.add(v, prio, tags, [None] * 5000)
        res.append(idx.search(q, 7, [0, 1, 2] * 3, [(), ("a",), ("b",)] * 3))
    assert [[r for r, _ in x] for x in res[0]] == [[r for r, _ in x] for x in res[1]]
    # same rows, scores equal up to the last bit of the final fp32 scaling (order of the two scale
    # multiplies differs between the GPU epilogue and the CPU reference)
    for a, b in zip(res[0], res[1]):
        for (_, sa), (_, sb) in zip(a, b):
            assert abs(sa - sb) <= 1e-6 * max(1.0, abs(sb))


def _small_index(gpu, storage="q16", n=3000, same=False):
    import numpy as np

    from pilottai_amd.memory.semantic_index import SemanticIndex

    v = np.random.default_rng(5).standard_normal((1 if same else n, 256)).astype(np.float32)
    idx = SemanticIndex(dim=256, capacity=n, device=gpu, storage=storage)
    idx.add(np.repeat(v, n, 0) if same else v, [i % 3 for i in range(n)], [()] * n, [None] * n)
    return idx, v


@pytest.mark.parametrize("storage", ["bf16", "q16"])
def test_search_takes_any_sequence_of_filters(gpu, storage):
    """Filters as numbers, as tensors on either device, and more of them than queries; fewer are refused, not repeated."""
    idx, v = _small_index(gpu, storage)
    q, none = v[:3], [()] * 3
    want = idx.search(q, 4, [0, 1, 2], none)
    for p in ((0, 1, 2), torch.tensor([0, 1, 2]), torch.tensor([0, 1, 2], device=gpu), [0, 1, 2, 0, 1], [0.5, 1.5, 2.0]):
        assert idx.search(q, 4, p, none) == want
    assert idx.search(q, 4, [0, 1, 2], [()] * 5) == want
    for p, t in (([1], none), ([0, 1, 2], [()])):
        with pytest.raises(ValueError):
            idx.search(q, 4, p, t)
    with pytest.raises((RuntimeError, OverflowError)):
        idx.search(q, 4, [0, 1, 1 << 40], none)


@pytest.mark.parametrize("storage", ["bf16", "q16"])
@pytest.mark.parametrize("Q", [1, 64, 65, 130])  # a pass, and several
def test_search_takes_queries_from_anywhere(gpu, storage, Q):
    """Queries as an array, as tensors of the host or the GPU, of other types and strides: the same results, in lists of plain
    numbers that end with the hits."""
    idx, v = _small_index(gpu, storage)
    q = torch.from_numpy(v[:Q])
    args = (3, [i % 3 for i in range(Q)], [()] * Q)
    want = idx.search(v[:Q], *args)
    assert [len(w) for w in want] == [3] * Q and all(type(r) is int and type(x) is float for w in want for r, x in w)
    assert all(w[0][0] == i for i, w in enumerate(want))
    for x in (q, q.double(), q.to(gpu), q.t().contiguous().t(), q.t().contiguous().to(gpu).t()):
        assert idx.search(x, *args) == want
    assert idx.search(q, 3, [2] * Q, [("unknown",)] * Q) == [[]] * Q


@pytest.mark.parametrize("D", [1984, 2048, 2112])  # around what a workgroup keeps of a query
def test_query_preparation_of_long_queries(gpu, D):
    q = torch.randn(3, D)
    assert torch.equal(ops.unit_queries(q.to(gpu)).cpu(), ops.unit_queries(q))
    assert all(torch.equal(a.cpu(), b) for a, b in zip(ops.q16_queries(q.to(gpu), True), ops.q16_queries(q, True)))


def test_search_times_its_second_pass_too(gpu, monkeypatch):
    """The events around a search that falls back to the exact scan lie around both passes."""
    idx, v = _small_index(gpu, n=40_000, same=True)
    idx.pass_events, ends, run = [], [], ops.q16_pass

    def noted(*args):
        run(*args)
        ends.append(torch.cuda.Event(enable_timing=True))
        ends[-1].record()
    monkeypatch.setattr(ops, "q16_pass", noted)
    idx.search(v, 5, [0], [()])
    assert idx.stats["q16_fallbacks"] == 1 and len(ends) == 2 and len(idx.pass_events) == 1
    (start, end), = idx.pass_events
    assert 0 < start.elapsed_time(ends[0]) < start.elapsed_time(ends[1]) <= start.elapsed_time(end)


@pytest.mark.parametrize("exact", [False, True])
def test_search_that_fails_waits_for_its_passes(gpu, monkeypatch, exact):
    """A pass that raises behind its launches, the first or the one that stands behind it: the pinned memory that the kernels
    write to stays until they are done."""
    idx, v = _small_index(gpu, n=40_000, same=True)
    idx.search(v, 5, [0], [()])
    run = ops.q16_pass

    def fails(*args):
        run(*args)
        if args[-2] == exact:
            torch.cuda._sleep(50_000_000)
            raise KeyError("pass")
    monkeypatch.setattr(ops, "q16_pass", fails)
    with pytest.raises(KeyError):
        idx.search(v, 5, [0], [()])
    assert idx._stream.query()
    monkeypatch.setattr(ops, "q16_pass", run)
    assert [r for r, _ in idx.search(v, 5, [0], [()])[0]]


def test_search_in_one_call(gpu):
    """A bf16 index and queries of the host: events lie around the pass, a call that raises has waited for its launches, and
    threads on streams of their own get what one gets."""
    from concurrent.futures import ThreadPoolExecutor

    idx, v = _small_index(gpu, "bf16")
    args = (3, [0] * 70, [()] * 70)
    want = idx.search(v[:70], *args)
    idx.pass_events = []
    assert idx.search(v[:70], *args) == want
    (start, end), = idx.pass_events
    assert start.elapsed_time(end) > 0
    idx.pass_events = None
    with pytest.raises(RuntimeError):  # (behind the queries' preparation)
        idx.search(v[:70, :32], *args)
    assert idx._stream.query()
    before = torch.cuda.current_stream(gpu)

    def one(i):
        with torch.cuda.stream(torch.cuda.Stream(gpu)):
            return idx.search(v[i:i + 1], 3, [0], [()])[0]
    with ThreadPoolExecutor(4) as pool:
        assert list(pool.map(one, range(70))) == want
    assert torch.cuda.current_stream(gpu) == before
