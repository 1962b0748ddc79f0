"""Numerics of the CDNA4 HIP kernels vs the fp32 PyTorch references (ops/reference.py)."""
import math

import numpy as np
import pytest
import torch

from pilottai_amd import ops
from pilottai_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _bf(*shape, dev, scale=1.0):
    return (torch.randn(*shape, device=dev) * scale).to(torch.bfloat16)


@pytest.mark.parametrize("D", [4096, 8192, 1024, 256, 4104])
def test_rmsnorm(gpu, D):
    torch.manual_seed(0)
    x = _bf(37, D, dev=gpu)
    w = _bf(D, dev=gpu)
    y = ops.rmsnorm(x, w, 1e-5)
    r = ref.rmsnorm(x.cpu(), w.cpu(), 1e-5)
    torch.testing.assert_close(y.cpu().float(), r.float(), atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("T,D", [(1, 4096), (5, 520), (64, 64), (67, 8192), (130, 4104)])
def test_first_and_last_rows(gpu, T, D):
    """Gathers inside the step's first launch and its last norm: the bits of the launches that they stand for."""
    gen = torch.Generator().manual_seed(T)
    emb = torch.randn(301, D + 8, generator=gen).to(torch.bfloat16).to(gpu)[:, :D]  # (rows that lie apart)
    ids = torch.randint(0, 301, (T,), generator=gen, dtype=torch.int32)
    ids[0], ids[-1] = 0, 300
    ss, zero = torch.full((2, T + 1), 7.0, device=gpu)
    h = ops.embed_rows(emb, ids.to(gpu), ss[:T], zero[:T])
    assert torch.equal(h.cpu(), emb.cpu()[ids.long()])
    assert torch.equal(ss[:T], ops.row_sumsq(h)) and not zero[:T].any() and ss[T] == zero[T] == 7
    assert torch.equal(ops.embed_rows(emb, ids.to(gpu)), h)
    w = torch.randn(D, generator=gen).to(torch.bfloat16).to(gpu)
    rows = torch.randint(0, T, (T + 3,), generator=gen, dtype=torch.int32).to(gpu)
    assert torch.equal(ops.rmsnorm(h, w, 1e-5, rows=rows), ops.rmsnorm(h.index_select(0, rows), w, 1e-5))


@pytest.mark.parametrize("D", [4096, 8192, 520])
def test_fused_add_rmsnorm(gpu, D):
    torch.manual_seed(1)
    x = _bf(19, D, dev=gpu)
    res = _bf(19, D, dev=gpu)
    w = _bf(D, dev=gpu)
    r_y, r_res = ref.fused_add_rmsnorm(res.cpu(), x.cpu(), w.cpu(), 1e-5)
    y = ops.fused_add_rmsnorm(res, x, w, 1e-5)
    torch.testing.assert_close(res.cpu().float(), r_res.float(), atol=1e-2, rtol=1e-2)
    torch.testing.assert_close(y.cpu().float(), r_y.float(), atol=2e-2, rtol=2e-2)


def test_silu_mul(gpu):
    torch.manual_seed(2)
    x = _bf(33, 2 * 14336, dev=gpu)
    y = ops.silu_mul(x)
    torch.testing.assert_close(y.cpu().float(), ref.silu_mul(x.cpu()).float(), atol=2e-2, rtol=2e-2)


def _make_cache(nblocks, KV, dev, blk=16):
    k = _bf(nblocks, KV, 16, blk, 8, dev=dev)
    v = _bf(nblocks, KV, 128, blk, dev=dev)
    return k, v


def test_rope_cache(gpu):
    torch.manual_seed(3)
    H, KV, T = 32, 8, 29
    qkv = _bf(T, (H + 2 * KV) * 128, dev=gpu)
    pos = torch.randint(0, 4000, (T,), dtype=torch.int32, device=gpu)
    slots = torch.randperm(64 * 16, device=gpu)[:T].int()
    slots[5] = -1  # padding token: must not be written
    cs = ref.rope_cos_sin(4096).to(gpu)
    kc, vc = _make_cache(64, KV, gpu)
    kc_r, vc_r = kc.cpu().clone(), vc.cpu().clone()
    q = torch.empty(T, H, 128, dtype=torch.bfloat16, device=gpu)
    q_r = torch.empty(T, H, 128, dtype=torch.bfloat16)
    ops.rope_cache(q, kc, vc, qkv, pos, slots, cs, H, KV)
    ref.rope_cache(q_r, kc_r, vc_r, qkv.cpu(), pos.cpu(), slots.cpu(), cs.cpu(), H, KV)
    torch.testing.assert_close(q.cpu().float(), q_r.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(kc.cpu().float(), kc_r.float(), atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(vc.cpu().float(), vc_r.float(), atol=0, rtol=0)


def _run_attention(gpu, H, KV, q_lens, ctx_lens, seed=0, split=True, part=512, qcols=128, pad=1,
                   launches=1, waves=4, split_keys=0):
    torch.manual_seed(seed)
    G = H // KV
    blk = 16
    ns = len(q_lens)
    nbs = [(c + blk - 1) // blk for c in ctx_lens]
    total_blocks = sum(nbs) + 4
    max_blocks = max(nbs)
    kc, vc = _make_cache(total_blocks, KV, gpu)
    perm = torch.randperm(total_blocks).tolist()
    bt = torch.zeros(ns, max_blocks, dtype=torch.int32)
    c = 0
    for s, nb in enumerate(nbs):
        bt[s, :nb] = torch.tensor(perm[c:c + nb], dtype=torch.int32)
        c += nb
    q_start = np.concatenate([[0], np.cumsum(q_lens)[:-1]]).astype(np.int32)
    T = int(sum(q_lens))
    q = _bf(T, H, 128, dev=gpu)
    items, nslots = ops.build_attention_items(q_lens, ctx_lens, G, split=split, part=part,
                                               qcols=qcols, wide_min_tokens=0, split_keys=split_keys)
    it = torch.tensor(items + [(0, 0, 0, 0)] * max(pad, nslots - len(items)), dtype=torch.int32, device=gpu)
    # per-(sequence, KV head) tickets, then -- with split prefill items, as the engine -- per-(partial
    # slot, KV head) ones; without them the kernel runs its instantiation with the partition
    # hand-off compiled out (both instantiations are covered: split_keys > 0 cases take the other)
    cnt = torch.zeros((ns + (it.shape[0] if split_keys else 0)) * KV, dtype=torch.int32, device=gpu)
    n_it = torch.tensor([len(items)], dtype=torch.int32, device=gpu)
    maxit = it.shape[0]
    part_o = torch.empty(maxit * KV * 16 * 128, dtype=torch.float32, device=gpu)
    part_ml = torch.empty(maxit * KV * 16 * 2, dtype=torch.float32, device=gpu)
    out = torch.zeros(T, H, 128, dtype=torch.bfloat16, device=gpu)
    scale = 1.0 / math.sqrt(128)
    dev_i = lambda a: torch.tensor(a, dtype=torch.int32, device=gpu)  # noqa: E731
    for _ in range(launches):  # the partition tickets must reset themselves for the next launch
        ops.paged_attention(out, part_o, part_ml, q, kc, vc, it, n_it, cnt, dev_i(q_start),
                            dev_i(q_lens), dev_i(ctx_lens), bt.to(gpu), scale, part_size=dev_i([part]),
                            waves=waves)
    torch.cuda.synchronize()
    assert int(cnt.abs().sum()) == 0, "partition tickets must be left zeroed"
    r = ref.paged_attention(q.cpu(), kc.cpu(), vc.cpu(), q_start, q_lens, ctx_lens, bt, scale)
    return out.cpu().float(), r.float()


@pytest.mark.parametrize("H,KV", [(32, 8), (8, 1), (16, 16)])
def test_attention_decode(gpu, H, KV):
    ctx = [1, 15, 16, 17, 33, 100, 511, 512, 513, 1500, 2049, 64]
    o, r = _run_attention(gpu, H, KV, [1] * len(ctx), ctx)
    torch.testing.assert_close(o, r, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("qcols", [32, 128])
@pytest.mark.parametrize("H,KV", [(32, 8), (8, 1)])
def test_attention_prefill_and_mixed(gpu, H, KV, qcols):
    """Prefill chunks of every length class next to decode rows; qcols 128 = the LDS-staged
    4-wave items (plus their 32-column / decode-path tails), 32 = one wave per item."""
    q_lens = [37, 1, 100, 3, 16, 5, 250, 129, 33]
    ctx = [37, 700, 164, 40, 16, 1029, 260, 1000, 2100]
    o, r = _run_attention(gpu, H, KV, q_lens, ctx, seed=5, qcols=qcols)
    torch.testing.assert_close(o, r, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("split_keys", [512, 1024])
@pytest.mark.parametrize("H,KV", [(32, 8), (64, 8), (8, 1)])
def test_attention_prefill_split_items(gpu, H, KV, split_keys):
    """the longest wide prefill items cut into 2-4 key partitions, merged
    in-kernel by the last partition (register-layout partials through the uncached slab),
    beside unsplit items and split decode rows; twice, so the tickets reset themselves."""
    q_lens = [2048, 1100, 300, 1, 700, 3]
    ctx = [2048, 1100, 1500, 900, 2600, 4000]
    G = H // KV
    items, _ = ops.build_attention_items(q_lens, ctx, G, qcols=128, wide_min_tokens=0, split_keys=split_keys)
    assert any((z >> 20) > 1 and (z & 0xFF) > 32 // G for _, _, z, _ in items), "no split prefill item"
    o, r = _run_attention(gpu, H, KV, q_lens, ctx, seed=13, split_keys=split_keys, launches=2)
    torch.testing.assert_close(o, r, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("H,KV", [(16, 16), (16, 8), (64, 8), (32, 8)])
def test_attention_prefill_tiles(gpu, H, KV):
    """q-split path: chunks spanning several 4 x 32/G-token tiles, cached prefixes,
    partial last tiles, plus decode rows in the same launch."""
    q_lens = [300, 129, 33, 1, 2, 77]
    ctx = [300, 1129, 65, 900, 18, 77 + 512]
    o, r = _run_attention(gpu, H, KV, q_lens, ctx, seed=11)
    torch.testing.assert_close(o, r, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("part", [128, 256])
def test_attention_small_partitions(gpu, part):
    """Per-step decode partition sizes chosen by the scheduler for small batches."""
    ctx = [1, 100, 127, 128, 129, 700, 2049, 64]
    o, r = _run_attention(gpu, 32, 8, [1, 1, 2, 1, 4, 1, 1, 3], ctx, seed=13, part=part)
    torch.testing.assert_close(o, r, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("case", ["decode", "mixed32", "mixed128", "tiles", "kv1", "kv16", "small_part", "step2048"])
def test_attention_repeated_padded_launches(gpu, case):
    """Three back-to-back launches on one ticket buffer with padded item lists, as the
    engine's graphs replay them: bit-identical to a single launch (the partition tickets
    reset themselves, the merge order is fixed) and equal to fp32."""
    cfg = {
        "decode": dict(H=32, KV=8, q=[1] * 12, c=[1, 15, 16, 17, 33, 100, 511, 512, 513, 1500, 2049, 64]),
        "mixed32": dict(H=32, KV=8, q=[37, 1, 100, 3, 16, 5, 250, 129, 33], c=[37, 700, 164, 40, 16, 1029, 260, 1000, 2100],
                        qcols=32),
        "mixed128": dict(H=32, KV=8, q=[37, 1, 100, 3, 16, 5, 250, 129, 33], c=[37, 700, 164, 40, 16, 1029, 260, 1000, 2100]),
        "tiles": dict(H=64, KV=8, q=[300, 129, 33, 1, 2, 77], c=[300, 1129, 65, 900, 18, 589]),
        "kv1": dict(H=8, KV=1, q=[37, 1, 100, 3, 16], c=[37, 700, 164, 40, 16]),
        "kv16": dict(H=16, KV=16, q=[1, 1, 40, 3], c=[100, 2049, 40, 700]),
        "small_part": dict(H=32, KV=8, q=[1, 1, 2, 1, 4, 1, 1, 3], c=[1, 100, 127, 128, 129, 700, 2049, 64], part=256),
        "step2048": dict(H=32, KV=8, q=[512] * 4 + [1] * 40, c=[768] * 4 + [600] * 40),
    }[case]
    kw = dict(seed=17, qcols=cfg.get("qcols", 128), part=cfg.get("part", 512), pad=200)
    og, r = _run_attention(gpu, cfg["H"], cfg["KV"], cfg["q"], cfg["c"], **kw)
    oq, _ = _run_attention(gpu, cfg["H"], cfg["KV"], cfg["q"], cfg["c"], launches=3, **kw)
    torch.testing.assert_close(oq, r, atol=2e-2, rtol=2e-2)
    assert torch.equal(oq, og)


@pytest.mark.parametrize("case", ["decode", "small_part", "mixed32", "mixed128_wide", "kv1", "rows9"])
def test_attention_eight_wave_workgroups(gpu, case):
    """512-thread workgroups (waves=8, the engine's decode-sized steps): decode items split
    their 32-key tiles over 8 waves, 32-column prefill items too, and wide (128-column)
    items run as their 32-column sub-items; equal to fp32 and to the 4-wave launch."""
    cfg = {
        "decode": dict(H=32, KV=8, q=[1] * 12, c=[1, 15, 16, 17, 33, 100, 511, 512, 513, 1500, 2049, 64]),
        "small_part": dict(H=32, KV=8, q=[1, 1, 2, 1, 4, 1, 1, 3], c=[1, 100, 127, 128, 129, 700, 2049, 64], part=256),
        "mixed32": dict(H=32, KV=8, q=[37, 1, 100, 3, 16, 5, 250, 129, 33], c=[37, 700, 164, 40, 16, 1029, 260, 1000, 2100],
                        qcols=32),
        "mixed128_wide": dict(H=32, KV=8, q=[37, 1, 100, 3, 16, 5, 250, 129, 33],
                              c=[37, 700, 164, 40, 16, 1029, 260, 1000, 2100]),
        "kv1": dict(H=8, KV=1, q=[1, 1, 2, 12, 1], c=[100, 600, 33, 40, 2000]),
        "rows9": dict(H=32, KV=8, q=[1] * 8 + [5], c=[600] * 8 + [300]),
    }[case]
    kw = dict(seed=23, qcols=cfg.get("qcols", 128), part=cfg.get("part", 256), pad=50)
    o4, r = _run_attention(gpu, cfg["H"], cfg["KV"], cfg["q"], cfg["c"], **kw)
    o8, _ = _run_attention(gpu, cfg["H"], cfg["KV"], cfg["q"], cfg["c"], waves=8, launches=2, **kw)
    torch.testing.assert_close(o8, r, atol=2e-2, rtol=2e-2)
    torch.testing.assert_close(o8, o4, atol=1e-2, rtol=1e-2)


def test_attention_nosplit_long(gpu):
    o, r = _run_attention(gpu, 32, 8, [1, 2], [3000, 1200], seed=7, split=False)
    torch.testing.assert_close(o, r, atol=2e-2, rtol=2e-2)


def test_sample_greedy_and_masks(gpu):
    torch.manual_seed(4)
    rows, V = 9, 128256
    logits = _bf(rows, V, dev=gpu, scale=3.0)
    words = (V + 31) // 32
    masks = torch.zeros(3, words, dtype=torch.int32)
    masks[0] = -1  # all allowed
    allowed = np.zeros(V, dtype=bool)
    allowed[[5, 77, 1000, 128000]] = True
    masks[1] = ref.pack_mask(allowed)
    temp = torch.zeros(rows)
    mcls = torch.tensor([-1, 0, 1, 1, -1, 0, 1, -1, 0], dtype=torch.int32)
    forced = torch.full((rows,), -1, dtype=torch.int32)
    forced[4] = 1234
    seeds = torch.arange(rows, dtype=torch.int64) * 7919
    offs = torch.arange(rows, dtype=torch.int32)
    tok = ops.sample(logits, temp.to(gpu), mcls.to(gpu), masks.to(gpu), seeds.to(gpu), offs.to(gpu),
                     forced.to(gpu))
    r = ref.sample(logits.cpu(), temp, mcls, masks, seeds, offs, forced)
    assert tok.cpu().tolist() == r.tolist()


def test_sample_temperature_matches_reference(gpu):
    torch.manual_seed(5)
    rows, V = 16, 32000
    logits = _bf(rows, V, dev=gpu, scale=2.0)
    masks = torch.full((1, (V + 31) // 32), -1, dtype=torch.int32)
    temp = torch.full((rows,), 0.7)
    mcls = torch.full((rows,), -1, dtype=torch.int32)
    seeds = torch.randint(0, 2 ** 62, (rows,), dtype=torch.int64)
    offs = torch.randint(0, 1000, (rows,), dtype=torch.int32)
    keys = torch.empty(rows, device=gpu)
    tok = ops.sample(logits, temp.to(gpu), mcls.to(gpu), masks.to(gpu), seeds.to(gpu), offs.to(gpu),
                     None, out_keys=keys)
    r, rk = ref.sample(logits.cpu(), temp, mcls, masks, seeds, offs, None, return_keys=True)
    # the hash is bit-identical; fast-math logs may flip near-ties only
    agree = (tok.cpu() == r).float().mean().item()
    assert agree >= 0.9
    torch.testing.assert_close(keys.cpu(), rk, atol=1e-2, rtol=5e-3)


def test_sample_distribution(gpu):
    """Gumbel-max samples follow softmax(logits / T)."""
    V = 64
    rows = 4096
    base = torch.linspace(-2, 2, V)
    logits = base.repeat(rows, 1).to(torch.bfloat16).to(gpu)
    masks = torch.full((1, 2), -1, dtype=torch.int32, device=gpu)
    temp = torch.full((rows,), 0.7, device=gpu)
    mcls = torch.full((rows,), -1, dtype=torch.int32, device=gpu)
    seeds = torch.full((rows,), 12345, dtype=torch.int64, device=gpu)
    offs = torch.arange(rows, dtype=torch.int32, device=gpu)
    tok = ops.sample(logits, temp, mcls, masks, seeds, offs, None).cpu()
    emp = torch.bincount(tok.long(), minlength=V).float() / rows
    exp = torch.softmax(base.to(torch.bfloat16).float() / 0.7, 0)
    assert (emp - exp).abs().max().item() < 0.03


@pytest.mark.parametrize("N,D,Q,K", [(20000, 1024, 5, 8), (150000, 256, 70, 64), (3000, 768, 17, 10),
                                     # short indexes: slices of 4, 5 and 8 tiles, a last tile of one row, every width of the kernel
                                     (1250, 96, 2, 64), (16384, 992, 16, 3), (16385, 288, 7, 33), (32768, 512, 15, 64), (32753, 64, 2, 1)])
def test_cosine_topk(gpu, N, D, Q, K):
    torch.manual_seed(6)
    idx = torch.nn.functional.normalize(torch.randn(N, D), dim=1).to(torch.bfloat16)
    qs = torch.nn.functional.normalize(torch.randn(Q, D), dim=1).to(torch.bfloat16)
    qs[1] = idx[1234]  # exact hit
    prio = torch.randint(0, 5, (N,), dtype=torch.int32)
    tags = torch.randint(0, 8, (N,), dtype=torch.int64)
    exp = torch.zeros(N)
    exp[::7] = 50.0  # expired at now=100
    qmin = torch.tensor([0, 0, 2, 4, 0] * ((Q + 4) // 5), dtype=torch.int32)[:Q]
    qt = torch.tensor([0, 0, 1, 2, 3] * ((Q + 4) // 5), dtype=torch.int64)[:Q]
    Np = (N + 15) // 16 * 16  # the index is stored in packed 16-row tiles
    packed = ops.pack_decode_weight(torch.cat([idx, torch.zeros(Np - N, D, dtype=idx.dtype)]).to(gpu))
    s, r = ops.cosine_topk(qs.to(gpu), packed, N, K, prio.to(gpu), tags.to(gpu), exp.to(gpu),
                           qmin.to(gpu), qt.to(gpu), 100.0)
    rs, rr = ref.cosine_topk(qs, idx, N, K, prio, tags, exp, qmin, qt, 100.0)
    torch.testing.assert_close(s.cpu(), rs, atol=2e-3, rtol=2e-3)
    # rows agree except for exact score ties
    assert (r.cpu() == rr).float().mean().item() > 0.95


@pytest.mark.parametrize("Q,N", [(1, 1000), (16, 32_768), (17, 32_768), (3, 32_769), (16, 20_000), (17, 20_000), (64, 300)])
def test_cosine_topk_workspace(gpu, Q, N):
    """A pass takes what it is said to need, is refused with less and leaves what lies behind alone; a short index needs its
    slices' lists and nothing else."""
    C, K, D = ops.kernels.require_native(), 7, 64
    need = C.cosine_topk_workspace_bytes(Q, N, K)
    if Q <= 16 and N <= 32_768:
        assert need <= Q * 256 * K * 8  # (a score and a row)
    g = torch.Generator(device=gpu).manual_seed(Q)
    rows = torch.nn.functional.normalize(torch.randn((N + 15) // 16 * 16, D, device=gpu, generator=g), dim=1).to(torch.bfloat16)
    q = torch.nn.functional.normalize(torch.randn(Q, D, device=gpu, generator=g), dim=1).to(torch.bfloat16)
    ints = lambda n, dt=torch.int32: torch.zeros(n, dtype=dt, device=gpu)  # noqa: E731
    room = torch.full((need + 4096,), 77, dtype=torch.uint8, device=gpu)
    s, r = torch.empty(Q, K, device=gpu), torch.empty(Q, K, dtype=torch.int32, device=gpu)
    args = (q, ops.pack_decode_weight(rows), N, K, ints(N), ints(N, torch.int64), torch.zeros(N, device=gpu), ints(Q), ints(Q, torch.int64), 0.0)
    C.cosine_topk(s, r, room[:need], *args)
    exact = (q.double() @ rows[:N].double().T).topk(K, 1).values
    torch.testing.assert_close(s.double(), exact, atol=64 * 2.0 ** -24, rtol=0)  # (sums of 64 products in fp32)
    assert bool((room[need:] == 77).all())
    with pytest.raises(RuntimeError, match="workspace too small"):
        C.cosine_topk(s, r, room[:need - 1], *args)


@pytest.mark.parametrize("Q", [65, 70, 80, 81, 128, 134])  # a last pass of 1 to 64 queries, on both sides of a short index's 16
@pytest.mark.parametrize("N", [1000, 20_000, 32_768, 32_769, 1_000_000])
def test_cosine_topk_workspace_of_passes(Q, N):
    C = ops.kernels.require_native()
    assert C.cosine_topk_workspace_bytes(Q, N, 9) == max(C.cosine_topk_workspace_bytes(n, N, 9) for n in (64, Q % 64 or 64))


@pytest.mark.parametrize("N,K", [(9000, 64), (20000, 33), (60000, 64), (60000, 5)])  # lists of up to 16,384 entries, of each width
def test_best_rows_lie_together(gpu, N, K):
    """The second stage of a lookup where the first's lists say little: all of the best in one slice, and all rows alike."""
    g = torch.Generator().manual_seed(N + K)
    idx = torch.nn.functional.normalize(torch.randn(N, 64, generator=g), dim=1)
    q = torch.nn.functional.normalize(torch.randn(2, 64, generator=g), dim=1).to(torch.bfloat16)
    idx[32:132] = torch.nn.functional.normalize(q[:1].float() + 0.02 * torch.randn(100, 64, generator=g), dim=1)
    idx = idx.to(torch.bfloat16)
    ints = lambda n, dt=torch.int32: torch.zeros(n, dtype=dt, device=gpu)  # noqa: E731
    for rows in (idx, idx[32:33].expand(N, -1)):
        packed = ops.pack_decode_weight(torch.cat([rows, rows[:-N % 16]]).to(gpu))
        s, r = ops.cosine_topk(q.to(gpu), packed, N, K, ints(N), ints(N, torch.int64), torch.zeros(N, device=gpu), ints(2),
                               ints(2, torch.int64), 0.0)
        exact = q.double() @ rows.double().T
        # (sums of 64 products in fp32)
        torch.testing.assert_close(s.double().cpu(), exact.topk(K, 1).values, atol=64 * 2.0 ** -24, rtol=0)
        r = r.long().cpu()
        assert all(len(set(x.tolist())) == K for x in r)
        torch.testing.assert_close(exact.gather(1, r), s.double().cpu(), atol=64 * 2.0 ** -24, rtol=0)


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (13, 6144, 4096), (64, 28672, 4096), (64, 4096, 14336),
                                   (100, 4096, 4096), (128, 1024, 512), (37, 128256, 4096)])
def test_skinny_gemm(gpu, M, N, K):
    from pilottai_amd.ops import kernels

    torch.manual_seed(8)
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=gpu)
    assert kernels.require_native().skinny_gemm(y, x, w)
    r = (x.float() @ w.float().T)
    torch.testing.assert_close(y.float(), r, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("V", [128256, 32000])
def test_topkp_threshold_matches_reference(gpu, V):
    torch.manual_seed(9)
    rows = 12
    logits = _bf(rows, V, dev=gpu, scale=4.0)
    words = (V + 31) // 32
    masks = torch.full((2, words), -1, dtype=torch.int32)
    allowed = np.zeros(V, dtype=bool)
    allowed[np.random.RandomState(0).choice(V, 5000, replace=False)] = True
    masks[1] = ref.pack_mask(allowed)
    temp = torch.tensor([0.7, 1.0, 0.5, 1.3, 0.0, 0.9, 1.0, 0.8, 1.0, 0.6, 1.0, 2.0])
    top_k = torch.tensor([0, 1, 5, 40, 10, 0, 200, 3, 0, 0, 64, 0], dtype=torch.int32)
    top_p = torch.tensor([0.9, 1.0, 1.0, 0.5, 0.9, 0.3, 1.0, 0.95, 1.0, 0.99, 0.8, 0.7])
    mcls = torch.tensor([-1, -1, 1, -1, -1, 1, -1, 1, -1, -1, 1, -1], dtype=torch.int32)
    tau = ops.topkp_threshold(logits, V, temp.to(gpu), top_k.to(gpu), top_p.to(gpu), mcls.to(gpu),
                              masks.to(gpu))
    r = ref.topkp_threshold(logits.cpu(), temp, top_k, top_p, mcls, masks)
    t = tau.cpu()
    for i in range(rows):
        if top_k[i] > 0 and top_p[i] >= 1.0:
            assert t[i].item() == r[i].item(), (i, t[i], r[i])  # top-k is exact
    assert (t == r).float().mean().item() >= 0.8  # top-p: fp32 vs fp64 mass at the boundary
    # sampling honours tau: every sampled token is allowed and >= tau
    seeds = torch.arange(rows, dtype=torch.int64) * 31 + 7
    offs = torch.zeros(rows, dtype=torch.int32)
    for trial in range(4):
        tok = ops.sample(logits, temp.to(gpu), mcls.to(gpu), masks.to(gpu), (seeds + trial).to(gpu),
                         offs.to(gpu), None, tau=tau).cpu()
        lg = logits.float().cpu()
        for i in range(rows):
            assert lg[i, tok[i]].item() >= t[i].item()
            if mcls[i] == 1:
                assert allowed[tok[i]]
        if trial == 0:
            assert tok[1].item() == int(lg[1].argmax())  # k = 1 is greedy


@pytest.mark.parametrize("M,N,K,epi,norm", [
    (1, 6144, 4096, "plain", True), (8, 4096, 4096, "resid", False), (13, 28672, 4096, "silu", True),
    (16, 4096, 14336, "resid", False), (5, 128256, 4096, "plain", False), (29, 6144, 4096, "plain", False),
    (64, 1024, 512, "silu", True), (40, 768, 512, "resid", False)])
def test_decode_gemm(gpu, M, N, K, epi, norm):
    """Packed-weight decode projection (csrc/ops/gemm_decode.hip) vs fp32: the
    folded RMSNorm, SwiGLU and residual epilogues, every default tile config."""
    torch.manual_seed(11)
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    resid = _bf(M, N, dev=gpu) if epi == "resid" else None
    wp = ops.pack_decode_gate_up(w) if epi == "silu" else ops.pack_decode_weight(w)
    y = ops.decode_gemm(x, wp, epi, norm=norm, resid=resid)
    acc = x.float() @ w.float().T
    if norm:
        acc = acc * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-5)
    if epi == "silu":
        acc = torch.nn.functional.silu(acc[:, :N // 2]) * acc[:, N // 2:]
    elif epi == "resid":
        acc = acc + resid.float()
    torch.testing.assert_close(y.float(), acc, atol=3e-2, rtol=2e-2)
    if epi == "resid":  # in place on the residual stream
        r2 = resid.clone()
        ops.decode_gemm(x, wp, "resid", resid=r2, out=r2)
        torch.testing.assert_close(r2, y, atol=0, rtol=0)


@pytest.mark.parametrize("M,N,K", [
    (17, 16, 32), (32, 4096, 96), (33, 2048, 544), (64, 2048, 8192), (64, 128256, 64), (31, 40_960, 160),  # up to 64 rows
    (33, 33_040, 96), (40, 114_416, 160), (64, 114_448, 32), (48, 131_072, 96), (64, 131_088, 64),  # 128 and 256 columns a tile
    (64, 98_304, 32), (40, 98_320, 96), (33, 229_376, 32), (64, 229_392, 32), (50, 262_144, 64), (64, 262_160, 32),  # the lines
    (65, 2064, 512), (96, 10368, 2048), (129, 4112, 1056), (512, 2048, 768), (1000, 1040, 64)])             # and more
def test_rows_gemm(gpu, M, N, K):
    """Every tile of dispatch_rows, at its edges: rows and columns past the tiles, k past the last stage. A bf16 result
    rounds by 2^-8 of itself at most, and a sum of K products in fp32 errs by K 2^-24 of their magnitudes at most."""
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = torch.randn(M, K + 8, device=gpu, generator=g).bfloat16()[:, :K]
    w = torch.randn(N, K, device=gpu, generator=g).bfloat16()
    buf = torch.full((M, N + 4), 7.0, device=gpu, dtype=torch.bfloat16)
    y = ops.rows_gemm(x, ops.pack_decode_weight(w), out=buf[:, :N])
    assert y is not None
    ref, size = x.float() @ w.float().T, x.float().abs() @ w.float().abs().T
    assert bool(((y.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * size).all())
    assert bool((buf[:, N:] == 7.0).all())
    assert ops.rows_gemm(torch.empty(513, 64, device=gpu, dtype=torch.bfloat16),
                         ops.pack_decode_weight(torch.zeros(4096, 64, device=gpu, dtype=torch.bfloat16))) is None


@pytest.mark.parametrize("M,N,K", [(24, 8192, 2048), (24, 8208, 2048), (24, 8208, 2016), (25, 2048, 736), (25, 2048, 768), (32, 64, 512),
                                   (33, 64, 512), (33, 4112, 512), (64, 80, 480), (40, 16384, 64), (40, 16400, 64), (17, 16, 14336)])
def test_decode_gemm_of_17_to_64_rows(gpu, M, N, K):
    """Both sides of the lines between its two kernels (rows_pay), with test_rows_gemm's bound."""
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x, w = torch.randn(M, K, device=gpu, generator=g).bfloat16(), torch.randn(N, K, device=gpu, generator=g).bfloat16()
    y = ops.decode_gemm(x, ops.pack_decode_weight(w))
    ref, size = x.float() @ w.float().T, x.float().abs() @ w.float().abs().T
    assert bool(((y.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("M,N,K", [(300, 512, 128), (300, 512, 8192), (300, 1408, 192), (300, 1408, 256), (128, 3072, 8192),
                                   (256, 2048, 4096), (256, 2048, 4160), (1600, 512, 3072), (1600, 512, 3136), (512, 3072, 3136)])
def test_packed_linear_of_many_rows(gpu, M, N, K):
    """Both sides of the lines between rows_gemm and prefill_gemm (rows_gemm_pays), with test_rows_gemm's bound."""
    from pilottai_amd.models.common import PackedLinear

    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x, w = torch.randn(M, K, device=gpu, generator=g).bfloat16(), torch.randn(N, K, device=gpu, generator=g).bfloat16()
    y = PackedLinear(w, torch.bfloat16, gpu)(x)
    ref, size = x.float() @ w.float().T, x.float().abs() @ w.float().abs().T
    assert bool(((y.float() - ref).abs() <= 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * size).all())


@pytest.mark.parametrize("nt,waves,splits", [(1, 8, 1), (1, 16, 1), (2, 8, 1), (2, 16, 1), (4, 8, 1), (4, 16, 1),
                                             (2, 8, 4), (4, 8, 2), (1, 16, 3), (2, 4, 8)])
def test_decode_gemm_configs(gpu, nt, waves, splits):
    """Every tile config, with split-K (sc1 slabs + last-arriver reduce) for the
    norm-folded, SwiGLU and residual epilogues; twice, for the self-resetting tickets."""
    torch.manual_seed(12)
    M, N, K = 13, 4096, 4096
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    y = ops.decode_gemm(x, ops.pack_decode_weight(w), "plain", nt=nt, waves=waves, splits=splits)
    torch.testing.assert_close(y.float(), x.float() @ w.float().T, atol=3e-2, rtol=2e-2)
    rs = torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-5)
    gu = (x.float() @ w.float().T) * rs
    want = torch.nn.functional.silu(gu[:, :N // 2]) * gu[:, N // 2:]
    resid = _bf(M, N, dev=gpu)
    for _ in range(2):
        if nt % 2 == 0:
            got = ops.decode_gemm(x, ops.pack_decode_gate_up(w), "silu", norm=True, nt=nt, waves=waves, splits=splits)
            torch.testing.assert_close(got.float(), want, atol=3e-2, rtol=2e-2)
        got = ops.decode_gemm(x, ops.pack_decode_weight(w), "resid", resid=resid, nt=nt, waves=waves, splits=splits)
        torch.testing.assert_close(got.float(), x.float() @ w.float().T + resid.float(), atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("M,H,KV,K,splits", [
    (7, 32, 8, 4096, 0), (16, 4, 1, 512, 0), (1, 8, 2, 1024, 0), (9, 32, 8, 4096, 2),
    # round 2's rare split-3 mismatch: fixed by the release + acquire hand-off (common.h
    # handoff_last); stressed with poisoned slabs in tests/test_handoff_gpu.py
    (9, 32, 8, 4096, 3), (16, 4, 1, 512, 2)])
def test_decode_qkv_rope(gpu, M, H, KV, K, splits):
    """Norm-folded QKV projection with RoPE + paged KV write in the epilogue vs the
    fp32 projection followed by the reference rope_cache."""
    torch.manual_seed(13)
    N = (H + 2 * KV) * 128
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    g = (torch.rand(K, device=gpu) + 0.5).to(torch.bfloat16)
    wp = ops.pack_decode_qkv_rope(w * g[None, :])
    NB = 8
    cos_sin = ref.rope_cos_sin(4096).to(gpu)
    pos = torch.randint(0, 4000, (M,), dtype=torch.int32, device=gpu)
    slots = torch.randperm(NB * 16, device=gpu)[:M].to(torch.int32)
    if M > 2:
        slots[1] = -1
    kc = torch.zeros(NB, KV, 16, 16, 8, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros(NB, KV, 128, 16, dtype=torch.bfloat16, device=gpu)
    q = torch.empty(M, H, 128, dtype=torch.bfloat16, device=gpu)
    ops.decode_qkv_rope(x, wp, 1e-5, q, kc, vc, pos, slots, cos_sin, H, KV, splits=splits)
    xn = x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-5) * g.float()
    qkv = (xn @ w.float().T).cpu()
    rq = torch.empty(M, H, 128, dtype=torch.float32)
    rk = torch.zeros(NB, KV, 16, 16, 8)
    rv = torch.zeros(NB, KV, 128, 16)
    ref.rope_cache(rq, rk, rv, qkv, pos.cpu(), slots.cpu(), cos_sin.cpu(), H, KV)
    torch.testing.assert_close(q.float().cpu(), rq, atol=3e-2, rtol=2e-2)
    torch.testing.assert_close(kc.float().cpu(), rk, atol=3e-2, rtol=2e-2)
    torch.testing.assert_close(vc.float().cpu(), rv, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("M,N,K,epi,norm,fm,fn,splits", [
    (64, 4096, 4096, "plain", False, 0, 0, 0), (128, 6144, 4096, "rope_perm", True, 0, 0, 0),
    (256, 28672, 4096, "silu", True, 0, 0, 0), (192, 4096, 14336, "resid", False, 0, 0, 0),
    (100, 1024, 512, "silu", True, 4, 2, 2), (77, 768, 512, "rope_perm", False, 2, 2, 1),
    (300, 4096, 4096, "resid", False, 8, 4, 3), (512, 6144, 4096, "plain", True, 8, 2, 1),
    (49, 2048, 1024, "plain", False, 2, 4, 8), (250, 4096, 4096, "plain", True, 4, 4, 4),
    (130, 1024, 1024, "silu", False, 8, 4, 2), (33, 512, 2048, "resid", False, 4, 2, 6),
    # 32-row tiles (17-32-token steps)
    (24, 4096, 4096, "resid", False, 1, 2, 4), (32, 28672, 4096, "silu", True, 1, 4, 1),
    (20, 6144, 4096, "rope_perm", True, 1, 2, 2), (48, 4096, 14336, "resid", False, 1, 2, 3),
    # 32-column tiles (fn = 1)
    (64, 4096, 4096, "resid", False, 1, 1, 1), (128, 4096, 14336, "resid", False, 2, 1, 1),
    (96, 4096, 4096, "plain", True, 2, 1, 2)])
def test_mid_gemm(gpu, M, N, K, epi, norm, fm, fn, splits):
    _check_mid(gpu, M, N, K, epi, norm, fm, fn, splits)


def _check_mid(gpu, M, N, K, epi, norm, fm, fn, splits):
    """Mid-size packed-weight GEMM (csrc/ops/gemm_mid.hip: LDS-DMA staged, C^T = W x^T)
    vs fp32, every epilogue and the folded row norm, partial row tiles, with and
    without split-K; run twice so the self-resetting split-K tickets are exercised."""
    torch.manual_seed(17)
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    resid = _bf(M, N, dev=gpu) if epi == "resid" else None
    pack = {"silu": ops.pack_decode_gate_up, "rope_perm": ops.pack_decode_qkv_rope}.get(epi, ops.pack_decode_weight)
    wp = pack(w)
    acc = x.float() @ w.float().T
    if norm:
        acc = acc * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-5)
    if epi == "silu":
        acc = torch.nn.functional.silu(acc[:, :N // 2]) * acc[:, N // 2:]
    elif epi == "resid":
        acc = acc + resid.float()
    for _ in range(2):
        y = ops.mid_gemm(x, wp, epi, resid=resid, norm=norm, fm=fm, fn=fn, splits=splits)
        torch.testing.assert_close(y.float(), acc, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("M,fm,fn,S", [(160, 0, 0, 1), (160, 0, 0, 4), (100, 2, 4, 3), (300, 8, 2, 2)])
def test_mid_gemm_resid_in_place_with_row_stats(gpu, M, fm, fn, S):
    """The residual epilogue may write over its residual input (h += x W^T) and accumulates
    the next norm's row statistics sum(h^2) of the written bf16 rows (ss_out), while zeroing
    another buffer (ss_zero); a following norm-folded projection consuming those statistics
    matches rmsnorm + GEMM."""
    torch.manual_seed(18)
    N, K = 4096, 4096
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    h = _bf(M, N, dev=gpu)
    want = h.float() + x.float() @ w.float().T
    hh = h.clone()
    ss = torch.zeros(M, dtype=torch.float32, device=gpu)
    junk = torch.full((M,), 7.0, device=gpu)
    ops.mid_gemm(x, ops.pack_decode_weight(w), "resid", resid=hh, out=hh, fm=fm, fn=fn, splits=S, ss_out=ss,
                 ss_zero=junk)
    torch.testing.assert_close(hh.float(), want, atol=3e-2, rtol=2e-2)
    torch.testing.assert_close(ss, hh.float().pow(2).sum(-1), rtol=1e-4, atol=1e-2)
    assert float(junk.abs().max()) == 0.0
    w2 = _bf(2048, N, dev=gpu, scale=0.05)
    g = (torch.rand(N, device=gpu) + 0.5).to(torch.bfloat16)
    wg = w2 * g[None, :]
    y = ops.mid_gemm(hh, ops.pack_decode_weight(wg), norm=True, ss_in=ss)
    xn = hh.float() * torch.rsqrt(hh.float().pow(2).mean(-1, keepdim=True) + 1e-5)
    ref_y = xn @ wg.float().T
    torch.testing.assert_close(y.float(), ref_y, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("M,H,KV,K,fm,fn,splits", [
    (64, 32, 8, 4096, 0, 0, 0), (200, 32, 8, 4096, 0, 0, 0), (96, 8, 2, 1024, 4, 2, 3),
    (300, 4, 1, 512, 8, 4, 1), (128, 32, 8, 4096, 4, 4, 5), (160, 32, 8, 4096, 8, 2, 2),
    (96, 8, 2, 1024, 2, 2, 1), (300, 4, 1, 512, 4, 4, 3), (200, 4, 1, 512, 8, 2, 2)])
def test_mid_qkv_rope(gpu, M, H, KV, K, fm, fn, splits):
    """Mid-size norm-folded QKV projection with RoPE + paged KV write in the epilogue vs
    the fp32 projection followed by the reference rope_cache (padding slots skipped)."""
    torch.manual_seed(19)
    N = (H + 2 * KV) * 128
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    g = (torch.rand(K, device=gpu) + 0.5).to(torch.bfloat16)
    wp = ops.pack_decode_qkv_rope(w * g[None, :])
    NB = (M + 15) // 16 + 4
    cos_sin = ref.rope_cos_sin(4096).to(gpu)
    pos = torch.randint(0, 4000, (M,), dtype=torch.int32, device=gpu)
    slots = torch.randperm(NB * 16, device=gpu)[:M].to(torch.int32)
    slots[1] = -1
    kc = torch.zeros(NB, KV, 16, 16, 8, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros(NB, KV, 128, 16, dtype=torch.bfloat16, device=gpu)
    q = torch.empty(M, H, 128, dtype=torch.bfloat16, device=gpu)
    for _ in range(2):
        ops.mid_qkv_rope(x, wp, 1e-5, q, kc, vc, pos, slots, cos_sin, H, KV, fm=fm, fn=fn, splits=splits)
    xn = x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-5) * g.float()
    qkv = (xn @ w.float().T).cpu()
    rq = torch.empty(M, H, 128, dtype=torch.float32)
    rk = torch.zeros(NB, KV, 16, 16, 8)
    rv = torch.zeros(NB, KV, 128, 16)
    ref.rope_cache(rq, rk, rv, qkv, pos.cpu(), slots.cpu(), cos_sin.cpu(), H, KV)
    torch.testing.assert_close(q.float().cpu(), rq, atol=3e-2, rtol=2e-2)
    torch.testing.assert_close(kc.float().cpu(), rk, atol=3e-2, rtol=2e-2)
    torch.testing.assert_close(vc.float().cpu(), rv, atol=3e-2, rtol=2e-2)


@pytest.mark.parametrize("storage", ["bf16", "q16"])
@pytest.mark.parametrize("N,Q,K", [(100, 3, 64), (81, 2, 40), (20_000, 16, 5), (20_000, 17, 33), (32_768, 16, 32), (32_769, 2, 9), (70_000, 5, 64)])
def test_lookup_begins_with_its_best(gpu, storage, N, Q, K):
    """The first round's threshold: rows of nothing but zeros (scores of 0), ties, rows that are not finite (they are never
    hits, and do not count as the best of their four), few rows that pass, and more queries than a short slice takes."""
    from pilottai_amd.memory.semantic_index import SemanticIndex

    g = torch.Generator().manual_seed(N + Q)
    v = torch.randn(N, 64, generator=g)
    v[N // 3:] = 0.0
    v[5:9] = v[4]
    odd = torch.tensor([1, 40, 77])
    idx = SemanticIndex(dim=64, capacity=N, device=gpu, growable=False, storage=storage)
    prio, tags = torch.ones(N, dtype=torch.int32), torch.ones(N, dtype=torch.int64)
    prio[odd] = 0
    bad = v.clone()
    bad[odd[0]], bad[odd[1], 3], bad[odd[2]] = float("nan"), float("nan"), float("inf")
    norm = lambda x: x / x.norm(dim=1, keepdim=True).clamp(min=1e-12)  # noqa: E731
    q = torch.cat([v[4:5], torch.zeros(1, 64), -v[:1], torch.randn(Q, 64, generator=g)])[:Q].numpy()
    idx.add_device(norm(bad).to(gpu), prio.to(gpu), tags.to(gpu), normalized=True)
    got, want = (idx.search(q, K, [p] * Q, [()] * Q) for p in (0, 1))  # (1: the odd rows are filtered out)
    scores = lambda hits: [[x for _, x in h] for h in hits]  # noqa: E731  (of rows that tie any may be the hits)
    assert scores(got) == scores(want) and all(len(h) == min(K, N - 3) for h in want)
    if storage == "bf16":  # (in fixed point they are rows of zeros)
        assert not any(r in odd.tolist() for h in got for r, _ in h)
    idx.priority[50:] = -1
    few = idx.search(q, K, [1] * Q, [()] * Q)
    assert all({r for r, _ in h} <= set(range(50)) - set(odd.tolist()) and len(h) == min(K, 48) for h in few)


def test_semantic_index_packed_storage(gpu):
    """SemanticIndex keeps rows in packed 16-row tiles: scattered and bulk writes
    (aligned and unaligned ranges, ring wrap) read back exactly, and the HIP
    search finds planted rows."""
    from pilottai_amd.memory.semantic_index import SemanticIndex

    torch.manual_seed(16)
    D = 256
    idx = SemanticIndex(dim=D, capacity=4096, device=gpu, growable=False)
    a = torch.nn.functional.normalize(torch.randn(37, D), dim=1)
    rows = idx.add(a.numpy(), [1] * 37, [[]] * 37, [None] * 37)
    b = torch.nn.functional.normalize(torch.randn(1003, D, device=gpu), dim=1).to(torch.bfloat16)
    idx.add_device(b, torch.ones(1003, dtype=torch.int32, device=gpu), torch.zeros(1003, dtype=torch.int64, device=gpu),
                   normalized=True)
    c = torch.nn.functional.normalize(torch.randn(1024, D, device=gpu), dim=1).to(torch.bfloat16)
    idx.size = 1024  # aligned bulk write at row 1024
    idx.add_device(c, torch.ones(1024, dtype=torch.int32, device=gpu), torch.zeros(1024, dtype=torch.int64, device=gpu),
                   normalized=True)
    assert rows == list(range(37))
    torch.testing.assert_close(idx.read_rows(0, 37).float().cpu(), a.to(torch.bfloat16).float(), atol=0, rtol=0)
    torch.testing.assert_close(idx.read_rows(37, 1024), b[:987], atol=0, rtol=0)
    torch.testing.assert_close(idx.read_rows(1024, 2048), c, atol=0, rtol=0)
    q = torch.stack([idx.row(5), idx.row(1500), idx.row(700)]).float().cpu().numpy()
    res = idx.search(q, 3, [0, 0, 0], [[], [], []])
    assert [r[0][0] for r in res] == [5, 1500, 700]
