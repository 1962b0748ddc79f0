"""Large-M packed-weight projections (csrc/ops/gemm_prefill.hip: 256 x 256, 256 x 192 and
256 x 128 MFMA tiles, LDS-DMA stages, fused epilogues) vs fp32 PyTorch references."""
import pytest
import torch

from pilottai_amd import ops
from pilottai_amd.ops import reference as ref

pytestmark = pytest.mark.gpu


def _bf(*shape, dev, scale=1.0):
    return (torch.randn(*shape, device=dev) * scale).to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K,epi,norm,full,splits", [
    # Llama-3-8B projections at prefill-step sizes (default plans: whole tiles + split tail)
    (2048, 28672, 4096, "silu", True, -1, 0), (2048, 6144, 4096, "rope_perm", True, -1, 0),
    (2048, 4096, 4096, "resid", False, -1, 0), (1024, 4096, 14336, "resid", False, -1, 0),
    # partial row tiles, explicit whole / split decompositions
    (300, 4096, 4096, "plain", False, -1, 1), (777, 6144, 4096, "plain", True, 0, 3),
    (513, 28672, 4096, "silu", True, 200, 2), (1536, 4096, 14336, "resid", False, 0, 4),
    (272, 2048, 1024, "plain", False, 3, 2), (64, 1024, 512, "silu", False, -1, 0),
    (1000, 1280, 8192, "rope_perm", True, 0, 2),  # 70B TP=8 QKV shard
    (17, 768, 128, "plain", True, -1, 1), (256, 512, 64, "resid", False, 0, 1),
    # more than one round of 256-wide tiles with a short tail (the default variant runs the
    # tail columns on 256 x 128 tiles in the same launch)
    (1024, 20480, 512, "rope_perm", True, -1, 0), (768, 24576, 256, "resid", False, -1, 0),
    (1000, 28672, 256, "plain", False, -1, 0),
    # blocks of row tiles, the last one smaller: whole columns, a split from amid a column on, whole and split columns
    (2100, 1280, 256, "plain", True, -1, 1), (2100, 1280, 512, "resid", False, 13, 2), (4000, 768, 512, "silu", False, 32, 2)])
@pytest.mark.parametrize("bn,variant", [(256, 3), (256, 9), (256, 1), (128, 3), (128, 1)])
def test_prefill_gemm(gpu, M, N, K, epi, norm, full, splits, bn, variant):
    """Every epilogue and the folded row norm; run twice so the self-resetting tickets of
    the split tail are exercised. Ping-pong kernels (variant 3, the default: two-phase
    256-wide / three-buffer 128-wide schedules; 9: without the mixed 128-wide tail) and the
    read-ahead / 3-stage kernels (variant 1, the fallback for < 2 k-tiles)."""
    from pilottai_amd.ops import kernels

    kernels.require_native().prefill_set_variant(variant)
    try:
        _check_prefill_gemm(gpu, M, N, K, epi, norm, full, splits, bn)
    finally:
        kernels.require_native().prefill_set_variant(-1)


def _check_prefill_gemm(gpu, M, N, K, epi, norm, full, splits, bn):
    torch.manual_seed(21)
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
        y = ops.prefill_gemm(x, wp, epi, resid=resid, norm=norm, full=full, splits=splits, bn=bn)
        torch.testing.assert_close(y.float(), acc, atol=4e-2, rtol=2e-2)


@pytest.mark.parametrize("M,N,K,epi,norm,full,splits", [
    # qkv of Llama-3-8B at 1,280 < M <= 2,048 (one round of 256 x 192 tiles)
    (2048, 6144, 4096, "rope_perm", True, -1, 0), (1536, 6144, 4096, "plain", False, -1, 1),
    (1300, 6144, 4096, "plain", True, -1, 0),
    # K-sliced items, every epilogue, partial row tiles, two k-tiles per item
    (777, 6144, 4096, "plain", True, 0, 3), (513, 6144, 4096, "silu", True, 10, 2),
    (1000, 6144, 14336, "resid", False, 0, 4), (300, 1536, 128, "resid", False, -1, 1),
    (2100, 11520, 512, "rope_perm", True, -1, 0), (64, 384, 256, "plain", False, 0, 2)])
def test_prefill_gemm_192(gpu, M, N, K, epi, norm, full, splits):
    """256 x 192 tiles (gemm_pingpong.h F = 6, `body6` schedule) vs fp32: whole tiles and
    K-slices, every register epilogue."""
    _check_prefill_gemm(gpu, M, N, K, epi, norm, full, splits, 192)


def test_prefill_gemm_192_refuses_other_widths(gpu):
    """bn = 192 needs N % 192 == 0 and the ping-pong schedule: anything else is refused at
    the launcher instead of running a partial tile."""
    x = _bf(512, 512, dev=gpu)
    wp = ops.pack_decode_weight(_bf(1024, 512, dev=gpu))
    with pytest.raises(ValueError, match="does not handle"):
        ops.prefill_gemm(x, wp, "plain", bn=192)


@pytest.mark.parametrize("M,N,K,bn", [
    (2817, 3072, 128, 192), (2816, 3072, 768, 192), (2560, 3072, 768, 128), (2561, 4096, 192, 256), (4096, 4096, 512, 256), (2304, 4096, 1024, 128),
    (2048, 4096, 256, 128), (500, 10752, 256, 128), (1000, 10752, 1024, 192), (500, 10752, 1024, 256), (1500, 10752, 256, 256),
    (2900, 1920, 128, 128), (2900, 3072, 64, 128)])
def test_prefill_gemm_default_width(gpu, M, N, K, bn):
    """The width that a call leaves open follows the rounds of its tiles, on both sides of the lines, and changes no bits; launches with slices of k
    and the kernels of fewer than two k-tiles keep the line by N."""
    from pilottai_amd.ops import kernels

    assert kernels.require_native().prefill_gemm_plan(M, N, K)[3] == bn
    _check_prefill_gemm(gpu, M, N, K, "plain", False, -1, 0, 0)
    x, wp = _bf(M, K, dev=gpu), ops.pack_decode_weight(_bf(N, K, dev=gpu, scale=0.05))
    line = 128 if N % 256 or N <= 6144 else 256
    assert torch.equal(ops.prefill_gemm(x, wp), ops.prefill_gemm(x, wp, bn=line))
    if K >= 128:
        _check_prefill_gemm(gpu, M, N, K, "plain", False, 0, 2, 0)


@pytest.mark.parametrize("variant", [3, 4, 8, 9])  # with a mixed tail and without
def test_prefill_gemm_default_width_of_a_family(gpu, variant):
    x, wp = _bf(3500, 1024, dev=gpu), ops.pack_decode_weight(_bf(6144, 1024, dev=gpu, scale=0.05))
    assert torch.equal(ops.prefill_gemm(x, wp, variant=variant), ops.prefill_gemm(x, wp, bn=128, variant=variant))


@pytest.mark.parametrize("bn,variant", [(256, -1), (192, -1), (128, -1), (256, 1)])
def test_prefill_gemm_asymmetric_identity(gpu, bn, variant):
    """x = I (rows), W asymmetric: the output must be exactly W^T's rows (catches a
    transposed or permuted C write, guide §3 'A = I-check with asymmetric B')."""
    M, N, K = 512, 1152 if bn == 192 else 1024, 512
    x = torch.zeros(M, K, device=gpu)
    x[torch.arange(M), torch.arange(M) % K] = 1.0
    w = (torch.arange(N * K, device=gpu, dtype=torch.float32).view(N, K) % 251 / 64.0).to(torch.bfloat16)
    y = ops.prefill_gemm(x.to(torch.bfloat16), ops.pack_decode_weight(w), "plain", full=-1, splits=1, bn=bn,
                         variant=variant)
    want = w.float().T[torch.arange(M) % K]
    assert torch.equal(y.float(), want.to(torch.bfloat16).float())


@pytest.mark.parametrize("M,S", [(700, 1), (700, 3), (2048, 2)])
@pytest.mark.parametrize("bn", [256, 128])
def test_prefill_gemm_resid_in_place_with_row_stats(gpu, M, S, bn):
    """h += x W^T in place, accumulating the next norm's row statistics (ss_out) of the
    written bf16 rows and zeroing another buffer (ss_zero); the following norm-folded
    projection consuming them matches rmsnorm + GEMM."""
    torch.manual_seed(22)
    N, K = 4096, 4096
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    h = _bf(M, N, dev=gpu)
    want = h.float() + x.float() @ w.float().T
    hh = h.clone()
    ss = torch.zeros(M, dtype=torch.float32, device=gpu)
    junk = torch.full((M,), 7.0, device=gpu)
    ops.prefill_gemm(x, ops.pack_decode_weight(w), "resid", resid=hh, out=hh, full=0 if S > 1 else -1,
                     splits=S, ss_out=ss, ss_zero=junk, bn=bn)
    torch.testing.assert_close(hh.float(), want, atol=4e-2, rtol=2e-2)
    torch.testing.assert_close(ss, hh.float().pow(2).sum(-1), rtol=1e-4, atol=1e-2)
    assert float(junk.abs().max()) == 0.0
    w2 = _bf(2048, N, dev=gpu, scale=0.05)
    g = (torch.rand(N, device=gpu) + 0.5).to(torch.bfloat16)
    wg = w2 * g[None, :]
    y = ops.prefill_gemm(hh, ops.pack_decode_weight(wg), norm=True, ss_in=ss, bn=bn)
    xn = hh.float() * torch.rsqrt(hh.float().pow(2).mean(-1, keepdim=True) + 1e-5)
    torch.testing.assert_close(y.float(), xn @ wg.float().T, atol=4e-2, rtol=2e-2)


@pytest.mark.parametrize("M,H,KV,K,full,splits", [
    (1024, 32, 8, 4096, -1, 0), (333, 32, 8, 4096, 0, 4), (600, 8, 2, 1024, -1, 1), (2048, 32, 8, 4096, 0, 2),
    (1792, 32, 8, 4096, -1, 0)])
@pytest.mark.parametrize("bn", [256, 192, 128])
def test_prefill_qkv_rope(gpu, M, H, KV, K, full, splits, bn):
    """Norm-folded QKV with RoPE + paged KV write vs fp32 projection + reference rope_cache."""
    torch.manual_seed(23)
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
        ops.prefill_qkv_rope(x, wp, 1e-5, q, kc, vc, pos, slots, cos_sin, H, KV, full=full, splits=splits, bn=bn)
    xn = x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-5) * g.float()
    qkv = (xn @ w.float().T).cpu()
    rq = torch.empty(M, H, 128, dtype=torch.float32)
    rk = torch.zeros(NB, KV, 16, 16, 8)
    rv = torch.zeros(NB, KV, 128, 16)
    ref.rope_cache(rq, rk, rv, qkv, pos.cpu(), slots.cpu(), cos_sin.cpu(), H, KV)
    torch.testing.assert_close(q.float().cpu(), rq, atol=4e-2, rtol=2e-2)
    torch.testing.assert_close(kc.float().cpu(), rk, atol=4e-2, rtol=2e-2)
    torch.testing.assert_close(vc.float().cpu(), rv, atol=4e-2, rtol=2e-2)


@pytest.mark.parametrize("M,H,KV,K", [(3500, 32, 8, 1024), (4096, 32, 8, 1024), (2900, 16, 4, 128), (1100, 64, 8, 1024)])
def test_prefill_qkv_rope_default_width(gpu, M, H, KV, K):
    """The width that a call leaves open: this epilogue has no mixed tail, so that a wider tile would bring slices of k. The bits are the
    line's by N."""
    N = (H + 2 * KV) * 128
    x, wp = _bf(M, K, dev=gpu), ops.pack_decode_qkv_rope(_bf(N, K, dev=gpu, scale=0.05))
    cos_sin, rows = ref.rope_cos_sin(4096).to(gpu), torch.arange(M, dtype=torch.int32, device=gpu)
    got = []
    for bn in (0, 128 if N % 256 or N <= 6144 else 256):
        q, kc, vc = (torch.zeros(*s, dtype=torch.bfloat16, device=gpu) for s in ((M, H, 128), (M // 16 + 1, KV, 16, 16, 8), (M // 16 + 1, KV, 128, 16)))
        ops.prefill_qkv_rope(x, wp, 1e-5, q, kc, vc, rows, rows, cos_sin, H, KV, bn=bn)
        got.append((q, kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("epi", ["plain", "resid"])
def test_prefill_gemm_strided_views(gpu, epi):
    """The plain / residual epilogues store (and read the residual) 16 B per lane: a padded
    output view with 16-byte rows is written correctly, a view whose rows are only 8-byte
    aligned is refused at the binding instead of issuing misaligned wide accesses."""
    torch.manual_seed(5)
    M, N, K = 300, 1024, 512
    x = _bf(M, K, dev=gpu)
    w = _bf(N, K, dev=gpu, scale=0.05)
    wp = ops.pack_decode_weight(w)
    want = x.float() @ w.float().T
    big = torch.zeros(M, N + 8, dtype=torch.bfloat16, device=gpu)  # padded rows, 16-B aligned
    resid = None
    if epi == "resid":
        rbig = _bf(M, N + 16, dev=gpu)
        resid = rbig[:, 8:8 + N]
        want = want + resid.float()
    y = ops.prefill_gemm(x, wp, epi, resid=resid, out=big[:, :N])
    torch.testing.assert_close(y.float(), want, atol=4e-2, rtol=2e-2)
    assert torch.equal(big[:, N:], torch.zeros_like(big[:, N:]))  # the padding is untouched
    odd = torch.zeros(M, N + 4, dtype=torch.bfloat16, device=gpu)[:, 4:]  # 8-byte aligned only
    with pytest.raises(RuntimeError, match="16-byte"):
        ops.prefill_gemm(x, wp, epi, resid=resid, out=odd)


@pytest.mark.parametrize("epi", ["plain", "resid", "silu"])
@pytest.mark.parametrize("M,live,N,K,bn", [(2049, 1, 512, 128, 0), (2304, 2047, 512, 192, 0), (2304, 2048, 1536, 512, 192),
                                           (2500, 2049, 512, 1024, 128), (3072, 2101, 7168, 256, 0), (4096, 0, 512, 128, 256)])
def test_prefill_tiles_without_a_token(gpu, M, live, N, K, bn, epi):
    """Whole tiles of 256 rows behind the last token stay as they were, on every tile width, in split tiles and in a mixed
    tail; all other rows are those of a launch that knows of no padding."""
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K, generator=g).to(gpu, torch.bfloat16)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(gpu, torch.bfloat16)
    slots = torch.arange(M, dtype=torch.int32)
    slots[live:] = -1
    NO = N // 2 if epi == "silu" else N
    kw = dict(bn=bn, resid=torch.randn(M, N, generator=g).to(gpu, torch.bfloat16) if epi == "resid" else None)
    wp = ops.pack_decode_weight(w)
    want = ops.prefill_gemm(x, wp, epi, **kw)
    got = torch.full((M, NO), 7.0, device=gpu, dtype=torch.bfloat16)
    ops.prefill_gemm(x, wp, epi, out=got, live=slots.to(gpu), **kw)
    edge = (live + 255) // 256 * 256
    assert torch.equal(got[:edge], want[:edge])
    assert (got[edge:] == 7.0).all()
    ops.prefill_gemm(x, wp, epi, out=got, **kw)  # (tickets of tiles left out are as they were)
    assert torch.equal(got, want)


@pytest.mark.parametrize("T,live", [(700, 300), (512, 256), (257, 256), (300, 0)])
def test_dense_unit_tiles_without_a_token(gpu, T, live):
    """The same of the gated unit's tiles of 256 rows (one group)."""
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, 256, generator=g).to(gpu, torch.bfloat16)
    w = (torch.randn(1, 512, 256, generator=g) / 16).to(gpu, torch.bfloat16)
    wp = ops.pack_groups(w, torch.bfloat16)
    tiles = torch.tensor([[0, i, min(256, T - i), 0] for i in range(0, T, 256)], dtype=torch.int32, device=gpu)
    n = torch.tensor([len(tiles)], dtype=torch.int32, device=gpu)
    order = torch.arange(T, dtype=torch.int32, device=gpu)
    slots = torch.where(order < live, order, -1)

    def run(**kw):
        out = torch.full((T, 256), 7.0, device=gpu, dtype=torch.bfloat16)
        return ops.expert_gemm(x, wp, out, tiles, n, order, T, x_div=0, out_order=False, tm=256, glu=(3e38, 1.0, 0.0), **kw)
    want, got, edge = run(), run(live=slots.to(torch.int32)), (live + 255) // 256 * 256
    assert torch.equal(got[:edge], want[:edge])
    assert (got[edge:] == 7.0).all()


@pytest.mark.parametrize("bn,variant", [(256, 3), (256, 1), (192, 3), (128, 3), (128, 1)])
@pytest.mark.parametrize("S", [3, 4])
def test_split_tiles_add_up_in_the_order_of_the_slices(gpu, bn, variant, S):
    """A split tile's sum does not depend on which slice arrives last. Slices of 2^30, 1, (1,) -2^30 are 0 in fp32 added in their
    order and 1 or 2 from the last one on; values of no such kind give the same bits on every run."""
    M, N, K = 700, 1536, S * 256
    x = torch.zeros(M, K, device=gpu, dtype=torch.bfloat16)
    for s in range(S):
        x[:, s * 256] = 2.0 ** 30 if s == 0 else -2.0 ** 30 if s == S - 1 else 1.0
    ones = ops.pack_decode_weight(torch.ones(N, K, device=gpu, dtype=torch.bfloat16))
    torch.manual_seed(S)
    y, w = _bf(M, K, dev=gpu), ops.pack_decode_weight(_bf(N, K, dev=gpu))
    kw = dict(full=0, splits=S, bn=bn, variant=variant)
    first = ops.prefill_gemm(y, w, **kw)
    for _ in range(20):
        assert not ops.prefill_gemm(x, ones, **kw).any()
        assert torch.equal(ops.prefill_gemm(y, w, **kw), first)
