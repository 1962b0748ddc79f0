"""Kernels of csrc/ops/{residual_norm, latent_cache, latent_attention, grouped_gemm}.hip against
plain fp32 formulas, in bf16 (MFMA) and fp32, at sizes that are not whole tiles."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DTYPES = [torch.bfloat16, torch.float32]


def tol(dt):
    return dict(rtol=2e-2, atol=2e-2) if dt == torch.bfloat16 else dict(rtol=2e-5, atol=2e-5)


def norm(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("D,K,add", [(192, 1, None), (100, 3, "add"), (2048, 6, "add"), (50, 2, "set"), (4096, 1, None)])
def test_residual_norm(gpu, dt, D, K, add):
    from pilottai_amd import ops

    g = torch.Generator().manual_seed(D + K)
    T, V, ld, eps = 9, 31, (D + 63) // 64 * 64, 1e-4
    r, y = torch.randn(T, D, generator=g), torch.randn(T * K, ld, generator=g).to(dt)
    wp, wn = torch.rand(D, generator=g) + 0.5, torch.rand(D, generator=g) + 0.5
    emb, ids = torch.randn(V, D, generator=g).to(dt), torch.randint(0, V, (T,), generator=g, dtype=torch.int32)
    kw = dict(y=y, partials=K, y_scale=1 / K, w_post=wp)
    want = r + norm(y.float()[:, :D].view(T, K, D).sum(1) / K, wp, eps)
    if add == "add":
        want, kw = want + emb[ids.long()].float(), dict(kw, emb=emb, ids=ids, emb_add=True)
    elif add == "set":
        want, kw = emb[ids.long()].float(), dict(emb=emb, ids=ids)
    kw = {k: v.to(gpu) if torch.is_tensor(v) else v for k, v in kw.items()}
    rows = torch.tensor([3, 0, 3, 8], dtype=torch.int32)
    rg = r.to(gpu)
    out = torch.full((4, ld), 7.0, dtype=dt, device=gpu)
    ops.residual_norm(rg, eps, w_next=wn.to(gpu), out=out, rows=rows.to(gpu), **kw)  # leaves the residual alone
    torch.testing.assert_close(rg.cpu(), r, rtol=0, atol=0)
    torch.testing.assert_close(out.float().cpu()[:, :D], norm(want, wn, eps)[rows.long()], **tol(dt))
    assert not out[:, D:].any()
    out = torch.full((T, ld), 7.0, dtype=dt, device=gpu)
    ops.residual_norm(rg, eps, w_next=wn.to(gpu), out=out, **kw)
    torch.testing.assert_close(rg.cpu(), want, rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(out.float().cpu()[:, :D], norm(want, wn, eps), **tol(dt))


@pytest.mark.parametrize("T,live,D", [(2049, 1, 512), (2500, 2046, 1024), (2304, 3, 2048), (2050, 2049, 4096), (2100, 77, 100)])
def test_residual_norm_leaves_rows_without_a_token(gpu, T, live, D):
    """One, two and four waves a row and widths that are no whole 8s; a workgroup with a token does all of its rows."""
    from pilottai_amd import ops

    g = torch.Generator().manual_seed(T)
    r, y, w = (torch.randn(*s, generator=g).to(gpu) for s in ((T, D), (T, D), (D,)))
    slots = torch.arange(T, dtype=torch.int32, device=gpu)
    slots[live:] = -1

    def run(**kw):
        rg, out = r.clone(), torch.full((T, D), 7.0, dtype=torch.bfloat16, device=gpu)
        ops.residual_norm(rg, 1e-5, y=y.to(torch.bfloat16), w_post=w, w_next=w, out=out, **kw)
        return rg, out
    (ra, a), (rb, b), edge = run(), run(live=slots), (live + 3) // 4 * 4
    assert torch.equal(ra[:live], rb[:live]) and torch.equal(a[:live], b[:live])
    assert torch.equal(rb[edge:], r[edge:]) and (b[edge:] == 7.0).all()


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("T", [1, 40, 130])
@pytest.mark.parametrize("G,N,K", [(3, 48, 32), (5, 208, 96), (2, 512, 128)])
def test_head_gemm(gpu, dt, T, G, N, K):
    from pilottai_amd import ops

    g = torch.Generator().manual_seed(T + N)
    x, w = torch.randn(T, G * (K + 32), generator=g).to(dt), (torch.randn(G, N, K, generator=g) / math.sqrt(K)).to(dt)
    out = torch.full((T, G * (N + 16)), 5.0, dtype=dt, device=gpu)
    ops.head_gemm(x.to(gpu), K + 32, ops.pack_groups(w, dt).to(gpu), out, N + 16)
    o = out.float().cpu().view(T, G, N + 16)
    want = torch.einsum("tgk,gnk->tgn", x.float().view(T, G, K + 32)[:, :, :K], w.float())
    torch.testing.assert_close(o[:, :, :N], want, **tol(dt))
    assert (o[:, :, N:] == 5.0).all()


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("T,G,N,K", [(32705, 1, 256, 32), (2049, 16, 272, 160), (1100, 33, 512, 256), (4095, 8, 512, 128), (4097, 16, 544, 256), (3100, 17, 256, 96)])
def test_head_gemm_of_many_rows(gpu, T, G, N, K, gated):
    """Two workgroups of 64 rows a CU and more: sizes that are no multiple of a tile, the widest inputs, beside rotated
    columns. Sums of K products in fp32 err by K 2^-24 of their magnitudes at most, a bf16 result rounds by 2^-8."""
    from pilottai_amd import ops

    g = torch.Generator(device=gpu).manual_seed(T)
    rnd = lambda *s: torch.randn(*s, device=gpu, generator=g)  # noqa: E731
    hs, r = K + 24, 16
    x, w = rnd(T, G * hs).bfloat16(), (rnd(G, N, K) / math.sqrt(K)).bfloat16()
    pos = torch.randint(0, 50, (T,), device=gpu, generator=g, dtype=torch.int32)
    ang = rnd(50, r // 2)
    cs = torch.cat([ang.cos(), ang.sin()], 1).contiguous()
    out = torch.full((T, G * (N + 32 + 8)), 5.0, dtype=torch.bfloat16, device=gpu)
    gate = rnd(T, G * (N + 40)).bfloat16() if gated else None
    ops.head_gemm(x, hs, ops.pack_groups(w, torch.bfloat16), out, N + 40, None if gated else (pos, cs, K, r, 32), gate)
    for h in range(G):
        xs, o = x[:, h * hs:(h + 1) * hs].float(), out[:, h * (N + 40):(h + 1) * (N + 40)].float()
        want, slack = xs[:, :K] @ w[h].float().T, K * 2.0 ** -24 * (xs[:, :K].abs() @ w[h].float().abs().T)
        if gated:
            s = torch.sigmoid(gate[:, h * (N + 40):h * (N + 40) + N].float())
            want, slack = want * s, slack * s + 2.0 ** -20 * want.abs()
        assert bool(((o[:, :N] - want).abs() <= 2.0 ** -8 * want.abs() + slack + 1e-30).all()) and bool((o[:, N + 32:] == 5.0).all())
        if not gated:
            u, v, c, sn = xs[:, K:K + r // 2], xs[:, K + r // 2:K + r], cs[pos.long(), :r // 2], cs[pos.long(), r // 2:]
            turned = torch.cat([u * c - v * sn, v * c + u * sn], 1)
            torch.testing.assert_close(o[:, N:N + r], turned, **tol(torch.bfloat16))
            assert not o[:, N + r:N + 32].any()


@pytest.mark.parametrize("T,layers", [(4096, [(64, 2), (2048, 3)]), (4097, [(64, 2), (5, 1)]), (1367, [(1025, 6), (7, 7)]), (9000, [(3, 2)])])
def test_table_route_slices(gpu, T, layers):
    """Up to two slices of positions and more, a layer with fewer slices than its neighbour, slices of padding alone: rows by
    expert and tiles of them, whatever the order of an expert's rows."""
    from pilottai_amd import ops

    g, V, tm = torch.Generator().manual_seed(T), 97, 64
    tabs = [torch.stack([torch.randperm(max(E, top), generator=g)[:top] % E for _ in range(V)]).int() for E, top in layers]
    ids, slots = torch.randint(0, V, (T,), generator=g, dtype=torch.int32), torch.arange(T, dtype=torch.int32)
    slots[T // 2: T // 2 + T // 5] = -1
    rows, o, t, tab = [], 0, 0, 0
    for E, top in layers:
        cap = T * top // tm + E
        rows.append([tab, V, top, E, o, t, cap, 0])
        tab, o, t = tab + V * top, o + T * top, t + cap
    desc = torch.tensor(rows, dtype=torch.int32)
    order, tiles, n = (torch.full(x, -7, dtype=torch.int32, device=gpu) for x in ((o,), (t, 4), (len(layers),)))
    for _ in range(2):
        ops.table_route(torch.cat([x.reshape(-1) for x in tabs]).to(gpu), desc.to(gpu), desc, ids.to(gpu), slots.to(gpu), T, tm, order, tiles, n)
    for k, (E, top) in enumerate(layers):
        expert = torch.where(slots[:, None] >= 0, tabs[k][ids.long()], -1).reshape(-1)
        got, at, listed = order[rows[k][4]:].cpu(), 0, []
        for e in range(E):
            want = torch.nonzero(expert == e).view(-1)
            assert torch.equal(got[at:at + len(want)].sort().values.long(), want)
            listed += [[e, at + b, min(tm, len(want) - b), 0] for b in range(0, len(want), tm)]
            at += len(want)
        assert int(n[k]) == len(listed) and tiles[rows[k][5]:][:len(listed)].tolist() == listed


@pytest.mark.parametrize("dt,tm", [(torch.bfloat16, 16), (torch.bfloat16, 64), (torch.bfloat16, 256), (torch.float32, 16)])
@pytest.mark.parametrize("T,E,top,ff,D", [(1, 5, 2, 40, 96), (900, 4, 2, 72, 200), (600, 2, 2, 128, 256), (77, 7, 3, 96, 160), (300, 12, 1, 64, 64), (130, 70, 5, 32, 128)])
def test_table_experts(gpu, dt, tm, T, E, top, ff, D):
    from pilottai_amd import ops
    from pilottai_amd.ops.latent import pad_to

    g = torch.Generator().manual_seed(T * E)
    V, lim, fp = 50, 0.7, pad_to(ff, 128 if tm == 256 else 32)
    tabs = [torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(V)]).int() for _ in range(2)]
    ids = torch.randint(0, V, (T,), generator=g, dtype=torch.int32)
    slots = torch.arange(T, dtype=torch.int32)
    slots[T // 3: T // 3 + T // 8] = -1  # padding rows go through no expert
    cap = T * top // tm + min(E, T * top)
    desc = torch.tensor([[i * V * top, V, top, E, i * T * top, i * cap, cap, 0] for i in range(2)], dtype=torch.int32)
    order = torch.empty(2 * T * top, dtype=torch.int32, device=gpu)
    tiles = torch.empty(2 * cap, 4, dtype=torch.int32, device=gpu)
    nt = torch.empty(2, dtype=torch.int32, device=gpu)
    ops.table_route(torch.cat([t.reshape(-1) for t in tabs]).to(gpu), desc.to(gpu), desc, ids.to(gpu), slots.to(gpu), T,
                    tm, order, tiles, nt)
    DK, DN = (pad_to(D, 128),) * 2 if tm == 256 else (pad_to(D, 32), pad_to(D, 16))
    x = torch.randn(T, pad_to(D, 128), generator=g).to(dt)
    w1, w3 = [(torch.randn(E, ff, D, generator=g) / math.sqrt(D) * 1.5).to(dt) for _ in range(2)]
    w2 = (torch.randn(E, D, ff, generator=g) / math.sqrt(ff)).to(dt)
    z = lambda a, b: torch.zeros(E, a, b, dtype=dt)  # noqa: E731
    g1, g3, g2 = z(fp, DK), z(fp, DK), z(DN, fp)
    g1[:, :ff, :D], g3[:, :ff, :D], g2[:, :D, :ff] = w1, w3, w2
    p13 = ops.pack_groups(ops.interleave_gate_up(g1, g3), dt).to(gpu)
    p2 = ops.pack_groups(g2, dt).to(gpu)
    for i, tab in enumerate(tabs):
        act = torch.empty(T * top, fp, dtype=dt, device=gpu)
        y = torch.full((T * top, DN), 3.0, dtype=dt, device=gpu)
        sel = (tiles[i * cap:(i + 1) * cap], nt[i:i + 1], order[i * T * top:(i + 1) * T * top], T * top)
        ops.expert_gemm(x.to(gpu), p13, act, *sel, x_div=top, out_order=False, tm=tm, glu=(lim, 1.702, 1.0))
        ops.expert_gemm(act, p2, y, *sel, x_div=0, out_order=True, tm=tm)
        y = y.float().cpu().view(T, top, -1)[:, :, :D]
        assert (y[slots < 0] == 3.0).all()
        es = tab[ids.long()].long()
        for e in range(E):
            t, k = torch.nonzero((es == e) & (slots >= 0)[:, None], as_tuple=True)
            v = x[t, :D].float()
            a, u = (v @ w1[e].float().T).clamp(max=lim), (v @ w3[e].float().T).clamp(-lim, lim)
            torch.testing.assert_close(y[t, k], (a * torch.sigmoid(1.702 * a) * (u + 1)) @ w2[e].float().T, **tol(dt))


def sorted_rows(gpu, tm, counts, N, K, always=0):
    """The grouped projections of sorted rows of one tile size: plain, the square of relu and gated with weights of rows,
    gathered and scattered. Sums of K products in fp32 err by K 2^-24 of their magnitudes at most, a bf16 result rounds by
    2^-8; silu(g) u moves by at most 1.1 |u| dg + |g| du."""
    from pilottai_amd import ops

    g = torch.Generator(device=gpu).manual_seed(N + K + len(counts))
    rnd = lambda *s: torch.randn(*s, device=gpu, generator=g)  # noqa: E731
    G, rows, top = len(counts), sum(counts), 2
    T = (rows + top - 1) // top
    x, w = rnd(T, K + 8).bfloat16()[:, :K], (rnd(G, N, K) / math.sqrt(K)).bfloat16()
    order = torch.randperm(T * top, device=gpu, generator=g)[:rows].int()
    tl, p = [], 0
    for e, n in enumerate(counts):
        tl += [[e, p + i, min(tm, n - i), 0] for i in range(0, n, tm)]
        p += n
    nt = torch.tensor([len(tl)], dtype=torch.int32, device=gpu)
    cap = rows // tm + min(G, rows)
    assert len(tl) <= cap
    tiles = torch.tensor(tl + [[0, 0, 0, 0]] * (cap - len(tl)), dtype=torch.int32, device=gpu)
    of = torch.repeat_interleave(torch.arange(G, device=gpu), torch.tensor(counts, device=gpu))
    xs = x.float()[order.long() // top]
    z, size = torch.empty(rows, N, device=gpu), torch.empty(rows, N, device=gpu)
    for e in range(G):
        z[of == e], size[of == e] = xs[of == e] @ w[e].float().T, xs[of == e].abs() @ w[e].float().abs().T
    slack = K * 2.0 ** -24 * size
    pw, args = ops.pack_groups(w, torch.bfloat16), (tiles, nt, order, rows)
    out = torch.full((T * top, N + 8), 9.0, dtype=torch.bfloat16, device=gpu)
    for relu2 in (False, True):
        want = z.clamp(min=0) ** 2 if relu2 else z
        err = 2.0 ** -8 * want.abs() + slack * ((2 * z.abs() + slack) if relu2 else 1)
        ops.expert_gemm(x, pw, out[:, :N], *args, x_div=top, out_order=True, tm=tm, relu2=relu2, always=always)
        assert bool(((out[order.long(), :N].float() - want).abs() <= err).all()) and bool((out[:, N:] == 9.0).all())
    if N % 32:
        return
    rw = torch.rand(T * top, device=gpu, generator=g) + 0.5
    zg = z.view(rows, N // 32, 2, 16) * rw[order.long(), None, None, None]
    sl = slack.view(rows, N // 32, 2, 16) * rw[order.long(), None, None, None] + 2.0 ** -22 * zg.abs()
    a, u = zg[:, :, 0], zg[:, :, 1]
    want = torch.nn.functional.silu(a) * u
    err = 2.0 ** -8 * want.abs() + 1.1 * u.abs() * sl[:, :, 0] + a.abs() * sl[:, :, 1] + 2.0 ** -20 * want.abs() + 1e-30
    out = torch.empty(rows, N // 2, dtype=torch.bfloat16, device=gpu)
    ops.expert_gemm(x, pw, out, *args, x_div=top, out_order=False, tm=tm, glu=(3e38, 1.0, 0.0), row_w=rw, always=always)
    assert bool(((out.float() - want.reshape(rows, -1)).abs() <= err.reshape(rows, -1)).all())


@pytest.mark.parametrize("tm", [16, 32, 64, 128])
@pytest.mark.parametrize("counts,N,K", [
    ([1, 0, 16, 17, 40, 130, 3], 96, 96),       # empty and single-row groups, remainders of every tile, k past no stage's end
    ([5, 33], 80, 2048), ([200] * 3, 2816, 32),  # an odd number of 16-row blocks; more blocks than XCDs
    ([7], 16384, 64), ([100], 16384, 320), ([300], 4096, 160), ([300], 16384, 96),   # one group: 4, 2 and 1 waves over k
    ([30, 1] * 20, 1040, 512), ([40] * 20, 1024, 512), ([7] * 100, 80, 1088), ([20, 2, 33], 288, 256)])  # few inputs, few outputs
def test_sorted_rows(gpu, tm, counts, N, K):
    sorted_rows(gpu, tm, counts, N, K)


@pytest.mark.parametrize("counts", [[1, 64, 65, 0, 128, 129], [192, 193, 256], [257, 320, 321, 2], [384, 385, 449]])
@pytest.mark.parametrize("N,K", [(256, 128), (384, 192), (512, 320)])  # 256 and 128 columns a tile; 2, 3 and 5 steps over k
def test_sorted_rows_of_whole_tiles(gpu, counts, N, K):
    """Tiles of 256 rows that hold every number of their 64-row parts."""
    sorted_rows(gpu, 256, counts, N, K)


@pytest.mark.parametrize("counts,always", [([3, 0, 70, 12] * 4 + [290], 1), ([40] * 3 + [1300], 1), ([9] * 5 + [600, 600], 2), ([0, 0, 513], 1),
                                           ([20, 30, 0], 1), ([1] * 7 + [16400], 1)])  # of no rows; of more than 64 tiles
@pytest.mark.parametrize("N,K", [(1280, 128), (384, 192)])
def test_tiles_of_groups_of_every_row(gpu, counts, always, N, K):
    sorted_rows(gpu, 256, counts, N, K, always)


@pytest.mark.parametrize("counts,always", [([3] * 70 + [0] * 40, 0), ([4] * 6 + [0] * 10, 0), ([70, 0] * 26 + [0] * 20 + [300], 1), ([9] * 64 + [0] * 40, 0)])
@pytest.mark.parametrize("N,K", [(1280, 128), (512, 320)])
def test_remainders_of_whole_rounds(gpu, counts, always, N, K):
    """Tiles behind an XCD's last 32, none and up to 16 of them, in halves."""
    sorted_rows(gpu, 256, counts, N, K, always)


def test_groups_of_every_row_are_some(gpu):
    from pilottai_amd import ops

    x, w = torch.zeros(4, 128, device=gpu).bfloat16(), ops.pack_groups(torch.zeros(2, 128, 128, device=gpu), torch.bfloat16)
    ints = lambda *n: torch.zeros(*n, dtype=torch.int32, device=gpu)  # noqa: E731
    for always in (-1, 2):
        with pytest.raises(RuntimeError):
            ops.expert_gemm(x, w, x.clone(), ints(1, 4), ints(1), ints(4), 4, x_div=0, out_order=False, tm=256, always=always)


@pytest.mark.parametrize("rows", [1, 257, 1024, 1025, 1600, 2049])  # below, at and past a block of four row tiles, a second block's 1 to 4
@pytest.mark.parametrize("N,K", [(1280, 128), (384, 192)])  # 5 columns of 256 and 3 of 128: XCDs start amid a block
def test_row_tiles_of_one_group(gpu, rows, N, K):
    sorted_rows(gpu, 256, [rows], N, K)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("NQ,R,r,rd,H", [(72, 104, 48, 48, 3), (50, 70, 24, 12, 5), (256, 512, 64, 64, 2)])
def test_latent_cache_and_query_rotation(gpu, dt, NQ, R, r, rd, H):
    from pilottai_amd import ops
    from pilottai_amd.ops import reference as ref
    from pilottai_amd.ops.latent import latent_pad, pad_to

    g = torch.Generator().manual_seed(R)
    T, Rp, rp, eps, base = 37, latent_pad(R), pad_to(r, 32), 1e-3, 900.0
    x = torch.randn(T, pad_to(NQ + R + r, 128), generator=g).to(dt)
    wq, wc = torch.rand(NQ, generator=g) + 0.5, torch.rand(R, generator=g) + 0.5
    pos = torch.arange(T, dtype=torch.int32) * 7 + 3
    slots = torch.randperm(5 * 16, generator=g)[:T].int()
    slots[5] = -1
    cs = ref.rope_cos_sin(400, rd, base)
    cq = torch.full((T, pad_to(NQ, 64)), 9.0, dtype=dt, device=gpu)
    pages = torch.full((5, (Rp + rp) // 8, 16, 8), 4.0, dtype=dt, device=gpu)
    ops.latent_cache(x.to(gpu), NQ, R, r, wq.to(gpu), wc.to(gpu), cq, pages, Rp, pos.to(gpu), slots.to(gpu), cs.to(gpu), eps)
    torch.testing.assert_close(cq.float().cpu()[:, :NQ], norm(x.float()[:, :NQ], wq, eps), **tol(dt))
    assert not cq[:, NQ:].any()

    def rot(v, p):  # [.., r]
        a = torch.tensor([p * base ** (-2.0 * i / rd) for i in range(rd // 2)], dtype=torch.float64)
        c, s = a.cos().float(), a.sin().float()
        u, w = v[..., :rd // 2], v[..., rd // 2:rd]
        return torch.cat([u * c - w * s, w * c + u * s, v[..., rd:]], -1)

    rows = pages.float().cpu().permute(0, 2, 1, 3).reshape(80, -1)
    for t in range(T):
        if slots[t] < 0:
            continue
        row = rows[slots[t]]
        torch.testing.assert_close(row[:R], norm(x[t].float()[NQ:NQ + R], wc, eps), **tol(dt))
        torch.testing.assert_close(row[Rp:Rp + r], rot(x[t].float()[NQ + R:NQ + R + r], int(pos[t])), **tol(dt))
        assert not row[R:Rp].any() and not row[Rp + r:].any()
    free = [s for s in range(80) if s not in slots.tolist()]
    assert (rows[free] == 4.0).all()
    # the queries' rotated part, beside their projection
    hs, N = 32 + rp, 48
    q, w = torch.randn(T, H * hs, generator=g).to(dt), (torch.randn(H, N, 32, generator=g) / 6).to(dt)
    dst = torch.full((T, H, N + rp + 16), 6.0, dtype=dt, device=gpu)
    ops.head_gemm(q.to(gpu), hs, ops.pack_groups(w, dt).to(gpu), dst.view(T, -1), N + rp + 16,
                  rot=(pos.to(gpu), cs.to(gpu), 32, r, rp))
    d = dst.float().cpu()
    assert (d[:, :, N + rp:] == 6.0).all() and not d[:, :, N + r:N + rp].any()
    torch.testing.assert_close(d[:, :, :N], torch.einsum("thk,hnk->thn", q.float().view(T, H, hs)[:, :, :32], w.float()), **tol(dt))
    for t in range(T):
        torch.testing.assert_close(d[t, :, N:N + r], rot(q[t].float().view(H, hs)[:, 32:32 + r], int(pos[t])), **tol(dt))


def fed_meta(gpu, H, reqs, split_target=384, window=0, nblocks=600, part=128, tiles=0):
    """Scheduler-built step: reqs [(cached tokens, new tokens)]; pages in scrambled order."""
    from pilottai_amd import _runtime

    group = min(H, 16)
    s = _runtime.Scheduler({"num_blocks": nblocks, "block_size": 16, "max_num_seqs": 16, "max_num_batched_tokens": 4096,
                            "max_model_len": 4096, "gqa_group": group, "kv_heads": 1, "att_qcols": 128,
                            "att_narrow_qcols": 128, "prefix_caching": False, "decode_part_target": split_target,
                            "att_max_keys": window, "att_min_part": part, "att_tile_target": tiles})
    L = s.layout()
    buf = np.zeros(L["total"], dtype=np.int32)
    junk = [(1000 + i, [1] * (16 * (1 + i % 3))) for i in range(8)]  # fragment the pool first
    s.schedule_fed(buf.ctypes.data, junk)
    s.commit(0, 0)
    for i in (1, 3, 4, 6):
        s.abort(1000 + i)
    for i, (c, _) in enumerate(reqs):
        if c:
            s.schedule_fed(buf.ctypes.data, [(i + 1, [1] * c)])
            s.commit(0, 0)
            if i < 4:
                s.abort([1000, 1002, 1005, 1007][i])
    T = s.schedule_fed(buf.ctypes.data, [(i + 1, [1] * n) for i, (_, n) in enumerate(reqs)])
    t = torch.from_numpy(buf)
    sl = lambda k, n: t[L[k]:L[k] + n].clone()  # noqa: E731
    ms, mb = L["max_seqs"], L["max_blocks"]
    m = dict(q_start=sl("q_start", ms), q_len=sl("q_len", ms), ctx_len=sl("ctx_len", ms),
             block_table=sl("block_table", ms * mb).view(ms, mb), items=sl("items", 4 * L["max_items"]).view(-1, 4),
             n_items=sl("n_items", 1))
    return T, m, 16 // group, 128 // group


def run_attention(gpu, dt, H, R, r, reqs, window, simple=False, split_target=384, seed=0, spike=None, **kw):
    from pilottai_amd import ops
    from pilottai_amd.ops.latent import latent_pad, pad_to

    g = torch.Generator().manual_seed(seed)
    Rp, rp = latent_pad(R), pad_to(r, 32)
    D = Rp + rp
    T, m, dec, tile = fed_meta(gpu, H, reqs, split_target, window, **kw)
    pages = torch.randn(600, D // 8, 16, 8, generator=g).to(dt)
    pages[:, R // 8:Rp // 8] = 0
    q = (torch.randn(T, H, D, generator=g) * 2).to(dt)
    if spike is not None:  # one key per query token answers loudly: it must be seen, or not, exactly
        spike(q, pages, m)
    NB, mi = (dec * H + 15) // 16, m["items"].shape[0]
    out = torch.full((T, H, Rp), 9.0, dtype=dt, device=gpu)
    po = torch.empty(mi * NB * 16 * Rp, dtype=torch.float32, device=gpu)
    pm = torch.empty(mi * NB * 32, dtype=torch.float32, device=gpu)
    mg = {k: v.to(gpu) for k, v in m.items()}
    scale = 1 / math.sqrt(R + r)
    ops.latent_attention(out, po, pm, q.to(gpu), pages.to(gpu), mg["items"], mg["n_items"], mg["q_start"],
                         mg["q_len"], mg["ctx_len"], mg["block_table"], scale, window, dec, tile, simple=simple)
    o = out.float().cpu()
    for i, (c, n) in enumerate(reqs):
        ctx, q0 = c + n, int(m["q_start"][i])
        rows = pages[m["block_table"][i, :(ctx + 15) // 16].long()].permute(0, 2, 1, 3).reshape(-1, D)[:ctx].float()
        sc = torch.einsum("thd,kd->htk", q[q0:q0 + n].float(), rows) * scale
        back = torch.arange(c, ctx)[:, None] - torch.arange(ctx)[None, :]
        sc = sc.masked_fill(~((back >= 0) & ((back < window) if window else True)), -math.inf)
        want = torch.einsum("htk,kd->thd", torch.softmax(sc, -1), rows[:, :Rp])
        torch.testing.assert_close(o[q0:q0 + n], want, **tol(dt), msg=lambda s, i=i: f"request {i} {reqs[i]}: {s}")


SHAPES = [(1, 32, 8), (3, 96, 24), (8, 100, 40), (16, 512, 64), (20, 256, 32), (40, 192, 64)]
STEPS = {"prompt": [(0, 75)], "decode": [(0, 1), (15, 1), (16, 1), (700, 1), (33, 1)], "two": [(130, 2), (0, 2)],
         "mixed": [(300, 1), (17, 40), (0, 3), (531, 130), (64, 1), (5, 2)]}


@pytest.mark.parametrize("window", [0, 1, 45, 128])
@pytest.mark.parametrize("step", list(STEPS))
@pytest.mark.parametrize("H,R,r", SHAPES)
def test_latent_attention_bf16(gpu, H, R, r, step, window):
    run_attention(gpu, torch.bfloat16, H, R, r, STEPS[step], window)


@pytest.mark.parametrize("window", [0, 45, 600])
@pytest.mark.parametrize("H,R,r", SHAPES)
def test_latent_attention_split_tiles(gpu, H, R, r, window):
    """Prompt portions cut over their keys: partitions of one item meet in the merge launch."""
    run_attention(gpu, torch.bfloat16, H, R, r, [(1500, 40), (900, 1), (0, 20), (700, 3)], window, tiles=64, part=256)
    tile = 128 // min(H, 16)  # and portions whose rest is as short as a decode row's tokens
    run_attention(gpu, torch.bfloat16, H, R, r, [(1500, tile + 1), (900, 2 * tile + 16 // min(H, 16))], window, tiles=64, part=256)


MERGED = {"one": [(2000, 1)], "two": [(1500, 1), (700, 1)], "rows": [(60 * i, 1) for i in range(15)], "portions": [(1500, 9), (3, 1), (700, 20), (0, 3)],
          "long": [(4000, 1)], "long rows": [(100 + 400 * i, 1) for i in range(6)]}


@pytest.mark.parametrize("step", list(MERGED))  # 1, 2 and more columns of 16 items, of one to more than 64 partitions; tokens of an item
@pytest.mark.parametrize("H,R,r,vp", [(16, 512, 64, 128), (20, 256, 32, 80), (3, 96, 24, 16), (40, 192, 64, 64)])
def test_merged_heads(gpu, H, R, r, vp, step):
    """The heads' products behind the merge, sums of Rp products in fp32: the bits of the merge and the products on their own."""
    from pilottai_amd import ops
    from pilottai_amd.ops.latent import latent_pad, pad_to

    g = torch.Generator(device=gpu).manual_seed(H + vp)
    rnd = lambda *s: torch.randn(*s, device=gpu, generator=g).bfloat16()  # noqa: E731
    Rp, rp = latent_pad(R), pad_to(r, 32)
    target, part = (192, 16) if step.startswith("long") else (64, 256)
    T, m, dec, tile = fed_meta(gpu, H, MERGED[step], target, 0, tiles=64, part=part)
    NB, mi, D = (dec * H + 15) // 16, m["items"].shape[0], Rp + rp
    assert step != "long" or H > 16 or int(m["items"][0, 2]) >> 20 > 64
    q, pages, uv = rnd(T, H, D), rnd(600, D // 8, 16, 8), rnd(H, vp, Rp) / Rp ** 0.5
    m = {k: v.to(gpu) for k, v in m.items()}
    f32 = lambda n: torch.empty(n, dtype=torch.float32, device=gpu)  # noqa: E731

    def run(**kw):
        out = torch.full((T, H, Rp), 9.0, dtype=torch.bfloat16, device=gpu)
        ops.latent_attention(out, f32(mi * NB * 16 * Rp), f32(mi * NB * 32), q, pages, m["items"], m["n_items"], m["q_start"], m["q_len"],
                             m["ctx_len"], m["block_table"], D ** -0.5, 0, dec, tile, **kw)
        return out
    y = torch.full((T, H * vp + 8), 7.0, dtype=torch.bfloat16, device=gpu)
    wp, two = ops.pack_groups(uv, torch.bfloat16), torch.zeros(T, H * vp, dtype=torch.bfloat16, device=gpu)
    run(heads=(wp, y[:, :H * vp]))
    oc = run()
    ops.head_gemm(oc.view(T, -1), Rp, wp, two, vp)
    assert torch.equal(y[:, :H * vp], two)
    o, w = oc.float(), uv.float()
    want, size = torch.einsum("thk,hvk->thv", o, w), torch.einsum("thk,hvk->thv", o.abs(), w.abs())
    err = (y[:, :H * vp].float().view(T, H, vp) - want).abs()
    assert bool((err <= 2.0 ** -8 * want.abs() + (2.0 ** -8 + Rp * 2.0 ** -24) * size).all()) and bool((y[:, H * vp:] == 7.0).all())


@pytest.mark.parametrize("R,r", [(256, 32), (512, 64)])
def test_latent_attention_item_rounds(gpu, R, r):
    """More items than workgroups, a round that is not full, decode rows among them."""
    run_attention(gpu, torch.bfloat16, 16, R, r, [(0, 2100), (33, 100), (500, 1), (200, 60)], 900)


@pytest.mark.parametrize("tiles,part", [(0, 128), (64, 256)])  # whole prompts, and cut over their keys
@pytest.mark.parametrize("H,R,r", [(16, 512, 64), (20, 256, 32), (8, 384, 0), (40, 192, 64)])
def test_latent_attention_of_peaked_scores(gpu, H, R, r, tiles, part):
    """Queries that point at one key, 2 to 6 nats above the others. The largest weight is exactly 1 where the running maximum
    is the true one, so of the weights only the others' roundings (2^-9 each) move the output; its own rounding averages out
    along the output's direction (6 sigma of steps of 2^-7 at most), and sums of 600 products in fp32 and the exponent of two
    err by 2^-14."""
    from pilottai_amd import ops
    from pilottai_amd.ops.latent import latent_pad, pad_to

    g, reqs, bf = torch.Generator().manual_seed(H + R), [(0, 300), (1000, 60)], torch.bfloat16
    Rp, rp = latent_pad(R), pad_to(r, 32)
    D, scale = Rp + rp, 1 / math.sqrt(R + r)
    T, m, dec, tile = fed_meta(gpu, H, reqs, tiles=tiles, part=part)
    pages = torch.randn(600, D // 8, 16, 8, generator=g).to(bf)
    q, rows = torch.zeros(T, H, D, dtype=bf), []
    for i, (c, n) in enumerate(reqs):
        rows.append(pages[m["block_table"][i, :(c + n + 15) // 16].long()].permute(0, 2, 1, 3).reshape(-1, D)[:c + n])
        at = (torch.rand(n, H, generator=g) * torch.arange(c + 1, c + n + 1)[:, None]).long()
        nats = torch.rand(n, H, 1, generator=g) * 4 + 2
        q[int(m["q_start"][i]):][:n] = (rows[i].float()[at] * nats / (scale * D)).to(bf)
    NB, mi = (dec * H + 15) // 16, m["items"].shape[0]
    out = torch.empty(T, H, Rp, dtype=bf, device=gpu)
    po, pm = torch.empty(mi * NB * 16 * Rp, device=gpu), torch.empty(mi * NB * 32, device=gpu)
    mg = {k: v.to(gpu) for k, v in m.items()}
    ops.latent_attention(out, po, pm, q.to(gpu), pages.to(gpu), mg["items"], mg["n_items"], mg["q_start"], mg["q_len"],
                         mg["ctx_len"], mg["block_table"], scale, 0, dec, tile)
    for i, (c, n) in enumerate(reqs):
        q0, k = int(m["q_start"][i]), rows[i].double()
        sc = torch.matmul(q[q0:q0 + n].double().transpose(0, 1).contiguous(), k.T.contiguous()) * scale  # [H, n, keys]
        sc.masked_fill_(torch.arange(c + n)[None, :] > torch.arange(c, c + n)[:, None], -math.inf)
        w = torch.softmax(sc, -1)
        want = torch.matmul(w, k[:, :Rp].contiguous())
        size = want.square().sum(-1)
        along = ((out[q0:q0 + n].double().cpu().transpose(0, 1) - want) * want).sum(-1) / size
        others = w.scatter(-1, w.argmax(-1, keepdim=True), 0.0)
        each = (others * torch.matmul(want, k[:, :Rp].T.contiguous()).abs()).sum(-1) / size
        rounding = 6 * 2.0 ** -7 / math.sqrt(12) * want.pow(4).sum(-1).sqrt() / size
        assert bool((along.abs() <= 2.0 ** -9 * each + rounding + 2.0 ** -14).all()), (reqs[i], float(along.abs().max()))


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("window", [0, 45])
@pytest.mark.parametrize("step", ["decode", "mixed"])
def test_latent_attention_any_size(gpu, dt, window, step):
    run_attention(gpu, dt, 5, 72, 8, STEPS[step], window, simple=True)


@pytest.mark.parametrize("R", [32, 64, 96, 128, 192, 256, 384, 512, 600])
def test_latent_attention_every_width(gpu, R):
    run_attention(gpu, torch.bfloat16, 6, R, 64 if R % 64 else 32, [(200, 1), (20, 30)], 77)


@pytest.mark.parametrize("edge", ["first", "before"])
@pytest.mark.parametrize("reqs", [[(500, 1)], [(470, 1), (300, 60)], [(100, 2)]])
def test_latent_attention_window_edge(gpu, edge, reqs):
    """The oldest visible key (or the one just before it) outscores all others by far."""
    W = 91

    def spike(q, pages, m):
        for i, (c, n) in enumerate(reqs):
            k = c + n - W - (edge == "before")
            if k < 0:
                continue
            pg, off = int(m["block_table"][i, k // 16]), k % 16
            last = int(m["q_start"][i]) + n - 1
            q[last] = (3.0 * pages[pg, :, off].reshape(1, -1).float()).to(q.dtype)
    run_attention(gpu, torch.bfloat16, 4, 128, 32, reqs, W, spike=spike)


# (cached, new) of a step's requests at the edges of the expanded form: tiles of 128 tokens, stages of 64 keys, 12 new tokens
# at least, keys split into parts (few tokens after many), none of them
EXPANDED = {"one": [(0, 300)], "edges": [(0, 128), (0, 129), (8, 64), (0, 63), (63, 155), (63, 65), (500, 1)],
            "parts": [(2100, 260), (700, 1), (0, 20)], "mixed": [(33, 1), (300, 300), (900, 20), (0, 700), (5, 1), (100, 64)],
            "few": [(900, 12), (70, 11), (0, 13)], "none": [(900, 11), (300, 1)], "many": [(37 * i % 200, 65 + 9 * i) for i in range(12)] + [(250, 1), (8, 9)]}


@pytest.mark.parametrize("window", [0, 45, 600])
@pytest.mark.parametrize("step", list(EXPANDED))
@pytest.mark.parametrize("H", [16, 5, 40])
def test_latent_attention_expanded(gpu, H, step, window):
    """Prompt portions whose keys are expanded per head, beside requests that keep the absorbed form: the step through both
    of a layer's head projections. Keys, values and weights have 16 bits (2^-9 each, and the outputs'), as the absorbed
    form's queries, rows and weights have."""
    from types import SimpleNamespace

    from pilottai_amd import ops
    from pilottai_amd.ops.latent import Expanded, ExpandPlan

    reqs = EXPANDED[step]
    want = [i for i, (c, n) in enumerate(reqs) if n >= 12]
    bf, R, n, r, V = torch.bfloat16, 512, 128, 64, 128
    g = torch.Generator().manual_seed(H + window)
    T, m, dec, tile = fed_meta(gpu, H, reqs, 384, window)
    T += 5  # rows of no request
    pages = torch.randn(600, (R + r) // 8, 16, 8, generator=g).to(bf)
    uk, uv = ((torch.randn(H, k, R, generator=g) * R ** -0.5).to(bf) for k in (n, V))
    q = torch.randn(T, H * (n + r), generator=g).to(bf)
    cs, scale = ops.angle_table(4096, r, 1e4), (n + r) ** -0.5
    d = lambda t: t.to(gpu)  # noqa: E731
    mg, pos = {k: d(v) for k, v in m.items()}, torch.zeros(T, dtype=torch.int32)
    for i, (c, k) in enumerate(reqs):
        pos[int(m["q_start"][i]):][:k] = torch.arange(c, c + k)
    out = torch.full((T, H * V), 9.0, dtype=bf, device=gpu)
    plan = ExpandPlan(SimpleNamespace(**mg), T, H, window)
    taken = [i for i in range(len(reqs)) if int(plan.lists[1][i]) > -(1 << 30)]
    assert taken == want and int(plan.form.sum()) == sum(reqs[i][1] for i in taken)
    qg, pg = d(q), d(pages)
    ex = Expanded(plan, pg, ops.pack_groups(d(uk), bf), ops.pack_groups(d(uv), bf), mg["block_table"], qg, d(cs), out)
    qa = torch.full((T, H, R + r), 7.0, dtype=bf, device=gpu)
    ops.head_gemm(qg, n + r, ops.pack_groups(d(uk.transpose(1, 2).contiguous()), bf), qa.view(T, -1), R + r,
                  rot=(d(pos), d(cs), n, r, r), skip=ex.skip)
    NB, mi = (dec * H + 15) // 16, m["items"].shape[0]
    po, pm = torch.empty(mi * NB * 16 * R, device=gpu), torch.empty(mi * NB * 32, device=gpu)
    oc = torch.zeros(T, H, R, dtype=bf, device=gpu)
    ops.latent_attention(oc, po, pm, qa, pg, mg["items"], mg["n_items"], mg["q_start"], mg["q_len"], mg["ctx_len"],
                         mg["block_table"], scale, window, dec, tile, expand=ex)
    ops.head_gemm(oc.view(T, -1), R, ops.pack_groups(d(uv), bf), out, V, skip=ex.skip)
    assert (out[-5:] == 9.0).all() and (qa[-5:] == 7.0).all()
    o = out.float().cpu().view(T, H, V)
    half = r // 2
    turn = lambda x, at: torch.cat([x[..., :half] * cs[at, :half] - x[..., half:] * cs[at, half:],  # noqa: E731
                                    x[..., half:] * cs[at, :half] + x[..., :half] * cs[at, half:]], -1)
    for i, (c, k) in enumerate(reqs):
        q0, ctx = int(m["q_start"][i]), c + k
        rows = pages[m["block_table"][i, :(ctx + 15) // 16].long()].permute(0, 2, 1, 3).reshape(-1, R + r)[:ctx].float()
        x = q[q0:q0 + k].float().view(k, H, n + r).transpose(0, 1)
        keys = torch.matmul(rows[:, :R], uk.float().transpose(1, 2))  # [H, keys, n]
        sc = torch.matmul(x[..., :n], keys.transpose(1, 2)) + torch.matmul(turn(x[..., n:], torch.arange(c, ctx)), rows[:, R:].T)
        back = torch.arange(c, ctx)[:, None] - torch.arange(ctx)[None, :]
        sc = (sc * scale).masked_fill(~((back >= 0) & ((back < window) if window else True)), -math.inf)
        want = torch.matmul(torch.softmax(sc, -1), torch.matmul(rows[:, :R], uv.float().transpose(1, 2))).transpose(0, 1)
        torch.testing.assert_close(o[q0:q0 + k], want, **tol(bf), msg=lambda s, i=i: f"request {i} {reqs[i]}: {s}")


def plan_of(gpu, reqs, H, window, rest=0):
    """(the plan of a step of [(cached, new)] and `rest` rows of no request, its rows)."""
    from types import SimpleNamespace

    from pilottai_amd.ops.latent import ExpandPlan

    new = torch.tensor([n for _, n in reqs] + [0] * 3, dtype=torch.int32)  # (slots without a request)
    meta = SimpleNamespace(q_len=new.to(gpu), q_start=(new.cumsum(0) - new).to(torch.int32).to(gpu),
                           ctx_len=torch.tensor([c + n for c, n in reqs] + [0] * 3, dtype=torch.int32, device=gpu))
    T = int(new.sum()) + rest
    return ExpandPlan(meta, T, H, window), T


@pytest.mark.parametrize("H,window,reqs,taken", [
    (16, 0, [(0, 64)] * 64, True), (16, 0, [(0, 64)] * 65, False), (16, 0, [(5, 1)] * 70 + [(0, 64)] * 64, True),  # X_REQS
    (16, 0, [(4096, 512)], True), (16, 0, [(4097, 512)], False),  # 288 blocks of keys are the room of 512 rows
    (16, 0, [(2500, 256)] * 2, False), (16, 600, [(2500, 256)] * 2, True), (40, 0, [(0, 300), (4000, 300)], True),
    (16, 0, [(0, 64)] * 7, True), (16, 0, [(0, 64)] * 6 + [(0, 63)], False),  # half of 112 units' columns
    (16, 0, [(0, 12)] * 2, True), (16, 0, [(0, 12)] * 3, False),  # two tiles, whatever they hold
    (16, 0, [(9, 1)] * 2 + [(9, 11)] * 3 + [(3, 70)], True), (16, 0, [(9, 1)] * 3 + [(9, 11)] * 3 + [(3, 70)], False),  # 35 other tokens
    (16, 0, [(70, 1)] * 1100 + [(0, 2200)], True), (16, 0, [(70, 1)] * 1101 + [(0, 2200)], False),
    (16, 0, [(900, 11), (3, 1)], False), (200, 45, [(0, 2000), (100, 700), (7, 1)], True), (1, 0, [(3000, 1000)], True)])
def test_expand_plan_takes_all_prompts_or_none(gpu, H, window, reqs, taken):
    """At the limits of requests, of keys and of units' fill; the work lists of what is taken name every block of its keys and
    every tile of its tokens once, inside the workspace."""
    plan, T = plan_of(gpu, reqs, H, window)
    counts, base, form, att, tiles = (t.cpu() for t in plan.lists)
    want = [i for i, (_, n) in enumerate(reqs) if n >= 12] if taken else []
    assert [i for i, b in enumerate(base.tolist()) if b > -(1 << 30)] == want
    assert form.tolist() == [int(i in want) for i, (_, n) in enumerate(reqs) for _ in range(n)]
    na, nt = counts.tolist()
    if not want:
        assert (na, nt) == (0, 0)
        return
    at, listed, first = 0, [], {}
    for i in want:
        c, n = reqs[i]
        first[i] = max(0, c - window + 1) // 64 * 4 if window else 0
        blocks = (c + n + 15) // 16 - first[i]
        assert int(base[i]) == at - first[i]
        listed += [[i, first[i] + j, min(4, blocks - j), at + j] for j in range(0, blocks, 4)]
        at += blocks
    assert at <= plan.blocks and nt == len(listed) <= len(tiles) and tiles[:nt].tolist() == listed
    parts = {}
    for i, tile, p, slot in att[:na].tolist():
        parts.setdefault((i, tile, p >> 16, slot if p >> 16 > 1 else -1), []).append(p & 0xffff)
    assert [k[:2] for k in parts] == [(i, t) for i in want for t in range((reqs[i][1] + 127) // 128)]
    assert all(v == list(range(k[2])) for k, v in parts.items())
    used = [slot + p for i, t, n, slot in parts for p in range(n) if n > 1]
    assert used == list(range(len(used))) and len(used) <= plan.slots


@pytest.mark.parametrize("H,reqs", [(130, [(0, 2100), (3, 20)]), (16, [(0, 17)]), (1, [(40, 4050)]), (5, [(0, 64), (70, 140)])])
def test_expanded_keys_and_values(gpu, H, reqs):
    """Every block of the plan's requests, whether a workgroup has none, one or more than 64 of them: products of 512 terms added
    up in fp32 and rounded to bf16, the rotated part as it is."""
    from pilottai_amd import ops
    from pilottai_amd.ops.latent import Expanded

    plan, T = plan_of(gpu, reqs, H, 0)
    g, bf, R = torch.Generator().manual_seed(H), torch.bfloat16, 512
    blocks = [(c + n + 15) // 16 for c, n in reqs]
    pages = torch.randn(sum(blocks) + 3, 72, 16, 8, generator=g).to(bf)
    table, ids = torch.zeros(len(reqs) + 3, max(blocks), dtype=torch.int32), torch.randperm(sum(blocks) + 3, generator=g).int()
    for i, n in enumerate(blocks):
        table[i, :n] = ids[sum(blocks[:i]):][:n]
    w = [(torch.randn(H, 128, R, generator=g) * R ** -0.5).to(bf) for _ in range(2)]
    ex = Expanded(plan, pages.to(gpu), *(ops.pack_groups(x.to(gpu), bf) for x in w), table.to(gpu),
                  torch.zeros(T, H * 192, dtype=bf, device=gpu), ops.angle_table(4608, 64, 1e4).to(gpu),
                  torch.zeros(T, H * 128, dtype=bf, device=gpu))
    base, kx, kr = plan.lists[1].tolist(), ex.kx.cpu(), ex.kr.cpu()
    both = torch.cat(w, 1).float()
    for i, n in enumerate(blocks):
        for b in range(n):
            page = pages[int(table[i, b])]
            assert torch.equal(kr[base[i] + b], page[R // 8:])
            x = page[:R // 8].permute(1, 0, 2).reshape(16, R).float()
            want, slack = both @ x.T, R * 2.0 ** -24 * (both.abs() @ x.abs().T)  # [H, 256, 16]
            got = kx[base[i] + b].float().permute(0, 1, 3, 2).reshape(H, 256, 16)
            assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 2 * slack).all()), (i, b)


@pytest.mark.parametrize("reqs", [[(0, 40)], [(9, 1), (3, 1020)], [(900, 11), (3, 1)]])  # taken, beside a decoding row, refused
@pytest.mark.parametrize("rest", [1, 13, 1100])
def test_rows_behind_the_last_request_are_left_out(gpu, reqs, rest):
    """A captured step's rows that no request has: the head products leave them out, whatever the plan takes."""
    plan, T = plan_of(gpu, reqs, 16, 0, rest)
    held = [int(n >= 12) for _, n in reqs for _ in range(n)]
    form = held if reqs[-1][1] >= 12 else [0] * len(held)
    assert plan.form.tolist() == form + [0] * rest and plan.skip.tolist() == form + [1] * rest and T == len(held) + rest


@pytest.mark.parametrize("T,G", [(9, 3), (70, 5), (300, 9), (2100, 16)])  # tiles of 16 and of 64 rows, rows through LDS
@pytest.mark.parametrize("N,K,r,rp", [(512, 128, 64, 64), (512, 128, 48, 64), (48, 32, 12, 32)])  # whole vectors, padding, pairs
def test_head_gemm_leaves_rows_out(gpu, T, G, N, K, r, rp):
    """Rows with an entry in `skip` stay as they are, their rotated columns too, in tiles with other rows and without; the
    others have the bits of a launch that leaves none out."""
    from pilottai_amd import ops

    bf, g = torch.bfloat16, torch.Generator().manual_seed(T + N)
    step = K + (r + 7) // 8 * 8
    x = torch.randn(T, G * step, generator=g).to(gpu, bf)
    w = ops.pack_groups(torch.randn(G, N, K, generator=g).to(gpu, bf) * K ** -0.5, bf)
    pos, cs = torch.randint(0, 64, (T,), generator=g, dtype=torch.int32).to(gpu), ops.angle_table(64, r, 100.0).to(gpu)
    skip = (torch.rand(T, generator=g) < 0.5).to(torch.int32)
    skip[64:128], skip[0], skip[T - 1] = 1, 1, 0

    def run(**kw):
        out = torch.full((T, G * (N + rp)), 7.0, dtype=bf, device=gpu)
        return ops.head_gemm(x, step, w, out, N + rp, rot=(pos, cs, K, r, rp), **kw)
    want, got, gone = run(), run(skip=skip.to(gpu)), skip.bool().to(gpu)
    assert (got[gone] == 7.0).all() and torch.equal(got[~gone], want[~gone])


@pytest.mark.parametrize("family,offered", [("bozupel", True), ("pusunex", False)])
def test_weights_of_expanded_keys_where_plans_are_made(gpu, family, offered):
    """Layers of the sizes that have the form hold the keys' weights only in a model whose steps have plans."""
    from pilottai_amd.models import bozupel, pusunex
    from pilottai_amd.models.latent import LatentAttentionSpec
    from pilottai_amd.models.registry import model_class

    spec = LatentAttentionSpec(heads=2, dim=128, rot_dim=64, vdim=128, q_rank=64, kv_rank=512, scale=0.07, rot_base=1e4, rot_dims=64)
    if family == "bozupel":
        cfg = bozupel.BozupelConfig("x", 512, 64, [bozupel.BozupelLayer(spec, None)])
    else:
        cfg = pusunex.PusunexConfig("x", 512, 64, [pusunex.PusunexLayer(spec, None)], norm_groups=4, side_dim=16)
    model = model_class(cfg)(cfg, gpu, max_len=64)
    L = model.layers[0]
    layer = L["attn"] if family == "bozupel" else L["mixer"].mixers[0]
    assert (layer.expand_key() == (2, 0)) == offered and len(layer.tensors()) == 3 + offered


def test_expanded_workspace_is_the_plans(gpu):
    """A workspace, partial results, a block table or a window other than the plan's are refused before any launch."""
    from pilottai_amd import ops
    from pilottai_amd.ops.latent import Expanded

    bf, H, d = torch.bfloat16, 2, dict(device=gpu)
    plan, T = plan_of(gpu, [(0, 300)], H, 0)
    S = plan.lists[1].numel()
    pages, table = torch.zeros(20, 72, 16, 8, dtype=bf, **d), torch.zeros(S, 19, dtype=torch.int32, **d)
    w, q, out = torch.zeros(H, 8, 16, 64, 8, dtype=bf, **d), torch.zeros(T, H * 192, dtype=bf, **d), torch.zeros(T, H * 128, dtype=bf, **d)
    cs = torch.zeros(400, 64, **d)

    def attend(ex, table=table, window=0):
        qa, oc = torch.zeros(T, H, 576, dtype=bf, **d), torch.zeros(T, H, 512, dtype=bf, **d)
        z, i = torch.zeros(1 << 20, **d), torch.zeros(4, 4, dtype=torch.int32, **d)
        n, one = torch.zeros(S, dtype=torch.int32, **d), torch.zeros(1, dtype=torch.int32, **d)
        ops.latent_attention(oc, z, z, qa, pages, i, one, n, n, n, table, 1.0, window, 8, 64, expand=ex)
    ex = Expanded(plan, pages, w, w, table, q, cs, out)
    with pytest.raises(RuntimeError, match="block table"):
        Expanded(plan, pages, w, w, table[:1], q, cs, out)
    with pytest.raises(RuntimeError, match="block table"):
        attend(ex, table[:1].contiguous())
    with pytest.raises(ValueError, match="window"):
        attend(ex, window=5)
    for name, match in (("kx", "workspace"), ("part_o", "too short"), ("part_ml", "too short")):
        whole = getattr(ex, name)
        setattr(ex, name, whole[:-1])
        if name == "kx":
            ex.kr = ex.kr[:-1]
        with pytest.raises(RuntimeError, match=match):
            attend(ex)
        setattr(ex, name, whole)
        if name == "kx":
            ex.kr = torch.zeros(len(whole), 8, 16, 8, dtype=bf, **d)
