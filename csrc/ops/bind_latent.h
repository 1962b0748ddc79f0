// Shared by the bindings of the modules with latent attention (_latent, _latent_linear): the fp32 residual, the latent cache
// and the attention over it.
#pragma once
#include "bind_grouped.h"
#include "latent_expand.h"

extern "C" {
int pa_residual_norm(int fp32, float* resid, const void* y, int K, int ldy, float y_scale, const float* w_post,
                     const void* emb, const int* ids, int vocab, int emb_add, const float* mix, float* hist,
                     long long hist_step, int n_hist, const float* w_next, void* out, int ldo, const int* rows, const int* live,
                     int n, int D, int post_groups, int next_groups, float eps, hipStream_t st);
int pa_latent_cache(int fp32, const void* x, int ldx, int NQ, int R, int r, int rd, const float* w_q, const float* w_c,
                    void* cq, int ldq, void* pages, int Rp, int D, const int* positions, const int* slots,
                    const float* cos_sin, float eps, int T, hipStream_t st);
int pa_latent_pad(int R);
int pa_latent_attention(int fp32, void* out, float* part_o, float* part_ml, const void* q, const void* pages,
                        const int* items, const int* n_items, int max_items, const int* q_start,
                        const int* q_len, const int* ctx_len, const int* block_table, int max_blocks, int H, int Rp,
                        int rp, int dec_tokens, int tile_tokens, int window, float scale_log2, int simple,
                        const pa::la::Expand* expand, const void* uv, void* y, int ldy, int vp, int T, hipStream_t st);
int pa_latent_plan(const pa::la::Expand* X, const int* q_start, const int* q_len, const int* ctx_len, int S, int T, int H, int window,
                   int room, int max_att, int max_tiles, int slots, int* skip, hipStream_t st);
int pa_latent_expand(const pa::la::Expand* X, const void* pages, const void* wk, const void* wv, const int* block_table, int max_blocks, int H, int D,
                     int max_tiles, hipStream_t st);
}

namespace {

void residual_norm(at::Tensor resid, Opt y, int64_t K, double y_scale, Opt w_post, Opt emb, Opt ids, bool emb_add,
                   Opt w_next, Opt out, Opt rows, double eps, int64_t post_groups, int64_t next_groups, Opt mix, Opt hist,
                   Opt live) {
  check_gpu(resid, "resid");
  check_dtype(resid, at::kFloat, "resid");
  TORCH_CHECK(resid.dim() == 2, "resid must be [T, D]");
  const int64_t T = resid.size(0), D = resid.size(1), n = rows.has_value() ? rows->numel() : T;
  at::ScalarType dt = at::kFloat;
  for (const Opt* o : {&y, &emb, &out})
    if (o->has_value()) dt = (*o)->scalar_type();
  int ldy = 0, ldo = 0;
  if (y.has_value()) {
    check_rows(*y, dt, "y");
    TORCH_CHECK(K >= 1 && y->size(0) == T * K && y->size(1) >= D, "y must be [T * K, >= D]");
    ldy = y->stride(0);
  }
  if (emb.has_value()) {
    check_gpu(*emb, "emb");
    check_dtype(*emb, dt, "emb");
    TORCH_CHECK(ids.has_value() && emb->dim() == 2 && emb->size(1) == D && emb->size(0) > 0, "emb must be [vocab, D]");
  }
  TORCH_CHECK(!w_next.has_value() || out.has_value(), "w_next needs out");
  long long hist_step = 0;
  int n_hist = 0;
  if (mix.has_value()) {  // weights of the embedding, the earlier results and this one
    n_hist = mix->numel() - 1;
    TORCH_CHECK(hist.has_value() && emb.has_value() && n_hist >= 1, "a depth average needs hist and the embedding");
    check_gpu(*hist, "hist");
    check_dtype(*hist, at::kFloat, "hist");
    TORCH_CHECK(hist->dim() == 3 && hist->size(0) >= n_hist && hist->size(1) >= T && hist->size(2) == D, "hist must be [>= n, T, D]");
    hist_step = hist->stride(0);
  }
  if (out.has_value()) {
    check_rows(*out, dt, "out");
    TORCH_CHECK(out->size(0) >= n && out->size(1) >= D && out->stride(0) == out->size(1), "out must be [>= n, >= D]");
    ldo = out->stride(0);
  }
  check_rc(pa_residual_norm(dt == at::kFloat, resid.data_ptr<float>(), y.has_value() ? y->data_ptr() : nullptr, (int)K,
                            ldy, (float)y_scale, opt_f32(w_post, D, "w_post"), emb.has_value() ? emb->data_ptr() : nullptr,
                            emb.has_value() ? ints(*ids, T, "ids") : nullptr, emb.has_value() ? emb->size(0) : 0,
                            emb_add ? 1 : 0, opt_f32(mix, 2, "mix"), n_hist ? hist->data_ptr<float>() : nullptr, hist_step,
                            n_hist, opt_f32(w_next, D, "w_next"), out.has_value() ? out->data_ptr() : nullptr,
                            ldo, rows.has_value() ? ints(*rows, n, "rows") : nullptr,
                            live.has_value() ? ints(*live, T, "live") : nullptr, (int)n, (int)D, (int)post_groups,
                            (int)next_groups, (float)eps, cur_stream()),
           "residual_norm");
}

// x [T, NQ | R | r ..]; NQ 0: no query latent (w_q, cq null), r 0: no rotated part (cos_sin null)
void latent_cache(at::Tensor x, int64_t NQ, int64_t R, int64_t r, Opt w_q, at::Tensor w_c, Opt cq, at::Tensor pages,
                  int64_t Rp, at::Tensor positions, at::Tensor slots, Opt cos_sin, double eps) {
  const int f = is_f32(x, "x");
  check_rows(x, x.scalar_type(), "x");
  check_gpu(pages, "pages");
  check_dtype(pages, x.scalar_type(), "pages");
  TORCH_CHECK(pages.dim() == 4 && pages.size(2) == 16 && pages.size(3) == 8, "pages must be [blocks, D/8, 16, 8]");
  const int64_t T = x.size(0), D = pages.size(1) * 8;
  TORCH_CHECK(x.size(1) >= NQ + R + r && NQ >= 0 && R > 0 && r >= 0 && R <= Rp && Rp + r <= D, "latent_cache sizes");
  TORCH_CHECK(f || ((uintptr_t)x.data_ptr() & 15) == 0, "latent_cache: 16-byte aligned rows");
  TORCH_CHECK((NQ > 0) == cq.has_value() && (NQ > 0) == w_q.has_value() && (r > 0) == cos_sin.has_value(), "latent_cache parts");
  int64_t rd = 0;
  if (cos_sin.has_value()) {
    TORCH_CHECK(cos_sin->dim() == 2 && cos_sin->size(1) % 2 == 0 && cos_sin->size(1) <= r, "cos_sin must be [max_pos, dims <= r]");
    rd = cos_sin->size(1);
  }
  if (cq.has_value()) {
    check_rows(*cq, x.scalar_type(), "cq");
    TORCH_CHECK(cq->size(0) == T && cq->size(1) >= NQ && cq->stride(0) == cq->size(1), "cq must be [T, >= NQ]");
  }
  check_rc(pa_latent_cache(f, x.data_ptr(), x.stride(0), NQ, R, r, rd, opt_f32(w_q, NQ, "w_q"), opt_f32(w_c, R, "w_c"),
                           cq.has_value() ? cq->data_ptr() : nullptr, cq.has_value() ? cq->stride(0) : 0, pages.data_ptr(), Rp,
                           D, ints(positions, T, "positions"), ints(slots, T, "slots"), opt_f32(cos_sin, 0, "cos_sin"),
                           (float)eps, T, cur_stream()),
           "latent_cache");
}

// What a step's plan of expanded requests holds: [counts, base, form, attention items, expansion tiles] (latent_expand.h)
using Tensors = std::vector<at::Tensor>;
pa::la::Expand expand_plan(const Tensors& p, int64_t S, int64_t T) {
  TORCH_CHECK(p.size() == 5 && p[3].dim() == 2 && p[3].size(1) == 4 && p[4].dim() == 2 && p[4].size(1) == 4,
              "a plan is [counts, base, form, items [n, 4], tiles [n, 4]]");
  pa::la::Expand X{};
  X.counts = (int*)ints(p[0], 2, "counts");
  X.base = (int*)ints(p[1], S, "base");
  X.form = (int*)ints(p[2], T, "form");
  X.att = (int4*)ints(p[3], 4, "items");
  X.tiles = (int4*)ints(p[4], 4, "tiles");
  return X;
}

// The workspace: kx [blocks, H, 32, 16, 8] and kr [blocks, 8, 16, 8], of at least the `room` blocks that the plan may give
// away; block_table: of all requests that the plan may name
void expand_room(pa::la::Expand& X, const Tensors& plan, const at::Tensor& kx, const at::Tensor& kr, const at::Tensor& block_table,
                 int64_t H, int64_t room) {
  for (auto* t : {&kx, &kr}) {
    check_gpu(*t, "workspace");
    check_dtype(*t, at::kBFloat16, "workspace");
  }
  TORCH_CHECK(kx.dim() == 5 && kx.size(1) == H && kx.size(2) * 8 == 2 * pa::la::X_DIM && kx.size(3) == 16 && kx.size(4) == 8 &&
                  kr.dim() == 4 && kr.size(0) == kx.size(0) && kr.size(1) * 8 == pa::la::X_ROT && kr.size(2) == 16 && kr.size(3) == 8,
              "workspace must be [blocks, H, 32, 16, 8] and [blocks, 8, 16, 8]");
  TORCH_CHECK(kx.size(0) >= room && room >= 1, "workspace of ", kx.size(0), " blocks for a plan of ", room);
  TORCH_CHECK(block_table.dim() == 2 && block_table.size(0) == plan[1].numel(), "a plan is for the requests of its block table");
  X.kx = kx.data_ptr();
  X.kr = kr.data_ptr();
}

// Decides which requests of the step have their keys expanded and writes the plan; `slots` partial results and `room` blocks
// are what the launches with this plan have.
void latent_plan(const Tensors& plan, at::Tensor q_start, at::Tensor q_len, at::Tensor ctx_len, int64_t T, int64_t H, int64_t window,
                 int64_t room, int64_t slots, at::Tensor skip) {
  const int64_t S = q_len.numel();
  const pa::la::Expand X = expand_plan(plan, S, T);
  TORCH_CHECK(T >= 1 && H >= 1 && room >= 1 && slots >= 0 &&
                  plan[3].size(0) >= T / pa::la::X_COLS + pa::la::X_REQS + slots, "latent_plan sizes");
  check_rc(pa_latent_plan(&X, ints(q_start, S, "q_start"), ints(q_len, S, "q_len"), ints(ctx_len, S, "ctx_len"), S, T, H, window, room,
                          plan[3].size(0), plan[4].size(0), slots, (int*)ints(skip, T, "skip"), cur_stream()),
           "latent_plan");
}

// keys and values of the planned requests from their pages: wk, wv [H, 8, 16, 64, 8], the heads' rows of W_uk and of W_uv;
// room: as the plan was made with
void latent_expand(const Tensors& plan, int64_t room, at::Tensor kx, at::Tensor kr, at::Tensor pages, at::Tensor wk, at::Tensor wv,
                   at::Tensor block_table) {
  pa::la::Expand X = expand_plan(plan, 0, 0);
  const int64_t H = wk.size(0);
  for (auto* t : {&pages, &wk, &wv}) {
    check_gpu(*t, "latent_expand arg");
    check_dtype(*t, at::kBFloat16, "latent_expand arg");
  }
  for (auto* w : {&wk, &wv})
    TORCH_CHECK(w->dim() == 5 && w->size(0) == H && w->size(1) * 16 == pa::la::X_DIM && w->size(2) * 32 == pa::la::X_RANK &&
                    w->size(3) == 64 && w->size(4) == 8, "weights must be packed [H, 8, 16, 64, 8]");
  TORCH_CHECK(pages.dim() == 4 && pages.size(1) * 8 == pa::la::X_RANK + pa::la::X_ROT && pages.size(2) == 16 && pages.size(3) == 8,
              "pages must be [blocks, 72, 16, 8]");
  expand_room(X, plan, kx, kr, block_table, H, room);
  check_rc(pa_latent_expand(&X, pages.data_ptr(), wk.data_ptr(), wv.data_ptr(), ints(block_table, 0, "block_table"), block_table.size(1),
                            H, pages.size(1) * 8, plan[4].size(0), cur_stream()),
           "latent_expand");
}

void latent_attention(at::Tensor out, at::Tensor part_o, at::Tensor part_ml, at::Tensor q,
                      at::Tensor pages, at::Tensor items, at::Tensor n_items, at::Tensor q_start, at::Tensor q_len,
                      at::Tensor ctx_len, at::Tensor block_table, int64_t dec_tokens, int64_t tile_tokens,
                      int64_t window, double scale, bool simple, const Tensors& plan, const Tensors& expand, int64_t room,
                      int64_t slots, Opt uv, Opt y) {
  const int f = is_f32(q, "q");
  for (auto* t : {&out, &q, &pages}) {
    check_gpu(*t, "latent_attention arg");
    check_dtype(*t, q.scalar_type(), "latent_attention arg");
  }
  TORCH_CHECK(q.dim() == 3 && out.dim() == 3 && out.size(0) == q.size(0) && out.size(1) == q.size(1),
              "q [T, H, D], out [T, H, Rp]");
  TORCH_CHECK(pages.dim() == 4 && pages.size(1) * 8 == q.size(2) && pages.size(2) == 16 && pages.size(3) == 8,
              "pages must be [blocks, D/8, 16, 8]");
  TORCH_CHECK(items.dim() == 2 && items.size(1) == 4 && block_table.dim() == 2, "items [n, 4], block_table [seqs, blocks]");
  const int64_t H = q.size(1), Rp = out.size(2), rp = q.size(2) - Rp, S = block_table.size(0), mi = items.size(0);
  const int64_t NB = (dec_tokens * H + 15) / 16;
  TORCH_CHECK(Rp > 0 && rp >= 0 && dec_tokens >= 1 && tile_tokens >= 1, "latent_attention sizes");
  TORCH_CHECK(part_o.numel() >= mi * NB * 16 * Rp && part_ml.numel() >= mi * NB * 32, "partition workspace too small");
  // uv: the heads' products with W_uv, to y [T, >= H vp] in place of out (which then holds anything)
  int ldy = 0, vp = 0;
  if (uv.has_value()) {
    check_gpu(*uv, "uv");
    check_dtype(*uv, at::kBFloat16, "uv");
    TORCH_CHECK(!f && y.has_value() && uv->dim() == 5 && uv->size(0) == H && uv->size(2) * 32 == Rp && uv->size(3) == 64 && uv->size(4) == 8,
                "uv must be packed [H, vp/16, Rp/32, 64, 8], with y");
    check_rows(*y, at::kBFloat16, "y");
    vp = uv->size(1) * 16;
    ldy = y->stride(0);
    TORCH_CHECK(y->size(0) == q.size(0) && y->size(1) >= H * vp && ldy % 4 == 0 && ((uintptr_t)y->data_ptr() & 7) == 0, "y must be [T, >= H vp], 8-byte aligned");
  }
  // expanded requests: expand = [kx, kr, q not yet absorbed or rotated, cos_sin, their outputs, partial outputs and (max, sum)];
  // room and slots: as the plan was made with
  pa::la::Expand X{};
  if (!expand.empty()) {
    const int64_t T = q.size(0), slot = H * pa::la::X_COLS;
    TORCH_CHECK(!f && expand.size() == 7 && Rp == pa::la::X_RANK && rp == pa::la::X_ROT, "latent_attention: expanded sizes");
    X = expand_plan(plan, S, T);
    expand_room(X, plan, expand[0], expand[1], block_table, H, room);
    const at::Tensor &xq = expand[2], &xo = expand[4];
    check_rows(xq, at::kBFloat16, "q");
    check_rows(xo, at::kBFloat16, "expanded out");
    TORCH_CHECK(xq.size(0) == T && xq.size(1) >= H * (pa::la::X_DIM + pa::la::X_ROT) && xq.stride(0) % 8 == 0 &&
                    ((uintptr_t)xq.data_ptr() & 15) == 0 && xo.size(0) == T && xo.size(1) >= H * pa::la::X_DIM &&
                    xo.stride(0) % 4 == 0 && ((uintptr_t)xo.data_ptr() & 7) == 0, "latent_attention: rows of expanded requests");
    TORCH_CHECK(expand[3].dim() == 2 && expand[3].size(1) == pa::la::X_ROT, "cos_sin must be [positions, 64]");
    X.q = xq.data_ptr();
    X.ldq = xq.stride(0);
    X.cos_sin = opt_f32(expand[3], 0, "cos_sin");
    X.out = xo.data_ptr();
    X.ldo = xo.stride(0);
    X.part_o = (float*)opt_f32(expand[5], slots * slot * pa::la::X_DIM, "partial outputs");
    X.part_ml = (float*)opt_f32(expand[6], slots * slot * 2, "partial sums");
  }
  check_rc(pa_latent_attention(f, out.data_ptr(), (float*)opt_f32(part_o, 0, "part_o"),
                               (float*)opt_f32(part_ml, 0, "part_ml"), q.data_ptr(),
                               pages.data_ptr(), ints(items, 0, "items"), ints(n_items, 1, "n_items"), mi,
                               ints(q_start, S, "q_start"), ints(q_len, S, "q_len"), ints(ctx_len, S, "ctx_len"),
                               ints(block_table, 0, "block_table"), block_table.size(1), H, Rp, rp, dec_tokens,
                               tile_tokens, window, (float)(scale * 1.4426950408889634), simple ? 1 : 0,
                               expand.empty() ? nullptr : &X, uv.has_value() ? uv->data_ptr() : nullptr,
                               uv.has_value() ? y->data_ptr() : nullptr, ldy, vp, q.size(0), cur_stream()),
           "latent_attention");
}

}  // namespace
