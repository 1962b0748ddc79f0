// Prompt portions of a latent attention in the expanded form: keys and values of every head, k_h = W_uk,h c and v_h =
// W_uv,h c, in a workspace, and an attention of heads of 128 + 64 (keys) and 128 (values) dimensions over them. A (query,
// key) pair and head then takes 2 (128 + 64 + 128) products instead of the absorbed form's 2 (512 + 64 + 512), and a key 2 *
// 512 * 256 once. Whether a step's prompts run so is decided on the device, step by step (expand_plan_kernel), since a captured
// step serves any mix of requests; the other requests keep the absorbed form, in the same launches.
//
// Workspace: kx [blocks of 16 keys][H][(128 + 128) / 8][16][8], a head's key then its value, both in the page layout;
// kr [blocks][64 / 8][16][8], the rotated key part that the heads share.
#pragma once
#include <hip/hip_runtime.h>

namespace pa {
namespace la {

constexpr int X_DIM = 128, X_ROT = 64, X_RANK = 512;  // sizes that have this form
constexpr int X_COLS = 128;                           // tokens of an attention unit
constexpr int X_PARTS = 8;                            // parts of a unit's keys, at most
constexpr int X_REQS = 64;                            // requests of a step that may take it
constexpr int X_NONE = -(1 << 30);

// what the plan of a step holds and the launches read; all null: no request takes the form
struct Expand {
  int* counts;  // attention items, expansion tiles
  int* base;    // [S] workspace block of the request's key block 0 (blocks before its window have none), or X_NONE
  int* form;    // [T] 1: the row belongs to an expanded request (the head products go by the plan's `skip`, 1 for rows of no request too)
  int4* att;    // {request, tile of X_COLS tokens, part | parts << 16, partial slot}
  int4* tiles;  // {request, first key block, blocks, workspace block}
  void *kx, *kr;
  const void* q;  // [T, >= H (128 + 64)], not yet rotated
  int ldq;
  const float* cos_sin;  // [positions, 64]
  void* out;             // [T, >= H 128]
  int ldo;
  float *part_o, *part_ml;  // [slots, H, X_COLS, 128], [slots, H, X_COLS, 2]
};

}  // namespace la
}  // namespace pa
