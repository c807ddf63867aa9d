// Host-side helpers shared by the C-ABI entry points: error reporting and
// launch checks. Every entry point returns 0 on success or one of the KF_E*
// codes declared in include/kotflash_amd.h; the message is kept per thread and
// read back through kf_last_error().
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/kotflash_amd.h"

namespace kf {

int set_error(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

// Translate the last HIP launch status into an error code.
int check_launch(const char* what);

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

// Padded head-dim tile (multiple of 32) for a real head dim D in [8, 128].
inline int head_tile(int64_t D) {
  if (D <= 32) return 32;
  if (D <= 64) return 64;
  if (D <= 96) return 96;
  return 128;
}

// Forms of the forward and dQ kernels: RB row blocks of 32 query rows times KG
// key groups, RB * KG waves per workgroup. A group's waves take every KG-th
// K/V tile of the workgroup's rows, and the groups' results are combined
// through LDS at the end. 4x1 moves the fewest K/V bytes per product and
// is the one for large problems; with few tiles the launch is as long as its
// longest chain of dependent tiles, and splitting the keys (and the rows into
// more workgroups) shortens it.
enum AttnForm { kForm4x1, kForm4x2, kForm2x2, kForm2x4, kForm1x4, kForm1x8, kNumForms };
struct FormShape {
  int rb, kg;
};
constexpr FormShape kFormShapes[kNumForms] = {{4, 1}, {4, 2}, {2, 2}, {2, 4}, {1, 4}, {1, 8}};

// Launch time of a form, us: `fixed` once, `round` for each round of workgroup
// slots (256 CUs times per_cu), and the K/V steps: a workgroup's step of 64
// keys per group takes `chain` when it has its CU to itself, and a CU retires
// one per `work` when several share it.
struct FormCost {
  float fixed, round, chain, work;
  int per_cu;  // resident workgroups per CU; 0: the form is not built
};

// Fitted to 580 shapes on MI355X (1 to 32 heads, batches of 1 to 16, 45 to
// 4096 queries, 45 to 6600 keys, up to 1024 tiles; rms error of one form's time
// 3 to 14%; which of two forms is faster is measured at attn_form).
constexpr FormCost kFwdCosts[4][kNumForms] = {  // by head-dim tile / 32 - 1; forms as in AttnForm
    {{3.39f, 0.00f, 0.58f, 0.44f, 2}, {0.90f, 2.98f, 0.83f, 0.87f, 1}, {3.38f, 0.28f, 0.59f, 0.46f, 2},
     {1.21f, 2.63f, 0.91f, 0.91f, 1}, {3.08f, 0.72f, 0.46f, 0.45f, 1}, {0, 0, 0, 0, 0}},
    {{4.19f, 0.00f, 0.70f, 0.59f, 2}, {0.00f, 5.05f, 1.02f, 1.07f, 1}, {0.04f, 4.21f, 0.79f, 0.59f, 2},
     {0.47f, 4.22f, 1.17f, 1.22f, 1}, {1.25f, 2.63f, 0.87f, 0.87f, 1}, {0.84f, 3.33f, 1.32f, 1.32f, 1}},
    {{0.00f, 4.62f, 0.84f, 0.85f, 3}, {0.00f, 5.53f, 1.16f, 1.31f, 1}, {0.85f, 3.68f, 1.01f, 1.05f, 1},
     {0, 0, 0, 0, 0}, {1.34f, 3.13f, 1.05f, 1.07f, 1}, {0, 0, 0, 0, 0}},
    {{0.00f, 5.13f, 1.06f, 1.08f, 2}, {0.00f, 6.74f, 1.43f, 1.77f, 1}, {0.00f, 5.28f, 1.17f, 1.36f, 1},
     {0, 0, 0, 0, 0}, {0.89f, 3.64f, 1.40f, 1.42f, 1}, {0, 0, 0, 0, 0}},
};
constexpr FormCost kDqCosts[4][kNumForms] = {  // by head-dim tile / 32 - 1; forms as in AttnForm
    {{3.72f, 0.21f, 0.56f, 0.44f, 2}, {0.78f, 3.54f, 0.77f, 0.85f, 1}, {2.46f, 1.68f, 0.58f, 0.44f, 2},
     {0.98f, 3.18f, 0.89f, 0.94f, 1}, {3.07f, 0.82f, 0.51f, 0.51f, 1}, {0, 0, 0, 0, 0}},
    {{0.00f, 5.09f, 0.75f, 0.81f, 2}, {0.00f, 6.25f, 1.19f, 1.33f, 1}, {0.19f, 5.15f, 0.85f, 0.79f, 2},
     {0.69f, 5.48f, 1.40f, 1.42f, 1}, {1.11f, 3.91f, 0.87f, 0.90f, 1}, {0.97f, 4.54f, 1.57f, 1.58f, 1}},
    {{0.00f, 4.69f, 0.94f, 1.03f, 2}, {0.00f, 6.12f, 1.44f, 1.79f, 1}, {0.43f, 4.69f, 1.11f, 1.17f, 1},
     {0, 0, 0, 0, 0}, {0.85f, 3.89f, 1.41f, 1.38f, 1}, {0, 0, 0, 0, 0}},
    {{0.00f, 6.97f, 1.32f, 1.34f, 2}, {0.00f, 9.65f, 2.06f, 2.58f, 1}, {0.00f, 7.17f, 1.47f, 1.58f, 1},
     {0, 0, 0, 0, 0}, {0.95f, 5.68f, 1.59f, 1.77f, 1}, {0, 0, 0, 0, 0}},
};

// The forms that the kernels are built in, by head-dim tile: exactly the priced
// ones. (dQ 4x2 at D=128 only causal: without the mask it costs more than 4x1
// up to 53 key tiles, and more than 0.92 of it beyond.)
constexpr bool form_built(int head_tile, int form) {
  return form == kForm2x4 ? head_tile <= 64 : form != kForm1x8 || head_tile == 64;
}
constexpr bool priced_forms_are_built(const FormCost (&costs)[4][kNumForms]) {
  for (int t = 0; t < 4; ++t)
    for (int f = 0; f < kNumForms; ++f)
      if ((costs[t][f].per_cu > 0) != form_built(32 * (t + 1), f)) return false;
  return true;
}
static_assert(priced_forms_are_built(kFwdCosts) && priced_forms_are_built(kDqCosts));

inline float attn_form_cost(const FormCost& c, const FormShape& f, int64_t heads, int64_t Sq, int64_t Sk,
                            bool causal) {
  const int rows = 32 * f.rb, keys = 64 * f.kg;
  const int64_t tiles = (Sq + rows - 1) / rows;
  const int64_t longest = causal && tiles * rows < Sk ? tiles * rows : Sk;
  const int64_t top = (longest + keys - 1) / keys;  // steps of the longest tile
  const int64_t wgs = tiles * heads, slots = 256 * c.per_cu;
  if (!causal) {
    // Equal workgroups: whole rounds, the last one perhaps with fewer per CU.
    const int64_t rest = wgs % slots;
    const float alone = top * c.chain, shared = top * c.work;
    float t = c.fixed + (wgs / slots) * (c.round + (alone > c.per_cu * shared ? alone : c.per_cu * shared));
    if (rest) {
      const float last = shared * ((rest + 255) / 256);
      t += c.round + (alone > last ? alone : last);
    }
    return t;
  }
  // Causal tile q sees min(Sk, (q + 1) rows) keys: those before tile m,
  // growing, then Sk (half a step on average for the last, partly filled one).
  // Unequal workgroups, longest first, fill in for one another.
  const float m = (float)(tiles < Sk / rows ? tiles : Sk / rows);
  const float steps = (rows * m * (m + 1.f) / 2.f + (tiles - m) * Sk) / keys + (f.kg > 1 || f.rb < 2 ? 0.5f * m : 0.f);
  const float rounds = (float)wgs / slots;
  const float chain = top * c.chain, work = steps * heads / 256.f * c.work;
  return c.fixed + c.round * (rounds > 1.f ? rounds : 1.f) + (chain > work ? chain : work);
}

// The form of a problem. The default is 1x4 for grids of 128-row tiles that
// leave most of the 256 CUs idle (at most 64 tiles, 128 when causal, whose
// tiles differ in length) and 4x1 for the others; another form is taken when
// the costs above make it at least 8% faster, up to two 4x1 workgroups per CU.
//
// Past one 4x1 workgroup per CU a non-causal grid takes only forms that also
// keep two on a CU: its tiles are equal, the second workgroup hides the latency
// that key groups would, and a form alone on its CU adds a round and a merge.
// The costs do not show that: they price 4x2 up to 15% ahead of 4x1 there, and
// it measured up to 23% behind (forward, 128 heads, 384 x 4343 D=128 bf16,
// 128.4 -> 157.6 us; dQ 2x2, 64 heads, 710 x 5854 D=80, 143.6 -> 166.4), while
// 2x2 at D=64, two per CU, is ahead (forward, 32 heads, 1195 x 3664, 70.1 ->
// 62.6). Causal tiles differ in length, and more workgroups even them out.
//
// Measured with every form over 1884 shapes of up to 640 tiles, against the
// default form: forward 6.5% and dQ 4.0% faster in the geometric mean; 3
// forwards got 4 to 8% slower (by 0.3 to 1.1 us) and 10 dQ 4 to 8% (by 0.3 to
// 0.9 us), most of them with one or two key tiles.
constexpr int64_t kFormMaxTiles = 512;

inline AttnForm attn_form(const FormCost (&costs)[kNumForms], int64_t heads, int64_t Sq, int64_t Sk, bool causal) {
  const int64_t tiles = (Sq + 127) / 128 * heads;
  if (tiles > kFormMaxTiles) return kForm4x1;
  const int resident = !causal && tiles > 256 ? 2 : 1;  // least workgroups per CU
  int best = Sk > 128 && tiles <= (causal ? 128 : 64) ? kForm1x4 : kForm4x1;
  float least = 0.92f * attn_form_cost(costs[best], kFormShapes[best], heads, Sq, Sk, causal);
  for (int f = 0; f < kNumForms; ++f) {
    if (costs[f].per_cu < resident) continue;
    const float t = attn_form_cost(costs[f], kFormShapes[f], heads, Sq, Sk, causal);
    if (t < least) {
      least = t;
      best = f;
    }
  }
  return (AttnForm)best;
}

// Whether a causal grid takes its tiles in fold_rank's order: when all its
// workgroups are resident at once, in more than one per CU, so that the
// pairing on a CU is decided by the order alone, and the tiles of a head
// differ enough in length. Measured over 47 forward and 41 dQ grids of the 4x1
// form, folded against unfolded, geometric means, forward / dQ: under 8 tiles
// per head 0.991 / 1.002 (the worst 1.026 and 1.027), 8 to 11 0.981 / 0.969,
// 12 to 23 0.967 / 0.954, 24 and more 0.967 / 0.940.
inline int fold_tiles(int64_t tiles_per_head, int64_t grid, int per_cu) {
  return tiles_per_head >= 8 && grid > 256 && grid <= 256 * per_cu;
}

}  // namespace kf
