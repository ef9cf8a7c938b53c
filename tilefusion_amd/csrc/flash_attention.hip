// Flash-attention forward: the C entry points, and which kernel instance (flash_attention.hpp) a call runs.
#include <algorithm>

#include "common.hpp"
#include "flash_attention_runs.hpp"
#include "jit_ops.hpp"

namespace tfk {

namespace {
// How a problem is dealt to workgroups: query rows per workgroup (256, 128 or 64) and, causal, pairs of query tiles
// (see the kernel) or single ones, whichever is expected to be done first.
//
// Fewer rows are more expensive per query (every wavefront reads the whole K and V tile from LDS for its 32 or 16
// queries) and pay where 256 leave CUs idle.  us, bf16, 256 / 128 / 64 rows: 8 slices of 512 x 512 x 64 12.2 / 8.9 / 7.7,
// 64 of 1337 x 1337 x 64 causal 30.0 / 26.7 / 29.4, 24 of 1024 x 1024 x 128 28.8 / 21.7 / 34.5, 64 of 2048 x 2048 x 128
// 118 / 152 / 232.  (4 wavefronts x 32 queries, which ran up to 128 rows before, were behind both smaller
// forms everywhere.)  Pairs do the same work each, in slice-major order, and pay where they fill whole rounds
// of the chip: bf16, D = 128, 256 rows, pairs / single tiles: 64 slices of 1024 x 1024 42 / 33 (half of the chip had nothing
// to do), 33 of 4096 213 / 137, 128 of 1024 48 / 51, 128 of 2048 142 / 156.
//
// Expected time of single tiles: a workgroup takes `tile` us a key tile while the chip is idle beside it, (1 + fill)
// times that with every CU taken, `full` where a CU works on several, and `start` us more for each further one.
// Work is handed out heaviest first: the (256 j + 1)-th workgroup shares its CU with j others that are no lighter.
// Causal tiles are of different weights, and `mean` us a tile is what the chip takes on average.  Pairs: the rounds
// they take.  Fitted to 210 problems without a mask and 710 causal ones (4..300 slices, 64..8192 keys); the pick is on
// average 0.2% and 1% behind the best, and 1.31x and 1.25x ahead of always taking 256 rows.  Small margins (`ahead`)
// keep 256 rows where the model cannot tell.
//
// With few keys a further workgroup starts sooner than with many, `few` + `per_tile` us a key tile after the one in front (us, fp16, D = 128, 256 / 128
// rows: 869 slices of 214 x 8 37.6 / 44.0, 58 of 1666 x 32 20.6 / 26.0, 503 of 465 x 208 65.5 / 77.0, 94 of 936 x 48 19.9 / 20.4; with
// `start` alone, fitted to many, all four took 128; over 55 problems of 280 to 1150 keys the pick is 0.1% behind the best, 4% before).
struct SingleCost { double fixed, tile, full, fill, start, mean, few = 1e9, per_tile = 0; };
struct PairCost { double fixed, tile, fill, start; };
struct HeadCost { SingleCost plain[3], causal[3]; PairCost pairs[3]; };
constexpr int kRowChoices[3] = {256, 128, 64};
constexpr HeadCost kHeadCost[3] = {
    // D = 64
    {{{5.2, 0.868, 0.956, 0.271, 6.9, 0}, {5.1, 0.505, 0.540, 0.261, 0.8, 0}, {4.9, 0.450, 0.348, 0.035, 1.2, 0}},
     {{6.2, 0.809, 0.837, 0.101, 6.0, 1.134}, {5.4, 0.443, 0.692, 0.390, 1.9, 0.606}, {5.1, 0.402, 0.0, 0.199, 2.2, 0.375}},
     {{2.7, 0.798, 0.183, 8.7}, {7.3, 0.531, 0.069, 0.9}, {6.7, 0.373, 0.0, 0.9}}},
    // 96
    {{{6.5, 1.013, 1.196, 0.378, 7.0, 0}, {5.5, 0.713, 0.809, 0.335, 5.8, 0}, {5.2, 0.659, 0.672, 0.125, 4.4, 0}},
     {{7.6, 0.982, 1.280, 0.176, 8.8, 1.440}, {6.2, 0.681, 0.880, 0.160, 6.5, 0.886}, {5.7, 0.643, 0.715, 0.078, 5.1, 0.734}},
     {{0.0, 0.991, 0.178, 13.7}, {1.5, 0.730, 0.061, 8.5}, {1.0, 0.667, 0.0, 7.4}}},
    // 128
    {{{7.0, 1.269, 1.218, 0.406, 25.6, 0, 9.0, 0.95}, {5.8, 0.885, 0.993, 0.309, 7.6, 0, 5.2, 0.15}, {5.3, 0.754, 0.802, 0.274, 4.6, 0}},
     {{8.3, 1.186, 1.636, 0.225, 9.8, 1.883}, {6.5, 0.873, 1.044, 0.125, 8.3, 1.121}, {6.0, 0.690, 0.368, 0.193, 6.4, 0.879}},
     {{7.2, 1.167, 0.536, 8.0}, {3.0, 0.835, 0.225, 8.7}, {1.0, 0.772, 0.0, 8.3}}}};

constexpr double kSplitMergeUs = 3.5, kSplitBytesPerUs = 2e6;

double expected_single(const SingleCost& c, int64_t batch, int64_t Lq, int64_t Lkv, bool causal, int rows) {
  const int64_t q_tiles = (Lq + rows - 1) / rows, items = q_tiles * batch, rounds = (items + 255) / 256;
  const int64_t all = (Lkv + 63) / 64;   // key tiles of a slice
  // key tiles of query tile i, all of them counted as full (fitted so; where CUs get several the kernel leaves a rest to the lightest)
  auto weight = [&](int64_t i) -> int64_t { return causal ? std::min(all, (i + 1) * rows / 64) : all; };
  double t = (double)weight(q_tiles - 1) * c.tile * (1.0 + c.fill * std::min(1.0, (double)items / 256.0));
  auto share = [&](int64_t j, int64_t i) {
    if (j > 0) t = std::max(t, (double)((j + 1) * weight(i)) * c.full + (double)j * std::min(c.start, c.few + c.per_tile * (double)weight(i)));
  };
  if (!causal) {
    share(rounds - 1, 0);
    return c.fixed + t;
  }
  // (of the workgroups of one weight the last to come is what counts)
  if (q_tiles < rounds) {
    for (int64_t i = 0; i < q_tiles; ++i) share(((q_tiles - i) * batch - 1) / 256, i);
  } else {
    for (int64_t j = 1; j < rounds; ++j) share(j, q_tiles - 1 - 256 * j / batch);
  }
  const int64_t growing = std::min(q_tiles, all * 64 / rows);
  const int64_t total = batch * (growing * (growing + 1) / 2 * (rows / 64) + (q_tiles - growing) * all);
  t = std::max(t, c.mean * (double)total / 256.0 + c.start * ((double)items / 256.0 - 1.0));
  return c.fixed + t;
}

double expected_pairs(const PairCost& c, int64_t batch, int64_t Lq, int64_t Lkv, int rows) {
  const int64_t q_tiles = (Lq + rows - 1) / rows, pairs = q_tiles / 2 * batch, rounds = (pairs + 255) / 256;
  const int64_t all = (Lkv + 63) / 64;
  // key tiles of the pair (i, q_tiles - 1 - i): the same for all, or most in the middle where Lq exceeds Lkv
  auto weight = [&](int64_t i) -> int64_t { return std::min(all, (i + 1) * rows / 64); };
  const int64_t tiles = std::max(weight(0) + weight(q_tiles - 1), weight(q_tiles / 2 - 1) + weight(q_tiles / 2));
  return c.fixed + (double)rounds * (c.start + (double)tiles * c.tile * (1.0 + c.fill * std::min(1.0, (double)pairs / 256.0)));
}

struct AttentionPlan { int rows; bool paired; };
AttentionPlan plan_attention(int64_t batch, int64_t Lq, int64_t Lkv, int64_t D, bool causal) {
  const HeadCost& cost = kHeadCost[D == 64 ? 0 : D == 96 ? 1 : 2];
  // forms that compute mostly beyond Lq, or less per fragment read with four rounds of the chip at hand, are left out
  const int first = Lq <= 64 ? 2 : Lq <= 128 ? 1 : 0;
  const int last = Lq > 128 && (Lq + 255) / 256 * batch >= 1024 ? 0 : 2;
  AttentionPlan plan = {kRowChoices[first], false};
  double best = 0;
  for (int i = first; i <= last; ++i) {
    const int rows = kRowChoices[i];
    const double ahead = i == 0 ? 1.0 : causal ? 1.05 : 1.03;
    const double single = ahead * expected_single(causal ? cost.causal[i] : cost.plain[i], batch, Lq, Lkv, causal, rows);
    if (i == first || single < best) {
      best = single;
      plan = {rows, false};
    }
    const int64_t q_tiles = (Lq + rows - 1) / rows;
    if (causal && q_tiles % 2 == 0 && (i == 0 || q_tiles > 2)) {   // (two small tiles: 1000 slices of 128 x 1024 x 64 21.0 / 18.5)
      const double paired = ahead * expected_pairs(cost.pairs[i], batch, Lq, Lkv, rows);
      if (paired < best) {
        best = paired;
        plan = {rows, true};
      }
    }
  }
  return plan;
}

// Keys in parts, workgroups of 64 queries: where the workgroups of whole problems leave CUs idle and the cost model, for `s` times
// as many slices of 1 / s of the keys plus the second kernel (a launch, and the fp32 rows written and read), sees more than 10%.
// 70 problems that it splits (1..110 slices, 16..4726 queries, 640..7732 keys): 1.06x to 4.8x, 1.86x on average, e.g. 17
// slices of 114 x 7732 x 128 99 / 27 us, 10 of 497 x 6123 x 128 80 / 36, 60 of 41 x 4096 x 128 55 / 28, 9 of 65 x 640 x 128
// 12.9 / 11.9; relative errors against 64 bits 0.96..1.05 of those in one piece (0.985 on average).
struct SplitPlan { int splits, chunk; };
SplitPlan plan_split(int64_t batch, int64_t Lq, int64_t Lkv, int64_t D) {
  const int64_t items = (Lq + 63) / 64 * batch, tiles = (Lkv + 63) / 64;
  if (items >= 256 || tiles < 8) return {1, 0};
  const HeadCost& cost = kHeadCost[D == 64 ? 0 : D == 96 ? 1 : 2];
  double best = 1e30;
  for (int i = Lq <= 64 ? 2 : Lq <= 128 ? 1 : 0; i < 3; ++i)
    best = std::min(best, expected_single(cost.plain[i], batch, Lq, Lkv, false, kRowChoices[i]));
  best *= 0.9;
  SplitPlan plan = {1, 0};
  const double row_us = (double)(batch * Lq * D * 4) / kSplitBytesPerUs;
  for (int64_t s = 2; s <= 16 && s <= tiles / 2 && s * items <= 1024; ++s) {
    const int64_t chunk = (tiles + s - 1) / s, parts = (tiles + chunk - 1) / chunk;
    if (parts != s) continue;
    const double t = expected_single(cost.plain[2], batch * s, Lq, 64 * chunk, false, 64) + kSplitMergeUs + (double)s * row_us;
    if (t < best) {
      best = t;
      plan = {(int)s, (int)(64 * chunk)};
    }
  }
  return plan;
}

bool is_wide(int64_t D) { return D == 160 || D == 192 || D == 256; }

// Head dimensions above 128, by the same rule: a workgroup takes `alone` us for 64 keys, `shared` where two are on a CU.  bf16, us,
// whole / in parts (how many): 16 slices of 64 x 4096 x 256 99.7 / 21.6 (13), 60 100 / 49.6 (4), 128 160 / 112 (2), 240 of 64 x
// 2048 97 / 112 (2, not taken), 100 of 128 x 1024 29.7 / 36.8 (2, not taken), 8 of 256 x 768 x 160 17.0 / 13.7 (4).
// 50 problems that it splits: 1.15x to 7.1x, 2.37x on average; errors against 64 bits as in one piece.
SplitPlan plan_split_wide(int64_t batch, int64_t Lq, int64_t Lkv, int64_t D) {
  const int64_t items = (Lq + 63) / 64 * batch, tiles = (Lkv + 63) / 64;
  if (items >= 256 || tiles < 8 || Lkv % 32 != 0) return {1, 0};
  const double alone = D == 160 ? 1.17 : D == 192 ? 1.32 : 1.53, shared = D == 160 ? 2.3 : D == 192 ? 2.6 : 3.2;
  SplitPlan plan = {1, 0};
  double best = 0.9 * (double)tiles * alone;
  const double row_us = (double)(batch * Lq * D * 4) / kSplitBytesPerUs;
  for (int64_t s = 2; s <= 16 && s <= tiles / 2 && s * items <= 512; ++s) {
    const int64_t chunk = (tiles + s - 1) / s;
    if ((tiles + chunk - 1) / chunk != s) continue;
    const double t = (double)chunk * (s * items <= 256 ? alone : shared) + kSplitMergeUs + (double)s * row_us;
    if (t < best) {
      best = t;
      plan = {(int)s, (int)(64 * chunk)};
    }
  }
  return plan;
}

int64_t next_tuned(int64_t D) { return D <= 64 ? 64 : D <= 96 ? 96 : D <= 128 ? 128 : D; }

// (any arguments: one part for what is not split)
SplitPlan plan_split_any(int64_t batch, int64_t Lq, int64_t Lkv, int64_t D) {
  if (batch <= 0 || batch >= 65536 || Lq <= 0 || Lq >= 1 << 21 || Lkv <= 0 || Lkv >= 1 << 24 || D <= 32 || (D > 128 && !is_wide(D)) ||
      D % 8 != 0)
    return {1, 0};
  return is_wide(D) ? plan_split_wide(batch, Lq, Lkv, D) : plan_split(batch, Lq, Lkv, next_tuned(D));
}

int run_by_head(const AttentionCall& c) {
  if (c.d == next_tuned(c.d)) return c.d == 128 ? run_attention_d128(c) : c.d == 96 ? run_attention_d96(c) : run_attention_d64(c);
  return c.d > 96 ? run_attention_below128(c) : c.d > 64 ? run_attention_below96(c) : run_attention_below64(c);
}

// the tuned kernels for D = Dv = 64, 96 or 128, and, K and V as they come, for multiples of 8 in between and above 32 (arguments
// already checked)
int run_tuned(const void* Q, const void* K, const void* V, void* O, bool bf16, int64_t batch, int64_t Lq, int64_t Lkv,
              int64_t D, bool k_transposed, bool v_transposed, double softmax_scale, bool causal, hipStream_t st) {
  const AttentionPlan plan = plan_attention(batch, Lq, Lkv, next_tuned(D), causal);
  const AttentionCall c = {Q, K, V, O, (int)batch, (int)Lq, (int)Lkv, (int)D, (float)(softmax_scale * 1.4426950408889634),
                           bf16, k_transposed, v_transposed, causal, plan.rows, plan.paired, st};
  return run_by_head(c);
}

// Head dimensions above 128 (V as it comes, whole key tiles): workgroups of 64 queries, two to a CU; 128 (8 wavefronts, one
// to a CU) where those are just one for every CU: the tiles come from the L2 half as often, and nothing is left for a second
// round.  bf16, 64 / 128 queries: 128 slices of 256 x 4096 x 160 162 / 147 us, 256 of 128 x 2048 x 192 106 / 99, 32 of 1000 x
// 1024 x 256 52 / 54; 320 workgroups of 128 are 25% behind.
// Causal: pairs of tiles where they fill rounds of two a CU, and single tiles, heaviest first, otherwise.  D = 256,
// singles / pairs: 341 slices of 384 (1024 pairs) 80 / 60, 150 of 384 (450) 32.7 / 30.5, 192 of 256 (384) 24.2 / 25.3, 320 of
// 1024 39 / 51.  (128 queries a workgroup are up to 30% behind the better of the two.)
AttentionPlan plan_wide(int64_t batch, int64_t Lq, bool causal) {
  const int64_t tiles = (Lq + 63) / 64;
  if (causal) {
    const int64_t pairs = tiles / 2 * batch, rounds = (pairs + 511) / 512;
    return {64, tiles % 2 == 0 && 100 * pairs >= 86 * 512 * rounds};
  }
  const int64_t large = (tiles + 1) / 2 * batch;
  return {tiles % 2 == 0 && large >= 244 && large <= 256 ? 128 : 64, false};
}

int check_attention_args(const char* who, const void* Q, const void* K, const void* V, const void* O, int64_t batch,
                         int64_t Lq, int64_t Lkv, int64_t D, int64_t Dv, int tile_length_q, int tile_length_kv,
                         int tile_hidden_qk, int tile_hidden_v, double softmax_scale) {
  TFK_REQUIRE(Q && K && V && O, TF_ERR_INVALID_ARG, "%s: null pointer", who);
  TFK_REQUIRE(batch > 0 && Lq > 0 && Lkv > 0 && D > 0 && Dv > 0, TF_ERR_INVALID_ARG, "%s: sizes must be positive", who);
  TFK_REQUIRE(batch < 65536 && Lq < (1 << 21) && Lkv < (1 << 24), TF_ERR_INVALID_ARG, "%s: dimension too large", who);
  TFK_REQUIRE(tile_length_q > 0 && tile_length_kv > 0 && tile_hidden_qk > 0 && tile_hidden_v > 0,
              TF_ERR_INVALID_ARG, "%s: tile sizes must be positive", who);
  TFK_REQUIRE(Lq % tile_length_q == 0 && Lkv % tile_length_kv == 0 && D % tile_hidden_qk == 0 &&
                  Dv % tile_hidden_v == 0,
              TF_ERR_INVALID_ARG, "%s: tile [%d,%d,%d,%d] does not divide problem [%lld,%lld,%lld,%lld]", who,
              tile_length_q, tile_length_kv, tile_hidden_qk, tile_hidden_v, (long long)Lq,
              (long long)Lkv, (long long)D, (long long)Dv);
  TFK_REQUIRE(softmax_scale == softmax_scale && softmax_scale - softmax_scale == 0.0,
              TF_ERR_INVALID_ARG, "%s: softmax_scale must be finite", who);
  return TF_OK;
}

// Head dimensions without a tuned kernel go to a run-time instantiation of the header kernel
// (any D %% 32 == 0, Dv %% 16 == 0 with V transposed, Lq %% 16 == 0, Lkv %% 32 == 0).
int attention_fallback(const char* who, const void* Q, const void* K, const void* V, void* O, int dtype,
                       int64_t batch, int64_t Lq, int64_t Lkv, int64_t D, int64_t Dv, int v_is_transposed,
                       int tq, int tkv, int thqk, int thv, double softmax_scale, int causal, hipStream_t st) {
  TFK_REQUIRE(jit_flash_attention_supports(Lq, Lkv, D, Dv, v_is_transposed), TF_ERR_UNSUPPORTED,
              "%s: no tuned kernel for head dims (D=%lld, Dv=%lld) (128/128, 96/96 and 64/64 have one), and the run-time "
              "compiled kernel needs a transposed V, D %% 32 == 0, Dv %% 16 == 0, Lq %% 16 == 0, Lkv %% 32 == 0 "
              "(got Lq=%lld Lkv=%lld, V %s); the torch op pads and transposes as needed",
              who, (long long)D, (long long)Dv, (long long)Lq, (long long)Lkv,
              v_is_transposed ? "transposed" : "in natural layout");
  return jit_flash_attention(Q, K, V, O, dtype, batch, Lq, Lkv, D, Dv, tq, tkv, thqk, thv, softmax_scale, causal, st);
}
}  // namespace
}  // namespace tfk

extern "C" int tf_flash_attention_fwd_f16(const void* Q, const void* K, const void* V, void* O,
                                          int64_t batch, int64_t Lq, int64_t Lkv, int64_t D,
                                          int64_t Dv, int v_is_transposed, int tile_length_q,
                                          int tile_length_kv, int tile_hidden_qk,
                                          int tile_hidden_v, double softmax_scale, int causal,
                                          void* stream) {
  using namespace tfk;
  if (int rc = check_attention_args("tf_flash_attention_fwd_f16", Q, K, V, O, batch, Lq, Lkv, D, Dv, tile_length_q,
                                    tile_length_kv, tile_hidden_qk, tile_hidden_v, softmax_scale))
    return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool tuned = D == Dv && (D == 128 || D == 96 || D == 64);
  if (!tuned)
    return attention_fallback("tf_flash_attention_fwd_f16", Q, K, V, O, TF_DTYPE_F16, batch, Lq, Lkv, D, Dv,
                              v_is_transposed, tile_length_q, tile_length_kv, tile_hidden_qk, tile_hidden_v,
                              softmax_scale, causal, st);
  TFK_REQUIRE(!v_is_transposed || Lkv % 8 == 0, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_f16: transposed V needs Lkv %% 8 == 0");
  return run_tuned(Q, K, V, O, false, batch, Lq, Lkv, D, false, v_is_transposed != 0, softmax_scale, causal != 0, st);
}

extern "C" int tf_flash_attention_fwd(const void* Q, const void* K, const void* V, void* O, int dtype, int64_t batch,
                                      int64_t Lq, int64_t Lkv, int64_t D, int64_t Dv, int v_is_transposed,
                                      int tile_length_q, int tile_length_kv, int tile_hidden_qk, int tile_hidden_v,
                                      double softmax_scale, int causal, void* stream) {
  using namespace tfk;
  if (dtype == TF_DTYPE_F16)
    return tf_flash_attention_fwd_f16(Q, K, V, O, batch, Lq, Lkv, D, Dv, v_is_transposed, tile_length_q, tile_length_kv,
                                      tile_hidden_qk, tile_hidden_v, softmax_scale, causal, stream);
  TFK_REQUIRE(dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  if (int rc = check_attention_args("tf_flash_attention_fwd", Q, K, V, O, batch, Lq, Lkv, D, Dv, tile_length_q,
                                    tile_length_kv, tile_hidden_qk, tile_hidden_v, softmax_scale))
    return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool tuned = D == Dv && (D == 128 || D == 96 || D == 64) && (!v_is_transposed || Lkv % 8 == 0);
  if (!tuned)
    return attention_fallback("tf_flash_attention_fwd", Q, K, V, O, dtype, batch, Lq, Lkv, D, Dv, v_is_transposed,
                              tile_length_q, tile_length_kv, tile_hidden_qk, tile_hidden_v, softmax_scale, causal, st);
  // the tuned kernels with the bf16 MFMA, bf16 weights and bf16 output
  return run_tuned(Q, K, V, O, true, batch, Lq, Lkv, D, false, v_is_transposed != 0, softmax_scale, causal != 0, st);
}

extern "C" int tf_flash_attention_fwd_wide(const void* Q, const void* K, const void* V, void* O, int dtype,
                                           int64_t batch, int64_t Lq, int64_t Lkv, int64_t D, double softmax_scale,
                                           int causal, void* stream) {
  using namespace tfk;
  if (int rc = check_attention_args("tf_flash_attention_fwd_wide", Q, K, V, O, batch, Lq, Lkv, D, D, 1, 1, 1, 1,
                                    softmax_scale))
    return rc;
  TFK_REQUIRE(dtype == TF_DTYPE_F16 || dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_wide: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  TFK_REQUIRE((D == 160 || D == 192 || D == 256) && Lkv % 32 == 0, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_wide: needs a head dimension of 160, 192 or 256 and Lkv %% 32 == 0 "
              "(got D=%lld Lkv=%lld)", (long long)D, (long long)Lkv);
  TFK_REQUIRE((reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(K) | reinterpret_cast<uintptr_t>(V) |
               reinterpret_cast<uintptr_t>(O)) % 16 == 0, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_wide: operands must start at a 16-byte boundary");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const AttentionPlan plan = plan_wide(batch, Lq, causal != 0);
  const AttentionCall c = {Q, K, V, O, (int)batch, (int)Lq, (int)Lkv, (int)D, (float)(softmax_scale * 1.4426950408889634),
                           dtype == TF_DTYPE_BF16, false, false, causal != 0, plan.rows, plan.paired, st};
  return run_attention_wide(c, (int)D);
}

extern "C" int tf_flash_attention_fwd_kt(const void* Q, const void* K, const void* V, void* O, int dtype,
                                         int64_t batch, int64_t Lq, int64_t Lkv, int64_t D, double softmax_scale,
                                         int causal, void* stream) {
  using namespace tfk;
  if (int rc = check_attention_args("tf_flash_attention_fwd_kt", Q, K, V, O, batch, Lq, Lkv, D, D, 1, 1, 1, 1,
                                    softmax_scale))
    return rc;
  TFK_REQUIRE(dtype == TF_DTYPE_F16 || dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_kt: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  TFK_REQUIRE((D == 64 || D == 96 || D == 128) && Lkv % 8 == 0, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_kt: needs a head dimension of 64, 96 or 128 and Lkv %% 8 == 0 "
              "(got D=%lld Lkv=%lld)", (long long)D, (long long)Lkv);
  TFK_REQUIRE((reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(K) | reinterpret_cast<uintptr_t>(V) |
               reinterpret_cast<uintptr_t>(O)) % 16 == 0, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_kt: operands must start at a 16-byte boundary");
  return run_tuned(Q, K, V, O, dtype == TF_DTYPE_BF16, batch, Lq, Lkv, D, true, false, softmax_scale, causal != 0,
                   static_cast<hipStream_t>(stream));
}

extern "C" int tf_flash_attention_fwd_d8(const void* Q, const void* K, const void* V, void* O, int dtype, int64_t batch,
                                         int64_t Lq, int64_t Lkv, int64_t D, double softmax_scale, int causal,
                                         void* stream) {
  using namespace tfk;
  if (int rc = check_attention_args("tf_flash_attention_fwd_d8", Q, K, V, O, batch, Lq, Lkv, D, D, 1, 1, 1, 1,
                                    softmax_scale))
    return rc;
  TFK_REQUIRE(dtype == TF_DTYPE_F16 || dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_d8: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  TFK_REQUIRE(D > 32 && D < 128 && D % 8 == 0 && D != 64 && D != 96, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_d8: needs a head dimension of 40..120, a multiple of 8 other than 64 and 96 "
              "(got %lld)", (long long)D);
  TFK_REQUIRE((reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(K) | reinterpret_cast<uintptr_t>(V) |
               reinterpret_cast<uintptr_t>(O)) % 16 == 0, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_d8: operands must start at a 16-byte boundary");
  return run_tuned(Q, K, V, O, dtype == TF_DTYPE_BF16, batch, Lq, Lkv, D, false, false, softmax_scale, causal != 0,
                   static_cast<hipStream_t>(stream));
}

extern "C" int64_t tf_flash_attention_split_workspace(int64_t batch, int64_t Lq, int64_t Lkv, int64_t D) {
  using namespace tfk;
  const SplitPlan plan = plan_split_any(batch, Lq, Lkv, D);
  return plan.splits > 1 ? (int64_t)plan.splits * batch * Lq * (next_tuned(D) + 2) * 4 : 0;
}

extern "C" int tf_flash_attention_fwd_split(const void* Q, const void* K, const void* V, void* O, int dtype, int64_t batch,
                                            int64_t Lq, int64_t Lkv, int64_t D, int k_is_transposed, double softmax_scale,
                                            void* workspace, void* stream) {
  using namespace tfk;
  if (int rc = check_attention_args("tf_flash_attention_fwd_split", Q, K, V, O, batch, Lq, Lkv, D, D, 1, 1, 1, 1,
                                    softmax_scale))
    return rc;
  TFK_REQUIRE(dtype == TF_DTYPE_F16 || dtype == TF_DTYPE_BF16, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_split: dtype must be TF_DTYPE_F16 or TF_DTYPE_BF16");
  const bool between = D != next_tuned(D);
  const SplitPlan plan = plan_split_any(batch, Lq, Lkv, D);
  TFK_REQUIRE(plan.splits > 1 && (!k_is_transposed || (Lkv % 8 == 0 && !between && !is_wide(D))),
              TF_ERR_UNSUPPORTED, "tf_flash_attention_fwd_split: the keys of [%lld, %lld, %lld, %lld] are not split",
              (long long)batch, (long long)Lq, (long long)Lkv, (long long)D);
  TFK_REQUIRE(workspace, TF_ERR_INVALID_ARG, "tf_flash_attention_fwd_split: null workspace");
  TFK_REQUIRE((reinterpret_cast<uintptr_t>(Q) | reinterpret_cast<uintptr_t>(K) | reinterpret_cast<uintptr_t>(V) |
               reinterpret_cast<uintptr_t>(O) | reinterpret_cast<uintptr_t>(workspace)) % 16 == 0, TF_ERR_UNSUPPORTED,
              "tf_flash_attention_fwd_split: operands must start at a 16-byte boundary");
  const AttentionCall c = {Q, K, V, O, (int)batch, (int)Lq, (int)Lkv, (int)D, (float)(softmax_scale * 1.4426950408889634),
                           dtype == TF_DTYPE_BF16, k_is_transposed != 0, false, false, 64, false,
                           static_cast<hipStream_t>(stream), static_cast<float*>(workspace), plan.splits, plan.chunk};
  return is_wide(D) ? run_attention_wide(c, (int)D) : run_by_head(c);
}

extern "C" int tf_flash_attention_rows(int64_t batch, int64_t Lq, int64_t Lkv, int64_t D, int causal) {
  if (batch <= 0 || Lq <= 0 || Lkv <= 0 || (D != 64 && D != 96 && D != 128)) return 0;
  return tfk::plan_attention(batch, Lq, Lkv, D, causal != 0).rows;
}

extern "C" int tf_flash_attention_pairs(int64_t batch, int64_t Lq, int64_t Lkv, int64_t D, int causal) {
  if (batch <= 0 || Lq <= 0 || Lkv <= 0 || (D != 64 && D != 96 && D != 128)) return 0;
  return tfk::plan_attention(batch, Lq, Lkv, D, causal != 0).paired;
}

extern "C" int tf_flash_attention_wide_rows(int64_t batch, int64_t Lq, int causal) {
  const tfk::AttentionPlan plan = tfk::plan_wide(batch, Lq, causal != 0);
  return plan.paired ? 2 * plan.rows : plan.rows;
}
