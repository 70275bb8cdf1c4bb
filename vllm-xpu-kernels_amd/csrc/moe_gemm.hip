// Kernel family of a grouped GEMM by recipe and expected slots per expert, and
// the launch of the chosen family.
#include <cstdlib>
#include <cstring>

#include "moe_gemm.h"

namespace mi355 {

namespace {
// Block size of the SMALL family by the expected slots per active expert, 0:
// beyond its range.  A block holds avg + 3 to 4 standard deviations where
// the padded block is cheap, so that most experts' weights stream once; beyond
// that larger blocks cost waves per SIMD.  Lines lie at a measured minimum, or
// 2 to 4 % beside it: bf16 16 (32 slots, 64 measured 230), int4 25 (64) and 125
// (W), w8a16 94 (96), each seen on one shape only.  us per layer, MI355X (block: 16 /
// 32 / 64 / 96 / 128, W the 320-slot kernel, - not measured):
//   bf16  Qwen3-30B   avg 4: 213 221 218 229 234   16: 247 234 230 238 244
//                     37: 351 302 251 255 262      56: 435 323 276 262 268 W 291
//                     87: 584 380 332 305 286 W 304   125: - - 384 385 367 W 325
//   fp8   rank of 8 of DeepSeek-V3  4: 246 245 258 269 -   12: 319 271 282 290 -
//                     31: 549 411 301 310 -   40: - - 316 - - W 320
//                     52: - - - 341 - W 332  58: - - - 352 - W 340
//         DeepSeek-V3 whole         40: - - 2164 - - W 2134   47: - - - 2242 - W 2174
//                                   58: - - 2479 2364 - W 2244
//   w8a16 rank of 8 of DeepSeek-V3  3: 241 244 249 270 -   16: 355 281 282 304 -
//                     32: 525 382 297 302 324 W 365   62: - - 421 376 386 W 437
//                     94: - - 467 476 498 W 509
//   int4  Qwen3-30B   4: 76 92 107 - - (fp16)  25: 121 118 123 - -
//                     44: 166 171 144 - - W 246   87: - - 240 215 231 W 281
//                     125: - - 299 295 316 W 303
//   mxfp4 gpt-oss-20b 8: 100 105 120 - -   16: 121 109 124 145 196
//                     25: 130 123 129 148 199   37: 182 153 144 160 212
//                     65: 256 207 217 188 245 W 306   112: - 285 278 320 297 W 342
//         uneven routing (probabilities rank^-0.6 / rank^-1.1; 16 / 32 / 64 / 96)
//                     25: 138 127 145 154 / 139 139 160 172   31: 156 131 154 154 / 161 146 164 182
//                     37: 162 150 168 178 / 174 156 170 207   50: 206 178 182 200 / 210 170 184 213
// mxfp4 keeps 32 slots to 40 per expert, though even routing has 64 the faster
// by up to a tenth: 64-slot blocks were up to 16 % slower there than the kernel
// before them where routing is uneven (200 tokens 128 -> 148, 250 131 -> 155).
int small_block(int recipe, int64_t avg, bool wide_ok) {
  if (recipe == MI355MOE_RECIPE_FP8BLOCK)
    return avg <= 4 ? 16 : avg <= 18 ? 32 : avg <= (wide_ok ? 44 : 46) ? 64
           : avg <= 60 && !wide_ok ? 96 : 0;
  if (is_w8a16_recipe(recipe))
    return avg <= 4 ? 16 : avg <= 17 ? 32 : avg <= 46 ? 64 : avg <= 100 ? 96 : 0;
  if (recipe == MI355MOE_RECIPE_INT4)
    return avg <= 10 ? 16 : avg <= 20 ? 32 : avg <= 48 ? 64 : avg <= 110 ? 96 : 0;
  if (recipe == MI355MOE_RECIPE_MXFP4)
    return avg <= 9 ? 16 : avg <= 40 ? 32 : avg <= 50 ? 64 : avg <= 78 ? 96 : avg <= 130 ? 64 : 0;
  return avg <= 8 ? 16 : avg <= 18 ? 32 : avg <= 46 ? 64 : avg <= 72 ? 96 : avg <= 104 ? 128 : 0;
}
}  // namespace

bool wide_ok_for(int recipe, int64_t a_rows, int64_t ldb_rows, int64_t K, bool w_kblock) {
  if (recipe == MI355MOE_RECIPE_BF16) return K % 32 == 0 && wide_offsets_fit(a_rows, ldb_rows, K);
  if (recipe == MI355MOE_RECIPE_FP8BLOCK) return wide8_shape_ok(a_rows, ldb_rows, K);
  if (recipe == MI355MOE_RECIPE_MXFP8)
    return w_kblock && ldb_rows % 4 == 0 && wide8_shape_ok(a_rows, ldb_rows, K);
  if (recipe == RECIPE_MX4A4)
    return w_kblock && ldb_rows % 4 == 0 && wide8_shape_ok_mx4(a_rows, ldb_rows, K);
  if (recipe == MI355MOE_RECIPE_MXFP4 || recipe == MI355MOE_RECIPE_INT4 ||
      is_w8a16_recipe(recipe))
    return w_kblock && wide4_shape_ok(a_rows, ldb_rows, ldb_rows, K);
  return false;
}

GemmTile pick_tile(int recipe, bool wide_ok, int64_t slots, int64_t local, int64_t num_experts,
                   int* bm) {
  // MI355MOE_GEMM_TILE forces a family (tests, measurements); read per call
  const int force = [] {
    const char* v = getenv("MI355MOE_GEMM_TILE");
    if (!v) return -1;
    if (!strcmp(v, "stream")) return static_cast<int>(TILE_STREAM);
    if (!strcmp(v, "small")) return static_cast<int>(TILE_SMALL);
    if (!strcmp(v, "big")) return static_cast<int>(TILE_BIG);
    if (!strcmp(v, "bigreg")) return static_cast<int>(TILE_BIGREG);
    if (!strcmp(v, "wide")) return static_cast<int>(TILE_WIDE);
    return -1;
  }();
  const int64_t active = local < num_experts ? local : num_experts;
  const int64_t avg = active > 0 ? local / active : 0;
  const int sb = small_block(recipe, avg, wide_ok);
  GemmTile t;
  int b;
  if ((recipe == MI355MOE_RECIPE_MXFP8 || recipe == RECIPE_MX4A4) && wide_ok && avg > 16) {
    // the 320-slot kernel with the e8m0 codes in the MFMA from 17 slots per
    // expert on (16-slot STREAM blocks would stream an expert's weights once
    // per block)
    t = TILE_WIDE, b = kWideBM;
  } else if (is_mx_recipe(recipe) || slots <= kStreamMaxSlots) {
    t = TILE_STREAM, b = 16;
  } else if (sb) {
    t = TILE_SMALL, b = sb;
  } else if (wide_ok) {
    t = TILE_WIDE, b = kWideBM;
  } else if (is_w8a16_recipe(recipe)) {  // (the BIG kernels do not read fp8 for 16-bit)
    t = TILE_SMALL, b = 128;
  } else {
    t = TILE_BIG, b = 128;
  }
  if (force >= 0 && !is_mx_recipe(recipe) && !is_w8a16_recipe(recipe)) {
    t = static_cast<GemmTile>(force);
    if (t == TILE_WIDE && !wide_ok) t = TILE_BIG;
    b = t == TILE_STREAM ? 16 : t == TILE_WIDE ? kWideBM : t == TILE_SMALL ? (sb ? sb : 64) : 128;
  }
  *bm = b;
  return t;
}

int launch_tile_gemm(GemmTile tile, int bm, int recipe, int epi, bool qout,
                     const GemmArgs& a, int64_t max_blocks, void* qs,
                     hipStream_t st) {
  MI_ARG(!a.w_kblock ||
             (recipe == MI355MOE_RECIPE_BF16 && a.K % 32 == 0 &&
              (tile == TILE_STREAM || tile == TILE_SMALL || tile == TILE_WIDE)) ||
             (recipe == MI355MOE_RECIPE_FP8BLOCK &&
              (tile == TILE_STREAM || tile == TILE_SMALL || tile == TILE_WIDE ||
               (tile == TILE_BIG && big8_supported(recipe, a)))) ||
             recipe == MI355MOE_RECIPE_MXFP4 || recipe == MI355MOE_RECIPE_INT4 ||
             is_mx_recipe(recipe) || (is_w8a16_recipe(recipe) && a.K % 32 == 0),
         "K-blocked weights need the bf16 (K % 32 == 0), fp8block, mxfp4, mxfp8 or "
         "per-expert fp8 (K % 32 == 0) recipe and a kernel family that reads them");
  MI_ARG(!is_mx_recipe(recipe) || tile == TILE_STREAM || tile == TILE_WIDE,
         "MX recipes run the STREAM and WIDE kernels");
  MI_CHECK(!is_w8a16_recipe(recipe) || tile == TILE_STREAM || tile == TILE_SMALL ||
               tile == TILE_WIDE,
           MI355MOE_ERR_UNSUPPORTED,
           "per-expert fp8 weights run the STREAM, SMALL and WIDE kernels");
  switch (tile) {
    case TILE_STREAM: return launch_moe_gemm_stream(recipe, epi, qout, a, max_blocks, qs, st);
    case TILE_BIG:
      if (big8_supported(recipe, a))
        return launch_moe_gemm_big8(recipe, epi, qout, a, max_blocks, qs, st);
      if (pipe_supported(recipe, a))
        return launch_moe_gemm_pipe(recipe, epi, qout, a, max_blocks, qs, st);
      return launch_moe_gemm_big(recipe, epi, qout, a, max_blocks, qs, st);
    case TILE_BIGREG: return launch_moe_gemm_big(recipe, epi, qout, a, max_blocks, qs, st);
    case TILE_WIDE:
      if (recipe == MI355MOE_RECIPE_FP8BLOCK || is_mx_recipe(recipe))
        return launch_moe_gemm_wide8(recipe, epi, qout, a, max_blocks, qs, st);
      MI_ARG(!qout, "wide GEMM: no fp8 activation output");
      if (recipe == MI355MOE_RECIPE_MXFP4 || recipe == MI355MOE_RECIPE_INT4 ||
          is_w8a16_recipe(recipe))
        return launch_moe_gemm_wide4(recipe, epi, a, max_blocks, st);
      return launch_moe_gemm_wide(recipe, epi, a, max_blocks, st);
    default: return launch_moe_gemm_mid(recipe, epi, qout, bm, a, max_blocks, qs, st);
  }
}

}  // namespace mi355
