// Grouped GEMM for batches of a few to about a hundred slots per expert (the
// SMALL family): an expert's weights are read once, or a few times from L2,
// and the weight stream is the bound.
//
// A workgroup holds MT * 16 sorted slots of one expert (16-slot tiles past its
// last slot are skipped) and WAVES * RT 16-row weight tiles (GLU: half of
// them gate rows, half their up rows).  Weights go straight from HBM to VGPRs
// in the MFMA's A layout, one 128-value K stage ahead; the activation stage
// is loaded two stages ahead into VGPRs and written one stage ahead to a
// two-slot LDS buffer that all waves read as the MFMA's B operand: one
// barrier a stage.  Four-wave workgroups and one stage in registers keep
// two (96 and 128 slots) to eight waves on a SIMD (bf16: 3.9 / 3.3 resident at
// 64 / 256 tokens of Qwen3-30B, fp8 5.5 at 64 of DeepSeek-V3), which hides the
// memory latency better than more stages in fewer waves did (two and four
// stages measured 3 to 10 % slower).  Loads are unconditional, from addresses limited to the expert's
// range (a load under a branch makes the compiler wait for all loads in
// flight where the branches join); what lies past K is zeroed before use.
//
// Measured per layer against the kernel before (one MFMA tile family, a wait
// for the whole stage): bf16 Qwen3-30B 250 tokens 247 -> 233 us (w13 141 us,
// 5.8 TB/s), fp8 DeepSeek-V3 512 tokens 2375 -> 1966, int4 Qwen3-30B fp16 61
// tokens 151 -> 76, mxfp4 gpt-oss-20b 400 tokens 280 -> 156.
#include <algorithm>
#include <string>

#include "mfma16.h"
#include "moe_gemm.h"

namespace mi355 {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

constexpr int KB = 128;  // K elements per stage

__device__ __forceinline__ f32x4 mfma_e4m3(uint4 a0, uint4 a1, uint4 b0, uint4 b1) {
  const i32x8 a = {(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w,
                   (int)a1.x, (int)a1.y, (int)a1.z, (int)a1.w};
  const i32x8 b = {(int)b0.x, (int)b0.y, (int)b0.z, (int)b0.w,
                   (int)b1.x, (int)b1.y, (int)b1.z, (int)b1.w};
  const f32x4 z = {0.f, 0.f, 0.f, 0.f};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, z, 0, 0, 0, 127, 0, 127);
}

// POST: int4 with its fp16 group scale applied to the fp32 partial sums of the
// group instead of to every weight.  The codes become fp16 integers in 9
// VALU per 8 values (sign bit flipped: u = v + 8; an e4m3 byte 0..15 is u *
// 2^-9, which the scaled conversion turns into u), in the order v0 v2 v4 v6
// v1 v3 v5 v7, in which the activation is staged too (even_odd); int4x8_to16,
// which rounds every product, takes 18.  The -8 per weight is one MFMA per
// step with a constant operand, shared by all weight rows.  16-slot blocks
// only (61 tokens of Qwen3-30B: 87 -> 76 us; with 32 slots equal).  Rounding
// no weight, it is the closer to 64 bits (layer of 61 tokens: 5.2e-4 against
// 6.0e-4); an infinite activation makes its slot's outputs NaN, where products
// of single weights give infinities, and NaN for weights of 0.
__device__ __forceinline__ uint4 int4x8_to_u16(uint32_t w) {
  const uint32_t t = w ^ 0x88888888u;
  const uint32_t lo = t & 0x0f0f0f0fu, hi = (t >> 4) & 0x0f0f0f0fu;
  auto u = [](auto v) { return __builtin_bit_cast(uint32_t, v); };
  return make_uint4(u(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, false)),
                    u(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, true)),
                    u(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, false)),
                    u(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, true)));
}
__device__ __forceinline__ uint4 even_odd(const uint4& v) {
  return make_uint4(__builtin_amdgcn_perm(v.y, v.x, 0x05040100u),
                    __builtin_amdgcn_perm(v.w, v.z, 0x05040100u),
                    __builtin_amdgcn_perm(v.y, v.x, 0x07060302u),
                    __builtin_amdgcn_perm(v.w, v.z, 0x07060302u));
}

// One stage of a lane's weight rows.
template <int RECIPE, bool POST, int RT>
struct MidFrag {                 // 16-bit: 4 MFMA steps x 8 values
  uint4 w[RT][4];
};
template <int RT>
struct MidFrag<MI355MOE_RECIPE_FP8BLOCK, false, RT> {  // 32 e4m3, the block scale
  uint4 w[RT][2];
  float ws[RT];
};
template <int RT>
struct MidFrag<MI355MOE_RECIPE_FP8, false, RT> {       // 32 fp8
  uint4 w[RT][2];
};
template <int RT>
struct MidFrag<MI355MOE_RECIPE_FP8E5M2, false, RT> : MidFrag<MI355MOE_RECIPE_FP8, false, RT> {};
template <int RT>
struct MidFrag<MI355MOE_RECIPE_MXFP4, false, RT> {     // 32 e2m1 and their scale code
  uint4 w[RT];
  uint32_t sc[RT];
};
template <int RT>
struct MidFrag<MI355MOE_RECIPE_INT4, false, RT> : MidFrag<MI355MOE_RECIPE_MXFP4, false, RT> {};
template <int RT>
struct MidFrag<MI355MOE_RECIPE_INT4, true, RT> {       // 32 int4; scales of the lane's output rows
  uint4 w[RT];
  uint2 sc[RT];
};

template <int RECIPE, int MT, int WAVES, int RT, int EPI, bool QOUT, bool F16, bool POST, bool GSC>
__global__ __launch_bounds__(WAVES * 64) void moe_gemm_mid_kernel(const GemmArgs a,
                                                                  void* __restrict__ qs) {
  constexpr bool kFp8 = RECIPE == MI355MOE_RECIPE_FP8BLOCK;
  constexpr bool kFp4 = RECIPE == MI355MOE_RECIPE_MXFP4 || RECIPE == MI355MOE_RECIPE_INT4;
  constexpr bool kInt4 = RECIPE == MI355MOE_RECIPE_INT4;
  constexpr bool kW8 = is_w8a16_recipe(RECIPE);
  constexpr bool kGlu = EPI == EPI_GLU;
  constexpr int BM = 16 * MT;
  constexpr int XB = kFp8 ? 1 : 2;            // bytes per activation element
  constexpr int NTH = WAVES * 64;
  constexpr int ROWB = KB * XB + 16;          // LDS row pitch
  constexpr int CPR = KB * XB / 16;      // 16-byte chunks per row
  constexpr int NCH = BM * CPR;
  constexpr int ACH = (NCH + NTH - 1) / NTH;  // per thread
  constexpr int NC = kGlu ? RT / 2 : RT;           // 16-column output tiles per wave
  constexpr int COLS = WAVES * 16 * NC;       // output columns per workgroup
  static_assert(NTH % CPR == 0, "one chunk column per thread");
  static_assert(!POST || (RECIPE == MI355MOE_RECIPE_INT4 && F16), "scales on the sums: int4, fp16");
  static_assert(!QOUT || (kFp8 && kGlu && COLS == 128), "128 activation columns per workgroup");

  __shared__ __attribute__((aligned(16))) uint8_t sX[2][BM * ROWB];
  __shared__ int s_arow[BM];
  __shared__ int s_drow[BM];
  __shared__ float s_xs[kFp8 ? 2 : 1][kFp8 ? BM : 1];
  __shared__ float s_amax[QOUT ? WAVES : 1][QOUT ? BM : 1];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, q = lane >> 4;
  // XCD x (workgroups go round-robin over the 8 XCDs) takes a contiguous range
  // of the (block, column tile) pairs, so that one L2 serves a block's
  // activation rows to all its column tiles
  const int n_tiles = static_cast<int>(gridDim.x);
  const int valid = (*a.ntp + BM - 1) / BM * n_tiles;
  const int lin = static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x);
  const int per = (valid + 7) / 8;
  const int tile = (lin & 7) * per + (lin >> 3);
  if ((lin >> 3) >= per || tile >= valid) return;  // uniform
  const int blk = tile / n_tiles, ntile = tile - blk * n_tiles;
  const int e = a.block_expert[blk];
  const int64_t K = a.K, N = a.N;
  const int rid = tid < BM ? a.row_ids[static_cast<int64_t>(blk) * BM + tid] : -1;

  // ---- this wave's weight rows.  Every load is the expert's base plus a
  // 32-bit lane offset (the launcher checks that an expert fits), advanced by
  // a uniform stage stride and limited to the expert's last bytes: lanes past
  // K, and stages prefetched past the end, read in-range data.
  const int64_t col0 = static_cast<int64_t>(ntile) * COLS + wave * (16 * NC);
  const int64_t wrow_bytes = kFp4 ? K / 2 : (kW8 ? K : K * XB);
  const uint8_t* wexp = static_cast<const uint8_t*>(a.B) +
                        static_cast<int64_t>(e) * a.ldb_rows * wrow_bytes;
  const WStride wst = kFp4 ? w_stride4(a)
                           : (kW8 ? w_stride8w(a) : (kFp8 ? w_stride8(a) : w_stride16(a)));
  const uint32_t kblk = static_cast<uint32_t>(wst.kblk);
  const uint32_t wstage = kFp8 ? kblk : 4 * kblk;
  const uint32_t wlim = static_cast<uint32_t>(a.ldb_rows * wrow_bytes) - 16u;
  const int nk = static_cast<int>((K + KB - 1) / KB);
  uint32_t woff[RT], soff[RT], sshift[RT];
  // scales: base of the expert, bytes per stage, last offset
  const uint8_t* sexp = nullptr;
  uint32_t sstage = 0, slim = 0;
  int sper = 0;  // int4: log2 of the stages (GSC: 32-value blocks) per group
  if constexpr (kFp8) {
    const int wsh = 7 - a.ws_rows64;
    const int64_t rows = a.ldb_rows >> wsh;
    sexp = static_cast<const uint8_t*>(a.b_scale) + e * rows * nk * 4;
    sstage = 4;
    slim = static_cast<uint32_t>(rows * nk * 4) - 4u;
  } else if constexpr (POST) {
    const int64_t groups = K / a.w_group;
    sper = a.w_group >> 8;  // 128: a group a stage, 256: two stages
    sexp = static_cast<const uint8_t*>(a.b_scale) + e * groups * a.ldb_rows * 2;
    sstage = static_cast<uint32_t>(a.ldb_rows * 2);
    slim = static_cast<uint32_t>(groups * a.ldb_rows * 2) - 8u;
  } else if constexpr (kInt4) {
    const int64_t groups = K / a.w_group;
    sexp = static_cast<const uint8_t*>(a.b_scale) + e * groups * a.ldb_rows * 2;
    slim = static_cast<uint32_t>(groups * a.ldb_rows * 2) - (GSC ? 2u : 4u);
    if constexpr (GSC) {  // lane block 4 s + q is in group (4 s + q) >> sper
      sper = 31 - __clz(a.w_group >> 5);
      sstage = a.w_kblock ? static_cast<uint32_t>(a.ldb_rows * 2) : 2u;  // per group
    } else {
      sper = a.w_group >> 8;
      sstage = static_cast<uint32_t>(a.ldb_rows * 2);
    }
  } else if constexpr (kFp4) {
    sexp = static_cast<const uint8_t*>(a.b_scale) + e * (K / 32) * a.ldb_rows;
    sstage = 4u * static_cast<uint32_t>(s_stride4(a).kblk);
    slim = static_cast<uint32_t>((K / 32) * a.ldb_rows) - (GSC ? 1u : 4u);
  }
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int64_t c = col0 + 16 * (t % NC);
    const int64_t up = t >= NC ? a.up_off : 0;
    // the lane's A row, and the first of its 4 output rows
    const uint32_t wrow = static_cast<uint32_t>(up + (c + l16 < N ? c + l16 : 0));
    const uint32_t orow = static_cast<uint32_t>(up + (c + 4 * q < N ? c + 4 * q : 0));
    woff[t] = wrow * static_cast<uint32_t>(wst.row) +
              (kFp8 ? 32u * q : kFp4 || kW8 ? q * kblk : 16u * q);
    soff[t] = sshift[t] = 0;
    if constexpr (kFp8) soff[t] = (orow >> (7 - a.ws_rows64)) * static_cast<uint32_t>(nk) * 4u;
    else if constexpr (POST) soff[t] = orow * 2u;
    else if constexpr (GSC && kInt4) {
      soff[t] = a.w_kblock ? 2u * wrow : 2u * wrow * static_cast<uint32_t>(K / a.w_group);
    } else if constexpr (GSC) {
      const WStride ss = s_stride4(a);
      soff[t] = wrow * static_cast<uint32_t>(ss.row) + q * static_cast<uint32_t>(ss.kblk);
    } else if constexpr (kInt4) {
      soff[t] = 2u * (wrow & ~1u);
      sshift[t] = 16u * (wrow & 1u);
    } else if constexpr (kFp4) {
      soff[t] = q * static_cast<uint32_t>(a.ldb_rows) + (wrow & ~3u);
      sshift[t] = 8u * (wrow & 3u);
    }
  }

  using Frag = MidFrag<RECIPE, POST, RT>;
  auto at = [&](const uint8_t* base, uint32_t off, uint32_t lim) {
    return base + (off < lim ? off : lim);
  };
  auto load_w = [&](Frag& f, int s) {
    const uint32_t so = static_cast<uint32_t>(s) * wstage;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      if constexpr (kFp8 || kW8) {
        const uint4* p = reinterpret_cast<const uint4*>(at(wexp, woff[t] + so, wlim - 16u));
        f.w[t][0] = p[0];
        f.w[t][1] = p[1];
      } else if constexpr (kFp4) {
        f.w[t] = *reinterpret_cast<const uint4*>(at(wexp, woff[t] + so, wlim));
      } else {
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
          f.w[t][s4] = *reinterpret_cast<const uint4*>(at(wexp, woff[t] + so + s4 * kblk, wlim));
      }
      if constexpr (kFp8)
        f.ws[t] = *reinterpret_cast<const float*>(at(sexp, soff[t] + s * sstage, slim));
      else if constexpr (POST)
        f.sc[t] = *reinterpret_cast<const uint2*>(at(sexp, soff[t] + (s >> sper) * sstage, slim));
      else if constexpr (GSC && kInt4)
        f.sc[t] = *reinterpret_cast<const uint16_t*>(
            at(sexp, soff[t] + ((4u * s + q) >> sper) * sstage, slim));
      else if constexpr (GSC)
        f.sc[t] = *at(sexp, soff[t] + s * sstage, slim);
      else if constexpr (kInt4)
        f.sc[t] = *reinterpret_cast<const uint32_t*>(at(sexp, soff[t] + (s >> sper) * sstage, slim));
      else if constexpr (kFp4)
        f.sc[t] = *reinterpret_cast<const uint32_t*>(at(sexp, soff[t] + s * sstage, slim));
    }
  };
  // the first weight stage is on its way before the slots are known
  Frag f;
  load_w(f, 0);

  if (tid < BM) {
    const bool ok = rid >= 0 && rid < a.num_valid;
    s_arow[tid] = ok ? (a.a_by_pos ? blk * BM + tid : rid / a.a_div) : -1;
    s_drow[tid] = ok ? (a.d_by_pos ? blk * BM + tid : rid) : -1;
  }
  __syncthreads();
  // 16-slot tiles past the last valid slot (a block's valid slots come first)
  int mtv = 0;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) mtv += s_arow[16 * mt] >= 0 ? 1 : 0;
  mtv = __builtin_amdgcn_readfirstlane(mtv);

  // the last stage of a K that is not a multiple of 128: what was re-read is zeroed
  auto clear_tail = [&](int64_t k0) {
    const uint4 z = make_uint4(0, 0, 0, 0);
    if constexpr (kFp4 || kW8) {
      if (k0 + 32 * q >= K) {
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          if constexpr (kFp4) {
            f.w[t] = z;
            if constexpr (!POST) f.sc[t] = 0;
          } else {
            f.w[t][0] = f.w[t][1] = z;
          }
        }
      }
    } else if constexpr (!kFp8) {
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
        if (k0 + 32 * s4 + 8 * q + 8 > K) {
#pragma unroll
          for (int t = 0; t < RT; ++t) f.w[t][s4] = z;
        }
    }
  };

  // ---- activation stage: thread's column xc, rows xrow
  constexpr int KE = 16 / XB;  // K elements per 16 bytes
  const uint32_t xc = (tid % CPR) * KE;
  const uint8_t* xrow[ACH];
  uint32_t xok = 0;
#pragma unroll
  for (int i = 0; i < ACH; ++i) {
    const int idx = tid + NTH * i;
    const int r = idx < NCH ? s_arow[idx / CPR] : -1;
    if (r >= 0) xok |= 1u << i;
    xrow[i] = static_cast<const uint8_t*>(a.A) + static_cast<int64_t>(r >= 0 ? r : 0) * K * XB;
  }
  uint4 av[ACH];
  float sv = 0.f;
  const uint32_t xlim = static_cast<uint32_t>(K * XB) - 16u;
  const int xsr = kFp8 && tid < BM ? s_arow[tid] : -1;
  const float* xsp = kFp8 ? a.a_scale + static_cast<int64_t>(xsr >= 0 ? xsr : 0) * nk : nullptr;
  auto load_x = [&](int s) {
    const uint32_t off0 = (static_cast<uint32_t>(s) * KB + xc) * XB;
    const uint32_t off = off0 < xlim ? off0 : xlim;
#pragma unroll
    for (int i = 0; i < ACH; ++i) av[i] = *reinterpret_cast<const uint4*>(xrow[i] + off);
    if constexpr (kFp8) sv = xsp[s < nk ? s : nk - 1];
  };
  auto store_x = [&](int s) {
    const bool kin = static_cast<uint32_t>(s) * KB + xc < static_cast<uint32_t>(K);
#pragma unroll
    for (int i = 0; i < ACH; ++i) {
      const int idx = tid + NTH * i;
      const uint32_t m = kin && (xok >> i & 1u) ? ~0u : 0u;
      uint4 v = make_uint4(av[i].x & m, av[i].y & m, av[i].z & m, av[i].w & m);
      if constexpr (POST) v = even_odd(v);
      if (NCH % NTH == 0 || idx < NCH)
        *reinterpret_cast<uint4*>(sX[s & 1] + (idx / CPR) * ROWB + (idx % CPR) * 16) = v;
    }
    if constexpr (kFp8) {
      if (tid < BM) s_xs[s & 1][tid] = xsr >= 0 ? sv : 0.f;
    }
  };

  f32x4 acc[MT][RT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[mt][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // f holds stage s and is reloaded with stage s + 1: packed weights as soon
  // as they are decoded, others after their last MFMA
  auto compute = [&](int s) {
    uint4 wf[kFp4 ? RT : 1][4];
    if constexpr (kFp4) {
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const uint32_t w4[4] = {f.w[t].x, f.w[t].y, f.w[t].z, f.w[t].w};
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          if constexpr (POST) wf[t][s4] = int4x8_to_u16(w4[s4]);
          else wf[t][s4] = w4_decode8<RECIPE, F16>(w4[s4], (f.sc[t] >> sshift[t]) & (kInt4 ? 0xffffu : 0xffu));
        }
      }
    }
    uint2 psc[RT];
    if constexpr (POST) {
#pragma unroll
      for (int t = 0; t < RT; ++t) psc[t] = f.sc[t];
    }
    // (the scheduler must not lift the loads above the last use of the
    // registers they go to: the copies it then makes wait for them)
    if constexpr (kFp4) {
      if constexpr (!POST) __builtin_amdgcn_sched_barrier(0);
      load_w(f, s + 1);
      if constexpr (!POST) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      if (mt > 0 && mt >= mtv) break;  // uniform
      const uint8_t* xr = sX[s & 1] + (mt * 16 + l16) * ROWB;
      if constexpr (kFp8) {
        const uint4 x0 = *reinterpret_cast<const uint4*>(xr + 32 * q);
        const uint4 x1 = *reinterpret_cast<const uint4*>(xr + 32 * q + 16);
        const float xs = s_xs[s & 1][mt * 16 + l16];
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          const f32x4 p = mfma_e4m3(f.w[t][0], f.w[t][1], x0, x1);
          acc[mt][t] += p * (xs * f.ws[t]);
        }
      } else {
        uint4 x[4];
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4)
          x[s4] = *reinterpret_cast<const uint4*>(
              xr + (kFp4 || kW8 ? 32 * q + 8 * s4 : 32 * s4 + 8 * q) * 2);
        if constexpr (POST) {
          constexpr uint32_t m8 = 0xC800C800u;  // -8, -8
          const uint4 c8 = make_uint4(m8, m8, m8, m8);
          f32x4 base = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s4 = 0; s4 < 4; ++s4) base = mfma16_16x16x32<F16>(c8, x[s4], base);
#pragma unroll
          for (int t = 0; t < RT; ++t) {
            f32x4 p = base;
#pragma unroll
            for (int s4 = 0; s4 < 4; ++s4) p = mfma16_16x16x32<F16>(wf[t][s4], x[s4], p);
            float sc[4];
            sc[0] = ld16<F16>(static_cast<uint16_t>(psc[t].x));
            sc[1] = ld16<F16>(static_cast<uint16_t>(psc[t].x >> 16));
            sc[2] = ld16<F16>(static_cast<uint16_t>(psc[t].y));
            sc[3] = ld16<F16>(static_cast<uint16_t>(psc[t].y >> 16));
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[mt][t][r] = fmaf(p[r], sc[r], acc[mt][t][r]);
          }
        } else {
#pragma unroll
          for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
            for (int t = 0; t < RT; ++t) {
              uint4 w;
              if constexpr (kFp4) {
                w = wf[t][s4];
              } else if constexpr (kW8) {
                constexpr bool k52 = RECIPE == MI355MOE_RECIPE_FP8E5M2;
                const uint4 v = f.w[t][s4 >> 1];
                w = fp8x8_to16<k52, F16>((s4 & 1) ? make_uint2(v.z, v.w) : make_uint2(v.x, v.y));
              } else {
                w = f.w[t][s4];
              }
              acc[mt][t] = mfma16_16x16x32<F16>(w, x[s4], acc[mt][t]);
            }
        }
      }
    }
    if constexpr (!kFp4) {
      __builtin_amdgcn_sched_barrier(0);
      load_w(f, s + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- K loop: stage s + 1 of the activation was requested a stage ago,
  // stage s + 2 is requested before the weights are reloaded
  load_x(0);
  store_x(0);
  load_x(1);
  __syncthreads();
  const int nfull = static_cast<int>(K / KB);
  for (int s = 0; s < nfull; ++s) {
    store_x(s + 1);
    load_x(s + 2);
    compute(s);
    __syncthreads();
  }
  if (nfull < nk) {  // uniform
    clear_tail(static_cast<int64_t>(nfull) * KB);
    compute(nfull);
  }

  // ---- epilogue: lane holds D[slot = mt*16 + l16][col0 + 16 j + 4 q + r]
  const int64_t bias_base = static_cast<int64_t>(e) * a.ldb_rows;
  const float es = a.expert_scale ? a.expert_scale[e] : 1.f;
  float outv[MT][NC][4];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int64_t n = col0 + j * 16 + 4 * q;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool nok = n + r < N;
        float v = acc[mt][j][r] * es;
        if (a.bias && nok) v += ld16<F16>(a.bias[bias_base + n + r]);
        v = rnd16<F16>(v);
        if constexpr (kGlu) {
          float u = acc[mt][kGlu ? j + NC : 0][r] * es;
          if (a.bias && nok) u += ld16<F16>(a.bias[bias_base + a.up_off + n + r]);
          u = rnd16<F16>(u);
          glu_clamp(a, n + r, v, u);
          v = rnd16<F16>(glu16<F16>(v, u, a.act, a.alpha, a.limit));
        }
        outv[mt][j][r] = nok ? v : 0.f;
      }
    }
  }

  if constexpr (QOUT) {
    // e4m3 output, one fp32 scale per (row, 128 columns): the workgroup's columns
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float m = 1e-10f;
#pragma unroll
      for (int j = 0; j < NC; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) m = fmaxf(m, fabsf(outv[mt][j][r]));
      m = max_over_rows(m);
      if (q == 0) s_amax[wave][mt * 16 + l16] = m;
    }
    __syncthreads();
    uint8_t* dq = static_cast<uint8_t*>(a.D);
    float* ds = static_cast<float*>(qs);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int row = mt * 16 + l16;
      const int drow = s_drow[row];
      if (drow < 0) continue;
      float am = s_amax[0][row];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) am = fmaxf(am, s_amax[w][row]);
      const float sc = fmaxf(am / 448.f, 1.0f / (448.f * 512.f));
      const float inv = 1.0f / sc;
      if (wave == 0 && q == 0) ds[static_cast<int64_t>(drow) * (N / 128) + ntile] = sc;
#pragma unroll
      for (int j = 0; j < NC; ++j)
        *reinterpret_cast<uint32_t*>(dq + static_cast<int64_t>(drow) * N + col0 + 16 * j + 4 * q) =
            e4m3x4_sat(outv[mt][j][0] * inv, outv[mt][j][1] * inv, outv[mt][j][2] * inv,
                       outv[mt][j][3] * inv);
    }
  } else {
    uint16_t* d = static_cast<uint16_t*>(a.D);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int drow = s_drow[mt * 16 + l16];
      if (drow < 0) continue;
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const int64_t n = col0 + j * 16 + 4 * q;
        uint16_t* dst = d + static_cast<int64_t>(drow) * N + n;
        if (n + 3 < N && (N & 3) == 0) {
          *reinterpret_cast<uint2*>(dst) = make_uint2(pack16x2<F16>(outv[mt][j][0], outv[mt][j][1]),
                                                      pack16x2<F16>(outv[mt][j][2], outv[mt][j][3]));
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < N) dst[r] = st16<F16>(outv[mt][j][r]);
        }
      }
    }
  }
}

// Row tiles per wave (a workgroup of 4 waves then has 64 RT weight rows):
// four where a fragment is small (4-bit weights, at most 32 slots: half the
// LDS reads per weight; mxfp4 gpt-oss layers of 64 tokens 104 -> 100 us; w2
// keeps two, 736 workgroups of its 2880 x 32 rows instead of 384) or converted (fp8 to 16 bits, 64 slots and more:
// DeepSeek-V3 rank of 8, 1024 tokens, 307 -> 297 us); otherwise two, which
// leave registers for more waves (bf16 Qwen3-30B, 64 tokens, 213 against 215
// us, 600 tokens of 96-slot blocks 255 against 282).
template <int RECIPE, int MT, int EPI, bool POST>
constexpr int mid_row_tiles() {
  if (POST) return 4;
  if (RECIPE == MI355MOE_RECIPE_MXFP4) return MT <= 2 && EPI == EPI_GLU ? 4 : 2;
  if (is_w8a16_recipe(RECIPE)) return MT == 4 || MT == 6 ? 4 : 2;
  return 2;
}

template <int RECIPE, int MT, int EPI, bool QOUT, bool POST, bool GSC>
int launch_mid_t(const GemmArgs& a, int64_t max_blocks, void* qs, hipStream_t st) {
  // e4m3 output needs the 128 activation columns of a scale in one workgroup
  constexpr int RT = QOUT ? 2 : mid_row_tiles<RECIPE, MT, EPI, POST>();
  constexpr int WAVES = QOUT ? 8 : 4;
  constexpr int COLS = WAVES * RT * (EPI == EPI_GLU ? 8 : 16);
  const int64_t nx = cdiv(a.N, COLS);
  // the kernel's XCD order takes tile (w % 8) * per + w / 8 in workgroup w:
  // the launch covers a multiple of 8 workgroups
  const int64_t ny = cdiv(cdiv(nx * max_blocks, 8) * 8, nx);
  const dim3 grid(static_cast<unsigned>(nx), static_cast<unsigned>(ny));
  if (a.out_f16)
    moe_gemm_mid_kernel<RECIPE, MT, WAVES, RT, EPI, QOUT, true, POST, GSC>
        <<<grid, dim3(WAVES * 64), 0, st>>>(a, qs);
  else if constexpr (!POST)
    moe_gemm_mid_kernel<RECIPE, MT, WAVES, RT, EPI, QOUT, false, POST, GSC>
        <<<grid, dim3(WAVES * 64), 0, st>>>(a, qs);
  MI_LAUNCH_CHECK();
  return MI355MOE_OK;
}
template <int RECIPE, int EPI, bool QOUT, bool GSC = false>
int launch_mid(int bm, const GemmArgs& a, int64_t max_blocks, void* qs, hipStream_t st) {
  switch (bm) {
    case 16: return launch_mid_t<RECIPE, 1, EPI, QOUT, false, GSC>(a, max_blocks, qs, st);
    case 32: return launch_mid_t<RECIPE, 2, EPI, QOUT, false, GSC>(a, max_blocks, qs, st);
    case 64: return launch_mid_t<RECIPE, 4, EPI, QOUT, false, GSC>(a, max_blocks, qs, st);
    case 96: return launch_mid_t<RECIPE, 6, EPI, QOUT, false, GSC>(a, max_blocks, qs, st);
    case 128:  // 16-bit and per-expert fp8 weights only (small_block)
      if constexpr (RECIPE == MI355MOE_RECIPE_BF16 || is_w8a16_recipe(RECIPE))
        return launch_mid_t<RECIPE, 8, EPI, QOUT, false, GSC>(a, max_blocks, qs, st);
      break;
    default: break;
  }
  return set_error(MI355MOE_ERR_INVALID, "no SMALL kernel of this recipe for blocks of " +
                                             std::to_string(bm) + " slots");
}

bool aligned(const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

}  // namespace

bool mid_fits(int64_t ldb_rows, int64_t K) {
  // an expert's bytes (16-bit elements bound every recipe) within 32-bit
  // offsets; what is addressed past them is limited to the range
  return ldb_rows <= (int64_t(1) << 30) / std::max<int64_t>(K, 1);
}

int launch_moe_gemm_mid(int recipe, int epi, bool qout, int bm, const GemmArgs& a,
                        int64_t max_blocks, void* qs, hipStream_t st) {
  if (max_blocks <= 0 || a.N <= 0) return MI355MOE_OK;
  MI_ARG(mid_fits(a.ldb_rows, a.K), "expert matrix too large for 32-bit offsets");
  if (qout) {
    MI_ARG(recipe == MI355MOE_RECIPE_FP8BLOCK && epi == EPI_GLU && a.N % 128 == 0,
           "fp8 activation output needs the fp8block recipe and I % 128 == 0");
    return launch_mid<MI355MOE_RECIPE_FP8BLOCK, EPI_GLU, true>(bm, a, max_blocks, qs, st);
  }
#define MI_MID(R, GSC)                                                                      \
  return epi == EPI_GLU ? launch_mid<R, EPI_GLU, false, GSC>(bm, a, max_blocks, qs, st)     \
                        : launch_mid<R, EPI_STORE, false, GSC>(bm, a, max_blocks, qs, st);
  switch (recipe) {
    case MI355MOE_RECIPE_BF16: MI_MID(MI355MOE_RECIPE_BF16, false)
    case MI355MOE_RECIPE_FP8BLOCK: MI_MID(MI355MOE_RECIPE_FP8BLOCK, false)
    case MI355MOE_RECIPE_FP8: MI_MID(MI355MOE_RECIPE_FP8, false)
    case MI355MOE_RECIPE_FP8E5M2: MI_MID(MI355MOE_RECIPE_FP8E5M2, false)
    case MI355MOE_RECIPE_MXFP4:
      // K-blocked codes, four rows' in an aligned word; otherwise one byte a lane
      if (a.w_kblock && a.ldb_rows % 4 == 0 && aligned(a.b_scale, 4)) {
        MI_MID(MI355MOE_RECIPE_MXFP4, false)
      }
      MI_MID(MI355MOE_RECIPE_MXFP4, true)
    case MI355MOE_RECIPE_INT4: {
      const bool rows = a.w_kblock && a.w_group % KB == 0 && a.ldb_rows % 4 == 0 &&
                        a.up_off % 4 == 0 && aligned(a.b_scale, 8);
      // POST, four rows' scales in one load: the same call in larger blocks,
      // row-major, or with scales off an 8-byte boundary rounds every weight
      // (6e-4 apart, relative to the layer's output)
      if (rows && a.out_f16 && bm == 16)
        return epi == EPI_GLU
                   ? launch_mid_t<MI355MOE_RECIPE_INT4, 1, EPI_GLU, false, true, false>(a, max_blocks, qs, st)
                   : launch_mid_t<MI355MOE_RECIPE_INT4, 1, EPI_STORE, false, true, false>(a, max_blocks, qs, st);
      if (rows) {
        MI_MID(MI355MOE_RECIPE_INT4, false)
      }
      MI_MID(MI355MOE_RECIPE_INT4, true)
    }
    default: break;
  }
#undef MI_MID
  return set_error(MI355MOE_ERR_INVALID, "unknown recipe");
}

}  // namespace mi355
