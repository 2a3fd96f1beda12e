// ftm_tile.hip -- the MoE expert stages above the token crossover as grouped
// bf16-MFMA tiles whose weights go straight from memory into registers.
//
// A tile is 64 pairs (rows) of one expert x 256 weight rows: four waves, each
// 64 rows x 64 weight rows over the whole K (stage A: 32 gate + 32 up
// channels of w13, so the activation needs no exchange; stage B: 64 output
// columns of w2).  A wave owns its weight rows, so the packed weights are
// loaded once per tile by buffer loads into VGPRs, one K step ahead of their
// use, and decoded there to exact bf16 codes; only the activations, which all
// four waves read, go through LDS: a three-stage ring filled by direct
// global->LDS copies two K steps ahead.  One barrier per K step of 128 (64
// for bf16 weights): 64 MFMAs a wave between barriers, two workgroups per CU.
// Quantisation-group scales multiply the fp32 partial sums of each group, as
// in the GEMV path.
//
// GPTQ: a nibble, zero-extended to a byte, is the e4m3 code of q * 2^-9 (0..15
// are the subnormals and the first binade), so v_cvt_scalef32_pk_bf16_fp8
// with the scale 512 turns two bytes into the bf16 values q exactly: 9 VALU a
// word in natural K order.  The zero points are taken out once per tile:
// every wave sums its share of the rows over each 128-wide group with one
// MFMA against ones per 32 K, the sums X[row][group] wait in LDS, and
// acc -= X . (s (z + 1)) runs on the fp32 16x16x4 MFMA at the end.
#include <type_traits>

#include "ftm_layer.h"

namespace ftm {

constexpr int kTM = 64;        // rows (pairs) per tile
constexpr int kTN = 256;       // weight rows per tile
constexpr int kTHPitch = 128 * 2 + 16;  // bytes of a staged h row (stage A's epilogue, 128 channels)
constexpr int kTStages = 2;    // activation stages in LDS

// How group scales enter: none (bf16; MXFP4's ride in the decode), one group
// over K (applied after the loop), one per K step of 128, one per 64.
enum { kScaleNone = 0, kScaleOne = 1, kScale128 = 2, kScale64 = 3 };

template <int FMT>
struct TileFmt {
  static constexpr int kKS = FMT == FTM_FMT_BF16 ? 64 : 128;                        // K per step
  static constexpr int kNL = FMT == FTM_FMT_MXFP4 ? 1 : 2;                          // 16-byte loads per row and step
  static constexpr int kARow = 2 * kKS;                                             // activation bytes per row and step
  static constexpr int kStage = kTM * kARow;
  static constexpr int kACopies = kStage / 1024 / 4;                                // 16-byte pieces per thread and step
  static constexpr int kRing = kTStages * kStage > kTM * kTHPitch ? kTStages * kStage : kTM * kTHPitch;
  static constexpr bool kPost = FMT == FTM_FMT_FP8_BLOCK || FMT == FTM_FMT_INT8_PACKED || FMT == FTM_FMT_GPTQ_INT4;
};

// Activation slot swizzle: slot s of row r holds 16-byte piece s ^ tile_fa(r)
// of its step, so that the 16 rows of one operand read hit distinct banks.
template <int FMT>
__device__ __forceinline__ int tile_fa(int r) {
  return TileFmt<FMT>::kKS == 128 ? (r & 15) : ((r >> 1) & 7);
}

// Tile row (weight row of the projection) of MFMA column block nj, lane
// column m, of a wave whose first rows are base[0] (nj 0, 1) and base[1] (2,
// 3): K-major formats 16 consecutive rows a block, GPTQ two neighbouring
// columns a lane (one 8-byte load).
template <int FMT>
__device__ __forceinline__ int tile_row(const int (&base)[2], int nj, int m) {
  return FMT == FTM_FMT_GPTQ_INT4 ? base[nj >> 1] + 2 * m + (nj & 1) : base[nj >> 1] + 16 * (nj & 1) + m;
}

// One step's packed weights of a wave and the raw words of its scales.
template <int FMT>
struct TileW {
  u32x4 w[4][TileFmt<FMT>::kNL];
  uint32_t s[2][4];  // FP8: [half-step][0 / 2]; INT8: [half-step][nj]; MXFP4: [0][nj], the lane's e8m0 byte
};
template <>
struct TileW<FTM_FMT_GPTQ_INT4> {
  u32x2 w[2][4];  // [half][q]: the words of columns 2m, 2m + 1 at K 32 q + 8 g
  uint32_t s[2];  // [half]: both columns' 16-bit scales
};

// Eight nibbles (low first) -> bf16 values q in natural order.
__device__ __forceinline__ u32x4 gptq_word_natural(uint32_t w) {
  const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;  // q0 q2 q4 q6 / q1 q3 q5 q7
  const uint32_t a = __builtin_amdgcn_perm(hi, lo, 0x05010400u);     // q0 q1 q2 q3
  const uint32_t b = __builtin_amdgcn_perm(hi, lo, 0x07030602u);     // q4 q5 q6 q7
  u32x4 r;
  r.x = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)a, 512.0f, false));
  r.y = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)a, 512.0f, true));
  r.z = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)b, 512.0f, false));
  r.w = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)b, 512.0f, true));
  return r;
}

// 16-bit scale word `hi` (0 / 1) of a pair -> its value (branch-free).
__device__ __forceinline__ float half_word(uint32_t w, int hi, int dt) {
  const uint32_t h = hi ? w >> 16 : w & 0xffffu;
  const float f = f16_to_f32((uint16_t)h), b = __uint_as_float(h << 16);
  return dt == FTM_DT_F16 ? f : b;
}

// The K loop: acc += A (16 MI rows) . W^T over the whole K.
//   arow[i]: start of the activation row of this thread's piece i
//   lds: two activation stages; Xs: GPTQ row sums [kTM][K / 128 + 1]
// Every step issues the same loads (past the last step through clamped or
// out-of-range offsets), so the compiler's counted waits are exact.
template <int FMT, int MODE, int MI>
__device__ __forceinline__ void tile_kloop(const ProjSlot& W, const int (&base)[2],
                                           const char* const (&arow)[TileFmt<FMT>::kACopies], char* lds, float* Xs,
                                           f32x4 (&acc)[MI][4]) {
  using F = TileFmt<FMT>;
  constexpr bool GQ = FMT == FTM_FMT_GPTQ_INT4;
  constexpr bool POST = MODE == kScale128 || MODE == kScale64;  // partial sums per step (or half step)
  constexpr int KS = F::kKS;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, m = lane & 15;
  const int K = W.K, N = W.N;
  const int nsteps = (K + KS - 1) / KS;

  // ---- activations: 16-byte pieces of the step's rows, one step ahead in
  // registers, then to LDS.  A piece past K re-reads one of the row's first
  // 64 elements (multiplied by zero weights, or skipped).
  constexpr int NA = F::kACopies, kPer = F::kARow / 16;
  // piece i is row (kBlock / kPer) i + tid / kPer: the swizzle is the same for every i
  const uint32_t aslot = (uint32_t)((tid / kPer) * F::kARow + 16 * ((tid % kPer) ^ tile_fa<FMT>(tid / kPer)));
  auto load_a = [&](int kb, u32x4 (&t)[NA]) {
    uint32_t off = (uint32_t)(kb < nsteps ? kb : nsteps - 1) * (uint32_t)F::kARow + 16u * (uint32_t)(tid % kPer);
    if (KS == 128) off = off < 2u * (uint32_t)K ? off : off & 127u;
#pragma unroll
    for (int i = 0; i < NA; ++i) t[i] = *(const u32x4*)(arow[i] + off);
  };
  auto store_a = [&](const u32x4 (&t)[NA], char* st) {
#pragma unroll
    for (int i = 0; i < NA; ++i) *(u32x4*)(st + aslot + i * (kBlock / kPer) * F::kARow) = t[i];
  };

  // ---- weights and scales
  const uint32_t rb = FMT == FTM_FMT_BF16 ? 2u * (uint32_t)K : FMT == FTM_FMT_MXFP4 ? (uint32_t)K / 2 : (uint32_t)K;
  const Rsrc wres = make_rsrc(W.w, GQ ? (uint32_t)(K / 8) * (uint32_t)N * 4u : rb * (uint32_t)N);
  const uint32_t sesz = W.s_dt == FTM_DT_F32 ? 4u : 2u;
  const int ngrp = F::kPost ? (K + W.group - 1) / W.group : 0;
  const Rsrc sres = make_rsrc(W.s, FMT == FTM_FMT_FP8_BLOCK ? (uint32_t)(((N + W.group - 1) / W.group) * ngrp) * sesz
                              : FMT == FTM_FMT_MXFP4        ? (uint32_t)N * (uint32_t)(K / 32)
                              : F::kPost                    ? (uint32_t)(N * ngrp) * sesz
                                                            : 0u);
  uint32_t woff[4], soff[4];
#pragma unroll
  for (int nj = 0; nj < 4; ++nj) {
    const int row = tile_row<FMT>(base, nj, m);
    soff[nj] = kOOB;
    if constexpr (GQ) {  // nj 0 and 2: the halves
      woff[nj] = row < N ? ((uint32_t)g * (uint32_t)N + (uint32_t)row) * 4u : kOOB;
      soff[nj] = row < N ? 2u * (uint32_t)row : kOOB;
    } else {
      woff[nj] = row < N ? (uint32_t)row * rb + 16u * (uint32_t)g : kOOB;
      if constexpr (FMT == FTM_FMT_FP8_BLOCK) soff[nj] = sesz * (uint32_t)((base[nj >> 1] / W.group) * ngrp);
      if constexpr (FMT == FTM_FMT_INT8_PACKED) soff[nj] = row < N ? sesz * (uint32_t)(row * ngrp) : kOOB;
      if constexpr (FMT == FTM_FMT_MXFP4)
        soff[nj] = row < N ? (uint32_t)row * (uint32_t)(K / 32) + (uint32_t)g : kOOB;
    }
  }
  // piece i of step kb's weights: 64 bytes of each row (GPTQ: half i)
  auto load_w = [&](int kb, int i, TileW<FMT>& t) {
    if constexpr (GQ) {
      const uint32_t o = woff[2 * i] + (kb < nsteps ? (uint32_t)kb * 64u * (uint32_t)N : kOOB);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        t.w[i][q] = __builtin_amdgcn_raw_buffer_load_b64(wres, o, 16u * (uint32_t)N * (uint32_t)q, 0);
    } else {
      constexpr uint32_t kStep = FMT == FTM_FMT_MXFP4 ? 64u : 128u;
      const int k0 = FMT == FTM_FMT_MXFP4 ? kb * KS + 32 * g : FMT == FTM_FMT_BF16 ? kb * KS + 32 * i : kb * KS + 64 * i;
      const uint32_t ko = k0 < K ? (uint32_t)kb * kStep + 64u * (uint32_t)i : kOOB;
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) t.w[nj][i] = bload16(wres, woff[nj] + ko);
    }
  };
  // byte offset of the scale of half-step i of step kb within its row
  auto sgrp = [&](int kb, int i) { return sesz * (uint32_t)((kb * 128 + 64 * i) / W.group); };
  auto load_s = [&](int kb, TileW<FMT>& t) {
    if constexpr (GQ) {
      const uint32_t go = kb < nsteps ? 2u * (uint32_t)(kb * 128 / W.group) * (uint32_t)N : kOOB;
#pragma unroll
      for (int h = 0; h < 2; ++h) t.s[h] = bload4(sres, soff[2 * h] + go);
    } else if constexpr (FMT == FTM_FMT_MXFP4) {
      const uint32_t go = kb * KS + 32 * g < K ? 4u * (uint32_t)kb : kOOB;
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) t.s[0][nj] = bload1(sres, soff[nj] + go);
    } else if constexpr (POST) {
#pragma unroll
      for (int i = 0; i < (MODE == kScale64 ? 2 : 1); ++i) {
        const uint32_t go = kb * KS + 64 * i < K ? sgrp(kb, i) : kOOB;
#pragma unroll
        for (int nj = 0; nj < 4; ++nj)
          if (FMT == FTM_FMT_INT8_PACKED || (nj & 1) == 0) t.s[i][nj] = bload4(sres, (soff[nj] + go) & ~3u);
      }
    }
  };

  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  auto afrag = [&](const char* st, int blk, int piece) {
    const int r = 16 * blk + m;
    return *(const u32x4*)(st + r * F::kARow + 16 * (piece ^ tile_fa<FMT>(r)));
  };

  // One K step: its weights in cur, the next step's loads into nxt and ra
  // first, so that they are in flight during the MFMAs.
  auto step = [&](int kb, const TileW<FMT>& cur, TileW<FMT>& nxt) {
    // stage kb is in LDS for every wave, and every wave is done with kb - 1
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    u32x4 ra[NA];
    load_a(kb + 1, ra);
    load_s(kb + 1, nxt);
#pragma unroll
    for (int i = 0; i < F::kNL; ++i) load_w(kb + 1, i, nxt);
    __builtin_amdgcn_sched_barrier(0);
    const char* st = lds + (kb & 1) * F::kStage;
    f32x4 p[MI][4], x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) p[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
    f32x4(&d)[MI][4] = POST ? p : acc;
    // one 32-wide sub-step: B operands bq against activation piece `piece` of every row
    auto mma = [&](int piece, const u32x4(&bq)[4]) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const u32x4 af = afrag(st, mi, piece);
#pragma unroll
        for (int nj = 0; nj < 4; ++nj) d[mi][nj] = mfma_bf16(af, bq[nj], d[mi][nj]);
      }
      if constexpr (GQ) x = mfma_bf16(afrag(st, wave, piece), ones, x);
    };
    // the partial sums of the step (kScale64: of half-step i) join acc
    auto fold = [&](int i, const auto& t) {
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) {
        const int sj = FMT == FTM_FMT_INT8_PACKED ? nj : nj & 2;
        const float s = decode_scalar_word(t.s[i][sj], (soff[sj] + sgrp(kb, i)) / sesz, W.s_dt);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
          acc[mi][nj] += p[mi][nj] * s;
          p[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
      }
    };
    if constexpr (GQ) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u32x4 bq[4];
#pragma unroll
        for (int nj = 0; nj < 4; ++nj)
          bq[nj] = gptq_word_natural((nj & 1) ? cur.w[nj >> 1][q].y : cur.w[nj >> 1][q].x);
        mma(4 * q + g, bq);
      }
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) {
        const float s = half_word(cur.s[nj >> 1], nj & 1, W.s_dt);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[mi][nj] += p[mi][nj] * s;
      }
      if (m == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) Xs[(16 * wave + 4 * g + r) * (nsteps + 1) + kb] = x[r];
      }
    } else if constexpr (FMT == FTM_FMT_MXFP4) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u32x4 bq[4];
#pragma unroll
        for (int nj = 0; nj < 4; ++nj) {
          const u32x4 r = cur.w[nj][0];
          bq[nj] = fp4x8_to_bf16(q == 0 ? r.x : q == 1 ? r.y : q == 2 ? r.z : r.w, e8m0_to_f32(cur.s[0][nj]));
        }
        mma(4 * g + q, bq);
      }
    } else if constexpr (FMT == FTM_FMT_BF16) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        u32x4 bq[4];
#pragma unroll
        for (int nj = 0; nj < 4; ++nj) bq[nj] = cur.w[nj][i];
        mma(4 * i + g, bq);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (i == 0 || kb * 128 + 64 < K) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            u32x4 bq[4];
#pragma unroll
            for (int nj = 0; nj < 4; ++nj) {
              const u32x4 r = cur.w[nj][i];
              bq[nj] = FMT == FTM_FMT_FP8_BLOCK ? fp8x8_to_bf16(h ? r.z : r.x, h ? r.w : r.y)
                                                : i8x8_to_bf16(h ? r.z : r.x, h ? r.w : r.y);
            }
            mma(8 * i + 2 * g + h, bq);
          }
          if (MODE == kScale64) fold(i, cur);
        }
      }
      if (MODE == kScale128) fold(0, cur);
    }
    __builtin_amdgcn_sched_barrier(0);
    store_a(ra, lds + ((kb + 1) & 1) * F::kStage);
  };

  TileW<FMT> w0, w1;
  {
    u32x4 ra[NA];
    load_a(0, ra);
    load_s(0, w0);
#pragma unroll
    for (int i = 0; i < F::kNL; ++i) load_w(0, i, w0);
    store_a(ra, lds);
  }
  for (int kb = 0; kb < nsteps; kb += 2) {
    step(kb, w0, w1);
    if (kb + 1 < nsteps) step(kb + 1, w1, w0);
  }
  if constexpr (MODE == kScaleOne) {
#pragma unroll
    for (int nj = 0; nj < 4; ++nj) {
      const float s = decode_scalar_word(bload4(sres, soff[nj] & ~3u), soff[nj] / sesz, W.s_dt);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) acc[mi][nj] *= s;
    }
  }
  // every wave is done with the stages and (GPTQ) has written its row sums
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if constexpr (GQ) {
    // acc -= X . (s (z + 1)): groups 4 t + g of row m / column (nj, m)
    const Rsrc zres = make_rsrc(W.z, (uint32_t)ngrp * (uint32_t)(N / 8) * 4u);
    for (int t = 0; t < nsteps; t += 4) {
      const int kb = t + g;
      const bool in = kb < nsteps;
      const uint32_t grp = (uint32_t)(kb * 128 / W.group);
      float c[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool ok = in && soff[2 * h] != kOOB;
        const uint32_t row = soff[2 * h] >> 1;
        const uint32_t sw = bload4(sres, ok ? 2u * grp * (uint32_t)N + soff[2 * h] : kOOB);
        const uint32_t zw = bload4(zres, ok ? 4u * (grp * (uint32_t)(N / 8) + row / 8u) : kOOB) >> (4u * (row & 7u));
        c[2 * h] = -half_word(sw, 0, W.s_dt) * (float)((zw & 15u) + 1u);
        c[2 * h + 1] = -half_word(sw, 1, W.s_dt) * (float)(((zw >> 4) & 15u) + 1u);
      }
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const float xa = in ? Xs[(16 * mi + m) * (nsteps + 1) + kb] : 0.0f;
#pragma unroll
        for (int nj = 0; nj < 4; ++nj) acc[mi][nj] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa, c[nj], acc[mi][nj], 0, 0, 0);
      }
    }
  }
}

// h = act(gate) * up for one 16 x 16 block pair, with the activation fixed at
// compile time (the selection stands outside the element loops).
template <int ACT>
__device__ __forceinline__ float tile_act(float g, float u, const LayerArgs& a) {
  return act_fn(ACT, g, u, a.L.swiglu_alpha, a.L.swiglu_limit);
}

template <int FMT, int MODE, int MI, bool STB>
__device__ __forceinline__ void tile_run(const LayerArgs& a, const ProjSlot& W, int Iu, int n0, int rows, char* lds,
                                         const int* s_pair, const float* s_w, float* s_bias, float* Xs) {
  using F = TileFmt<FMT>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, m = lane & 15;
  const int KP = a.KP, H = a.L.hidden;
  const size_t arb = STB ? (size_t)a.Imax * 2u : (size_t)H * 2u;
  const char* abase = STB ? a.hbuf : (const char*)a.x;
  const char* arow[F::kACopies];
#pragma unroll
  for (int i = 0; i < F::kACopies; ++i) {
    constexpr int kPer = F::kARow / 16;
    const int r = (kBlock / kPer) * i + tid / kPer;
    const int pr = s_pair[r < rows ? r : 0];  // padding rows repeat the first (their outputs are dropped)
    arow[i] = abase + (size_t)(STB ? pr : pr / KP) * arb;
  }
  const int base[2] = {n0 + (STB ? 64 : 32) * wave, STB ? n0 + 64 * wave + 32 : Iu + n0 + 32 * wave};
  // the tile's biases as fp32 in LDS (read in the epilogue)
  const int brow = STB || tid < kTN / 2 ? n0 + tid : Iu + n0 + tid - kTN / 2;
  s_bias[tid] = W.bias != nullptr && brow < W.N ? load_scalar(W.bias, brow, W.bias_dt) : 0.0f;
  f32x4 acc[MI][4];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int nj = 0; nj < 4; ++nj) acc[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
  tile_kloop<FMT, MODE, MI>(W, base, arow, lds, Xs, acc);

  const int lb[2] = {(STB ? 64 : 32) * wave, STB ? 64 * wave + 32 : kTN / 2 + 32 * wave};
  float bf[4];
#pragma unroll
  for (int nj = 0; nj < 4; ++nj) bf[nj] = s_bias[tile_row<FMT>(lb, nj, m)];
  if constexpr (STB) {
    // router-weighted fp32 rows into the slot buffer
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * mi + 4 * g + r;
        if (row < rows) {
          float* y = a.ybuf + (size_t)s_pair[row] * H;
          const float w = s_w[row];
#pragma unroll
          for (int nj = 0; nj < 4; ++nj) {
            const int col = tile_row<FMT>(base, nj, m);
            if (col < W.N) y[col] = (acc[mi][nj][r] + bf[nj]) * w;
          }
        }
      }
  } else {
    // h rows staged in the ring, then copied out in 16-byte pieces
    auto stage = [&](auto act) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const float h = tile_act<decltype(act)::value>(acc[mi][j][r] + bf[j], acc[mi][2 + j][r] + bf[2 + j], a);
            const int ch = tile_row<FMT>(base, j, m) - n0;
            *(uint16_t*)(lds + (16 * mi + 4 * g + r) * kTHPitch + 2 * ch) = f32_to_bf16(h);
          }
    };
    switch (a.L.act) {
      case FTM_ACT_SILU: stage(std::integral_constant<int, FTM_ACT_SILU>{}); break;
      case FTM_ACT_GELU: stage(std::integral_constant<int, FTM_ACT_GELU>{}); break;
      case FTM_ACT_RELU: stage(std::integral_constant<int, FTM_ACT_RELU>{}); break;
      default: stage(std::integral_constant<int, FTM_ACT_SWIGLU_OAI>{}); break;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    for (int q = tid; q < 16 * MI * 16; q += kBlock) {
      const int row = q >> 4, pc = q & 15;
      if (row < rows && n0 + 8 * pc < Iu)
        *(u32x4*)(a.hbuf + ((size_t)s_pair[row] * a.Imax + n0 + 8 * pc) * 2u) =
            *(const u32x4*)(lds + row * kTHPitch + 16 * pc);
    }
  }
}

// One item: a tile of 64 rows x 128 channels (stage A) or 256 columns (B).
// Items run expert by expert (ascending compact index), within an expert over
// its M tiles first: the workgroups in flight on an XCD then share an
// expert's weight columns and its activation rows in that XCD's L2.
template <int FMT, int MODE, bool STB>
__device__ __forceinline__ void tile_rows(const LayerArgs& a, const ProjSlot& W, int Iu, int n0, int rows, char* lds,
                                          const int* s_pair, const float* s_w, float* s_bias, float* Xs) {
  if (rows > 32) tile_run<FMT, MODE, 4, STB>(a, W, Iu, n0, rows, lds, s_pair, s_w, s_bias, Xs);
  else tile_run<FMT, MODE, 2, STB>(a, W, Iu, n0, rows, lds, s_pair, s_w, s_bias, Xs);
}

extern __shared__ __attribute__((aligned(16))) char ftm_tile_lds[];

// Dynamic LDS: activation stages, the tile's pairs, router weights and biases, GPTQ row sums.
template <int FMT>
constexpr int tile_ring(bool shared) {
  return shared && TileFmt<FTM_FMT_BF16>::kRing > TileFmt<FMT>::kRing ? TileFmt<FTM_FMT_BF16>::kRing
                                                                      : TileFmt<FMT>::kRing;
}

template <int FMT, int MODE, bool STB>
__global__ __launch_bounds__(kBlock, 2) void k_tile(const LayerArgs a, int ring) {
  char* lds = ftm_tile_lds;
  int* s_pair = (int*)(lds + ring);
  float* s_w = (float*)(s_pair + kTM);
  float* s_bias = s_w + kTM;
  float* Xs = s_bias + kTN;
  const int tid = threadIdx.x, lane = tid & 63;
  const int item = xcd_item(blockIdx.x, gridDim.x);
  const int I = a.L.inter, Is = a.L.shared_inter, H = a.L.hidden;
  const int ntn = STB ? (H + kTN - 1) / kTN : (I + kTN / 2 - 1) / (kTN / 2);
  // lane l owns compact experts 8 l .. 8 l + 7 (E <= 512)
  const Rsrc cres = make_rsrc(a.ucnt, (uint32_t)((a.L.num_experts + 8) / 8) * 32u);
  const u32x4 c0 = bload16(cres, 32u * (uint32_t)lane), c1 = bload16(cres, 32u * (uint32_t)lane + 16u);
  const int nRouted = a.ctrl[kCtrlNRouted];
  const uint32_t cw[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  int cnt8[8], lsum = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    cnt8[j] = 8 * lane + j < nRouted ? (int)cw[j] : 0;
    lsum += (cnt8[j] + kTM - 1) / kTM;
  }
  int incl = lsum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off);
    if (lane >= off) incl += o;
  }
  const int routed = __builtin_amdgcn_readlane(incl, 63) * ntn;
  const int32_t* list = nullptr;
  int m0, cnt, n0, slot = 0;
  bool shared = false;
  if (item < routed) {
    int b = (incl - lsum) * ntn, fu = -1, fl = 0, fc = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int v = (cnt8[j] + kTM - 1) / kTM * ntn;
      if (fu < 0 && item >= b && item < b + v) {
        fu = 8 * lane + j;
        fl = item - b;
        fc = cnt8[j];
      }
      b += v;
    }
    const int src = (int)__builtin_ctzll(__ballot(fu >= 0));
    const int u = __builtin_amdgcn_readlane(fu, src), loc = __builtin_amdgcn_readlane(fl, src);
    cnt = __builtin_amdgcn_readlane(fc, src);
    const int mt = (cnt + kTM - 1) / kTM;
    m0 = (loc % mt) * kTM;
    n0 = loc / mt;
    const int e = __builtin_amdgcn_readfirstlane(a.uniq[u]);
    list = a.lists + (size_t)e * a.T;
    slot = __builtin_amdgcn_readfirstlane(a.L.slot_of_expert ? a.L.slot_of_expert[e] : e);
  } else {
    const int nts = STB ? ntn : (Is + kTN / 2 - 1) / (kTN / 2), mts = (a.T + kTM - 1) / kTM;
    const int loc = item - routed;
    if (Is == 0 || loc >= nts * mts) return;
    m0 = (loc % mts) * kTM;
    n0 = loc / mts;
    cnt = a.T;
    shared = true;
  }
  n0 *= STB ? kTN : kTN / 2;
  const int rows = cnt - m0 < kTM ? cnt - m0 : kTM;
  if (tid < kTM) {
    const int p = tid < rows ? (list != nullptr ? list[m0 + tid] : (m0 + tid) * a.KP + a.L.topk) : 0;
    s_pair[tid] = p;
    if (STB) s_w[tid] = tid < rows ? a.wts[p] : 0.0f;
  }
  __syncthreads();
  if (shared) {
    const ProjSlot W = STB ? shared_view(a.L.shared_w2, H, Is) : shared_view(a.L.shared_w13, 2 * Is, H);
    tile_rows<FTM_FMT_BF16, kScaleNone, STB>(a, W, Is, n0, rows, lds, s_pair, s_w, s_bias, Xs);
    return;
  }
  const ftm_proj& PW = STB ? a.L.w2 : a.L.w13;
  if (slot < 0 || slot >= PW.num_slots) {
    if (STB) {  // non-resident expert: its rows contribute zeros
      for (int idx = tid; idx < kTM * kTN; idx += kBlock) {
        const int row = idx / kTN, col = n0 + idx % kTN;
        if (row < rows && col < H) a.ybuf[(size_t)s_pair[row] * H + col] = 0.0f;
      }
    }
    if (tid == 0) atomicOr(&a.ctrl[kCtrlError], 1);
    return;
  }
  tile_rows<FMT, MODE, STB>(a, proj_slot(PW, slot), I, n0, rows, lds, s_pair, s_w, s_bias, Xs);
}

// ---------------------------------------------------------------- launch
// Dynamic LDS of one projection's tiles.
template <int FMT>
static size_t tile_lds(const ftm_moe_layer& L, bool stb) {
  const int K = stb ? L.inter : L.hidden;
  const size_t x = FMT == FTM_FMT_GPTQ_INT4 ? (size_t)kTM * (size_t)((K + 127) / 128 + 1) * 4u : 0u;
  return (size_t)tile_ring<FMT>(L.shared_inter > 0) + (size_t)kTM * 8u + (size_t)kTN * 4u + x;
}

// GPTQ layers the tiles take: 128-wide groups (or multiples), 16-bit scales,
// whole K steps, and row sums that fit the LDS beside the ring.
bool tile_gptq_ok(const ftm_moe_layer& L) {
  if (L.w13.fmt != FTM_FMT_GPTQ_INT4 || L.act_dtype != FTM_DT_BF16) return false;
  if (L.w13.group % 128 != 0 || L.w2.group % 128 != 0 || L.hidden % 128 != 0 || L.inter % 128 != 0) return false;
  if (L.w13.s_dtype == FTM_DT_F32 || L.w2.s_dtype == FTM_DT_F32) return false;
  return tile_lds<FTM_FMT_GPTQ_INT4>(L, false) <= 160u * 1024u && tile_lds<FTM_FMT_GPTQ_INT4>(L, true) <= 160u * 1024u;
}

template <int FMT, int MODE, bool STB>
static void launch_tile_t(const LayerArgs& a, hipStream_t st) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_tile<FMT, MODE, STB>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr = true;
  }
  const ftm_moe_layer& L = a.L;
  const long pairs = (long)a.T * L.topk;
  const long maxU = L.num_experts < pairs ? L.num_experts : pairs;
  const int I = L.inter, Is = L.shared_inter, H = L.hidden;
  const long ntn = STB ? (H + kTN - 1) / kTN : (I + kTN / 2 - 1) / (kTN / 2);
  const long nts = Is == 0 ? 0 : STB ? ntn : (Is + kTN / 2 - 1) / (kTN / 2);
  const long items = (pairs / kTM + maxU) * ntn + (long)((a.T + kTM - 1) / kTM) * nts;
  hipLaunchKernelGGL((k_tile<FMT, MODE, STB>), dim3((unsigned)items), dim3(kBlock), tile_lds<FMT>(L, STB), st, a,
                     tile_ring<FMT>(Is > 0));
}

void launch_tile_gptq(const LayerArgs& a, hipStream_t st, int which) {
  if (which & 1) launch_tile_t<FTM_FMT_GPTQ_INT4, kScale128, false>(a, st);
  if (which & 2) launch_tile_t<FTM_FMT_GPTQ_INT4, kScale128, true>(a, st);
}

}  // namespace ftm
