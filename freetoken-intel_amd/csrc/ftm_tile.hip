// ftm_tile.hip -- the MoE expert stages above the token crossover as grouped
// MFMA tiles whose weights go straight from memory into registers: k_tile
// (bf16 MFMAs: GPTQ, INT8 and bf16 experts, FP8 ones of fewer than 16 tokens)
// and, further down, k_gemm_mx (scaled MFMAs: MXFP4 and FP8 experts).
//
// A tile is 64 pairs (rows) of one expert x 256 weight rows: four waves, each
// 64 rows x 64 weight rows over the whole K (stage A: 32 gate + 32 up
// channels of w13, so the activation needs no exchange; stage B: 64 output
// columns of w2).  A wave owns its weight rows, so the weights are loaded once
// per tile by buffer loads into VGPRs, one K step ahead of their use (in the
// loops whose second step of a pair is behind a branch, bf16, INT8 with one
// scale and MXFP4, in every second step only: in the other the compiler waits
// for a step's weights before it requests the next); only the activations,
// which all four waves read, go through LDS: a three-stage ring filled by
// direct global->LDS copies two K steps ahead.  One barrier per K
// step of 128 (64 for bf16 weights), two workgroups per CU (MXFP4: three).
// Quantisation-group scales multiply the fp32 partial sums of each group, as
// in the GEMV path.
//
// Bound by the bytes a CU keeps in flight where an expert has about a tile of
// rows, by LDS reads and MFMA issue where it has many.  Measured on MI355X, us
// per layer, LDS-ring tiles (GPTQ: GEMV stages) before / these: 256 FP8
// experts of 512 + shared at 512 / 2048 tokens 352 / 549 and 223 / 355; 32
// MXFP4 experts of 2880 at 256 / 4096 340 / 1287 and 189 / 972; 128 GPTQ
// experts of 768 at 1000 / 4096 466 / 1613 and 213 / 550; 64 INT8 experts of
// 1024 at 256 / 2048 237 / 523 and 127 / 259; 128 bf16 experts of 768 at 333
// 334 and 284.
//
// GPTQ's activations stay the bf16 values that the GEMV stages read (a
// two-term e4m3 split of them takes the same time, 209 us at 1000 tokens, but
// drops what lies 2^13 below a 32-block's largest: with one channel of 128 at
// 1e4 and weights that do not read it the others' result is off by 0.3).  The
// zero points leave after the loop, acc -= X . (s (z + 1)) on fp32 MFMAs, X the
// row sums of each step, which a wave takes for its share of the rows by MFMAs
// against ones and keeps in LDS.
#include <type_traits>

#include "ftm_layer.h"

namespace ftm {

constexpr int kTM = 64;        // rows (pairs) per tile
constexpr int kTN = 256;       // weight rows per tile
constexpr int kTHPitch = 128 * 2 + 16;  // bytes of a staged h row (stage A's epilogue, 128 channels)
constexpr int kTStages = 3;    // activation stages in LDS

// How group scales enter: none (bf16), one group over K (applied after the
// loop), one per K step of 128 (GPTQ: with its zero points after the loop).
enum { kScaleNone = 0, kScaleOne = 1, kScale128 = 2 };

template <int FMT>
struct TileFmt {
  static constexpr int kKS = FMT == FTM_FMT_BF16 ? 64 : 128;  // K per step
  static constexpr int kSub = kKS / 32;                       // MFMA sub-steps
  static constexpr int kARow = 2 * kKS;                       // activation bytes per row and step
  static constexpr int kStage = kTM * kARow;
  static constexpr int kACopies = kStage / 1024 / 4;          // 1 KiB copies per wave and step
  static constexpr int kRing = kTStages * kStage > kTM * kTHPitch ? kTStages * kStage : kTM * kTHPitch;
};

// Activation slot swizzle: slot s of row r holds 16-byte piece s ^ tile_fa(r)
// of its step, so that the 16 rows of one operand read hit distinct banks.
template <int FMT>
__device__ __forceinline__ int tile_fa(int r) {
  return TileFmt<FMT>::kKS == 128 ? (r & 15) : ((r >> 1) & 7);
}

// Tile row (weight row of the projection) of MFMA column block nj, lane
// column m, of a wave whose first rows are base[0] (nj 0, 1) and base[1] (2,
// 3): two neighbouring rows a lane (GPTQ: one 8-byte load of two columns), so
// that a lane's results are neighbours too.
__device__ __forceinline__ int tile_row(const int (&base)[2], int nj, int m) {
  return base[nj >> 1] + 2 * m + (nj & 1);
}

// 16-bit scale word `hi` (0 / 1) of a pair -> its value (branch-free).
__device__ __forceinline__ float half_word(uint32_t w, int hi, int dt) {
  const uint32_t h = hi ? w >> 16 : w & 0xffffu;
  const float f = f16_to_f32((uint16_t)h), b = __uint_as_float(h << 16);
  return dt == FTM_DT_F16 ? f : b;
}

// One step's packed weights of a wave and the raw words of its scales.
template <int FMT>
struct TileW {
  u32x4 w[4][2];
  uint32_t s[4];
};
template <>
struct TileW<FTM_FMT_GPTQ_INT4> {
  u32x2 w[2][4];  // [half][q]: the words of columns 2m, 2m + 1 at K 32 q + 8 g
  uint32_t s[2];  // [half]: both columns' 16-bit scales
};

// Eight nibbles (low first) -> the bf16 values 0..15 in natural order, 9 VALU:
// a nibble, zero-extended to a byte, is the e4m3 code of q 2^-9 (0..15 are the
// subnormals and the first binade), which the scaled convert makes q exactly.
__device__ __forceinline__ u32x4 gptq_word_natural(uint32_t w) {
  const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;  // q0 q2 q4 q6 / q1 q3 q5 q7
  const uint32_t a = __builtin_amdgcn_perm(hi, lo, 0x05010400u);     // q0 q1 q2 q3
  const uint32_t b = __builtin_amdgcn_perm(hi, lo, 0x07030602u);     // q4 q5 q6 q7
  auto pair = [](uint32_t v, auto hi_half) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8((int)v, 512.0f, hi_half()));
  };
  using L = std::integral_constant<bool, false>;
  using H = std::integral_constant<bool, true>;
  return (u32x4){pair(a, L{}), pair(a, H{}), pair(b, L{}), pair(b, H{})};
}

// The bf16 operand of column block nj in sub-step q.
template <int FMT>
__device__ __forceinline__ u32x4 tile_weights(const TileW<FMT>& t, int nj, int q) {
  if constexpr (FMT == FTM_FMT_GPTQ_INT4) {
    return gptq_word_natural((nj & 1) ? t.w[nj >> 1][q].y : t.w[nj >> 1][q].x);
  } else if constexpr (FMT == FTM_FMT_INT8_PACKED) {
    const u32x4 r = t.w[nj][q >> 1];
    return i8x8_to_bf16(q & 1 ? r.z : r.x, q & 1 ? r.w : r.y);
  } else if constexpr (FMT == FTM_FMT_FP8_BLOCK) {
    const u32x4 r = t.w[nj][q >> 1];
    return fp8x8_to_bf16(q & 1 ? r.z : r.x, q & 1 ? r.w : r.y);
  } else {
    return t.w[nj][q];
  }
}

// Activation sources of a wave's copies: byte offsets into the buffer (BIG:
// addresses).
template <int N>
struct TileSrc {
  uint64_t p[N];
};

// The K loop of the bf16 tiles: acc += A (16 MI rows) . W^T over the whole K.
// Every step issues the same loads (past the last step through clamped or
// out-of-range offsets), so the counted waits are exact.
// bf16 weights, MFMA sub-step q, lane group g: stage A takes activation piece
// 2 g + q of the step, stage B piece 4 q + g.  Those are the sums, in their
// order, of the LDS tiles (k_gemm_a_ring, k_gemm_b), so a token's output does
// not depend on which of the two the batch's size chose.
template <int FMT, int MODE, int MI, bool STB, bool BIG>
__device__ __forceinline__ void tile_kloop(const ProjSlot& W, const int (&base)[2], const char* abase, uint32_t abytes,
                                           const TileSrc<TileFmt<FMT>::kACopies>& src, char* lds, float* Xs,
                                           f32x4 (&acc)[MI][4]) {
  using F = TileFmt<FMT>;
  constexpr bool I8 = FMT == FTM_FMT_INT8_PACKED, GQ = FMT == FTM_FMT_GPTQ_INT4, F8 = FMT == FTM_FMT_FP8_BLOCK;
  constexpr bool BYTES = I8 || F8;  // a lane's 16 bytes are 16 K of its weight row
  constexpr bool ONESET = MODE == kScale128;  // one register set of weights (below)
  constexpr bool PAIR = FMT == FTM_FMT_BF16 && !STB;  // a lane's two pieces are neighbours
  constexpr int KS = F::kKS, NA = F::kACopies;
  constexpr int NW = 8 + (GQ || F8 ? 2 : MODE == kScale128 ? 4 : 0);  // weight and scale loads a step
  typedef __attribute__((address_space(1))) const void* GPtr;
  typedef __attribute__((address_space(3))) void* LPtr;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, m = lane & 15;
  const int K = W.K, N = W.N;
  const int nsteps = (K + KS - 1) / KS;

  // a last half step's copies read past the row (another row, or zeros past
  // the buffer): nothing uses them
  const Rsrc ares = make_rsrc(abase, abytes);
  auto issue_a = [&](int kb, int slot) {
    const uint32_t ko = (uint32_t)(kb < nsteps ? kb : nsteps - 1) * (uint32_t)F::kARow;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      char* dst = lds + slot * F::kStage + 1024 * (wave * NA + i);
      if constexpr (BIG) {
        // the piece's K must exist: an address has no range check
        const uint32_t pc = (uint32_t)((lane % (F::kARow / 16)) ^ tile_fa<FMT>((64 * (wave * NA + i) + lane) / (F::kARow / 16)));
        const uint32_t over = KS == 128 && ko + 16u * pc >= 2u * (uint32_t)K ? 128u : 0u;
        __builtin_amdgcn_global_load_lds((GPtr)(src.p[i] + ko - over), (LPtr)dst, 16, 0, 0);
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, (LPtr)dst, 16, (int)((uint32_t)src.p[i] + ko), 0, 0, 0);
      }
    }
  };

  using Wgt = TileW<FMT>;
  const uint32_t rb = BYTES ? (uint32_t)K : 2u * (uint32_t)K;
  const Rsrc wres = make_rsrc(W.w, GQ ? (uint32_t)(K / 8) * (uint32_t)N * 4u : rb * (uint32_t)N);
  const uint32_t sesz = W.s_dt == FTM_DT_F32 ? 4u : 2u;
  const int ngrp = I8 || GQ ? K / W.group : 0;
  const int nkb = K / 128;  // FP8: fp32 scales of 128 x 128 blocks
  const Rsrc sres = make_rsrc(W.s, F8 ? 4u * (uint32_t)((N + 127) / 128 * nkb) : (uint32_t)(N * ngrp) * sesz);
  uint32_t woff[4];  // GPTQ: [0] and [2], the halves' first columns in word row g
#pragma unroll
  for (int nj = 0; nj < 4; ++nj) {
    const int row = tile_row(base, nj, m);
    woff[nj] = row >= N ? kOOB
               : GQ     ? 4u * (uint32_t)(g * N + row)
                        : (uint32_t)row * rb + (PAIR ? 32u : 16u) * (uint32_t)g;
  }
  // index of the scale of block nj in step kb (rows past N: past the end)
  auto sidx = [&](int kb, int nj) {
    return (uint32_t)(tile_row(base, nj, m) * ngrp) + (MODE == kScaleOne ? 0u : (uint32_t)(kb * 128 / W.group));
  };
  auto load_s = [&](int kb, Wgt& t) {
    if constexpr (GQ) {
      const uint32_t go = kb < nsteps ? 2u * (uint32_t)(kb * 128 / W.group) * (uint32_t)N : kOOB;
#pragma unroll
      for (int h = 0; h < 2; ++h) t.s[h] = bload4(sres, 2u * (uint32_t)tile_row(base, 2 * h, m) + go);
    } else if constexpr (F8) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
        t.s[2 * h] = bload4(sres, 4u * (uint32_t)(base[h] / 128 * nkb + (kb < nsteps ? kb : 0)));
    } else if constexpr (MODE == kScale128) {
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) t.s[nj] = bload4(sres, (sesz * sidx(kb < nsteps ? kb : 0, nj)) & ~3u);
    }
  };
  auto load_w = [&](int kb, int i, Wgt& t) {  // 64 bytes of each row (bf16: K is whole steps); GPTQ: sub-step i
    if constexpr (GQ) {
      const uint32_t ko = kb < nsteps ? (uint32_t)kb * 64u * (uint32_t)N : kOOB;
#pragma unroll
      for (int h = 0; h < 2; ++h)
        t.w[h][i] = __builtin_amdgcn_raw_buffer_load_b64(wres, woff[2 * h] + ko, 16u * (uint32_t)N * (uint32_t)i, 0);
    } else {
      const uint32_t ko = kb * KS + (BYTES ? 64 : 32) * i < K ? (uint32_t)kb * 128u + (PAIR ? 16u : 64u) * (uint32_t)i : kOOB;
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) t.w[nj][i] = bload16(wres, woff[nj] + ko);
    }
  };
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // bf16 1.0

  // ONESET holds one register set beside its partial sums: cur and nxt are the
  // same, a piece is requested again as soon as its last MFMA has read it
  auto step = [&](int kb, int slot, Wgt& cur, Wgt& nxt) {
    // the copies of stage kb have landed (younger: this step's weights, the
    // copies of stage kb + 1), then every wave's have, and every wave is done
    // reading stage kb - 1
    wait_vm<NW + NA>();
    asm volatile("s_barrier" ::: "memory");
    issue_a(kb + 2, slot == 0 ? 2 : slot - 1);
    uint32_t sw[std::extent<decltype(cur.s)>::value];
#pragma unroll
    for (int j = 0; j < (int)std::extent<decltype(cur.s)>::value; ++j) sw[j] = cur.s[j];
    load_s(kb + 1, nxt);
    if constexpr (!ONESET) {
      load_w(kb + 1, 0, nxt);
      load_w(kb + 1, 1, nxt);
    }
    __builtin_amdgcn_sched_barrier(0);
    const char* st = lds + slot * F::kStage;
    f32x4 p[ONESET ? MI : 1][4];
#pragma unroll
    for (auto& r : p)
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) r[nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // sub-step q's operand of row block blk: activation piece 4 q + g (PAIR: 2 g
    // + q; BYTES: 8 (q / 2) + 2 g + q % 2, the 16 K of a lane's weight bytes)
    auto row = [&](int blk, int q) {
      const int piece = BYTES ? 8 * (q >> 1) + 2 * g + (q & 1) : PAIR ? 2 * g + q : 4 * q + g;
      const int r = 16 * blk + m;
      return *(const u32x4*)(st + r * F::kARow + 16 * (piece ^ tile_fa<FMT>(r)));
    };
    // all row blocks of a sub-step, read during the MFMAs of the one before
    auto frag = [&](int q, u32x4(&a)[MI]) {
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) a[mi] = row(mi, q);
    };
    auto mma = [&](int q, const u32x4(&a)[MI]) {
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) {
        const u32x4 b = tile_weights<FMT>(cur, nj, q);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
          acc[mi][nj] = mfma_bf16(a[mi], b, acc[mi][nj]);
        }
      }
    };
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    u32x4 a0[MI], a1[MI];
    if constexpr (!ONESET) frag(0, a0);
    if constexpr (ONESET) {
      // a sub-step's four operands, their registers requested again for the
      // next step as soon as all are decoded, against one row block after the
      // other, whose activations are read two blocks ahead (the accumulators
      // leave no room for a sub-step's at once); GPTQ: beside the products, the
      // sums of row block `wave` over the step (the same in every column), for
      // the zero points
      u32x4 a[3] = {row(0, 0), row(1, 0)};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u32x4 xa;
        if constexpr (GQ) xa = row(wave, q);
        u32x4 b[4];
#pragma unroll
        for (int nj = 0; nj < 4; ++nj) b[nj] = tile_weights<FMT>(cur, nj, q);
        if (GQ) load_w(kb + 1, q, nxt);
        else if (q & 1) load_w(kb + 1, q >> 1, nxt);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
          const int i = MI * q + mi;
          if (i + 2 < 4 * MI) a[(i + 2) % 3] = row((i + 2) % MI, (i + 2) / MI);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int nj = 0; nj < 4; ++nj) p[mi][nj] = mfma_bf16(a[i % 3], b[nj], p[mi][nj]);
        }
        if constexpr (GQ) x = mfma_bf16(xa, ones, x);
      }
    } else if constexpr (I8) {
      // INT8: K may end in a half step, whose zero bytes would decode to -128
      frag(1, a1);
      __builtin_amdgcn_sched_barrier(0);
      mma(0, a0);
      frag(2, a0);
      __builtin_amdgcn_sched_barrier(0);
      mma(1, a1);
      if (kb * 128 + 64 < K) {
        frag(3, a1);
        __builtin_amdgcn_sched_barrier(0);
        mma(2, a0);
        mma(3, a1);
      }
    } else {
      frag(1, a1);
      __builtin_amdgcn_sched_barrier(0);
      mma(0, a0);
      mma(1, a1);
    }
    if constexpr (ONESET) {
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) {
        float sv;
        if constexpr (GQ) sv = half_word(sw[nj >> 1], nj & 1, W.s_dt);
        else if constexpr (F8) sv = __uint_as_float(sw[nj & 2]);
        else sv = decode_scalar_word(sw[nj], sidx(kb, nj), W.s_dt);
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[mi][nj] += p[mi][nj] * sv;
      }
    }
    if constexpr (GQ) {
      // the sums exist before the branch: the compiler has sunk their MFMAs
      // (and the operand moves, which then skip the masked lanes) into it
      asm volatile("" : "+v"(x));
      if (m == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) Xs[(16 * wave + 4 * g + r) * (nsteps + 1) + kb] = x[r];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  Wgt w0, w1;
  issue_a(0, 0);
  load_s(0, w0);
#pragma unroll
  for (int i = 0; i < (GQ ? 4 : 2); ++i) load_w(0, i, w0);
  issue_a(1, 1);
  int slot = 0;
  auto next = [&] { slot = slot == 2 ? 0 : slot + 1; };
  if constexpr (ONESET) {
    for (int kb = 0; kb < nsteps; ++kb) {
      step(kb, slot, w0, w0);
      next();
    }
  } else {
    for (int kb = 0; kb < nsteps; kb += 2) {
      step(kb, slot, w0, w1);
      next();
      if (kb + 1 < nsteps) step(kb + 1, slot, w1, w0);
      next();
    }
  }
  if constexpr (MODE == kScaleOne) {
#pragma unroll
    for (int nj = 0; nj < 4; ++nj) {
      const uint32_t idx = sidx(0, nj);
      const float sv = decode_scalar_word(bload4(sres, (sesz * idx) & ~3u), idx, W.s_dt);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) acc[mi][nj] *= sv;
    }
  }
  // the copies past the last step have landed and every wave is done with the
  // ring and (GPTQ) has written its row sums
  wait_vm<0>();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if constexpr (GQ) {
    // the zero points: acc -= X . (s (z + 1)), steps t + g of row m / column (nj, m)
    const Rsrc zres = make_rsrc(W.z, (uint32_t)ngrp * (uint32_t)(N / 8) * 4u);
    for (int t = 0; t < nsteps; t += 4) {
      const int kb = t + g;
      const bool in = kb < nsteps;
      const uint32_t grp = (uint32_t)(kb * 128 / W.group);
      float c[4];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t row = (uint32_t)tile_row(base, 2 * h, m);
        const bool ok = in && row < (uint32_t)N;
        const uint32_t sw = bload4(sres, ok ? 2u * (grp * (uint32_t)N + row) : kOOB);
        const uint32_t zw = bload4(zres, ok ? 4u * (grp * (uint32_t)(N / 8) + row / 8u) : kOOB) >> (4u * (row & 7u));
        c[2 * h] = -half_word(sw, 0, W.s_dt) * (float)((zw & 15u) + 1u);
        c[2 * h + 1] = -half_word(sw, 1, W.s_dt) * (float)(((zw >> 4) & 15u) + 1u);
      }
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        const float xa = in ? Xs[(16 * mi + m) * (nsteps + 1) + kb] : 0.0f;
#pragma unroll
        for (int nj = 0; nj < 4; ++nj)
          acc[mi][nj] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa, c[nj], acc[mi][nj], 0, 0, 0);
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

template <class F>
__device__ __forceinline__ void tile_with_act(int act, F&& f) {
  switch (act) {
    case FTM_ACT_SILU: f(std::integral_constant<int, FTM_ACT_SILU>{}); break;
    case FTM_ACT_GELU: f(std::integral_constant<int, FTM_ACT_GELU>{}); break;
    case FTM_ACT_RELU: f(std::integral_constant<int, FTM_ACT_RELU>{}); break;
    default: f(std::integral_constant<int, FTM_ACT_SWIGLU_OAI>{}); break;
  }
}

// Stage A's epilogue: h = bf16(act(gate + b_g) * (up + b_u)) of the tile in
// LDS rows of kTHPitch bytes.
template <int FMT, int MI>
__device__ __forceinline__ void tile_stage_h(const LayerArgs& a, int n0, const float (&bf)[4], char* lds,
                                             const f32x4 (&acc)[MI][4]) {
  const int lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  auto stage = [&](auto act) {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float h0 = tile_act<decltype(act)::value>(acc[mi][0][r] + bf[0], acc[mi][2][r] + bf[2], a);
        const float h1 = tile_act<decltype(act)::value>(acc[mi][1][r] + bf[1], acc[mi][3][r] + bf[3], a);
        *(uint32_t*)(lds + (16 * mi + 4 * g + r) * kTHPitch + 64 * wave + 4 * m) = pack_bf16x2(h0, h1);
      }
  };
  tile_with_act(a.L.act, stage);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Stage B's epilogue: router-weighted fp32 rows into the slot buffer.
template <int FMT, int MI>
__device__ __forceinline__ void tile_store_y(const LayerArgs& a, const ProjSlot& W, const int (&base)[2],
                                             const float (&bf)[4], int rows, const int* s_pair, const float* s_w,
                                             const f32x4 (&acc)[MI][4]) {
  const int lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * mi + 4 * g + r;
      if (row < rows) {
        float* y = a.ybuf + (size_t)s_pair[row] * a.L.hidden;
        const float w = s_w[row];
#pragma unroll
        for (int nj = 0; nj < 4; nj += 2) {  // N is a multiple of 64: both columns of a lane or none
          const int col = tile_row(base, nj, m);
          if (col < W.N) *(f32x2*)(y + col) = (f32x2){(acc[mi][nj][r] + bf[nj]) * w, (acc[mi][nj + 1][r] + bf[nj + 1]) * w};
        }
      }
    }
}

template <int FMT, int MODE, int MI, bool STB, bool BIG>
__device__ __forceinline__ void tile_run(const LayerArgs& a, const ProjSlot& W, int Iu, int n0, int rows, char* lds,
                                         const int* s_pair, const float* s_w, const float* s_bias, float* Xs) {
  using F = TileFmt<FMT>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15;
  const int KP = a.KP, H = a.L.hidden;
  const uint32_t arb = 2u * (uint32_t)(STB ? a.Imax : H);
  const char* abase = STB ? a.hbuf : (const char*)a.x;
  TileSrc<F::kACopies> src;
#pragma unroll
  for (int i = 0; i < F::kACopies; ++i) {
    constexpr int kPer = F::kARow / 16;
    const int r = (64 * (wave * F::kACopies + i) + lane) / kPer;
    const int pr = s_pair[r < rows ? r : 0];  // padding rows repeat the first (their outputs are dropped)
    const uint64_t off = (uint64_t)(STB ? pr : pr / KP) * arb + 16 * ((lane % kPer) ^ tile_fa<FMT>(r));
    src.p[i] = BIG ? (uint64_t)(uintptr_t)abase + off : off;
  }
  const uint32_t abytes = BIG ? 0u : (uint32_t)(STB ? a.T * KP : a.T) * arb;
  const int base[2] = {n0 + (STB ? 64 : 32) * wave, STB ? n0 + 64 * wave + 32 : Iu + n0 + 32 * wave};
  f32x4 acc[MI][4];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int nj = 0; nj < 4; ++nj) acc[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
  tile_kloop<FMT, MODE, MI, STB, BIG>(W, base, abase, abytes, src, lds, Xs, acc);

  const int lb[2] = {(STB ? 64 : 32) * wave, STB ? 64 * wave + 32 : kTN / 2 + 32 * wave};
  float bf[4];
#pragma unroll
  for (int nj = 0; nj < 4; ++nj) bf[nj] = s_bias[tile_row(lb, nj, m)];
  if constexpr (STB) {
    tile_store_y<FMT, MI>(a, W, base, bf, rows, s_pair, s_w, acc);
  } else {
    tile_stage_h<FMT, MI>(a, n0, bf, lds, acc);
    for (int q = tid; q < 16 * MI * 16; q += kBlock) {
      const int row = q >> 4, pc = q & 15;
      if (row < rows && n0 + 8 * pc < Iu)
        *(u32x4*)(a.hbuf + ((size_t)s_pair[row] * a.Imax + n0 + 8 * pc) * 2u) =
            *(const u32x4*)(lds + row * kTHPitch + 16 * pc);
    }
  }
}

// The tile on the instantiation for its number of 16-row blocks.
template <int FMT, int MODE, bool STB, bool BIG>
__device__ __forceinline__ void tile_rows(const LayerArgs& a, const ProjSlot& W, int Iu, int n0, int rows, char* lds,
                                          const int* s_pair, const float* s_w, const float* s_bias,
                                          float* Xs = nullptr) {
  if (rows > 32) tile_run<FMT, MODE, 4, STB, BIG>(a, W, Iu, n0, rows, lds, s_pair, s_w, s_bias, Xs);
  else tile_run<FMT, MODE, 2, STB, BIG>(a, W, Iu, n0, rows, lds, s_pair, s_w, s_bias, Xs);
}

extern __shared__ __attribute__((aligned(16))) char ftm_tile_lds[];

// One item: a tile of 64 rows x 128 channels (stage A) or 256 columns (B).
// Items run expert by expert (ascending compact index), within an expert over
// its M tiles first: the workgroups in flight on an XCD then share an
// expert's weight columns and its activation rows in that XCD's L2.  The
// shared expert's items come first.  rows <= 0: no item.
struct TileItem {
  const int32_t* list;  // the expert's pairs (null: the shared expert)
  int m0, rows, n0, slot;
  bool shared;
};

template <bool STB>
__device__ __forceinline__ TileItem tile_item(const LayerArgs& a) {
  const int lane = threadIdx.x & 63;
  const int I = a.L.inter, Is = a.L.shared_inter, H = a.L.hidden;
  constexpr int tn = STB ? kTN : kTN / 2;
  const int ntn = ((STB ? H : I) + tn - 1) / tn;
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
  const int nts = Is == 0 ? 0 : ((STB ? H : Is) + tn - 1) / tn, mts = (a.T + kTM - 1) / kTM;
  // the grid is an upper bound: both kinds are spread over the XCDs by the
  // items there are (spread over the grid, the last XCDs would find none)
  const int bid = (int)blockIdx.x - nts * mts;
  TileItem t = {nullptr, 0, 0, 0, 0, false};
  if (bid >= routed) return t;
  if (bid >= 0) {
    const int item = xcd_item(bid, routed);
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
    const int cnt = __builtin_amdgcn_readlane(fc, src);
    const int mt = (cnt + kTM - 1) / kTM;
    t.n0 = loc / mt;
    t.m0 = (loc - t.n0 * mt) * kTM;
    t.rows = cnt - t.m0;
    const int e = __builtin_amdgcn_readfirstlane(a.uniq[u]);
    t.list = a.lists + (size_t)e * a.T;
    t.slot = __builtin_amdgcn_readfirstlane(a.L.slot_of_expert ? a.L.slot_of_expert[e] : e);
  } else {
    const int loc = xcd_item(blockIdx.x, nts * mts);
    t.n0 = loc / mts;
    t.m0 = (loc - t.n0 * mts) * kTM;
    t.rows = a.T - t.m0;
    t.shared = true;
  }
  t.rows = t.rows < kTM ? t.rows : kTM;
  t.n0 *= tn;
  return t;
}

// The tile's pairs, biases (fp32) and (stage B) router weights in LDS.
template <bool STB>
__device__ __forceinline__ void tile_tables(const LayerArgs& a, const TileItem& t, int* s_pair, float* s_w,
                                            float* s_bias) {
  const int tid = threadIdx.x;
  const ftm_proj& PW = STB ? a.L.w2 : a.L.w13;
  float bias = 0.0f;
  if (!t.shared && PW.bias != nullptr && t.slot >= 0 && t.slot < PW.num_slots) {
    const int row = STB || tid < kTN / 2 ? t.n0 + tid : a.L.inter + t.n0 + tid - kTN / 2;
    if (row < PW.N) bias = load_scalar((const char*)PW.bias + (int64_t)t.slot * PW.bias_stride, row, PW.bias_dtype);
  }
  if (tid < kTM) {
    const int p = tid < t.rows ? (t.list != nullptr ? t.list[t.m0 + tid] : (t.m0 + tid) * a.KP + a.L.topk) : 0;
    s_pair[tid] = p;
    if (STB) s_w[tid] = tid < t.rows ? a.wts[p] : 0.0f;
  }
  s_bias[tid] = bias;
  __syncthreads();
}

// A non-resident expert's tile: its rows contribute zeros (stage B), and the
// error word says so.
template <bool STB>
__device__ __forceinline__ void tile_missing(const LayerArgs& a, const TileItem& t, const int* s_pair) {
  if (STB) {
    const int H = a.L.hidden;
    for (int idx = threadIdx.x; idx < kTM * kTN; idx += kBlock) {
      const int row = idx / kTN, col = t.n0 + idx % kTN;
      if (row < t.rows && col < H) a.ybuf[(size_t)s_pair[row] * H + col] = 0.0f;
    }
  }
  if (threadIdx.x == 0) atomicOr(&a.ctrl[kCtrlError], 1);
}

template <int FMT, int MODE, bool STB, bool BIG>
__global__ __launch_bounds__(kBlock, 2) void k_tile(const LayerArgs a) {
  char* lds = ftm_tile_lds;
  int* s_pair = (int*)(lds + TileFmt<FMT>::kRing);
  float* s_w = (float*)(s_pair + kTM);
  float* s_bias = s_w + kTM;
  const TileItem t = tile_item<STB>(a);
  if (t.rows <= 0) return;
  tile_tables<STB>(a, t, s_pair, s_w, s_bias);
  const int H = a.L.hidden, I = a.L.inter, Is = a.L.shared_inter;
  if (t.shared) {
    const ProjSlot W = STB ? shared_view(a.L.shared_w2, H, Is) : shared_view(a.L.shared_w13, 2 * Is, H);
    tile_rows<FTM_FMT_BF16, kScaleNone, STB, BIG>(a, W, Is, t.n0, t.rows, lds, s_pair, s_w, s_bias);
    return;
  }
  const ftm_proj& PW = STB ? a.L.w2 : a.L.w13;
  if (t.slot < 0 || t.slot >= PW.num_slots) {
    tile_missing<STB>(a, t, s_pair);
    return;
  }
  tile_rows<FMT, MODE, STB, BIG>(a, proj_slot(PW, t.slot), I, t.n0, t.rows, lds, s_pair, s_w, s_bias, s_bias + kTN);
}

// ---------------------------------------------------------------- scaled-MFMA tiles
// The routed experts of MXFP4 and FP8 (128 x 128 blocks) layers: the same tile
// on v_mfma_scale_f32_16x16x128_f8f6f4 with the decode path's operand layouts
// (ftm_moe.hip).  The weights go in as stored, straight from the buffer loads
// (e4m3, or e2m1 with e8m0 as scale_b); the activations as their two-term e4m3
// split (kMxChunk bytes per row and 128 K: the input by token from the router
// launch, h by pair from stage A's epilogue).  One K step is one MFMA pair per
// 16 x 16 block, so FP8's block scale multiplies the pair's sums and no second
// accumulator set is held.
//
// The activation rows are requested two K steps ahead, by direct buffer->LDS
// copies into a ring of three stages (buffer copies, not the global ones:
// those count as FLAT accesses, after which the compiler waits for every load
// in flight before it uses any), the weights one step ahead into one of two
// register sets.
constexpr int kXRow = 256;                           // hi and lo terms of a row and step
constexpr int kXStage = kTM * kXRow + kTM * 16;      // + the rows' scale bytes, 16 a row
constexpr int kXStages = 3;
constexpr int kXbSteps = 4;  // k_gemm_mxb_f8: K of at most this many steps, a stage for each

template <int FMT>
struct MxW {
  u32x4 w[4][FMT == FTM_FMT_MXFP4 ? 1 : 2];
  uint32_t s[4];  // MXFP4: the lane's e8m0 byte of block nj; FP8: [0] / [2], the halves' fp32 block scales
};

// Copy i of a wave covers rows 16 wave + 4 i + lane / 16 (16-byte pieces,
// swizzled), its last one the scale bytes of rows 16 wave + lane / 4.
using MxRows = TileSrc<5>;

// Wait until at most NW + NA n vector-memory operations are in flight (n < 4).
template <int NW, int NA>
__device__ __forceinline__ void wait_n(int n) {
  if (n == 3) wait_vm<NW + 3 * NA>();
  else if (n == 2) wait_vm<NW + 2 * NA>();
  else if (n == 1) wait_vm<NW + NA>();
  else wait_vm<NW>();
}

// One K step of a wave: 16 MI activation rows of the LDS stage st against its
// 64 weight rows, into acc.
template <int FMT, int MI>
__device__ __forceinline__ void mx_step(const char* st, const MxW<FMT>& cur, f32x4 (&acc)[MI][4]) {
  constexpr bool F8 = FMT == FTM_FMT_FP8_BLOCK;  // the step's products are scaled into acc
  const int lane = threadIdx.x & 63, g = lane >> 4, m = lane & 15;
  i32x8 bw[4];
  int sb[4];
#pragma unroll
  for (int nj = 0; nj < 4; ++nj) {
    if constexpr (F8) {
      const u32x4 r0 = cur.w[nj][0], r1 = cur.w[nj][1];
      bw[nj] = (i32x8){(int)r0.x, (int)r0.y, (int)r0.z, (int)r0.w, (int)r1.x, (int)r1.y, (int)r1.z, (int)r1.w};
      sb[nj] = 127;
    } else {
      const u32x4 r0 = cur.w[nj][0];
      bw[nj] = (i32x8){(int)r0.x, (int)r0.y, (int)r0.z, (int)r0.w, 0, 0, 0, 0};
      sb[nj] = (int)cur.s[nj];
    }
  }
  // each term of a row block is read from LDS during the MFMAs of the term
  // before it, and FP8's products of block mi are scaled into acc during
  // block mi + 1's
  struct Term {
    u32x4 a, b;
  };
  auto term = [&](int mi, int lo) {
    const char* cb = st + (16 * mi + m) * kXRow;
    Term t;
    t.a = *(const u32x4*)(cb + 16 * ((8 * lo + g) ^ m));
    t.b = *(const u32x4*)(cb + 16 * ((8 * lo + 4 + g) ^ m));
    return t;
  };
  auto scales = [&](int mi) { return (uint32_t)*(const uint16_t*)(st + kTM * kXRow + 16 * (16 * mi + m) + 2 * g); };
  f32x4 tq[2][4];
  auto fold = [&](int mi) {
    if constexpr (F8) {
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) acc[mi][nj] += tq[mi & 1][nj] * __uint_as_float(cur.s[nj & 2]);
    }
  };
  constexpr int kB = F8 ? 0 : 4;  // B format: e4m3 or e2m1
  auto mma = [&](int mi, const Term& t, int scale, bool first) {
    const i32x8 av = {(int)t.a.x, (int)t.a.y, (int)t.a.z, (int)t.a.w, (int)t.b.x, (int)t.b.y, (int)t.b.z, (int)t.b.w};
#pragma unroll
    for (int nj = 0; nj < 4; ++nj) {
      f32x4& d = F8 ? tq[mi & 1][nj] : acc[mi][nj];
      const f32x4 z = {0.f, 0.f, 0.f, 0.f};
      d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bw[nj], F8 && first ? z : d, 0, kB, 0, scale, 0, sb[nj]);
    }
  };
  Term hi = term(0, 0);
  uint32_t sc = scales(0);
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const Term lo = term(mi, 1);
    __builtin_amdgcn_sched_barrier(0);
    mma(mi, hi, (int)(sc & 0xffu), true);
    const int slo = (int)(sc >> 8);
    __builtin_amdgcn_sched_barrier(0);
    if (mi + 1 < MI) {
      hi = term(mi + 1, 0);
      sc = scales(mi + 1);
    }
    if (mi > 0) fold(mi - 1);
    __builtin_amdgcn_sched_barrier(0);
    mma(mi, lo, slo, false);
  }
  fold(MI - 1);
}

template <int FMT, int MI, bool BIG, bool SHORT>
__device__ __forceinline__ void mx_kloop(const ProjSlot& W, const int (&base)[2], const char* abase, uint32_t abytes,
                                         const MxRows& rows, char* lds, f32x4 (&acc)[MI][4]) {
  constexpr bool F8 = FMT == FTM_FMT_FP8_BLOCK;
  constexpr int NA = 5, NW = F8 ? 10 : 8;  // copies / loads a step
  typedef __attribute__((address_space(1))) const void* GPtr;
  typedef __attribute__((address_space(3))) void* LPtr;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4, m = lane & 15;
  const int K = W.K, N = W.N;
  const int nsteps = (K + 127) / 128;
  const Rsrc ares = make_rsrc(abase, abytes);
  uint32_t aoff[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) aoff[i] = (uint32_t)rows.p[i];
  auto issue_a = [&](int kb, int slot) {
    const uint32_t so = (uint32_t)(kb < nsteps ? kb : nsteps - 1) * (uint32_t)kMxChunk;
    char* st = lds + slot * kXStage;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      char* dst = i < 4 ? st + (16 * wave + 4 * i) * kXRow : st + kTM * kXRow + 256 * wave;
      if constexpr (BIG) {
        if (i < 4) __builtin_amdgcn_global_load_lds((GPtr)(rows.p[i] + so), (LPtr)dst, 16, 0, 0);
        else __builtin_amdgcn_global_load_lds((GPtr)(rows.p[i] + so), (LPtr)dst, 4, 0, 0);
      } else {
        if (i < 4) __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, (LPtr)dst, 16, (int)aoff[i], (int)so, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(ares, (LPtr)dst, 4, (int)aoff[i], (int)so, 0, 0);
      }
    }
  };

  const uint32_t rb = F8 ? (uint32_t)K : (uint32_t)K / 2;
  const int nkb = K / 128;
  const Rsrc wres = make_rsrc(W.w, rb * (uint32_t)N);
  const Rsrc sres = make_rsrc(W.s, F8 ? 4u * (uint32_t)((N + 127) / 128) * (uint32_t)nkb : (uint32_t)N * (uint32_t)(K / 32));
  uint32_t woff[4];
#pragma unroll
  for (int nj = 0; nj < 4; ++nj) {
    const int row = tile_row(base, nj, m);
    woff[nj] = row < N ? (uint32_t)row * rb + 16u * (uint32_t)g : kOOB;
  }
  auto load_w = [&](int kb, MxW<FMT>& t) {
    const int k0 = F8 ? kb * 128 : kb * 128 + 32 * g;  // FP8: K is whole steps
    const uint32_t so = k0 < K ? 4u * (uint32_t)kb : kOOB;
    const uint32_t ko = k0 < K ? (uint32_t)kb * (F8 ? 128u : 64u) : kOOB;
    if constexpr (F8) {
#pragma unroll
      for (int h = 0; h < 4; h += 2) t.s[h] = bload4(sres, 4u * (uint32_t)(base[h >> 1] / 128 * nkb) + so);
    } else {
      // the e8m0 byte of a 16-byte piece sits at a sixteenth of its offset
      // (rows past N: past the scales' end as well)
#pragma unroll
      for (int nj = 0; nj < 4; ++nj) t.s[nj] = bload1(sres, (woff[nj] >> 4) + so);
    }
#pragma unroll
    for (int nj = 0; nj < 4; ++nj)
#pragma unroll
      for (int i = 0; i < (F8 ? 2 : 1); ++i) t.w[nj][i] = bload16(wres, woff[nj] + ko + 64u * (uint32_t)i);
  };

  MxW<FMT> w0, w1;
  if constexpr (SHORT) {
    // at most kXbSteps steps: every stage's copies go out at once, each step
    // waits for its own
    issue_a(0, 0);
    load_w(0, w0);
#pragma unroll
    for (int kb = 1; kb < kXbSteps; ++kb) issue_a(kb, kb);
#pragma unroll
    for (int kb = 0; kb < kXbSteps; ++kb) {
      if (kb < nsteps) {
        const MxW<FMT>& cur = kb & 1 ? w1 : w0;
        // younger than stage kb's copies: this step's weights, the later stages' copies
        wait_n<NW, NA>(kXbSteps - 1 - kb);
        asm volatile("s_barrier" ::: "memory");
        if (kb + 1 < kXbSteps) load_w(kb + 1, kb & 1 ? w0 : w1);
        __builtin_amdgcn_sched_barrier(0);
        mx_step<FMT, MI>(lds + kb * kXStage, cur, acc);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  } else {
    auto step = [&](int kb, int slot, const MxW<FMT>& cur, MxW<FMT>& nxt) {
      // the copies of stage kb have landed (younger: this step's weights, the
      // copies of stage kb + 1), then every wave's have, and every wave is
      // done reading stage kb - 1
      wait_vm<NW + NA>();
      asm volatile("s_barrier" ::: "memory");
      issue_a(kb + 2, slot == 0 ? 2 : slot - 1);
      load_w(kb + 1, nxt);
      __builtin_amdgcn_sched_barrier(0);
      mx_step<FMT, MI>(lds + slot * kXStage, cur, acc);
      __builtin_amdgcn_sched_barrier(0);
    };
    issue_a(0, 0);
    load_w(0, w0);
    issue_a(1, 1);
    int slot = 0;
    auto next = [&] { slot = slot == 2 ? 0 : slot + 1; };
    if constexpr (F8) {
      // an odd last step of its own: with a branch round the second step of a
      // pair the compiler waits for this step's weights before it requests the
      // next ones (MXFP4 has no registers for the third copy of the step)
      int kb = 0;
      for (; kb + 1 < nsteps; kb += 2) {
        step(kb, slot, w0, w1);
        next();
        step(kb + 1, slot, w1, w0);
        next();
      }
      if (kb < nsteps) step(kb, slot, w0, w1);
    } else {
      for (int kb = 0; kb < nsteps; kb += 2) {
        step(kb, slot, w0, w1);
        next();
        if (kb + 1 < nsteps) step(kb + 1, slot, w1, w0);
        next();
      }
    }
  }
  // the copies past the last step have landed and every wave is done with the ring
  wait_vm<0>();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <bool STB, bool BIG>
__device__ __forceinline__ MxRows mx_rows(const LayerArgs& a, int rows, const int* s_pair) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const uint32_t arb = (uint32_t)mx_row_bytes(STB ? a.Imax : a.L.hidden);
  const char* abase = (const char*)(STB ? a.hq : a.xq);
  // padding rows repeat the first (their outputs are dropped)
  MxRows ar;
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int r = 16 * wave + (i < 4 ? 4 * i + (lane >> 4) : lane >> 2);
    const int pr = s_pair[r < rows ? r : 0];
    const uint64_t off = (uint64_t)(STB ? pr : pr / a.KP) * arb +
                         (i < 4 ? 16 * ((lane & 15) ^ (r & 15)) : 256 + 4 * (lane & 3));
    ar.p[i] = BIG ? (uint64_t)(uintptr_t)abase + off : off;
  }
  return ar;
}

template <int FMT, int MI, bool STB, bool BIG, bool SHORT>
__device__ __forceinline__ void mx_run(const LayerArgs& a, const ProjSlot& W, int Iu, int n0, int rows, char* lds,
                                       const int* s_pair, const float* s_w, const float* s_bias) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15;
  const int KP = a.KP, H = a.L.hidden;
  const uint32_t arb = (uint32_t)mx_row_bytes(STB ? a.Imax : H);
  const char* abase = (const char*)(STB ? a.hq : a.xq);
  const MxRows ar = mx_rows<STB, BIG>(a, rows, s_pair);
  const uint32_t abytes = BIG ? 0u : (uint32_t)(STB ? a.T * KP : a.T) * arb;
  const int base[2] = {n0 + (STB ? 64 : 32) * wave, STB ? n0 + 64 * wave + 32 : Iu + n0 + 32 * wave};
  f32x4 acc[MI][4];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int nj = 0; nj < 4; ++nj) acc[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
  mx_kloop<FMT, MI, BIG, SHORT>(W, base, abase, abytes, ar, lds, acc);

  const int lb[2] = {(STB ? 64 : 32) * wave, STB ? 64 * wave + 32 : kTN / 2 + 32 * wave};
  float bf[4];
#pragma unroll
  for (int nj = 0; nj < 4; ++nj) bf[nj] = s_bias[tile_row(lb, nj, m)];
  if constexpr (STB) {
    tile_store_y<FMT, MI>(a, W, base, bf, rows, s_pair, s_w, acc);
  } else {
    // h = bf16(act(gate) up) to LDS rows of 128 channels, then split into
    // e4m3 hi + lo, 8 channels a thread and one 32-channel block a quad of
    // lanes (channels past I are zeros: the tile is one whole chunk)
    tile_stage_h<FMT, MI>(a, n0, bf, lds, acc);
    const size_t hrow = (size_t)mx_row_bytes(a.Imax);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int row = 16 * i + (tid >> 4), pc = tid & 15;
      u32x4 v = *(const u32x4*)(lds + row * kTHPitch + 16 * pc);
      if (n0 + 8 * pc >= Iu) v = (u32x4){0u, 0u, 0u, 0u};
      const MxPiece q = mx_piece(v);
      if (row < rows) {
        uint8_t* o = a.hq + (size_t)s_pair[row] * hrow + (size_t)(n0 / 128) * kMxChunk;
        *(u32x2*)(o + 8 * pc) = q.hi;
        *(u32x2*)(o + 128 + 8 * pc) = q.lo;
        if ((pc & 3) == 0) *(uint16_t*)(o + 256 + (pc >> 1)) = (uint16_t)q.sc;
      }
    }
  }
}

template <int FMT, bool STB, bool BIG, bool SHORT>
__device__ __forceinline__ void mx_tile(const LayerArgs& a, int ring) {
  char* lds = ftm_tile_lds;
  int* s_pair = (int*)(lds + ring);
  float* s_w = (float*)(s_pair + kTM);
  float* s_bias = s_w + kTM;
  const TileItem t = tile_item<STB>(a);
  if (t.rows <= 0) return;
  tile_tables<STB>(a, t, s_pair, s_w, s_bias);
  const int H = a.L.hidden, I = a.L.inter, Is = a.L.shared_inter;
  if (t.shared) {
    const ProjSlot W = STB ? shared_view(a.L.shared_w2, H, Is) : shared_view(a.L.shared_w13, 2 * Is, H);
    tile_rows<FTM_FMT_BF16, kScaleNone, STB, BIG>(a, W, Is, t.n0, t.rows, lds, s_pair, s_w, s_bias);
    return;
  }
  const ftm_proj& PW = STB ? a.L.w2 : a.L.w13;
  if (t.slot < 0 || t.slot >= PW.num_slots) {
    tile_missing<STB>(a, t, s_pair);
    return;
  }
  const ProjSlot W = proj_slot(PW, t.slot);
  if (t.rows > 32) mx_run<FMT, 4, STB, BIG, SHORT>(a, W, I, t.n0, t.rows, lds, s_pair, s_w, s_bias);
  else mx_run<FMT, 2, STB, BIG, SHORT>(a, W, I, t.n0, t.rows, lds, s_pair, s_w, s_bias);
}

template <int FMT, bool STB, bool BIG>
__global__ __launch_bounds__(kBlock, FMT == FTM_FMT_MXFP4 ? 3 : 2) void k_gemm_mx(const LayerArgs a) {
  mx_tile<FMT, STB, BIG, false>(a, kXStages * kXStage);
}

// FP8 stage B with K = I of at most kXbSteps steps (the layer of 256 experts
// of 512): an LDS stage for every step, so no copy is issued past the last.
// Products, scales and epilogue are k_gemm_mx's, in the same order: the
// output is the same bits.
__global__ __launch_bounds__(kBlock, 2) void k_gemm_mxb_f8(const LayerArgs a) {
  mx_tile<FTM_FMT_FP8_BLOCK, true, false, true>(a, kXbSteps * kXStage);
}

// ---------------------------------------------------------------- launch
// Dynamic LDS: activation stages, the tile's pairs, router weights and biases,
// k_tile on GPTQ: its row sums.
constexpr size_t kTileTables = (size_t)kTM * 8u + (size_t)kTN * 4u;
constexpr size_t kMxLds = (size_t)kXStages * kXStage + kTileTables;
template <int FMT>
static size_t tile_lds(const ftm_moe_layer& L, bool stb) {
  const size_t x = FMT == FTM_FMT_GPTQ_INT4 ? (size_t)kTM * (size_t)((stb ? L.inter : L.hidden) / 128 + 1) * 4u : 0u;
  return (size_t)TileFmt<FMT>::kRing + kTileTables + x;
}

// GPTQ layers the tiles take: 128-wide groups (or multiples), 16-bit scales,
// whole K steps, and row sums that fit the LDS beside the ring.
bool tile_gptq_ok(const ftm_moe_layer& L) {
  if (L.w13.fmt != FTM_FMT_GPTQ_INT4 || L.act_dtype != FTM_DT_BF16) return false;
  if (L.w13.group <= 0 || L.w2.group <= 0 || L.w13.group % 128 != 0 || L.w2.group % 128 != 0) return false;
  if (L.hidden % 128 != 0 || L.inter % 128 != 0 || L.hidden % L.w13.group != 0 || L.inter % L.w2.group != 0) return false;
  if (L.w13.s_dtype == FTM_DT_F32 || L.w2.s_dtype == FTM_DT_F32) return false;
  return tile_lds<FTM_FMT_GPTQ_INT4>(L, false) <= 160u * 1024u && tile_lds<FTM_FMT_GPTQ_INT4>(L, true) <= 160u * 1024u;
}

// The layers the bf16 tiles take: GPTQ (tile_gptq_ok); FP8 128 x 128 below 16
// tokens per expert (mx_gemm_ok); INT8 groups of whole K steps, or
// one over K; bf16 weights where there is a stage-A tile for every CU.  Below
// that the ring tiles' 64 x 64 channels fill twice as many CUs: 16 bf16 experts
// of 1024 x 512, top-2, at 256 / 400 / 700 / 1100 / 1500 / 2048 tokens 53.3 /
// 54.2 / 56.7 / 59.6 / 63.8 / 90.6 us a layer there against 58.4 / 59.7 / 60.1 /
// 61.8 / 63.8 / 86.5 here.  (INT8 wins from 128 tokens of 16 experts on: its
// ring tiles decode every weight after an LDS read, 50.3 against 39.2 us.)
constexpr long kTileBf16MinItems = 256;
bool tile_bf16_ok(const ftm_moe_layer& L, int T) {
  if (L.act_dtype != FTM_DT_BF16) return false;
  if (L.w13.fmt == FTM_FMT_BF16) {
    const long pairs = (long)T * L.topk;
    const long maxU = L.num_experts < pairs ? L.num_experts : pairs;
    return (pairs / kTM + maxU) * ((L.inter + kTN / 2 - 1) / (kTN / 2)) >= kTileBf16MinItems;
  }
  if (L.w13.fmt == FTM_FMT_GPTQ_INT4) return tile_gptq_ok(L);
  if (L.w13.fmt == FTM_FMT_FP8_BLOCK) return mx_fmt(L) && !mx_gemm_ok(L, T);
  auto ok = [](const ftm_proj& P) { return P.group == P.K || (P.group % 128 == 0 && P.group > 0); };
  return L.w13.fmt == FTM_FMT_INT8_PACKED && ok(L.w13) && ok(L.w2);
}

// Items of one stage, an upper bound: every routed expert's last M tile may
// be partly filled.
template <bool STB>
static unsigned tile_items(const LayerArgs& a) {
  const ftm_moe_layer& L = a.L;
  const long pairs = (long)a.T * L.topk;
  const long maxU = L.num_experts < pairs ? L.num_experts : pairs;
  const int I = L.inter, Is = L.shared_inter, H = L.hidden;
  constexpr long tn = STB ? kTN : kTN / 2;
  const long ntn = ((STB ? H : I) + tn - 1) / tn, nts = Is == 0 ? 0 : ((STB ? H : Is) + tn - 1) / tn;
  return (unsigned)((pairs / kTM + maxU) * ntn + (long)((a.T + kTM - 1) / kTM) * nts);
}

template <class K>
static void tile_attr(K* kernel, DeviceBits& done) {
  (void)allow_lds(done, reinterpret_cast<const void*>(kernel), 160 * 1024);
}

// BIG: activation rows past what one buffer descriptor's 32-bit offsets span.
static bool tile_big(const LayerArgs& a, bool stb, size_t row_bytes) {
  return (stb ? (double)a.T * a.KP : (double)a.T) * (double)row_bytes >= 4294967296.0;
}

template <int FMT, int MODE, bool STB, bool BIG>
static void launch_tile_t(const LayerArgs& a, hipStream_t st) {
  static DeviceBits attr;
  tile_attr(&k_tile<FMT, MODE, STB, BIG>, attr);
  static_assert(TileFmt<FMT>::kRing >= TileFmt<FTM_FMT_BF16>::kRing, "the shared expert's stages fit");
  hipLaunchKernelGGL((k_tile<FMT, MODE, STB, BIG>), dim3(tile_items<STB>(a)), dim3(kBlock),
                     tile_lds<FMT>(a.L, STB), st, a);
}

template <int FMT, int MODE, bool STB>
static void launch_tile_s(const LayerArgs& a, hipStream_t st) {
  if (tile_big(a, STB, 2u * (size_t)(STB ? a.Imax : a.L.hidden))) launch_tile_t<FMT, MODE, STB, true>(a, st);
  else launch_tile_t<FMT, MODE, STB, false>(a, st);
}

void launch_tile_bf16(const LayerArgs& a, hipStream_t st, int which) {
  const int f = a.L.w13.fmt;
  const bool i8 = f == FTM_FMT_INT8_PACKED;
  if (which & 1) {
    if (f == FTM_FMT_GPTQ_INT4) launch_tile_s<FTM_FMT_GPTQ_INT4, kScale128, false>(a, st);
    else if (f == FTM_FMT_FP8_BLOCK) launch_tile_s<FTM_FMT_FP8_BLOCK, kScale128, false>(a, st);
    else if (!i8) launch_tile_s<FTM_FMT_BF16, kScaleNone, false>(a, st);
    else if (a.L.w13.group == a.L.w13.K) launch_tile_s<FTM_FMT_INT8_PACKED, kScaleOne, false>(a, st);
    else launch_tile_s<FTM_FMT_INT8_PACKED, kScale128, false>(a, st);
  }
  if (which & 2) {
    if (f == FTM_FMT_GPTQ_INT4) launch_tile_s<FTM_FMT_GPTQ_INT4, kScale128, true>(a, st);
    else if (f == FTM_FMT_FP8_BLOCK) launch_tile_s<FTM_FMT_FP8_BLOCK, kScale128, true>(a, st);
    else if (!i8) launch_tile_s<FTM_FMT_BF16, kScaleNone, true>(a, st);
    else if (a.L.w2.group == a.L.w2.K) launch_tile_s<FTM_FMT_INT8_PACKED, kScaleOne, true>(a, st);
    else launch_tile_s<FTM_FMT_INT8_PACKED, kScale128, true>(a, st);
  }
}

template <int FMT, bool STB, bool BIG>
static void launch_mx_t(const LayerArgs& a, hipStream_t st) {
  static DeviceBits attr;
  tile_attr(&k_gemm_mx<FMT, STB, BIG>, attr);
  static_assert(kXStages * kXStage >= TileFmt<FTM_FMT_BF16>::kRing, "the shared expert's stages fit");
  hipLaunchKernelGGL((k_gemm_mx<FMT, STB, BIG>), dim3(tile_items<STB>(a)), dim3(kBlock), kMxLds, st, a);
}

template <int FMT, bool STB>
static void launch_mx_s(const LayerArgs& a, hipStream_t st) {
  if (tile_big(a, STB, (size_t)mx_row_bytes(STB ? a.Imax : a.L.hidden))) launch_mx_t<FMT, STB, true>(a, st);
  else launch_mx_t<FMT, STB, false>(a, st);
}

// k_gemm_mxb_f8's layers; FTM_PROJ_RING_B asks for k_gemm_mx.
bool tile_mxb_ok(const ftm_moe_layer& L, int T) {
  const int KP = L.topk + (L.shared_inter > 0 ? 1 : 0);
  const int imax = L.inter > L.shared_inter ? L.inter : L.shared_inter;
  return L.w2.fmt == FTM_FMT_FP8_BLOCK && (L.w2.flags & FTM_PROJ_RING_B) == 0 && L.inter % 128 == 0 &&
         L.inter <= 128 * kXbSteps && (double)T * KP * mx_row_bytes(imax) < 4294967296.0;
}

static void launch_mxb(const LayerArgs& a, hipStream_t st) {
  static DeviceBits attr;
  tile_attr(&k_gemm_mxb_f8, attr);
  hipLaunchKernelGGL(k_gemm_mxb_f8, dim3(tile_items<true>(a)), dim3(kBlock),
                     (size_t)kXbSteps * kXStage + kTileTables, st, a);
}

void launch_tile_mx(const LayerArgs& a, hipStream_t st, int which) {
  const int f = a.L.w13.fmt;
  if (which & 1) {
    if (f == FTM_FMT_FP8_BLOCK) launch_mx_s<FTM_FMT_FP8_BLOCK, false>(a, st);
    else launch_mx_s<FTM_FMT_MXFP4, false>(a, st);
  }
  if (which & 2) {
    if (f == FTM_FMT_FP8_BLOCK && tile_mxb_ok(a.L, a.T)) launch_mxb(a, st);
    else if (f == FTM_FMT_FP8_BLOCK) launch_mx_s<FTM_FMT_FP8_BLOCK, true>(a, st);
    else launch_mx_s<FTM_FMT_MXFP4, true>(a, st);
  }
}

}  // namespace ftm
