// ftm_gemm.hip -- the dispatch of the expert stages above the token crossover,
// and the LDS-tiled bf16-MFMA GEMMs (v_mfma_f32_16x16x32_bf16) for the layers
// the register-fed tiles (ftm_tile.hip) do not take: FP8 blocks other than
// 128 x 128 with fp32 scales, FP8 with H or I not a multiple of 128, INT8 with
// groups other than K or whole 128s, bf16 layers with fewer tiles than CUs.
//
// Below the crossover every expert sees a handful of tokens and the stages are
// weight-streaming GEMVs (ftm_moe.hip).  Above it (prefill) each expert's
// weights are reused by many tokens, so a tile of 64 tokens x 64 channels
// loads its weights once per K step into LDS, decoded to bf16 exactly (FP8
// e4m3 and INT8 codes are exact in bf16), and four waves run 16x16x32 MFMAs
// out of LDS.  FP8 block and INT8 group scales multiply the fp32 partial sums
// of each quantisation group, as in the GEMV path, so both paths share one
// numerical contract.
//
// Tiles: the routed experts' token lists are cut into 64-row M tiles
// (ascending compact expert index u), then the shared expert's tokens.  Stage
// A (w13 + activation): a tile covers 64 channels, i.e. the 64 gate rows and
// the matching 64 up rows of w13, and writes h.  Stage B (w2): a tile covers
// 64 output columns and writes router-weighted fp32 rows into the slot buffer
// that k_combine reduces.
#include "ftm_layer.h"

namespace ftm {

constexpr int kGM = 64;            // tokens per tile
constexpr int kGK = 64;            // K per step
constexpr int kGPitch = kGK + 8;   // LDS row pitch in bf16 (144 B: rows do not share a bank period)
// Crossover, in average tokens per routed expert: 16 where the tiles' grid is
// small (a tile's latency is then the stage's: 16 INT8 experts of 512 take
// 26.6 us on the GEMV stages against 34.6 at 8 tokens per expert, 50 against
// 37 at 16) and for MXFP4 (its token-resident stages win below).
constexpr int kGemmMinRows = 16;
// Register-fed tiles that cover the chip (at least kGemmWideItems stage-A
// tiles, one per CU) read the weights once at a higher rate than the GEMV
// stages, which read them again for every few tokens.  Measured on MI355X (us
// per layer, GEMV stages / tiles): GPTQ 128 experts of 768 at 3 / 8 tokens per
// expert 126 / 139 against 103 / 111; 64 INT8 experts of 1024 at 2 / 8 132 /
// 172 against 113 / 123; 64 FP8 experts of 1024 at 4 / 9 / 15 160 / 205 / 284
// against 145 / 152 / 157; bf16 at 2 / 3 220 / 253 against 241 / 248.
constexpr int kGemmMinRowsWide = 3;
constexpr int kGemmWideItems = 256;
// The lean FP8 shape (256 experts of 512): 2 / 3 / 4 / 5 / 6 / 8 tokens per
// expert 150 / 172 / 193 / 213 / 231 / 266 us on its own stages against 180 /
// 193 / 206 / 208 / 212 / 219 on the tiles.  The tiles would win from 5 on; the
// line lies past 8 because the kernels of this shape are named up to 256 tokens
// (ftm_moe_stage_kernel, pinned by the dispatch test).
constexpr int kGemmMinRowsLean = 9;

// Weight bytes per element and 16-byte pieces per tile row per K step.
template <int WFMT>
struct GemmW {
  static constexpr int kPieces = WFMT == FTM_FMT_BF16 ? 8 : 4;
  static constexpr int kElems = kGK / kPieces;  // elements per piece
  static constexpr bool kPostScale = WFMT == FTM_FMT_FP8_BLOCK || WFMT == FTM_FMT_INT8_PACKED;
  __device__ static uint32_t row_bytes(int K) {
    return WFMT == FTM_FMT_BF16 ? 2u * (uint32_t)K : (uint32_t)K;
  }
};

// M tile -> (compact expert u, first row, token count).  u == nRouted is the
// shared expert; u < 0: past the last tile.  Every lane of the calling wave
// gets the same answer (wave-uniform, no LDS).
struct GemmTile {
  int u, m0, cnt;
};

template <int MT = kGM>
__device__ __forceinline__ GemmTile gemm_find_tile(const LayerArgs& a, int mtile, int nRouted, bool shared) {
  const int lane = threadIdx.x & 63;
  // lane l owns compact experts 8l .. 8l+7 (E <= 512)
  const Rsrc cres = make_rsrc(a.ucnt, (uint32_t)(a.L.num_experts + 1) * 4u);
  int v[8], c[8];
  int lsum = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int u = 8 * lane + j;
    c[j] = u < nRouted ? (int)bload4(cres, 4u * (uint32_t)u) : 0;
    v[j] = (c[j] + MT - 1) / MT;
    lsum += v[j];
  }
  // exclusive prefix over lanes
  int incl = lsum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int o = __shfl_up(incl, off);
    if (lane >= off) incl += o;
  }
  const int total = __shfl(incl, 63);
  GemmTile t = {-1, 0, 0};
  if (mtile < total) {
    int base = incl - lsum;
    int found_u = -1, found_m0 = 0, found_cnt = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (found_u < 0 && mtile >= base && mtile < base + v[j]) {
        found_u = 8 * lane + j;
        found_m0 = (mtile - base) * MT;
        found_cnt = c[j];
      }
      base += v[j];
    }
    const uint64_t who = __ballot(found_u >= 0);
    const int src = (int)__builtin_ctzll(who);
    t.u = __shfl(found_u, src);
    t.m0 = __shfl(found_m0, src);
    t.cnt = __shfl(found_cnt, src);
  } else if (shared) {
    const int st = mtile - total;
    if (st * MT < a.T) {
      t.u = nRouted;
      t.m0 = st * MT;
      t.cnt = a.T;
    }
  }
  return t;
}

// Routed M tiles (device total) for the item -> tile mapping of a stage whose
// routed part has ntn N tiles per M tile.
template <int MT = kGM>
__device__ __forceinline__ int gemm_routed_mtiles(const LayerArgs& a, int nRouted) {
  const int lane = threadIdx.x & 63;
  const Rsrc cres = make_rsrc(a.ucnt, (uint32_t)(a.L.num_experts + 1) * 4u);
  int lsum = 0;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int u = 8 * lane + j;
    lsum += u < nRouted ? ((int)bload4(cres, 4u * (uint32_t)u) + MT - 1) / MT : 0;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) lsum += __shfl_xor(lsum, off);
  return lsum;
}

// One 64-token x (NWR weight rows) tile over the whole K range.
//   WFMT: weight format; NWR = 128 (stage A: 64 gate + 64 up rows) or 64 (stage B)
//   grow(r): global weight row of tile row r
//   arow[i]: byte offset of the activation row of A piece i of this thread (kOOB = zero row)
//   acc[mi][nj]: wave (wm, wn) tile: tokens 32wm + 16mi, tile rows nrow(nj)
template <int WFMT, int NWR, int AXB>
struct GemmTileRun {
  static constexpr int NB = NWR == 128 ? 4 : 2;  // 16-column MFMA blocks per wave
  static constexpr int kWPieces = NWR * GemmW<WFMT>::kPieces;
  static constexpr int kWLoads = (kWPieces + kBlock - 1) / kBlock;

  // tile row of MFMA column block nj of wave column wn
  __device__ static int nrow(int nj, int wn) {
    if constexpr (NWR == 128) return nj < 2 ? 32 * wn + 16 * nj : 64 + 32 * wn + 16 * (nj - 2);
    return 32 * wn + 16 * nj;
  }
};

template <int WFMT, int NWR>
__device__ __forceinline__ void gemm_tile(const ProjSlot& W, int c0, int Iu, Rsrc ares, const uint32_t (&arow)[2],
                                          uint16_t* sA, uint16_t* sB, f32x4 (&acc)[2][NWR == 128 ? 4 : 2]) {
  using G = GemmW<WFMT>;
  using R = GemmTileRun<WFMT, NWR, 2>;
  constexpr int NB = R::NB;
  constexpr int kSA = kGM * kGPitch, kSB = NWR * kGPitch;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int K = W.K;
  const int nsteps = (K + kGK - 1) / kGK;
  auto grow = [&](int r) { return NWR == 128 ? (r < 64 ? c0 + r : Iu + c0 + (r - 64)) : c0 + r; };

  const uint32_t rb = G::row_bytes(K);
  const Rsrc wres = make_rsrc(W.w, rb * (uint32_t)W.N);
  uint32_t woff[R::kWLoads];
  int wtr[R::kWLoads], wpc[R::kWLoads];
#pragma unroll
  for (int i = 0; i < R::kWLoads; ++i) {
    const int c = tid + kBlock * i;
    wtr[i] = c / G::kPieces;
    wpc[i] = c % G::kPieces;
    const int r = grow(wtr[i]);
    woff[i] = (c < R::kWPieces && r < W.N) ? (uint32_t)r * rb + (uint32_t)wpc[i] * 16u : kOOB;
  }
  // post-scale sources: FP8 block rows (uniform per column block), INT8 rows (per lane)
  const int lpg = G::kPostScale ? W.group / kGK : 1;
  int srow[NB];
#pragma unroll
  for (int nj = 0; nj < NB; ++nj) srow[nj] = grow(R::nrow(nj, wn));
  const uint32_t sesz = W.s_dt == FTM_DT_F32 ? 4u : 2u;
  Rsrc i8res = wres;
  if constexpr (WFMT == FTM_FMT_INT8_PACKED) i8res = make_rsrc(W.s, (uint32_t)(W.N * (K / W.group)) * sesz);

  u32x4 rw[R::kWLoads], ra[2];
  auto issue = [&](int kb) {
    const uint32_t kbyte = (uint32_t)kb * (uint32_t)(kGK * (WFMT == FTM_FMT_BF16 ? 2 : 1));
#pragma unroll
    for (int i = 0; i < R::kWLoads; ++i) rw[i] = bload16(wres, woff[i] != kOOB ? woff[i] + kbyte : kOOB);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int piece = (tid + kBlock * i) & 7;
      ra[i] = bload16(ares, arow[i] != kOOB ? arow[i] + (uint32_t)(kb * kGK + piece * 8) * 2u : kOOB);
    }
  };
  auto stage = [&](int buf) {
    uint16_t* a_ = sA + buf * kSA;
    uint16_t* b_ = sB + buf * kSB;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int c = tid + kBlock * i;
      *(u32x4*)(a_ + (c >> 3) * kGPitch + (c & 7) * 8) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < R::kWLoads; ++i) {
      if (tid + kBlock * i >= R::kWPieces) continue;
      uint16_t* dst = b_ + wtr[i] * kGPitch + wpc[i] * G::kElems;
      if constexpr (WFMT == FTM_FMT_FP8_BLOCK) {
        *(u32x4*)dst = fp8x8_to_bf16(rw[i].x, rw[i].y);
        *(u32x4*)(dst + 8) = fp8x8_to_bf16(rw[i].z, rw[i].w);
      } else if constexpr (WFMT == FTM_FMT_INT8_PACKED) {
        *(u32x4*)dst = i8x8_to_bf16(rw[i].x, rw[i].y);
        *(u32x4*)(dst + 8) = i8x8_to_bf16(rw[i].z, rw[i].w);
      } else {
        *(u32x4*)dst = rw[i];
      }
    }
  };

  f32x4 tmp[2][NB];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int nj = 0; nj < NB; ++nj) tmp[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};

  issue(0);
  for (int kb = 0; kb < nsteps; ++kb) {
    const int buf = kb & 1;
    stage(buf);
    __syncthreads();
    if (kb + 1 < nsteps) issue(kb + 1);
    const uint16_t* a_ = sA + buf * kSA;
    const uint16_t* b_ = sB + buf * kSB;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int ko = ks * 32 + 8 * (lane >> 4);
      u32x4 af[2], bf[NB];
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) af[mi] = *(const u32x4*)(a_ + (32 * wm + 16 * mi + (lane & 15)) * kGPitch + ko);
#pragma unroll
      for (int nj = 0; nj < NB; ++nj) bf[nj] = *(const u32x4*)(b_ + (R::nrow(nj, wn) + (lane & 15)) * kGPitch + ko);
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int nj = 0; nj < NB; ++nj) tmp[mi][nj] = mfma_bf16(af[mi], bf[nj], tmp[mi][nj]);
    }
    if constexpr (G::kPostScale) {
      // end of a quantisation group: acc += group partial * scale (straight-line)
      const bool last = ((kb + 1) % lpg == 0) | (kb + 1 == nsteps);
      const int grp = kb / lpg;
#pragma unroll
      for (int nj = 0; nj < NB; ++nj) {
        float s;
        if constexpr (WFMT == FTM_FMT_FP8_BLOCK) {
          const int nkb = (K + W.group - 1) / W.group;
          const uint32_t idx = (uint32_t)((srow[nj] / W.group) * nkb + grp);
          s = decode_scalar_word(sload4(W.s, (idx * sesz) & ~3u), idx, W.s_dt);
        } else {
          const uint32_t idx = (uint32_t)((srow[nj] + (lane & 15)) * (K / W.group) + grp);
          s = decode_scalar_word(bload_scalar_word(i8res, idx, W.s_dt, srow[nj] + (lane & 15) < W.N), idx, W.s_dt);
        }
        const float f = last ? s : 0.0f;
        const float keep = last ? 0.0f : 1.0f;
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
          acc[mi][nj] += tmp[mi][nj] * f;
          tmp[mi][nj] *= keep;
        }
      }
    }
  }
  if constexpr (!G::kPostScale) {
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int nj = 0; nj < NB; ++nj) acc[mi][nj] += tmp[mi][nj];
  }
  __syncthreads();  // the LDS tiles are reused by the caller's next tile
}

// ---------------------------------------------------------------- LDS ring tiles (stage A)
// The stage A tiles for FP8 / INT8 / bf16 weights, fed by a ring of up to
// four LDS stages that direct global-to-LDS copies (global_load_lds, 16 B per
// lane) fill three K steps ahead of the MFMAs.  Activations (bf16) and the raw
// weight bytes both land in LDS undecoded; a wave decodes its own weight rows
// after its LDS read.  Each 1 KiB copy writes 64 consecutive 16-byte slots, so
// the bank-conflict swizzle is applied on the read side of the copy: the lane
// filling slot s of row r fetches piece s ^ f(r) of that row, and a reader
// finds piece p of row r in slot p ^ f(r).  With f below, the rows one MFMA
// operand read touches (16 rows, one piece each) hit distinct 16-byte bank
// groups.  The tile's quantisation-group scales are copied to LDS once, before
// the K loop, so no scale load waits inside it.

// Raw weight bytes per row per K step and rows per 1 KiB copy.
template <int WFMT>
struct RingW {
  static constexpr int kRowBytes = WFMT == FTM_FMT_BF16 ? 2 * kGK : kGK;
  static constexpr int kRowsPerCopy = 1024 / kRowBytes;
};
// Ring bytes per workgroup: 64 KiB (FP8/INT8: 4 stages, bf16: 2).  The
// tile's scales follow the ring (at most kRingScaleBytes; the launch sizes the
// dynamic LDS to what the layer needs).
constexpr int kRingA = 64 * 1024;
constexpr int kRingScaleBytes = 16 * 1024;

template <int WFMT, int NWR, int RB>
struct RingPlan {
  static constexpr int kA = kGM * 2 * kGK;  // 64 token rows x 64 bf16
  static constexpr int kW = NWR * RingW<WFMT>::kRowBytes;
  static constexpr int kStage = kA + kW;
  static constexpr int kStages = RB / kStage < 4 ? RB / kStage : 4;
  static constexpr int kALoads = kA / 1024 / 4;  // 1 KiB copies per wave per stage
  static constexpr int kWLoads = kW / 1024 / 4;
  static constexpr int kLoads = kALoads + kWLoads;
  static_assert(kStages >= 2 && kA % 4096 == 0 && kW % 4096 == 0, "ring shape");
};

__device__ __forceinline__ int ring_fa(int r) { return (r ^ (r >> 3)) & 7; }         // 8 pieces per row
__device__ __forceinline__ int ring_fw(int r) { return ((r >> 1) ^ (r >> 3)) & 3; }  // 4 pieces per row

// Wait until at most `stages` ring stages of this wave's copies are in flight.
template <int LOADS, int MAXS>
__device__ __forceinline__ void wait_ring(int stages) {
  if (MAXS >= 3 && stages >= 3) wait_vm<3 * LOADS>();
  else if (MAXS >= 2 && stages == 2) wait_vm<2 * LOADS>();
  else if (stages == 1) wait_vm<LOADS>();
  else wait_vm<0>();
}

// One 64-token x NWR-row tile over the whole K range (FP8, INT8 or bf16
// weights).  Wave w owns tile rows 64 j + 16 w .. + 15 (j < NWR / 64: for
// stage A the gate rows and the matching up rows) for all 64 tokens, so each
// weight byte is decoded once.  LPG: K steps per quantisation group, the loop
// unrolled so the group partial is scaled once, straight after the group's
// last MFMAs (2: 128-wide groups); 0: no intermediate scaling (bf16, or one
// group over K); -1: any group size (scaled with selects every step).
//   arow[i]: activation row of this lane's slot in A copy i (always a valid row;
//            padding rows repeat a real one and their outputs are dropped)
//   acc[mi][j]: tokens 16 mi + 4 (lane / 16) + r, tile row 64 j + 16 w + lane % 16
template <int WFMT, int NWR, int RB, int LPG>
__device__ __forceinline__ void gemm_tile_ring(const ProjSlot& W, int c0, int Iu,
                                               const char* const (&arow)[RingPlan<WFMT, NWR, RB>::kALoads],
                                               char* lds, f32x4 (&acc)[4][NWR / 64]) {
  using P = RingPlan<WFMT, NWR, RB>;
  using RW = RingW<WFMT>;
  typedef __attribute__((address_space(1))) const void* GPtr;
  typedef __attribute__((address_space(3))) void* LPtr;
  constexpr int NB = NWR / 64;
  constexpr int S = P::kStages;
  constexpr bool kPost = WFMT == FTM_FMT_FP8_BLOCK || WFMT == FTM_FMT_INT8_PACKED;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = W.K;
  const int nsteps = K / kGK;
  auto grow = [&](int r) { return NWR == 128 ? (r < 64 ? c0 + r : Iu + c0 + (r - 64)) : c0 + r; };
  const uint32_t rb = GemmW<WFMT>::row_bytes(K);
  float* sS = (float*)(lds + RB);

  // ---- this lane's copy sources (K offset added per step)
  const char* asrc[P::kALoads];
#pragma unroll
  for (int i = 0; i < P::kALoads; ++i) {
    const int r = 8 * (wave * P::kALoads + i) + (lane >> 3);
    asrc[i] = arow[i] + 16 * ((lane & 7) ^ ring_fa(r));
  }
  const char* wsrc[P::kWLoads];
#pragma unroll
  for (int i = 0; i < P::kWLoads; ++i) {
    const int j = wave * P::kWLoads + i;
    int r, piece;
    if constexpr (WFMT == FTM_FMT_BF16) {
      r = 8 * j + (lane >> 3);
      piece = (lane & 7) ^ ring_fa(r);
    } else {
      r = 16 * j + (lane >> 2);
      piece = (lane & 3) ^ ring_fw(r);
    }
    wsrc[i] = W.w + (size_t)grow(r) * rb + 16 * piece;
  }
  auto issue = [&](int kb, int slot) {
    char* st = lds + slot * P::kStage;
#pragma unroll
    for (int i = 0; i < P::kALoads; ++i)
      __builtin_amdgcn_global_load_lds((GPtr)(asrc[i] + kb * 2 * kGK),
                                       (LPtr)(st + 1024 * (wave * P::kALoads + i)), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < P::kWLoads; ++i)
      __builtin_amdgcn_global_load_lds((GPtr)(wsrc[i] + kb * RW::kRowBytes),
                                       (LPtr)(st + P::kA + 1024 * (wave * P::kWLoads + i)), 16, 0, 0);
  };

  // ---- group scales of the tile -> LDS as fp32 (FP8: one row per 64-row
  // half, INT8: one row per tile row), loads issued before the ring prologue
  const int ngroups = kPost ? (K + W.group - 1) / W.group : 0;
  constexpr int kScaleRows = WFMT == FTM_FMT_INT8_PACKED ? NWR : NWR / 64;
  constexpr int kScalePer = WFMT == FTM_FMT_INT8_PACKED ? (kRingScaleBytes / 4 + kBlock - 1) / kBlock : 1;
  uint32_t sw[kScalePer];
  uint32_t sidx[kScalePer];
  if constexpr (kPost) {
    const uint32_t sesz = W.s_dt == FTM_DT_F32 ? 4u : 2u;
    const int nsc = kScaleRows * ngroups;
    const Rsrc sres = make_rsrc(W.s, WFMT == FTM_FMT_FP8_BLOCK
                                         ? (uint32_t)(((W.N + W.group - 1) / W.group) * ngroups) * sesz
                                         : (uint32_t)(W.N * ngroups) * sesz);
#pragma unroll
    for (int q = 0; q < kScalePer; ++q) {
      const int e = tid + kBlock * q;
      const int sr = e / (ngroups > 0 ? ngroups : 1), g = e - sr * ngroups;
      const int wrow = WFMT == FTM_FMT_FP8_BLOCK ? grow(64 * sr) / W.group : grow(sr);
      sidx[q] = (uint32_t)(wrow * ngroups + g);
      sw[q] = bload_scalar_word(sres, sidx[q], W.s_dt, e < nsc);
    }
  }
  const int pro = nsteps < S - 1 ? nsteps : S - 1;
  for (int kb = 0; kb < pro; ++kb) issue(kb, kb);
  if constexpr (kPost) {
    wait_ring<P::kLoads, S - 1>(pro);
#pragma unroll
    for (int q = 0; q < kScalePer; ++q) {
      const int e = tid + kBlock * q;
      if (e < kScaleRows * ngroups) sS[e] = decode_scalar_word(sw[q], sidx[q], W.s_dt);
    }
  }

  const int g4 = lane >> 4;
  int arr[4], wrr[NB];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) arr[mi] = 16 * mi + (lane & 15);
#pragma unroll
  for (int nj = 0; nj < NB; ++nj) wrr[nj] = 64 * nj + 16 * wave + (lane & 15);

  // one K step into d: wait for its stage, refill the ring, LDS -> MFMAs
  auto step = [&](int kb, f32x4 (&d)[4][NB]) {
    const int ahead = nsteps - 1 - kb < S - 2 ? nsteps - 1 - kb : S - 2;
    wait_ring<P::kLoads, S - 2>(ahead);
    __syncthreads();  // stage kb is in LDS for every wave; every wave is done with stage kb - 1
    if (kb + S - 1 < nsteps) issue(kb + S - 1, (kb + S - 1) % S);
    const char* st = lds + (kb % S) * P::kStage;
    u32x4 b0[NB], b1[NB];
#pragma unroll
    for (int nj = 0; nj < NB; ++nj) {
      const char* row = st + P::kA + wrr[nj] * RW::kRowBytes;
      if constexpr (WFMT == FTM_FMT_BF16) {
        b0[nj] = *(const u32x4*)(row + 16 * ((2 * g4) ^ ring_fa(wrr[nj])));
        b1[nj] = *(const u32x4*)(row + 16 * ((2 * g4 + 1) ^ ring_fa(wrr[nj])));
      } else {
        const u32x4 raw = *(const u32x4*)(row + 16 * (g4 ^ ring_fw(wrr[nj])));
        if constexpr (WFMT == FTM_FMT_FP8_BLOCK) {
          b0[nj] = fp8x8_to_bf16(raw.x, raw.y);
          b1[nj] = fp8x8_to_bf16(raw.z, raw.w);
        } else {
          b0[nj] = i8x8_to_bf16(raw.x, raw.y);
          b1[nj] = i8x8_to_bf16(raw.z, raw.w);
        }
      }
    }
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
      const char* row = st + arr[mi] * (2 * kGK);
      const u32x4 a0 = *(const u32x4*)(row + 16 * ((2 * g4) ^ ring_fa(arr[mi])));
      const u32x4 a1 = *(const u32x4*)(row + 16 * ((2 * g4 + 1) ^ ring_fa(arr[mi])));
#pragma unroll
      for (int nj = 0; nj < NB; ++nj) {
        d[mi][nj] = mfma_bf16(a0, b0[nj], d[mi][nj]);
        d[mi][nj] = mfma_bf16(a1, b1[nj], d[mi][nj]);
      }
    }
  };
  auto scale_of = [&](int nj, int grp) {
    return sS[(WFMT == FTM_FMT_FP8_BLOCK ? nj : wrr[nj]) * ngroups + grp];
  };

  if constexpr (!kPost) {
    for (int kb = 0; kb < nsteps; ++kb) step(kb, acc);
  } else {
    f32x4 tmp[4][NB];
#pragma unroll
    for (int mi = 0; mi < 4; ++mi)
#pragma unroll
      for (int nj = 0; nj < NB; ++nj) tmp[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
    if constexpr (LPG > 0) {
      // nsteps % LPG == 0 (checked at launch): whole groups per iteration
      for (int kb = 0, grp = 0; kb < nsteps; kb += LPG, ++grp) {
#pragma unroll
        for (int q = 0; q < LPG; ++q) step(kb + q, tmp);
#pragma unroll
        for (int nj = 0; nj < NB; ++nj) {
          const float sc = scale_of(nj, grp);
#pragma unroll
          for (int mi = 0; mi < 4; ++mi) {
            acc[mi][nj] += tmp[mi][nj] * sc;
            tmp[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
          }
        }
      }
    } else if constexpr (LPG == 0) {
      for (int kb = 0; kb < nsteps; ++kb) step(kb, tmp);
#pragma unroll
      for (int nj = 0; nj < NB; ++nj) {
        const float sc = scale_of(nj, 0);
#pragma unroll
        for (int mi = 0; mi < 4; ++mi) acc[mi][nj] += tmp[mi][nj] * sc;
      }
    } else {
      const int lpg = W.group / kGK;
      for (int kb = 0; kb < nsteps; ++kb) {
        step(kb, tmp);
        // end of a quantisation group: acc += group partial * scale (straight-line)
        const bool last = ((kb + 1) % lpg == 0) | (kb + 1 == nsteps);
        const int grp = kb / lpg;
#pragma unroll
        for (int nj = 0; nj < NB; ++nj) {
          const float sc = scale_of(nj, grp);
          const float f = last ? sc : 0.0f;
          const float keep = last ? 0.0f : 1.0f;
#pragma unroll
          for (int mi = 0; mi < 4; ++mi) {
            acc[mi][nj] += tmp[mi][nj] * f;
            tmp[mi][nj] *= keep;
          }
        }
      }
    }
  }
  __syncthreads();  // the ring is reused by the caller's next tile
}

// K-loop group structure of a projection: 2 (128-wide groups), 0 (one group
// over K, or no scales), -1 (other).
__host__ __device__ __forceinline__ int ring_lpg(int fmt, int group, int K) {
  if (fmt != FTM_FMT_FP8_BLOCK && fmt != FTM_FMT_INT8_PACKED) return 0;
  if (group >= K) return 0;
  if (group == 2 * kGK && (K / kGK) % 2 == 0) return 2;
  return -1;
}

// Stage A body on the ring tiles: item -> rows, tile, activation epilogue.
template <int WFMT, int LPG>
__device__ void gemm_a_ring_body(const LayerArgs& a, const ProjSlot& W, int Iu, int c0, int m0, int cnt,
                                 const int32_t* list, int shared_col, char* lds) {
  using P = RingPlan<WFMT, 128, kRingA>;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = a.L.hidden, KP = a.KP;
  const Rsrc lres = make_rsrc(list, list ? (uint32_t)a.T * 4u : 0u);
  const int p0 = pair_of_row(lres, list != nullptr, m0, cnt, KP, shared_col);
  const char* ap[P::kALoads];
#pragma unroll
  for (int i = 0; i < P::kALoads; ++i) {
    int p = pair_of_row(lres, list != nullptr, m0 + 8 * (wave * P::kALoads + i) + (lane >> 3), cnt, KP, shared_col);
    p = p >= 0 ? p : p0;
    ap[i] = (const char*)a.x + (size_t)(p / KP) * (size_t)H * 2u;
  }
  f32x4 acc[4][2];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int nj = 0; nj < 2; ++nj) acc[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
  gemm_tile_ring<WFMT, 128, kRingA, LPG>(W, c0, Iu, ap, lds, acc);
  const int ch = c0 + 16 * wave + (lane & 15);
  const float bg = W.bias != nullptr ? load_scalar(W.bias, ch, W.bias_dt) : 0.0f;
  const float bu = W.bias != nullptr ? load_scalar(W.bias, Iu + ch, W.bias_dt) : 0.0f;
#pragma unroll
  for (int mi = 0; mi < 4; ++mi)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int pe = pair_of_row(lres, list != nullptr, m0 + 16 * mi + 4 * (lane >> 4) + r, cnt, KP, shared_col);
      if (pe >= 0) {
        const float h = act_fn(a.L.act, acc[mi][0][r] + bg, acc[mi][1][r] + bu, a.L.swiglu_alpha, a.L.swiglu_limit);
        store_scalar(a.hbuf, (size_t)pe * a.Imax + ch, FTM_DT_BF16, h);
      }
    }
}

// ---------------------------------------------------------------- stage A (w13 + activation)
template <int WFMT>
__device__ void gemm_a_body(const LayerArgs& a, const ProjSlot& W, int Iu, int c0, int m0, int cnt,
                            const int32_t* list, int shared_col, uint16_t* sA, uint16_t* sB) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int H = a.L.hidden, KP = a.KP;
  const Rsrc lres = make_rsrc(list, list ? (uint32_t)a.T * 4u : 0u);
  const Rsrc xres = make_rsrc(a.x, (uint32_t)a.T * (uint32_t)H * 2u);
  uint32_t arow[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = pair_of_row(lres, list != nullptr, m0 + ((tid + kBlock * i) >> 3), cnt, KP, shared_col);
    arow[i] = p >= 0 ? (uint32_t)(p / KP) * (uint32_t)H * 2u : kOOB;
  }
  int pe[2][4];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      pe[mi][r] = pair_of_row(lres, list != nullptr, m0 + 32 * wm + 16 * mi + 4 * (lane >> 4) + r, cnt, KP,
                              shared_col);
  float bg[2], bu[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int ch = c0 + 32 * wn + 16 * j + (lane & 15);
    bg[j] = W.bias != nullptr ? load_scalar(W.bias, ch, W.bias_dt) : 0.0f;
    bu[j] = W.bias != nullptr ? load_scalar(W.bias, Iu + ch, W.bias_dt) : 0.0f;
  }
  f32x4 acc[2][4];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int nj = 0; nj < 4; ++nj) acc[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
  gemm_tile<WFMT, 128>(W, c0, Iu, xres, arow, sA, sB, acc);
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int ch = c0 + 32 * wn + 16 * j + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (pe[mi][r] >= 0) {
          const float h = act_fn(a.L.act, acc[mi][j][r] + bg[j], acc[mi][2 + j][r] + bu[j], a.L.swiglu_alpha,
                                 a.L.swiglu_limit);
          store_scalar(a.hbuf, (size_t)pe[mi][r] * a.Imax + ch, FTM_DT_BF16, h);
        }
      }
    }
}

// Stage A ring body by K-loop group structure (ring_lpg): FP8 128x128 blocks
// take LPG 2; INT8 per-channel (one group over K) 0, 128-wide groups 2; bf16 0.
template <int WFMT>
__device__ __forceinline__ void ring_a(const LayerArgs& a, const ProjSlot& W, int Iu, int c0, int m0, int cnt,
                                       const int32_t* list, int shared_col, char* lds) {
  const int lpg = ring_lpg(WFMT, W.group, W.K);
  if constexpr (WFMT == FTM_FMT_BF16) {  // no group post-scale
    gemm_a_ring_body<WFMT, 0>(a, W, Iu, c0, m0, cnt, list, shared_col, lds);
  } else if constexpr (WFMT == FTM_FMT_FP8_BLOCK) {
    if (lpg == 2) gemm_a_ring_body<WFMT, 2>(a, W, Iu, c0, m0, cnt, list, shared_col, lds);
    else gemm_a_ring_body<WFMT, -1>(a, W, Iu, c0, m0, cnt, list, shared_col, lds);
  } else {
    if (lpg == 0) gemm_a_ring_body<WFMT, 0>(a, W, Iu, c0, m0, cnt, list, shared_col, lds);
    else if (lpg == 2) gemm_a_ring_body<WFMT, 2>(a, W, Iu, c0, m0, cnt, list, shared_col, lds);
    else gemm_a_ring_body<WFMT, -1>(a, W, Iu, c0, m0, cnt, list, shared_col, lds);
  }
}

template <int FMT, bool RING>
__device__ __forceinline__ void gemm_a_item(const LayerArgs& a, int item, uint16_t* sA, uint16_t* sB) {
  const int I = a.L.inter, Is = a.L.shared_inter;
  const int nRouted = a.ctrl[kCtrlNRouted];
  const int ntn = I / 64;
  const int routed_items = gemm_routed_mtiles(a, nRouted) * ntn;
  if (item < routed_items) {
    const GemmTile t = gemm_find_tile(a, item / ntn, nRouted, false);
    if (t.u < 0) return;
    const int e = a.uniq[t.u];
    const int slot = a.L.slot_of_expert ? a.L.slot_of_expert[e] : e;
    if (slot < 0 || slot >= a.L.w13.num_slots) {
      if (threadIdx.x == 0) atomicOr(&a.ctrl[kCtrlError], 1);
      return;
    }
    const ProjSlot W = proj_slot(a.L.w13, slot);
    if constexpr (RING)
      ring_a<FMT>(a, W, I, (item % ntn) * 64, t.m0, t.cnt, a.lists + (size_t)e * a.T, 0, (char*)sA);
    else
      gemm_a_body<FMT>(a, W, I, (item % ntn) * 64, t.m0, t.cnt, a.lists + (size_t)e * a.T, 0, sA, sB);
  } else if (Is > 0) {
    const int sitem = item - routed_items, nts = Is / 64;
    const int m0 = (sitem / nts) * kGM;
    if (m0 >= a.T) return;
    const ProjSlot W = shared_view(a.L.shared_w13, 2 * Is, a.L.hidden);
    if constexpr (RING)
      ring_a<FTM_FMT_BF16>(a, W, Is, (sitem % nts) * 64, m0, a.T, nullptr, a.L.topk, (char*)sA);
    else
      gemm_a_body<FTM_FMT_BF16>(a, W, Is, (sitem % nts) * 64, m0, a.T, nullptr, a.L.topk, sA, sB);
  }
}

template <int FMT>
__global__ __launch_bounds__(kBlock) void k_gemm_a(const LayerArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t sA[2 * kGM * kGPitch];
  __shared__ __attribute__((aligned(16))) uint16_t sB[2 * 128 * kGPitch];
  gemm_a_item<FMT, false>(a, blockIdx.x, sA, sB);
}

extern __shared__ __attribute__((aligned(16))) uint16_t ftm_ring_lds[];

// The ring tiles (dynamic LDS: ring + the layer's tile scales), items in
// XCD-aware order.
template <int FMT>
__global__ __launch_bounds__(kBlock) void k_gemm_a_ring(const LayerArgs a) {
  gemm_a_item<FMT, true>(a, xcd_item(blockIdx.x, gridDim.x), ftm_ring_lds, nullptr);
}

// ---------------------------------------------------------------- stage B (w2 -> slot buffer)
template <int WFMT>
__device__ void gemm_b_body(const LayerArgs& a, const ProjSlot& W, int n0, int m0, int cnt, const int32_t* list,
                            int shared_col, uint16_t* sA, uint16_t* sB) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int H = a.L.hidden, KP = a.KP;
  const Rsrc lres = make_rsrc(list, list ? (uint32_t)a.T * 4u : 0u);
  const Rsrc hres = make_rsrc(a.hbuf, (uint32_t)a.T * (uint32_t)KP * (uint32_t)a.Imax * 2u);
  const Rsrc wres = make_rsrc(a.wts, (uint32_t)a.T * (uint32_t)KP * 4u);
  uint32_t arow[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = pair_of_row(lres, list != nullptr, m0 + ((tid + kBlock * i) >> 3), cnt, KP, shared_col);
    arow[i] = p >= 0 ? (uint32_t)p * (uint32_t)a.Imax * 2u : kOOB;
  }
  int pe[2][4];
  float we[2][4];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      pe[mi][r] = pair_of_row(lres, list != nullptr, m0 + 32 * wm + 16 * mi + 4 * (lane >> 4) + r, cnt, KP,
                              shared_col);
      we[mi][r] = __uint_as_float(bload4(wres, pe[mi][r] >= 0 ? 4u * (uint32_t)pe[mi][r] : kOOB));
    }
  float bn[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + 32 * wn + 16 * j + (lane & 15);
    bn[j] = W.bias != nullptr ? load_scalar(W.bias, n, W.bias_dt) : 0.0f;
  }
  f32x4 acc[2][2];
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int nj = 0; nj < 2; ++nj) acc[mi][nj] = (f32x4){0.f, 0.f, 0.f, 0.f};
  gemm_tile<WFMT, 64>(W, n0, 0, hres, arow, sA, sB, acc);
#pragma unroll
  for (int mi = 0; mi < 2; ++mi)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + 32 * wn + 16 * j + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (pe[mi][r] >= 0) {
          float y = acc[mi][j][r];
          if (W.bias != nullptr) y += bn[j];
          a.ybuf[(size_t)pe[mi][r] * H + n] = y * we[mi][r];
        }
    }
}

template <int FMT>
__device__ __forceinline__ void gemm_b_item(const LayerArgs& a, int item, uint16_t* sA, uint16_t* sB) {
  const int H = a.L.hidden, Is = a.L.shared_inter;
  const int nRouted = a.ctrl[kCtrlNRouted];
  const int ntn = H / 64;
  const int routed_items = gemm_routed_mtiles(a, nRouted) * ntn;
  if (item < routed_items) {
    const GemmTile t = gemm_find_tile(a, item / ntn, nRouted, false);
    if (t.u < 0) return;
    const int e = a.uniq[t.u];
    const int32_t* list = a.lists + (size_t)e * a.T;
    const int slot = a.L.slot_of_expert ? a.L.slot_of_expert[e] : e;
    const int n0 = (item % ntn) * 64;
    if (slot < 0 || slot >= a.L.w2.num_slots) {
      // non-resident expert: its rows contribute zeros
      for (int idx = threadIdx.x; idx < kGM * 64; idx += kBlock) {
        const int m = t.m0 + idx / 64;
        if (m < t.cnt) a.ybuf[(size_t)list[m] * H + n0 + idx % 64] = 0.0f;
      }
      if (threadIdx.x == 0) atomicOr(&a.ctrl[kCtrlError], 1);
      return;
    }
    const ProjSlot W = proj_slot(a.L.w2, slot);
    gemm_b_body<FMT>(a, W, n0, t.m0, t.cnt, list, 0, sA, sB);
  } else if (Is > 0) {
    const int sitem = item - routed_items;
    const int m0 = (sitem / ntn) * kGM;
    if (m0 >= a.T) return;
    const ProjSlot W = shared_view(a.L.shared_w2, H, Is);
    gemm_b_body<FTM_FMT_BF16>(a, W, (sitem % ntn) * 64, m0, a.T, nullptr, a.L.topk, sA, sB);
  }
}

template <int FMT>
__global__ __launch_bounds__(kBlock) void k_gemm_b(const LayerArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t sA[2 * kGM * kGPitch];
  __shared__ __attribute__((aligned(16))) uint16_t sB[2 * 64 * kGPitch];
  gemm_b_item<FMT>(a, blockIdx.x, sA, sB);
}

// ---------------------------------------------------------------- launch
bool gemm_path_ok(const ftm_moe_layer& L, int T) {
  if (L.act_dtype != FTM_DT_BF16) return false;
  const int f = L.w13.fmt;
  if (f != FTM_FMT_FP8_BLOCK && f != FTM_FMT_INT8_PACKED && f != FTM_FMT_MXFP4 && f != FTM_FMT_BF16 && !tile_gptq_ok(L))
    return false;
  if (L.hidden % 64 != 0 || L.inter % 64 != 0 || (L.shared_inter > 0 && L.shared_inter % 64 != 0)) return false;
  if ((f == FTM_FMT_FP8_BLOCK || f == FTM_FMT_INT8_PACKED) &&
      (L.w13.group % kGK != 0 || L.w2.group % kGK != 0))
    return false;
  if (L.apply_router_weight_on_input) return false;
  // above the crossover: on average at least that many tokens per routed
  // expert (MXFP4: more than that, up to which its scaled-MFMA decode path wins)
  const long pairs = (long)T * L.topk;
  const long maxU = L.num_experts < pairs ? L.num_experts : pairs;
  if (f == FTM_FMT_MXFP4 && T <= kXlMaxTMx) return pairs > (long)kGemmMinRows * maxU;
  long rows = kGemmMinRows;
  if (f != FTM_FMT_MXFP4 && (mx_gemm_ok(L, T) || tile_bf16_ok(L, T)) && maxU * ((L.inter + 127) / 128) >= kGemmWideItems)
    rows = lean_shape(L) ? kGemmMinRowsLean : kGemmMinRowsWide;
  return pairs >= rows * maxU;
}

// Whether the ring tiles take this layer: weights whose tile scales fit the
// LDS scale area (INT8: one fp32 per tile row and group).
static bool ring_ok(const ftm_moe_layer& L) {
  const int f = L.w13.fmt;
  if (f == FTM_FMT_INT8_PACKED || f == FTM_FMT_FP8_BLOCK) {
    const long g13 = (L.hidden + L.w13.group - 1) / L.w13.group;
    if (f == FTM_FMT_INT8_PACKED && 128 * g13 * 4 > kRingScaleBytes) return false;
    if (f == FTM_FMT_FP8_BLOCK && 2 * g13 > kBlock) return false;  // one scale per thread
  }
  return true;
}

// Dynamic LDS of the ring kernels for this layer: ring + tile scales.
static size_t ring_lds_a(const ftm_moe_layer& L) {
  const int f = L.w13.fmt;
  const int g = (L.hidden + L.w13.group - 1) / (L.w13.group > 0 ? L.w13.group : 1);
  const int rows = f == FTM_FMT_FP8_BLOCK ? 2 : f == FTM_FMT_INT8_PACKED ? 128 : 0;
  return (size_t)kRingA + (size_t)rows * g * 4;
}

// FP8 between the wide crossover and 16 tokens per expert runs on the bf16
// tiles, which read the activations as the GEMV stages below do; the scaled
// tiles' two-term split keeps only what lies within 2^13 of a 32-block's
// largest (one channel of 128 at 1e6 that no weight reads: the layer is off by
// 0.1).  us a layer there, bf16 / scaled: 64 experts of 1024 at 4 / 15 tokens
// per expert 145 / 157 against 131 / 146, 256 of 512 at 9 / 16 220 / 233
// against 209 / 224.
bool mx_gemm_ok(const ftm_moe_layer& L, int T) {
  const long pairs = (long)T * L.topk;
  const long maxU = L.num_experts < pairs ? L.num_experts : pairs;
  return mx_fmt(L) && (L.w13.fmt != FTM_FMT_FP8_BLOCK || pairs >= kGemmMinRows * maxU);
}

const char* gemm_a_kernel_name(const ftm_moe_layer& L, int T) {
  return mx_gemm_ok(L, T) ? "k_gemm_mx" : tile_bf16_ok(L, T) ? "k_tile" : ring_ok(L) ? "k_gemm_a_ring" : "k_gemm_a";
}

template <int FMT>
static void ring_lds_attr() {
  static DeviceBits done;
  (void)allow_lds(done, reinterpret_cast<const void*>(&k_gemm_a_ring<FMT>), kRingA + kRingScaleBytes);
}

const char* gemm_b_kernel_name(const ftm_moe_layer& L, int T) {
  if (tile_bf16_ok(L, T)) return "k_tile";
  if (!mx_gemm_ok(L, T)) return "k_gemm_b";
  return tile_mxb_ok(L, T) ? "k_gemm_mxb_f8" : "k_gemm_mx";
}

template <int FMT>
static void launch_gemm_t(const LayerArgs& a, hipStream_t st, int which) {
  const ftm_moe_layer& L = a.L;
  const long pairs = (long)a.T * L.topk;
  const long maxU = L.num_experts < pairs ? L.num_experts : pairs;
  const long mt_routed = pairs / kGM + maxU + 1;
  const long mt_shared = L.shared_inter > 0 ? (a.T + kGM - 1) / kGM : 0;
  const long items_a = mt_routed * (L.inter / 64) + mt_shared * (L.shared_inter > 0 ? L.shared_inter / 64 : 0);
  const long items_b = (mt_routed + mt_shared) * (L.hidden / 64);
  // Stage A on the ring tiles where they apply (us a layer on MI355X, ring /
  // register-staged: 16 INT8 experts of 1024 with 64-wide groups at 256 / 1024
  // tokens 70 / 110 against 73 / 125, 64 of 2048 at 512 / 2048 468 / 936 against
  // 471 / 1087; 16 bf16 experts of 512 at 256 / 700 52.0 / 55.6 against 55.4 /
  // 57.5).  Stage B keeps the register-staged tiles: with K = I its tiles are a
  // few K steps long and 4 workgroups per CU beat the deeper ring (256 FP8
  // experts of 512, 2048 tokens, w2 259 us against 377).
  const bool ring = ring_ok(L);
  if (which & 1) {
    if (ring) {
      ring_lds_attr<FMT>();
      hipLaunchKernelGGL((k_gemm_a_ring<FMT>), dim3((unsigned)items_a), dim3(kBlock), ring_lds_a(L), st, a);
    } else {
      hipLaunchKernelGGL((k_gemm_a<FMT>), dim3((unsigned)items_a), dim3(kBlock), 0, st, a);
    }
  }
  if (which & 2) hipLaunchKernelGGL((k_gemm_b<FMT>), dim3((unsigned)items_b), dim3(kBlock), 0, st, a);
}

void launch_gemm_stages(const ftm_moe_layer& L, const void* x, int T, void* out, char* ws, const WsLayout& wl,
                        hipStream_t st, int which, bool xq_ready) {
  const LayerArgs a = make_args(L, x, out, T, ws, wl);
  if (mx_gemm_ok(L, T)) {
    // stage A over the quantised input, writing h quantised the same way for stage B
    if ((which & 1) && !xq_ready) launch_quant_mx(x, T, L.hidden, a.xq, st);
    launch_tile_mx(a, st, which);
    return;
  }
  if (tile_bf16_ok(L, T)) {
    launch_tile_bf16(a, st, which);
    return;
  }
  if (L.w13.fmt == FTM_FMT_FP8_BLOCK) launch_gemm_t<FTM_FMT_FP8_BLOCK>(a, st, which);
  else if (L.w13.fmt == FTM_FMT_INT8_PACKED) launch_gemm_t<FTM_FMT_INT8_PACKED>(a, st, which);
  else launch_gemm_t<FTM_FMT_BF16>(a, st, which);
}

}  // namespace ftm
