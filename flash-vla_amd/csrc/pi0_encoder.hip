// Prefix-encoder kernels for gfx950: M = 768..816 token rows at width 2048.
//
// At these shapes the GEMMs are MFMA-bound (2 * 768 * 2048 * 32768 flops for the
// gated FFN alone), so the design is the classic LDS-tiled one:
//   * tile_gemm_kernel<BM, BN, EPI, DUAL>: 4 waves in a 2 x 2 grid, BM x BN
//     output block, K consumed 64 at a time through a ring of steps. A (row-major
//     activations) goes to LDS in whole 128-byte step rows, 16-byte chunks
//     XOR-swizzled by row; B is the packed weight stream, already in MFMA
//     fragment order. One barrier per 64-deep step.
//   * tiles are assigned so that the workgroups dispatched to one XCD (the
//     hardware deals workgroups round-robin over the 8 XCDs) cover consecutive
//     tiles -- all row blocks of a weight column block, or of a group of them
//     where the rows are many (tile_group) -- so each weight block
//     is read into one XCD's L2 once.
//   * split-K (ffn-down, K = 16384) writes fp32 partials and a second launch
//     sums them in split order and applies the residual epilogue.
// Epilogues (reference file:line, backends/tilelang/):
//   TE_STORE     C                      plain projection
//   TE_BIAS      C + b                  encoder_projector GEMM (wrappers.py:336-344)
//   TE_RES       out += C               encoder o-proj / ffn-down (wrappers.py:366-392)
//   TE_GATE      gelu(C_g) * C_u        encoder gated FFN (kernels/base.py:508-549)
//   TE_QKV_ROPE  bf16(C), RoPE on the rounded values, scatter Q / K / V
//                                       (kernels/base.py:672-726)
//   TE_PARTIAL   fp32 split-K partial
//   TE_BIAS_RES  C + b + R               vision o-proj / ffn-down / patch embedding
//                                       (kernels/base.py:197-270)
//   TE_BIAS_GELU gelu_tanh(C + b)        vision ffn-up (kernels/base.py:273-300)
#include "pi0_common.h"
#include "pi0_hip.h"

#include <algorithm>
#include <cmath>
#include <initializer_list>

namespace pi0 {

enum TileEpi {
  TE_STORE = 0, TE_BIAS = 1, TE_RES = 2, TE_GATE = 3, TE_QKV_ROPE = 4, TE_PARTIAL = 5,
  TE_BIAS_RES = 6,    // C + b + R[row % res_mod or row]   (vision residual GEMMs, patch embedding)
  TE_BIAS_GELU = 7    // gelu_tanh(C + b)                   (vision FFN up)
};

struct TileArgs {
  const __bf16* a; int lda;
  const __bf16* w0; const __bf16* w1;   // packed B fragments ([nt][kt] tiles of 32 k x 16 n)
  const __bf16* bias;
  __bf16* out; int ldo;
  __bf16* out_k; __bf16* out_v; int ldkv;
  const __bf16* rope;
  float* part;                          // TE_PARTIAL: [splitk][M][N] fp32
  const __bf16* res; int ldres, res_mod;  // TE_BIAS_RES residual (may alias out); res_mod 0 = row
  int n_valid;                          // output columns stored (<= N; the rest is padding)
  int rows_per_batch;                   // TE_QKV_ROPE: prefix rows per request (RoPE position
  long long kv_bstride;                 //   = row % rows_per_batch), cache stride per request
  int M, N, K;                          // N, K = the packed (padded) weight's shape
  int tiles_m, tiles_n, splitk, ksteps; // ksteps = 64-deep steps per split
  int heads, head_dim;
  int xcd_remap;
  int group;                            // column tiles per group of the tile order (tile_of)
};

// Row and column tile (and K split) of tile index `id`, the order in which an XCD's workgroups
// take them: groups of a.group column tiles, row by row inside a group. The 32 tiles that an
// XCD works on at a time then draw about as many bytes of rows as of columns through its L2.
// (A group of one is all row tiles of a column tile: with 26 of those every XCD streams all of
// the activations.)
__device__ __forceinline__ void tile_of(const TileArgs& a, int id, int& mt, int& nt, int& ks) {
  const int all = a.tiles_m * a.tiles_n, per = a.tiles_m * a.group;
  ks = id / all;
  id -= ks * all;
  const int g = id / per, rem = id - g * per, w = min(a.group, a.tiles_n - g * a.group);
  mt = rem / w;
  nt = g * a.group + rem - mt * w;
}


__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Epilogue of 8 consecutive columns col .. col + 7 of output row grow: v holds the fp32
// products, b8 / r8 the bias and residual pieces (where the form has them).
template <int EPI>
__device__ __forceinline__ void tile_store(const TileArgs& a, int grow, int col, float* v, bf16x8 b8,
                                           bf16x8 r8) {
  __bf16* dst;
  if constexpr (EPI == TE_QKV_ROPE) {
    const int hd = a.head_dim, qdim = a.heads * hd;
    const int bq = grow / a.rows_per_batch, tq = grow - bq * a.rows_per_batch;
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = round_bf(v[q]);
    if (col < qdim + hd) {          // rotate the rounded pairs (2p, 2p + 1)
      const bf16x8 rp = load8(a.rope + (size_t)tq * hd + (col % hd));
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const float cs_ = bf2f(rp[2 * p]), sn = bf2f(rp[2 * p + 1]);
        const float x0 = v[2 * p], x1 = v[2 * p + 1];
        v[2 * p] = x0 * cs_ - x1 * sn;
        v[2 * p + 1] = x1 * cs_ + x0 * sn;
      }
    }
    const size_t kv = (size_t)bq * a.kv_bstride + (size_t)tq * a.ldkv;
    if (col < qdim) dst = a.out + (size_t)grow * qdim + col;
    else if (col < qdim + hd) dst = a.out_k + kv + (col - qdim);
    else dst = a.out_v + kv + (col - qdim - hd);
  } else {
    dst = a.out + (size_t)grow * a.ldo + col;
    if constexpr (EPI == TE_BIAS) {
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] += bf2f(b8[q]);
    }
    if constexpr (EPI == TE_RES) {
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] += bf2f(r8[q]);
    }
    if constexpr (EPI == TE_BIAS_RES || EPI == TE_BIAS_GELU) {
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] += bf2f(b8[q]);
    }
    if constexpr (EPI == TE_BIAS_RES) {
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] += bf2f(r8[q]);
    }
    if constexpr (EPI == TE_BIAS_GELU) {
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = gelu_tanh_rcp(v[q]);
    }
  }
  bf16x8 o;
#pragma unroll
  for (int q = 0; q < 8; ++q) o[q] = f2bf(v[q]);
  *reinterpret_cast<bf16x8*>(dst) = o;
}

// v_mfma_f32_32x32x16_bf16 is used because one wave per SIMD sustains ~90% of the
// MFMA peak with it (the 16x16x32 form stalls near 55-60% at this occupancy).
// Fragment layouts (lane l, j = 0..7, e = 0..15):
//   A (32 rows x 16 k): A[l % 32][8 (l / 32) + j]
//   B (16 k x 32 cols): B[8 (l / 32) + j][l % 32]      (pi0hip_pack_weight32 order)
//   C (32 x 32):        C[8 (e / 4) + 4 (l / 32) + e % 4][l % 32]
//
// Workgroup = 4 waves side by side along N; each wave owns all BM rows of the
// block and WN of its B columns. Both operands run D 64-deep steps ahead:
//   * A (activations, shared by the 4 waves) goes global -> LDS directly
//     (buffer_load ... lds, 16 bytes per lane) into a D-slot ring; the buffer
//     resource ends at row M so the rows of a ragged last block load as zeros.
//     An instruction reads 8 rows x 128 bytes, whole cache lines: reading one
//     32 x 16 fragment instead (32 lines, 32 bytes of each, every line touched by
//     four instructions) held the load path back. Encoder down at M = 768 71.6 ->
//     58.8 us, o-proj 18.4 -> 15.4, vision QKV 14.2 -> 11.8, FFN-up 20.8 -> 18.0;
//     vision at 3072 rows QKV 47.6 -> 36.2, FFN-down 54.8 -> 43.9. The swizzle
//     (chunk c of row r sits at c ^ (r / 2 % 8)) puts the fragment reads of 16
//     neighbouring rows on distinct 16-byte slots of LDS's 64 banks: fragments read
//     at 448 bytes a nanosecond per CU, as fast as linear ones, against 287 with
//     c ^ (r % 8), where 16 rows meet on 8 slots (down 58.8 -> 57.4 us);
//   * B (the packed weight stream, private to the wave) goes global -> VGPRs
//     into a D-slot register ring, so no weight byte passes through LDS.
// The step count is a multiple of D (the host checks), so the ring unrolls with
// static slots; every step issues the same number of loads (steps past the end
// re-load the last step into the free slot), so "A of step s has landed" is the
// fixed count vmcnt <= LB + (D - 2) * (LA + LB) of loads issued after it; a plain
// s_barrier (no fence: the fence would wait for every prefetch) then publishes it.
//
// RMS = 1 fuses the decoder's RMS pre-norm for its batched gated FFN (fused_norm.py:26-78):
// the block sees every k of its rows, so each row's sum of squares is accumulated from
// the A fragments it already reads (v_dot2 on bf16 pairs; row tile i by wave i % 4),
// f = bf16(rsqrt(mean(x^2) + 1e-6)) goes to LDS and the epilogue forms
// gelu(f * x@Wg) * (f * x@Wu) from the fp32 accumulators.
template <int BM, int WN, int D, int EPI, bool DUAL, int OCC, int RMS = 0>
__global__ __launch_bounds__(256, OCC) void tile_gemm_kernel(TileArgs a) {
  constexpr int BN = 4 * WN;               // B columns per workgroup
  constexpr int FM = BM / 32;              // 32-row fragments (every wave holds all rows)
  constexpr int FN = WN / 32;              // 32-column B tiles per wave
  constexpr int TA = FM * 4;               // A fragments per 64-deep step (4 x k16)
  constexpr int LA = TA / 4;               // ... loaded by each wave
  constexpr int LB = FN * 4;               // B fragments per wave per step
  constexpr int AWAIT = LB + (D - 2) * (LA + LB);
  constexpr int PF = 3;                    // A-fragment register ring
  static_assert(BM % 32 == 0 && WN % 32 == 0 && (!DUAL || WN % 64 == 0), "tile shape");
  static_assert(D >= 2 && AWAIT < 64, "pipeline depth");
  constexpr int OUTC = DUAL ? BN / 2 : BN;           // output columns of the block
  constexpr int CP = OUTC + 4;                       // fp32 pitch of the parked tile
  constexpr int RING = D * TA * 64;                  // 16-byte slots of the operand ring
  constexpr int PARK = (BM * CP * 4 + 15) / 16;
  __shared__ bf16x8 lds[RING > PARK ? RING : PARK];
  __shared__ float rms_f[RMS ? BM : 1];

  PI0_PROBE(0);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  float ssr[FM];
#pragma unroll
  for (int i = 0; i < FM; ++i) ssr[i] = 0.f;
  int id = blockIdx.x;
  if (a.xcd_remap) id = (id & 7) * (gridDim.x >> 3) + (id >> 3);
  int mt, ntile, ks;
  tile_of(a, id, mt, ntile, ks);
  const int m0 = mt * BM;
  const int KT = a.K >> 4;                 // 16-deep k tiles
  const int step0 = ks * a.ksteps, nsteps = a.ksteps;

  const int arows = max(min(BM, a.M - m0), 0);
  const __amdgpu_buffer_rsrc_t ar =
      rows_rsrc_sgpr(a.a + (size_t)m0 * a.lda, arows * a.lda * (int)sizeof(__bf16));
  // copy i of wave w covers block rows (4 i + w) * 8 .. + 7 whole 128-byte step rows (full
  // cache lines); LDS word (row, c) receives the row's 16-byte chunk c ^ (row / 2 % 8)
  const int aoff = ((wave * 8 + (lane >> 3)) * a.lda +
                    ((lane & 7) ^ ((wave & 1) * 4 + (lane >> 4))) * 8) * (int)sizeof(__bf16);
  const int arow_step = 32 * a.lda * (int)sizeof(__bf16);
  // ... so this lane's piece of A fragment (row tile i, slice kq) is word i * 256 + (afrag ^ 2 kq)
  const int afrag = (lane & 31) * 8 + ((lane >> 5) ^ ((lane >> 1) & 7));
  // this wave's 32-column B tiles: for the gated FFN, FN / 2 gate tiles then FN / 2 up tiles
  const __bf16* bptr[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    if constexpr (DUAL) {
      const int half = FN / 2, jj = j < half ? j : j - half;
      const int ntg = ntile * (BN / 64) + wave * half + jj;
      bptr[j] = (j < half ? a.w0 : a.w1) + (size_t)ntg * KT * 512 + lane * 8;
    } else {
      const int ntg = ntile * (BN / 32) + wave * FN + j;
      bptr[j] = a.w0 + (size_t)ntg * KT * 512 + lane * 8;
    }
  }

  // the epilogue's bias / residual pieces (8 columns of a row per thread and pass) do not
  // depend on the product: they are loaded right after the ring's first steps are issued
  // and land while the k loop runs
  constexpr int C8 = OUTC / 8, NEP = (BM * C8 + 255) / 256;
  constexpr bool EB = EPI == TE_BIAS || EPI == TE_BIAS_RES || EPI == TE_BIAS_GELU;
  constexpr bool ER = EPI == TE_RES || EPI == TE_BIAS_RES;
  bf16x8 epb[EB ? NEP : 1], epr[ER ? NEP : 1];
  bf16x8 breg[D][FN][4];
  auto issue = [&](int s, int slot) {
    const int st = min(s, nsteps - 1) + step0;   // past the end: a harmless re-load
    const int abase = st * 64 * (int)sizeof(__bf16);
#pragma unroll
    for (int i = 0; i < LA; ++i)
      buf_load16_lds_u(ar, &lds[(slot * TA + i * 4 + wave) * 64], aoff, abase + i * arow_step);
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int kq = 0; kq < 4; ++kq) breg[slot][j][kq] = load8(bptr[j] + ((size_t)st * 4 + kq) * 512);
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

#pragma unroll
  for (int u = 0; u < D - 1; ++u) issue(u, u);
  if constexpr (EB || ER) {
    // unconditional loads through bounded resources (pieces past the end read as zeros and
    // are never stored), so no divergent branch makes the compiler wait on the ring above
    const __amdgpu_buffer_rsrc_t br = rows_rsrc_sgpr(a.bias, EB ? a.n_valid * (int)sizeof(__bf16) : 0);
    const int rrows = EPI == TE_RES ? a.M : (a.res_mod ? a.res_mod : a.M);
    const int rld = EPI == TE_RES ? a.ldo : a.ldres;
    const __amdgpu_buffer_rsrc_t rr =
        rows_rsrc_sgpr(EPI == TE_RES ? (const void*)a.out : (const void*)a.res,
                       ER ? rrows * rld * (int)sizeof(__bf16) : 0);
#pragma unroll
    for (int k = 0; k < NEP; ++k) {
      const int idx = t + 256 * k, row = idx / C8, c = (idx - row * C8) * 8;
      const int grow = m0 + row, col = ntile * OUTC + c;
      const bool in = idx < BM * C8;
      if constexpr (EB) epb[k] = buf_load8(br, in ? col * (int)sizeof(__bf16) : INT_MAX - 64);
      if constexpr (ER) {
        const int rrow = EPI == TE_BIAS_RES && a.res_mod ? grow % a.res_mod : grow;
        epr[k] = buf_load8(rr, in && rrow < rrows ? (rrow * rld + col) * (int)sizeof(__bf16) : INT_MAX - 64);
      }
    }
  }

  PI0_PROBE(1);

  for (int s0 = 0; s0 < nsteps; s0 += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const int s = s0 + u;
      __builtin_amdgcn_s_waitcnt(PI0_VMCNT(AWAIT));
      __builtin_amdgcn_s_barrier();
      PI0_PROBE(8 + s);
      issue(s + D - 1, (u + D - 1) % D);
      // A fragments through a PF-deep register ring (f = kq * FM + i): the read of
      // fragment f + PF - 1 is issued before the MFMAs of fragment f.
      const bf16x8* st = lds + u * TA * 64;
      bf16x8 ap[PF];
#pragma unroll
      for (int p = 0; p < PF - 1; ++p) ap[p] = st[(p % FM) * 256 + (afrag ^ (p / FM * 2))];
#pragma unroll
      for (int f = 0; f < 4 * FM; ++f) {
        const int kq = f / FM, i = f % FM;
        if (f + PF - 1 < 4 * FM) {
          const int fn = f + PF - 1;
          ap[(f + PF - 1) % PF] = st[(fn % FM) * 256 + (afrag ^ (fn / FM * 2))];
        }
        __builtin_amdgcn_sched_barrier(0);   // keep the prefetch ahead of these MFMAs
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = mfma32(ap[f % PF], breg[u][j][kq], acc[i][j]);
        if constexpr (RMS) {
          if (wave == (i & 3)) {
            typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
            const bf16x8 v = ap[f % PF];
#pragma unroll
            for (int p = 0; p < 4; ++p) {
              const bf16x2_t q = {v[2 * p], v[2 * p + 1]};
              ssr[i] = __builtin_amdgcn_fdot2_f32_bf16(q, q, ssr[i], false);
            }
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  PI0_PROBE(2);
  __builtin_amdgcn_s_waitcnt(PI0_VMCNT(0));   // drain the dummy tail loads before exit
  if constexpr (RMS) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if (wave != (i & 3)) continue;
      const float ss = ssr[i] + __shfl_xor(ssr[i], 32);    // the two k halves of row lane % 32
      if (lane < 32) rms_f[i * 32 + lane] = round_bf(rsqrtf(ss / (float)a.K + 1e-6f));
    }
  }

  // ---- epilogue through LDS (the ring is free now): the waves park their fp32 tiles
  // row-major, then every thread finishes 8 consecutive output columns of a row with
  // 16-byte loads and stores (residual, RoPE table, outputs, split-K partials).
  // Lane holds C[8 (e / 4) + 4 (lane / 32) + e % 4][lane % 32] of each fragment.
  __syncthreads();
  float* cs = reinterpret_cast<float*>(lds);
  {
    const int r = lane & 31, h = lane >> 5;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = i * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
        if constexpr (DUAL) {
          const float fr = RMS ? rms_f[row] : 1.f;
#pragma unroll
          for (int j = 0; j < FN / 2; ++j)
            cs[row * CP + (wave * (FN / 2) + j) * 32 + r] =
                RMS ? gelu_tanh(fr * acc[i][j][e]) * (fr * acc[i][FN / 2 + j][e])
                    : gelu_tanh_rcp(acc[i][j][e]) * acc[i][FN / 2 + j][e];
        } else {
#pragma unroll
          for (int j = 0; j < FN; ++j) cs[row * CP + (wave * FN + j) * 32 + r] = acc[i][j][e];
        }
      }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NEP; ++k) {
    const int idx = t + 256 * k;
    if (idx >= BM * C8) continue;
    const int row = idx / C8, c = (idx - row * C8) * 8;
    const int grow = m0 + row;
    if (grow >= a.M) continue;
    const f32x4 lo = *reinterpret_cast<const f32x4*>(&cs[row * CP + c]);
    const f32x4 hi = *reinterpret_cast<const f32x4*>(&cs[row * CP + c + 4]);
    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    const int col = ntile * OUTC + c;
    if (col >= a.n_valid) continue;            // padded weight columns
    if constexpr (EPI == TE_PARTIAL) {
      float* dst = a.part + ((size_t)ks * a.M + grow) * a.N + col;
      *reinterpret_cast<f32x4*>(dst) = lo;
      *reinterpret_cast<f32x4*>(dst + 4) = hi;
      continue;
    }
    tile_store<EPI>(a, grow, col, v, epb[EB ? k : 0], epr[ER ? k : 0]);
  }
  PI0_PROBE(3);
}

// ---- 8-wave blocks, both operands staged in LDS ------------------------------------------
// Workgroup = WMC x WNC waves over WMC FM 32 rows x WNC FN 32 packed B columns (DUAL: half of
// them gate, half the matching up columns); wave (wm, wn) owns FM x FN fragments. Steps are
// 32 deep in a ring of D slots (256 x 256: 32 KB each, three steps in flight while one is
// multiplied). A instructions copy 16 rows x 64 bytes, B instructions one packed fragment.
// Two things set the pace beside the MFMAs, and the loop is built around them:
//   * the load path takes a copy in tens of clocks, so a burst of a step's copies blocks the
//     waves that should be multiplying: half of a step's copies go out between the MFMAs of
//     each k16 slice (256 x 256, K 2048: 87.5 -> 80.2k clocks, the MFMAs alone 65.5k);
//   * a slice's fragments are read while the one before it is multiplied, into a second set
//     of registers, across the step's barrier too: the barrier stands before the last slice,
//     whose fragments are in registers, so it has MFMAs queued on both sides. Past it the
//     step's slot is free for the step D - 1 ahead.
// The k order of every accumulation is the strip kernel's: bitwise-equal products.
template <int WMC, int WNC, int FM, int FN, int EPI, bool DUAL>
__global__ __launch_bounds__(64 * WMC * WNC, 1) void block_gemm_kernel(TileArgs a) {
  constexpr int D = 4, NW = WMC * WNC;
  constexpr int BM = WMC * FM * 32, NBF = WNC * FN;      // rows, 32-column B fragments
  constexpr int HT = DUAL ? NBF / 2 : NBF;               // B fragment columns per weight
  constexpr int TA = BM / 16, TB = NBF * 2;              // copies of a step ...
  constexpr int CC = (TA + TB + NW - 1) / NW, CH = CC / 2;   // ... per wave, in the last slice
  // 16-byte LDS words: D slots of B, then D of A (fragment reads reach every B slot from one
  // address register)
  constexpr int SA = BM * 4, SB = NBF * 128, A0 = D * SB;
  constexpr int OUTC = DUAL ? NBF * 16 : NBF * 32, CP = OUTC + 4, C8 = OUTC / 8;
  constexpr int PR = WMC * 32;                           // rows parked per epilogue pass
  constexpr int PARK = (PR * CP * 4 + 15) / 16;
  constexpr int NEP = PR * C8 / (64 * NW);               // 8-column pieces per thread and pass
  static_assert(!DUAL || FN % 2 == 0, "gate and up tiles of one wave");
  static_assert(!DUAL || TA % NW == 0 || HT * 2 >= NW, "a mixed copy holds gate tiles only");
  static_assert(FM * FN >= CC - CH, "a slice's copies between its MFMAs");
  static_assert(NEP * 64 * NW == PR * C8 && BM % 16 == 0, "tile shape");
  __shared__ bf16x8 lds[D * (SA + SB) > PARK ? D * (SA + SB) : PARK];

  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave / WNC, wn = wave % WNC;
  // XCD-contiguous tile order for any grid: workgroup b runs on XCD b % 8
  int id;
  {
    const int b = blockIdx.x, x = b & 7, q = gridDim.x >> 3, r = gridDim.x & 7;
    id = x * q + min(x, r) + (b >> 3);
  }
  int mt, ntile, ks;
  tile_of(a, id, mt, ntile, ks);
  const int m0 = mt * BM, KT = a.K >> 4, nsteps = a.ksteps, step0 = ks * a.ksteps;

  const int arows = max(min(BM, a.M - m0), 0);
  const __amdgpu_buffer_rsrc_t ar =
      rows_rsrc_sgpr(a.a + (size_t)m0 * a.lda, arows * a.lda * (int)sizeof(__bf16));
  const int btile = KT * 512 * (int)sizeof(__bf16);
  const __amdgpu_buffer_rsrc_t gr =
      rows_rsrc_sgpr(a.w0 + (size_t)ntile * HT * KT * 512, HT * btile);
  const __amdgpu_buffer_rsrc_t ur =
      rows_rsrc_sgpr((DUAL ? a.w1 : a.w0) + (size_t)ntile * HT * KT * 512, HT * btile);
  // A copy: row 16 q + lane / 4, LDS chunk lane % 4 of the row's four; chunk c of row r sits
  // at c ^ (r / 4 % 4), so the fragment reads of 16 neighbouring rows hit distinct banks
  const int avoff = ((lane >> 2) * a.lda + ((lane & 3) ^ (lane >> 4)) * 8) * (int)sizeof(__bf16);
  const int afrag = (lane & 31) * 4 + ((lane >> 5) ^ ((lane >> 2) & 3));
  const int bvoff = lane * 16, arow16 = 16 * a.lda * (int)sizeof(__bf16);
  // copy i of this wave for step s: A rows first, then B fragments (tile q / 2, slice q % 2);
  // a count that the waves do not divide repeats the last fragment
  auto copy = [&](int s, int slot, int i) {
    const int st = min(s, nsteps - 1) + step0;           // past the end: a harmless re-load
    const int q = min(i * NW + wave, TA + TB - 1);
    const int qb = q - TA, tile = qb >> 1;
    const bool isa = q < TA, up = DUAL && tile >= HT;
    const int soff = isa ? st * 64 + q * arow16
                         : st * 2048 + (qb & 1) * 1024 + (up ? tile - HT : tile) * btile;
    bf16x8* const da = &lds[A0 + slot * SA + q * 64];
    bf16x8* const db = &lds[slot * SB + qb * 64];
    if (i * NW + NW <= TA)
      buf_load16_lds_u(ar, da, avoff, soff);
    else if (i * NW >= TA)
      buf_load16_lds_u(up ? ur : gr, db, bvoff, soff);
    else                                                 // both kinds: B's first tiles
      buf_load16_lds_u(isa ? ar : gr, isa ? da : db, isa ? avoff : bvoff, soff);
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // fragment sets: A two, B two where the accumulators leave the registers for it; else B's
  // next fragment follows each column's last MFMA into the same registers
  constexpr bool B2 = FM * FN <= 10;
  bf16x8 fa[2][FM], fb[B2 ? 2 : 1][FN];
  auto read_a = [&](int slot, int kq, int b) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
      fa[b][i] = lds[A0 + slot * SA + (wm * FM + i) * 128 + (afrag ^ (kq * 2))];
  };
  auto read_b = [&](int slot, int kq, int b, int j) {
    const int tile = DUAL ? (j < FN / 2 ? 0 : HT) + wn * (FN / 2) + j % (FN / 2) : wn * FN + j;
    fb[B2 ? b : 0][j] = lds[slot * SB + (tile * 2 + kq) * 64 + lane];
  };
  // one slice: read the next one's fragments (slot rs, slice b ^ 1), multiply set b, with
  // copies c0 .. c1 - 1 of step s spread between the MFMAs
  auto slice = [&](int b, int rs, int s, int slot, int c0, int c1) {
    constexpr int EV = FM * FN / (CC - CH) > 0 ? FM * FN / (CC - CH) : 1;
    read_a(rs, b ^ 1, b ^ 1);
    if constexpr (B2) {
#pragma unroll
      for (int j = 0; j < FN; ++j) read_b(rs, b ^ 1, b ^ 1, j);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const int n = j * FM + i;
        acc[i][j] = mfma32(fa[b][i], fb[B2 ? b : 0][j], acc[i][j]);
        if (n % EV == EV / 2 && c0 + n / EV < c1) {
          __builtin_amdgcn_sched_barrier(0);
          copy(s, slot, c0 + n / EV);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if constexpr (!B2) {
        __builtin_amdgcn_sched_barrier(0);
        read_b(rs, b ^ 1, 0, j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

#pragma unroll
  for (int u = 0; u < D; ++u)
#pragma unroll
    for (int c = 0; c < (u < D - 1 ? CC : CH); ++c) copy(u, u, c);
  __builtin_amdgcn_s_waitcnt(PI0_VMCNT((D - 2) * CC + CH));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read_a(0, 0, 0);
#pragma unroll
  for (int j = 0; j < FN; ++j) read_b(0, 0, 0, j);
  for (int s0 = 0; s0 < nsteps; s0 += D) {
#pragma unroll
    for (int p = 0; p < D; ++p) {
      const int s = s0 + p;
      slice(0, p, s + D - 1, (p + D - 1) % D, CH, CC);   // the rest of that step's copies
      // this wave's copies of step s + 1 have landed and its reads of step s are done; past
      // the barrier the same holds for every wave
      __builtin_amdgcn_s_waitcnt(PI0_VMCNT((D - 2) * CC) & ~(0xF << 8));
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      slice(1, (p + 1) % D, s + D, p, 0, CH);
    }
  }

  // ---- epilogue, FM passes of one row fragment of every wave: fp32 parked row-major, then 8
  // columns of a row per thread with 16-byte loads and stores
  __builtin_amdgcn_s_waitcnt(PI0_VMCNT(0));              // drain the harmless re-loads
  constexpr bool EB = EPI == TE_BIAS || EPI == TE_BIAS_RES || EPI == TE_BIAS_GELU;
  constexpr bool ER = EPI == TE_RES || EPI == TE_BIAS_RES;
  const __amdgpu_buffer_rsrc_t br = rows_rsrc_sgpr(a.bias, EB ? a.n_valid * (int)sizeof(__bf16) : 0);
  const int rrows = EPI == TE_RES ? a.M : (a.res_mod ? a.res_mod : a.M);
  const int rld = EPI == TE_RES ? a.ldo : a.ldres;
  const __amdgpu_buffer_rsrc_t rr =
      rows_rsrc_sgpr(EPI == TE_RES ? (const void*)a.out : (const void*)a.res,
                     ER ? rrows * rld * (int)sizeof(__bf16) : 0);
  float* cs = reinterpret_cast<float*>(lds);
  const int r = lane & 31, h = lane >> 5;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    bf16x8 epb[EB ? NEP : 1], epr[ER ? NEP : 1];
#pragma unroll
    for (int k = 0; k < NEP; ++k) {
      const int idx = t + 64 * NW * k, prow = idx / C8, col = ntile * OUTC + (idx - prow * C8) * 8;
      const int grow = m0 + (prow >> 5) * (FM * 32) + i * 32 + (prow & 31);
      if constexpr (EB) epb[k] = buf_load8(br, col * (int)sizeof(__bf16));
      if constexpr (ER) {
        const int rrow = EPI == TE_BIAS_RES && a.res_mod ? grow % a.res_mod : grow;
        epr[k] = buf_load8(rr, rrow < rrows ? (rrow * rld + col) * (int)sizeof(__bf16) : INT_MAX - 64);
      }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      float* row = cs + (wm * 32 + 8 * (e >> 2) + 4 * h + (e & 3)) * CP + r;
      if constexpr (DUAL) {
#pragma unroll
        for (int j = 0; j < FN / 2; ++j)
          row[(wn * (FN / 2) + j) * 32] = gelu_tanh_rcp(acc[i][j][e]) * acc[i][FN / 2 + j][e];
      } else {
#pragma unroll
        for (int j = 0; j < FN; ++j) row[(wn * FN + j) * 32] = acc[i][j][e];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NEP; ++k) {
      const int idx = t + 64 * NW * k, prow = idx / C8, c = (idx - prow * C8) * 8;
      const int grow = m0 + (prow >> 5) * (FM * 32) + i * 32 + (prow & 31);
      const int col = ntile * OUTC + c;
      if (grow >= a.M || col >= a.n_valid) continue;     // ragged rows, padded weight columns
      const f32x4 lo = *reinterpret_cast<const f32x4*>(&cs[prow * CP + c]);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(&cs[prow * CP + c + 4]);
      if constexpr (EPI == TE_PARTIAL) {
        float* dst = a.part + ((size_t)ks * a.M + grow) * a.N + col;
        *reinterpret_cast<f32x4*>(dst) = lo;
        *reinterpret_cast<f32x4*>(dst + 4) = hi;
      } else {
        float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        tile_store<EPI>(a, grow, col, v, epb[EB ? k : 0], epr[ER ? k : 0]);
      }
    }
  }
}

// ---- residual GEMM of a few hundred rows: 32 x 32 outputs over the whole K ----------------
// out += x @ W for the batched decoder's o-proj and down (M = 204, N = 1024): as tiles of any
// size these are too few to fill the chip without splitting K over workgroups, and the split
// pays a second launch for its sum. Here the 8 waves of a workgroup split K and are summed
// through LDS. What bounds it is the CU's load path, (32 + 32) K values per workgroup, so all
// of it is asked for at once: each wave copies its x slice to LDS (whole 128-byte lines, four
// 64-deep chunks, refilled in place once) and reads its packed W fragments into registers,
// and multiplies a chunk as soon as the loads up to it have landed. The row blocks of a column
// tile sit on one XCD, which then reads that weight tile from HBM once.
template <int KT>     // k16 fragments per wave: K = 128 KT
__global__ __launch_bounds__(512, 1) void rows32_res_kernel(TileArgs a, int nrb, int xcd_map) {
  constexpr int NW = 8, NCH = KT / 4, SL = NCH < 4 ? NCH : 4;   // 64-deep chunks, LDS slots
  static_assert(KT % 4 == 0 && NCH <= 2 * SL && 4 * SL + KT < 64, "chunks in flight");
  __shared__ bf16x8 lds[NW * SL * 256];                        // 4 KB per chunk and wave
  static_assert(sizeof(float) * NW * 1024 <= sizeof(lds), "reduction area");
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int nt, rb;
  if (xcd_map) {            // column tiles congruent to the XCD index, all row blocks each
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
    nt = (j / nrb) * 8 + xcd;
    rb = j - (j / nrb) * nrb;
  } else {
    nt = blockIdx.x / nrb;
    rb = blockIdx.x - nt * nrb;
  }
  const int m0 = rb * 32, rows = min(32, a.M - m0);
  const __amdgpu_buffer_rsrc_t xr =
      rows_rsrc_sgpr(a.a + (size_t)m0 * a.lda, rows * a.lda * (int)sizeof(__bf16));
  // the residual pair this thread finishes (row t / 16, columns 2 (t % 16) ..): first, so that
  // every wait below covers it
  const __amdgpu_buffer_rsrc_t orr =
      rows_rsrc_sgpr(a.out + (size_t)m0 * a.ldo, rows * a.ldo * (int)sizeof(__bf16));
  const int ooff = ((t >> 4) * a.ldo + nt * 32 + (t & 15) * 2) * (int)sizeof(__bf16);
  const uint32_t res = __builtin_amdgcn_raw_buffer_load_b32(orr, ooff, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
  // chunk copies: 8 rows x 128 bytes an instruction, 16-byte chunk c of row r at c ^ (r / 2 % 8)
  bf16x8* const xs = lds + wave * SL * 256;
  const int kw0 = wave * KT * 16;
  const int xoff = ((lane >> 3) * a.lda + kw0) * (int)sizeof(__bf16);
  auto copy = [&](int c) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      buf_load16_lds_u(xr, xs + (c % SL) * 256 + i * 64,
                       xoff + ((lane & 7) ^ ((i & 1) * 4 + (lane >> 4))) * 16,
                       c * 128 + i * 8 * a.lda * (int)sizeof(__bf16));
  };
  const __bf16* wp = a.w0 + ((size_t)nt * (a.K >> 4) + wave * KT) * 512 + lane * 8;
  bf16x8 bv[KT];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    if (c < SL) copy(c);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) bv[c * 4 + i] = load8(wp + (c * 4 + i) * 512);
    __builtin_amdgcn_sched_barrier(0);
  }
  f32x16 acc[2];            // even and odd fragments: two chains
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[0][e] = acc[1][e] = 0.f;
  const int frag = (lane & 31) * 8 + ((lane >> 5) ^ ((lane >> 1) & 7));
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    // operations issued after chunk c's last: the later chunks' of the first pass, and the
    // refills issued so far
    constexpr int first = SL * 4 + KT;
    const int pos = c < SL ? 8 * (c + 1) : first + 4 * (c - SL + 1);
    const int issued = first + 4 * (NCH > SL ? min(c, NCH - SL) : 0);
    __builtin_amdgcn_sched_barrier(0);
    switch (issued - pos) {         // folds to one wait once the loop is unrolled
#define PI0_W(n) case n: __builtin_amdgcn_s_waitcnt(PI0_VMCNT(n)); break;
      PI0_W(0) PI0_W(4) PI0_W(8) PI0_W(12) PI0_W(16) PI0_W(20) PI0_W(24) PI0_W(28) PI0_W(32)
      PI0_W(36) PI0_W(40) PI0_W(44)
#undef PI0_W
      default: __builtin_amdgcn_s_waitcnt(PI0_VMCNT(0)); break;
    }
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 av[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) av[i] = xs[(c % SL) * 256 + (frag ^ (i * 2))];
    if (c + SL < NCH) {             // this wave's own slot: free once its reads are done
      __builtin_amdgcn_s_waitcnt(0xC07F);                       // lgkmcnt(0)
      __builtin_amdgcn_sched_barrier(0);
      copy(c + SL);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i & 1] = mfma32(av[i], bv[c * 4 + i], acc[i & 1]);
  }
  __syncthreads();                  // every wave is done with its slice
  float (*red)[16][PI0_WAVE] = reinterpret_cast<float (*)[16][PI0_WAVE]>(lds);
#pragma unroll
  for (int e = 0; e < 16; ++e) red[wave][e][lane] = acc[0][e] + acc[1][e];
  __syncthreads();
  const int row = t >> 4, col = (t & 15) * 2;
  if (row >= rows) return;
  // C lane 32 h + col holds rows 8 (e / 4) + 4 h + e % 4
  const int e = (row >> 3) * 4 + (row & 3), l = ((row >> 2) & 1) * 32 + col;
  float v0 = 0.f, v1 = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float* p = &red[w][e][l];
    v0 += p[0];
    v1 += p[1];
  }
  const bf16x2 r2 = __builtin_bit_cast(bf16x2, res);
  const bf16x2 o = {f2bf(v0 + bf2f(r2[0])), f2bf(v1 + bf2f(r2[1]))};
  *reinterpret_cast<bf16x2*>(a.out + (size_t)(m0 + row) * a.ldo + nt * 32 + col) = o;
}

// W[batch][K][N] -> 32x32x16 B fragments: tile (nt, kt) of 16 k x 32 n is 64 lanes x 8 bf16,
// lane = (k % 16 / 8) * 32 + n % 32, element k % 8; tiles ordered [nt][kt].
// K_pad x N_pad (multiples of 16 / 32) with zeros outside the K x N source.
__global__ void pack_weight32_kernel(const __bf16* __restrict__ w, __bf16* __restrict__ p,
                                     int K, int N, int K_pad, int N_pad, long long total_frags) {
  const long long f = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= total_frags) return;
  const long long per = (long long)(K_pad / 16) * (N_pad / 32) * 64;
  const long long b = f / per;
  long long rem = f - b * per;
  const int lane = (int)(rem & 63);
  rem >>= 6;
  const int KT = K_pad / 16;
  const int kt = (int)(rem % KT), nt = (int)(rem / KT);
  const int n = nt * 32 + (lane & 31);
  const int k0 = kt * 16 + (lane >> 5) * 8;
  const __bf16* src = w + b * (long long)K * N + (long long)k0 * N + n;
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = (n < N && k0 + j < K) ? src[(long long)j * N] : __bf16(0.f);
  *reinterpret_cast<bf16x8*>(p + f * 8) = v;
}

// Split-K second pass: sum the partials in split order, add the residual, round once. The
// split count is a compile-time one so that all partials of a piece are requested together
// (0: any count).
template <int S>
__global__ __launch_bounds__(256) void tile_reduce_res_kernel(TileArgs a) {
  const int id = blockIdx.x * 256 + threadIdx.x;
  const int per_row = a.N >> 2;
  const int row = id / per_row, col = (id - row * per_row) * 4;
  if (row >= a.M) return;
  const float* src = a.part + (size_t)row * a.N + col;
  const size_t stride = (size_t)a.M * a.N;
  __bf16* dst = a.out + (size_t)row * a.ldo + col;
  const bf16x4 rv = *reinterpret_cast<const bf16x4*>(dst);
  f32x4 s = zero4();
  if constexpr (S > 0) {
    f32x4 p[S];
#pragma unroll
    for (int k = 0; k < S; ++k) p[k] = *reinterpret_cast<const f32x4*>(src + k * stride);
#pragma unroll
    for (int k = 0; k < S; ++k) s += p[k];
  } else {
    for (int k = 0; k < a.splitk; ++k) s += *reinterpret_cast<const f32x4*>(src + k * stride);
  }
  const bf16x4 o = {f2bf(s[0] + bf2f(rv[0])), f2bf(s[1] + bf2f(rv[1])),
                    f2bf(s[2] + bf2f(rv[2])), f2bf(s[3] + bf2f(rv[3]))};
  *reinterpret_cast<bf16x4*>(dst) = o;
}

// ---- encoder RMSNorm: out = bf16(x * rsqrt(mean(x^2) + 1e-6)), one wave per row
// (kernels/base.py:373-403; the Gemma 1 + w weight is folded into the next GEMM).
template <int CPL>   // 16-byte chunks per lane: K = CPL * 512
__global__ __launch_bounds__(256) void rms_norm_kernel(const __bf16* __restrict__ x, int ldx,
                                                       __bf16* __restrict__ out, int ldo, int M,
                                                       int K) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const __bf16* xr = x + (size_t)row * ldx;
  bf16x8 v[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) v[c] = load8(xr + (c * 64 + lane) * 8);
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CPL; ++c)
#pragma unroll
    for (int j = 0; j < 8; ++j) { const float f = bf2f(v[c][j]); ss += f * f; }
  ss = warp_sum(ss);
  const float f = rsqrtf(ss / (float)K + 1e-6f);
  __bf16* orow = out + (size_t)row * ldo;
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bf(bf2f(v[c][j]) * f);
    *reinterpret_cast<bf16x8*>(orow + (c * 64 + lane) * 8) = o;
  }
}

// ---- LayerNorm: out = bf16((x - mean) * rsqrt(E[x^2] - mean^2 + eps) * w + b), one wave
// per row, statistics in fp32 (kernels/base.py:405-447; the vision tower's final norm in
// encoder_projector, wrappers.py:336-344). K % 8 == 0, K <= 2048.
__global__ __launch_bounds__(256) void layer_norm_kernel(const __bf16* __restrict__ x, int ldx,
                                                         const __bf16* __restrict__ w,
                                                         const __bf16* __restrict__ b,
                                                         __bf16* __restrict__ out, int ldo, int M,
                                                         int K, float eps) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const int chunks = K >> 3;
  const __bf16* xr = x + (size_t)row * ldx;
  bf16x8 v[4], wv[4], bv[4];
  // the row and the affine parameters are requested together: one memory round trip
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int ch = c * 64 + lane;
    v[c] = ch < chunks ? load8(xr + ch * 8) : zero8();
    wv[c] = ch < chunks ? load8(w + ch * 8) : zero8();
    bv[c] = ch < chunks ? load8(b + ch * 8) : zero8();
  }
  float s = 0.f, ss = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int j = 0; j < 8; ++j) { const float f = bf2f(v[c][j]); s += f; ss += f * f; }
  }
  s = warp_sum(s);
  ss = warp_sum(ss);
  const float mean = s / (float)K;
  const float inv = rsqrtf(ss / (float)K - mean * mean + eps);
  __bf16* orow = out + (size_t)row * ldo;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int ch = c * 64 + lane;
    if (ch >= chunks) continue;
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = f2bf((bf2f(v[c][j]) - mean) * inv * bf2f(wv[c][j]) + bf2f(bv[c][j]));
    *reinterpret_cast<bf16x8*>(orow + ch * 8) = o;
  }
}

// ---- encoder multi-query attention (attention.py:29-34): every flat query row
// (token * heads + head) attends over all keys of the one KV head, no mask.
//
// Workgroup = 32 query rows; wave w takes the 32-key blocks b with b % 4 == w, so
// each K / V byte is read once per workgroup, straight from L2 into registers
// (no LDS staging, no barriers in the key loop). Per block, with 32x32x16 MFMAs:
//   S^T[32 keys][32 q] = K Q^T      A = K rows (16 B loads), B = Q^T (held all along)
//   online softmax per query in the log2 domain (the logits are rounded to bf16
//   first, as the reference's bf16 matmul output is); each lane owns one query
//   and 16 of its keys, the other 16 sit in lane ^ 32;
//   O^T[256 d][32 q] += V^T P^T     A = V^T (rows of the transposed V, pre-pass
//   below), B = P^T, which is exactly the S^T accumulator's layout once the key
//   slots of V^T are permuted the same way -- P never moves between lanes and
//   the per-query rescale is lane-local.
// The 4 waves' partial (m, l, O^T) are merged through LDS at the end.
constexpr int EA_HD = 256;

struct EncAttnArgs {
  const __bf16* q; int ldq;
  const __bf16* kp;                     // K in fragment order (see pack_kv_kernel)
  const __bf16* vp;                     // V^T in fragment order
  int ldvt;                             // keys zero-padded to a multiple of 64
  __bf16* out; int ldo;
  int rows, keys;                       // per request (grid.y = requests)
  float scale_log2;
  long long kv_bstride;                 // elements between two requests' K
};

// Attention pre-pass: K and V of one request in the order enc_attn_kernel's MFMA fragments
// read them, so every fragment load of the attention is one contiguous 1 KB per wave (from
// row-major K / V^T each 16-byte fragment sits on its own cache line). For 32-key block b:
//   kp[((b * 16 + kk) * 64 + l) * 8 ..]          = K[32 b + l % 32][16 kk + 8 (l / 32) ..]
//   vp[(((b * 8 + dt) * 2 + c) * 64 + l) * 8 ..] = V^T[32 dt + l % 32][slots 32 b + 16 c + 8 (l / 32) ..]
// where V^T's key slots follow, inside every 16-key chunk, the order the P^T operand uses,
// {0-3, 8-11, 4-7, 12-15}. Keys past `keys` (up to ldvt, a multiple of 64) are zero.
// One workgroup: a 64-key x 64-dim tile of K (copied) and of V (transposed through LDS).
__global__ __launch_bounds__(256) void pack_kv_kernel(const __bf16* __restrict__ k,
                                                      const __bf16* __restrict__ v, int ldkv,
                                                      __bf16* __restrict__ kp, __bf16* __restrict__ vp,
                                                      int ldvt, int keys, long long kv_bstride) {
  __shared__ __attribute__((aligned(16))) __bf16 tile[64][72];
  const int k0 = blockIdx.x * 64, d0 = blockIdx.y * 64;
  k += (size_t)blockIdx.z * kv_bstride;
  v += (size_t)blockIdx.z * kv_bstride;
  kp += (size_t)blockIdx.z * EA_HD * ldvt;
  vp += (size_t)blockIdx.z * EA_HD * ldvt;
  const int t = threadIdx.x;
  // 16-byte loads: key row kr, dims d0 + 8 c .. + 7 (keys past the end read as zeros)
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = t + 256 * j, kr = i >> 3, c = (i & 7) * 8, key = k0 + kr, d = d0 + c;
    const bool in = key < keys;
    const bf16x8 kx = in ? load8(k + (size_t)key * ldkv + d) : zero8();
    const bf16x8 vx = in ? load8(v + (size_t)key * ldkv + d) : zero8();
    const int l = ((d & 15) >> 3) * 32 + (key & 31);
    *reinterpret_cast<bf16x8*>(kp + (((size_t)(key >> 5) * 16 + (d >> 4)) * 64 + l) * 8) = kx;
    *reinterpret_cast<bf16x8*>(&tile[kr][c]) = vx;
  }
  __syncthreads();
  // V^T row d, storage slots s .. s + 7 (each slot's key permuted into the P^T order)
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int i = t + 256 * j, dr = i >> 3, c = (i & 7) * 8;
    bf16x8 o;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int kc = c + q, sl = kc & 15;
      const int key = (kc & ~15) + ((sl & 4) ? 8 : 0) + ((sl & 8) ? 4 : 0) + (sl & 3);
      o[q] = tile[key][dr];
    }
    const int d = d0 + dr, sl0 = k0 + c;                       // slot of o[0]
    const int l = ((sl0 & 15) >> 3) * 32 + (d & 31);
    const size_t frag = ((size_t)(sl0 >> 5) * 8 + (d >> 5)) * 2 + ((sl0 & 31) >> 4);
    *reinterpret_cast<bf16x8*>(vp + (frag * 64 + l) * 8) = o;
  }
}

__global__ __launch_bounds__(256, 1) void enc_attn_kernel(EncAttnArgs a) {
  constexpr int DP = EA_HD + 4;                        // fp32 pitch of a parked O row
  __shared__ __attribute__((aligned(16))) float ob[4][32][DP];   // per wave: O[q][d]; first Q^T
  __shared__ float ml[4][2][32];                       // per wave: m and l of each query

  PI0_PROBE(0);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int q0 = blockIdx.x * 32;
  {                                     // request blockIdx.y: its rows, K and V^T
    const int bq = blockIdx.y;
    a.q += (size_t)bq * a.rows * a.ldq;
    a.out += (size_t)bq * a.rows * a.ldo;
    a.kp += (size_t)bq * EA_HD * a.ldvt;
    a.vp += (size_t)bq * EA_HD * a.ldvt;
  }

  const int nblk = (a.keys + 31) / 32;
  const int mine = nblk > wave ? (nblk - wave + 3) / 4 : 0;     // blocks b = wave + 4 i
  // Staggered single buffers: V^T of block i is requested before its S^T MFMAs, and
  // K of block i + 1 right after them (into the registers they just consumed), so
  // each load has the other phase's 16 MFMAs to land.
  bf16x8 kf[16], vf[8][2];
  auto blk = [&](int i) { return wave + 4 * min(i, mine - 1); };   // past the end: re-load
  // fragment-ordered K / V^T: each fragment is one contiguous 1 KB wave load
  auto load_k = [&](int i) {
    const __bf16* src = a.kp + ((size_t)blk(i) * 16 * 64 + lane) * 8;
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) kf[kk] = load8(src + kk * 64 * 8);
  };
  auto load_v = [&](int i) {
    const __bf16* src = a.vp + ((size_t)blk(i) * 16 * 64 + lane) * 8;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int c = 0; c < 2; ++c) vf[dt][c] = load8(src + (dt * 2 + c) * 64 * 8);
  };
  if (mine > 0) load_k(0);                  // block 0's K is in flight during the Q staging

  // Q^T fragments (B operand, 16 d each; lane holds Q[q0 + r][16 kk + 8 h .. + 7]) are
  // shared by the 4 waves: staged once in LDS (in the merge buffer's space)
  bf16x8* qs = reinterpret_cast<bf16x8*>(&ob[0][0][0]);    // [16 kk][64 lanes]
  {
    const __amdgpu_buffer_rsrc_t qr =
        rows_rsrc_sgpr(a.q + (size_t)q0 * a.ldq, max(min(32, a.rows - q0), 0) * a.ldq * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kk = wave * 4 + i;
      qs[kk * 64 + lane] = buf_load8(qr, (r * a.ldq + kk * 16 + h * 8) * 2);
    }
  }
  __syncthreads();
  PI0_PROBE(1);

  float m_run = -1.0e30f, l_run = 0.f;
  f32x16 o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;

  for (int i = 0; i < mine; ++i) {
    const int key0 = (wave + 4 * i) * 32;
    PI0_PROBE(8 + i);
    load_v(i);
    bf16x8 qv[16];
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) qv[kk] = qs[kk * 64 + lane];
    __builtin_amdgcn_sched_barrier(0);     // keep the V^T and Q requests ahead of the S^T MFMAs
    f32x16 st;
#pragma unroll
    for (int e = 0; e < 16; ++e) st[e] = 0.f;
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) st = mfma32(kf[kk], qv[kk], st);
    __builtin_amdgcn_sched_barrier(0);
    load_k(i + 1);
    __builtin_amdgcn_sched_barrier(0);     // and the next K requests ahead of the softmax
    // lane holds S^T[key 8 (e / 4) + 4 h + e % 4][query r]
    float sv[16], mx = -1.0e30f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int key = key0 + 8 * (e >> 2) + 4 * h + (e & 3);
      sv[e] = key < a.keys ? round_bf(st[e]) * a.scale_log2 : -1.0e30f;
      mx = fmaxf(mx, sv[e]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, PI0_WAVE));
    const float m_new = fmaxf(m_run, mx);
    const float alpha = fast_exp2(m_run - m_new);
    float ps = 0.f;
    bf16x8 pf[2];                                      // P^T for chunk c = e / 8
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float pv = fast_exp2(sv[e] - m_new);
      ps += pv;
      pf[e >> 3][e & 7] = f2bf(pv);
    }
    ps += __shfl_xor(ps, 32, PI0_WAVE);
    l_run = l_run * alpha + ps;
    m_run = m_new;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      f32x16 acc = o[dt] * alpha;
#pragma unroll
      for (int c = 0; c < 2; ++c) acc = mfma32(vf[dt][c], pf[c], acc);
      o[dt] = acc;
    }
  }
  PI0_PROBE(2);
  __syncthreads();                                     // every wave is done with qs

  // ---- merge the 4 waves' partials: O = sum_w 2^(m_w - M) O_w / sum_w 2^(m_w - M) l_w.
  // Every wave parks its O rows (lane: query r, 4 consecutive d per 16-byte store), then
  // wave w finishes head dims 64 w .. 64 w + 63 of all 32 rows, summing the waves in order.
  if (h == 0) { ml[wave][0][r] = m_run; ml[wave][1][r] = l_run; }
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      const f32x4 v4 = {o[dt][e4 * 4], o[dt][e4 * 4 + 1], o[dt][e4 * 4 + 2], o[dt][e4 * 4 + 3]};
      *reinterpret_cast<f32x4*>(&ob[wave][r][dt * 32 + 8 * e4 + 4 * h]) = v4;
    }
  __syncthreads();
  float M = -1.0e30f;
#pragma unroll
  for (int w = 0; w < 4; ++w) M = fmaxf(M, ml[w][0][r]);
  float wgt[4], L = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    wgt[w] = fast_exp2(ml[w][0][r] - M);     // 0 for a wave that saw no key
    L += wgt[w] * ml[w][1][r];
  }
  const float inv = __builtin_amdgcn_rcpf(L);
  const int row = q0 + r;
  if (row >= a.rows) return;
  __bf16* orow = a.out + (size_t)row * a.ldo;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {           // 4 consecutive d per load and store
      const int d0 = (2 * wave + j) * 32 + 8 * e4 + 4 * h;
      f32x4 v = *reinterpret_cast<const f32x4*>(&ob[0][r][d0]) * wgt[0];
#pragma unroll
      for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(&ob[w][r][d0]) * wgt[w];
      const bf16x4 pk = {f2bf(v[0] * inv), f2bf(v[1] * inv), f2bf(v[2] * inv), f2bf(v[3] * inv)};
      *reinterpret_cast<bf16x4*>(orow + d0) = pk;
    }
  PI0_PROBE(3);
}


// The same attention for many requests: workgroup = 128 query rows, one 32-row tile per wave,
// all keys. A 32-row workgroup pulls every K and V byte through its CU for itself (835 KB at
// 816 keys, two of three rounds of the chip at batch 4); here the four waves share each 32-key
// block in LDS (fragment order, 32 KB, four slots filled by buffer loads with the LDS
// destination), and the next block's S^T MFMAs are issued ahead of this block's softmax.
// A wave sees all keys, so there is no merge. The reference of the exponents moves only when a
// row's maximum has outgrown it by 2^8 (P then stays below 2^8, the same relative rounding),
// which saves the rescale of O (62.8 us with it at 4 x 816); the sum is that of the rounded P,
// and the logits stay in fp32, which outweighs that no P is exactly 1 any more. Used from 128
// workgroups on; fewer leave too much of the chip idle. With the K / V pre-pass, 32-row
// workgroups -> these: 3 x 816 rows 59.5 -> 42.4 us, 4 x 816 76.5 -> 45.2, 8 x 816 130 -> 80.6;
// distance from 64 bits at 4 x 816 4.2e-3 -> 2.3e-3.
__global__ __launch_bounds__(256, 1) void enc_attn_wide_kernel(EncAttnArgs a) {
  constexpr int D = 4, SLOT = 32 * 64;                 // slots, 16-byte words (16 K + 16 V^T fragments)
  __shared__ bf16x8 ring[D * SLOT];
  const int t = threadIdx.x, lane = t & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int bq = blockIdx.y, q0 = blockIdx.x * 128 + wave * 32;
  a.q += (size_t)bq * a.rows * a.ldq;
  a.out += (size_t)bq * a.rows * a.ldo;
  const int kvbytes = EA_HD * a.ldvt * (int)sizeof(__bf16);
  const __amdgpu_buffer_rsrc_t kr = rows_rsrc_sgpr(a.kp + (size_t)bq * EA_HD * a.ldvt, kvbytes);
  const __amdgpu_buffer_rsrc_t vr = rows_rsrc_sgpr(a.vp + (size_t)bq * EA_HD * a.ldvt, kvbytes);
  const int nblk = (a.keys + 31) / 32;
  // wave w copies fragments w, w + 4, .. of K and of V^T (blocks past the end: the last again)
  auto issue = [&](int b) {
    bf16x8* dst = ring + (b & (D - 1)) * SLOT + wave * 64;
    const int so = min(b, nblk - 1) * 16384 + wave * 1024;
#pragma unroll
    for (int i = 0; i < 4; ++i) buf_load16_lds_s(kr, dst + i * 256, lane * 16, so + i * 4096);
#pragma unroll
    for (int i = 0; i < 4; ++i) buf_load16_lds_s(vr, dst + 1024 + i * 256, lane * 16, so + i * 4096);
  };
  bf16x8 qf[16];
  {
    const __amdgpu_buffer_rsrc_t qr =
        rows_rsrc_sgpr(a.q + (size_t)q0 * a.ldq, max(min(32, a.rows - q0), 0) * a.ldq * 2);
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) qf[kk] = buf_load8(qr, (r * a.ldq + kk * 16 + h * 8) * 2);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int b = 0; b < D - 1; ++b) issue(b);
  auto scores = [&](int b) {                           // S^T of block b: keys x queries
    const bf16x8* k = ring + (b & (D - 1)) * SLOT + lane;
    f32x16 s;
#pragma unroll
    for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) s = mfma32(k[kk * 64], qf[kk], s);
    return s;
  };
  float m_ref = -1.0e30f, l = 0.f;
  f32x16 o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
  __builtin_amdgcn_s_waitcnt(PI0_VMCNT(16));           // Q and block 0
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  f32x16 st = scores(0);
  for (int b = 0; b < nblk; ++b) {
    // block b + 1 has landed in every wave, and every wave is past block b - 1, whose slot
    // takes block b + 3
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(PI0_VMCNT(8) & ~(0xF << 8));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    issue(b + D - 1);
    __builtin_amdgcn_sched_barrier(0);
    const f32x16 next = scores(b + 1);                 // past the end: a block computed, not used
    float sv[16], mx = -1.0e30f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {     // (masking behind a branch for the last block: 10% slower)
      const int key = b * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
      sv[e] = key < a.keys ? st[e] * a.scale_log2 : -1.0e30f;
      mx = fmaxf(mx, sv[e]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, PI0_WAVE));
    if (__any(mx > m_ref + 8.f)) {
      const float m_new = fmaxf(m_ref, mx), alpha = fast_exp2(m_ref - m_new);
      m_ref = m_new;
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) o[dt] = o[dt] * alpha;
    }
    bf16x8 pf[2];                                      // P^T for chunk c = e / 8
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      pf[e >> 3][e & 7] = f2bf(fast_exp2(sv[e] - m_ref));
      l += bf2f(pf[e >> 3][e & 7]);
    }
    const bf16x8* v = ring + (b & (D - 1)) * SLOT + 1024 + lane;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int c = 0; c < 2; ++c) o[dt] = mfma32(v[(dt * 2 + c) * 64], pf[c], o[dt]);
    st = next;
  }
  __builtin_amdgcn_s_waitcnt(PI0_VMCNT(0));            // the re-loads past the end
  l += __shfl_xor(l, 32, PI0_WAVE);
  const float inv = __builtin_amdgcn_rcpf(l);
  if (q0 + r >= a.rows) return;
  __bf16* orow = a.out + (size_t)(q0 + r) * a.ldo;
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      const bf16x4 pk = {f2bf(o[dt][e4 * 4] * inv), f2bf(o[dt][e4 * 4 + 1] * inv),
                         f2bf(o[dt][e4 * 4 + 2] * inv), f2bf(o[dt][e4 * 4 + 3] * inv)};
      *reinterpret_cast<bf16x4*>(orow + dt * 32 + 8 * e4 + 4 * h) = pk;
    }
}


// ---- SigLIP vision tower pieces (pipeline.py:21-54) -----------------------------

// images [views][224][224][3] -> patch rows [views * 256][ldo]: row = view * 256 + py * 16 + px,
// column (iy * 14 + ix) * 3 + c for the 14 x 14 x 3 patch, zero for columns 588 .. ldo - 1
// (the patchify of vision_patch_embed, wrappers.py:257-269).
__global__ __launch_bounds__(256) void im2col_patches_kernel(const __bf16* __restrict__ img,
                                                             __bf16* __restrict__ out, int ldo,
                                                             int rows) {
  const int id = blockIdx.x * 256 + threadIdx.x;
  const int chunks = ldo >> 3;
  const int row = id / chunks, c0 = (id - row * chunks) * 8;
  if (row >= rows) return;
  const int view = row >> 8, py = (row >> 4) & 15, px = row & 15;
  bf16x8 v;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int k = c0 + j;
    __bf16 x = __bf16(0.f);
    if (k < 588) {
      const int iy = k / 42, r = k - iy * 42;           // 42 = 14 columns x 3 channels
      x = img[(((size_t)view * 224 + py * 14 + iy) * 224 + px * 14) * 3 + r];
    }
    v[j] = x;
  }
  *reinterpret_cast<bf16x8*>(out + (size_t)row * ldo + c0) = v;
}

// Multi-head vision attention (attention.py:20-26, SDPA over each view's 256 tokens,
// 16 heads of 72). A workgroup stages one (view, head)'s K and V in LDS straight from the
// packed QKV rows (buffer loads with the LDS destination, rows of 144 bytes: nine 16-byte
// chunks, an odd count, so the fragment reads of 16 neighbouring rows hit distinct banks) and
// takes 2 tiles of 32 queries, each over 2 halves of the keys: wave = (query tile, key half).
// S^T = K Q^T and O^T = V^T P^T on 32x32x16 MFMAs (head_dim zero-padded to 80 for the k16
// steps), softmax in fp32 with P rounded to bf16 and normalised by the rounded P's sum. All of
// a wave's scores are held at once, so there is one maximum and no rescaling. V^T comes from row-major V by transposing LDS reads:
// within a 16-lane group lane 4 k + c points at 4 columns of key k and lane j receives 4 keys
// of column j, which is half of an A fragment in the key order that P^T has in the S^T
// accumulator. A launch that transposed V through memory, waves reading both from L2 and an
// online softmax took 13.8 us at 3 views and 35.9 at 12; this takes 6.6 and 21.5, at the same
// distance from 64 bits (2.15e-3). One 4-tile workgroup over all keys: 7.2 and 20.6, but
// 2.19e-3 (a maximum over more keys leaves fewer P that are exactly 1).
constexpr int VA_TOK = 256, VA_HD = 72;

struct VisAttnArgs {
  const __bf16* qkv; int ldqkv;
  __bf16* out; int ldo;
  int dim;
  float scale_log2;
};

constexpr int VA_QT = 2, VA_KS = 2;                     // query tiles, key parts per workgroup

// WIDE: rows too far apart for 32-bit offsets over a whole view; every copy then has a resource
// of its own, from its first row on.
template <bool WIDE>
__global__ __launch_bounds__(64 * VA_QT * VA_KS, 1) void vision_attn_kernel(VisAttnArgs a) {
  constexpr int QT = VA_QT, KS = VA_KS, NW = QT * KS, CH = VA_HD / 8, WORDS = VA_TOK * CH, CI = WORDS / (64 * NW);
  constexpr int NB = VA_TOK / 32 / KS;                  // 32-key blocks of a wave
  static_assert(CI * 64 * NW == WORDS && NB * 32 * KS == VA_TOK, "staging and key split");
  // K, then V; the padded head dims of V's last rows are read (and not used) past the end
  __shared__ bf16x8 kv[2 * WORDS + 32];
  PI0_PROBE(0);
  const int t = threadIdx.x, lane = t & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), qi = wave / KS, kp = wave % KS;
  const int head = blockIdx.y, view = blockIdx.z;
  const __bf16* base = a.qkv + (size_t)view * VA_TOK * a.ldqkv + head * VA_HD;
  if constexpr (WIDE) {
#pragma unroll
    for (int i = 0; i < 2 * CI; ++i) {                  // K, then V
      const int w0 = (i % CI * NW + wave) * 64, row0 = w0 / CH, row = (w0 + lane) / CH;
      const __bf16* src = base + (i < CI ? 1 : 2) * a.dim + (size_t)row0 * a.ldqkv;
      const int rows = min(63 / CH + 2, VA_TOK - row0); // that a copy's 64 chunks can touch
      const __amdgpu_buffer_rsrc_t r =
          rows_rsrc_sgpr(src, ((rows - 1) * a.ldqkv + VA_HD) * (int)sizeof(__bf16));
      buf_load16_lds(r, &kv[(i < CI ? 0 : WORDS) + w0],
                     ((row - row0) * a.ldqkv + (w0 + lane - row * CH) * 8) * (int)sizeof(__bf16));
    }
  } else {
    const int nbytes = ((VA_TOK - 1) * a.ldqkv + VA_HD) * (int)sizeof(__bf16);
    const __amdgpu_buffer_rsrc_t kr = rows_rsrc_sgpr(base + a.dim, nbytes);
    const __amdgpu_buffer_rsrc_t vr = rows_rsrc_sgpr(base + 2 * a.dim, nbytes);
    int off[CI];
#pragma unroll
    for (int i = 0; i < CI; ++i) {
      const int id = (i * NW + wave) * 64 + lane, row = id / CH;
      off[i] = (row * a.ldqkv + (id - row * CH) * 8) * (int)sizeof(__bf16);
      buf_load16_lds(kr, &kv[(i * NW + wave) * 64], off[i]);
    }
#pragma unroll
    for (int i = 0; i < CI; ++i) buf_load16_lds(vr, &kv[WORDS + (i * NW + wave) * 64], off[i]);
  }
  __builtin_amdgcn_sched_barrier(0);
  // Q^T fragments: lane holds Q[q][16 kk + 8 h .. + 7] (zero past d = 72)
  const int q = (blockIdx.x * QT + qi) * 32 + r;
  bf16x8 qf[5];
#pragma unroll
  for (int kk = 0; kk < 5; ++kk) {
    const int d = kk * 16 + h * 8;
    qf[kk] = d < VA_HD ? load8(base + (size_t)q * a.ldqkv + d) : zero8();
  }
  f32x16 st[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) st[b][e] = 0.f;
  __syncthreads();                                      // waits for every copy
  PI0_PROBE(1);
  const int key0 = kp * NB * 32;
#pragma unroll
  for (int kk = 0; kk < 5; ++kk)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      bf16x8 kf = kv[(key0 + b * 32 + r) * CH + kk * 2 + (kk < 4 ? h : 0)];
      if (kk == 4 && h) kf = zero8();                   // head dims 72 .. 79
      st[b] = mfma32(kf, qf[kk], st[b]);
    }
  // lane holds S^T[key 32 b + 8 (e / 4) + 4 h + e % 4][query r]
  float mx = -1.0e30f, l = 0.f;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) { st[b][e] *= a.scale_log2; mx = fmaxf(mx, st[b][e]); }
  mx = fmaxf(mx, __shfl_xor(mx, 32, PI0_WAVE));
  f32x16 o[3];
#pragma unroll
  for (int dt = 0; dt < 3; ++dt)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[dt][e] = 0.f;
  typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
  const __bf16* vs = reinterpret_cast<const __bf16*>(kv + WORDS);
  const int vlane = (key0 + 4 * h + ((lane & 15) >> 2)) * VA_HD + (lane & 16) + (lane & 3) * 4;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    bf16x8 pf[2];                                       // P^T for chunk c = e / 8
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      pf[e >> 3][e & 7] = f2bf(fast_exp2(st[b][e] - mx));
      l += bf2f(pf[e >> 3][e & 7]);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int dt = 0; dt < 3; ++dt) {
        const int at = vlane + (b * 32 + c * 16) * VA_HD + dt * 32;
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vs + at));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(vs + at + 8 * VA_HD));
        const bf16x8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        o[dt] = mfma32(vf, pf[c], o[dt]);
      }
  }
  l += __shfl_xor(l, 32, PI0_WAVE);
  PI0_PROBE(2);
  {                                                     // join the key halves
    static_assert(KS == 2, "one part parked per query tile");
    float* park = reinterpret_cast<float*>(kv) + qi * 50 * PI0_WAVE + lane;
    __syncthreads();                                    // every wave is done with K and V
    if (kp == 1) {
      park[0] = mx;
      park[PI0_WAVE] = l;
#pragma unroll
      for (int dt = 0; dt < 3; ++dt)
#pragma unroll
        for (int e = 0; e < 16; ++e) park[(2 + dt * 16 + e) * PI0_WAVE] = o[dt][e];
    }
    __syncthreads();
    if (kp == 1) return;
    const float m1 = park[0], m = fmaxf(mx, m1);
    const float w0 = fast_exp2(mx - m), w1 = fast_exp2(m1 - m);
    l = l * w0 + park[PI0_WAVE] * w1;
#pragma unroll
    for (int dt = 0; dt < 3; ++dt)
#pragma unroll
      for (int e = 0; e < 16; ++e) o[dt][e] = o[dt][e] * w0 + park[(2 + dt * 16 + e) * PI0_WAVE] * w1;
  }
  // lane holds O^T[d = 32 dt + 8 (e / 4) + 4 h + e % 4][query r]
  const float inv = __builtin_amdgcn_rcpf(l);
  __bf16* orow = a.out + ((size_t)view * VA_TOK + q) * a.ldo + head * VA_HD;
#pragma unroll
  for (int dt = 0; dt < 3; ++dt)
#pragma unroll
    for (int e4 = 0; e4 < 4; ++e4) {
      const int d = dt * 32 + 8 * e4 + 4 * h;
      if (d < VA_HD) {
        const bf16x4 pk = {f2bf(o[dt][e4 * 4] * inv), f2bf(o[dt][e4 * 4 + 1] * inv),
                           f2bf(o[dt][e4 * 4 + 2] * inv), f2bf(o[dt][e4 * 4 + 3] * inv)};
        *reinterpret_cast<bf16x4*>(orow + d) = pk;
      }
    }
  PI0_PROBE(3);
}


// Prompt embedding (the reference takes precomputed embeddings,
// spec.py:46): out[b * rows_per_batch + row0 + j] = bf16(table[ids[b][j]] * scale).
__global__ __launch_bounds__(256) void embed_tokens_kernel(const int* __restrict__ ids, int n_tok,
                                                           const __bf16* __restrict__ table,
                                                           int vocab, int dim, float scale,
                                                           __bf16* __restrict__ out, int ldo,
                                                           int row0, int rows_per_batch,
                                                           int total) {
  const int per_row = dim >> 3;
  const int id = blockIdx.x * 256 + threadIdx.x;
  if (id >= total * per_row) return;
  const int tok = id / per_row, c = (id - tok * per_row) * 8;
  const int b = tok / n_tok, j = tok - b * n_tok;
  const int v = min(max(ids[tok], 0), vocab - 1);      // out-of-range ids clamp (checked on host)
  const bf16x8 e = load8(table + (size_t)v * dim + c);
  bf16x8 o;
#pragma unroll
  for (int q = 0; q < 8; ++q) o[q] = f2bf(bf2f(e[q]) * scale);
  *reinterpret_cast<bf16x8*>(out + ((size_t)b * rows_per_batch + row0 + j) * ldo + c) = o;
}

}  // namespace pi0

using namespace pi0;

// ---- host-side launch helpers ----------------------------------------------------

// Column tiles per group of the tile order (tile_of): as many as balance the rows and columns
// of the 32 tiles that an XCD holds, from 1536 rows on. us per launch in the plain order /
// grouped (cold weights): 3072 rows vision QKV 36.2 / 31.7, encoder down 209 / 189; 6528 rows
// encoder gate 748 / 711, QKV 81.7 / 76.0; 4096 rows vision down 78.0 / 65.7; 1536 rows vision
// QKV 18.4 / 17.9, encoder o-proj 19.2 / 18.4. Below that few row tiles share the columns and
// the groups cost more than they save: 1280 rows vision QKV 18.2 / 20.0, FFN-up 21.4 / 22.3,
// 1072 rows encoder gate 139 / 145, 1024 rows vision QKV 12.5 / 13.1; 816 rows are level.
static int tile_group(const TileArgs& a, int bm, int bn) {
  if (a.M < 1536) return 1;
  return std::max(1, std::min(a.tiles_n, (int)lroundf(sqrtf(32.f * bm / bn))));
}

template <int BM, int WN, int D, int EPI, bool DUAL, int OCC, int RMS = 0>
static int launch_tile(TileArgs a, hipStream_t s) {
  a.tiles_m = (a.M + BM - 1) / BM;
  const int bn_out = DUAL ? 2 * WN : 4 * WN;
  if (a.N % bn_out) return PI0HIP_ERR_SHAPE;
  a.tiles_n = a.N / bn_out;
  const int steps = a.K / 64;
  if (a.K % 64 || steps % a.splitk || (steps / a.splitk) % D) return PI0HIP_ERR_SHAPE;
  a.ksteps = steps / a.splitk;
  a.group = tile_group(a, BM, 4 * WN);
  const int grid = a.tiles_m * a.tiles_n * a.splitk;
  // XCD-contiguous tile order needs a grid divisible by the 8 XCDs
  a.xcd_remap = (grid % 8 == 0) ? 1 : 0;
  hipLaunchKernelGGL((tile_gemm_kernel<BM, WN, D, EPI, DUAL, OCC, RMS>), dim3(grid), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}

// Pipeline depth: the deepest even ring (<= DMAX) whose depth divides the per-split step count.
template <int BM, int WN, int DMAX, int EPI, bool DUAL, int OCC = 1, int RMS = 0>
static int launch_tile_auto(TileArgs a, hipStream_t s) {
  if (a.K % 64 || a.splitk < 1 || (a.K / 64) % a.splitk) return PI0HIP_ERR_SHAPE;
  const int steps = a.K / 64 / a.splitk;
  if (DMAX >= 8 && steps % 8 == 0) return launch_tile<BM, WN, (DMAX >= 8 ? 8 : 2), EPI, DUAL, OCC, RMS>(a, s);
  if (DMAX >= 6 && steps % 6 == 0) return launch_tile<BM, WN, (DMAX >= 6 ? 6 : 2), EPI, DUAL, OCC, RMS>(a, s);
  if (DMAX >= 4 && steps % 4 == 0) return launch_tile<BM, WN, (DMAX >= 4 ? 4 : 2), EPI, DUAL, OCC, RMS>(a, s);
  if (steps % 2 == 0) return launch_tile<BM, WN, 2, EPI, DUAL, OCC, RMS>(a, s);
  return PI0HIP_ERR_SHAPE;
}

// Pipeline depth preferring 4 (measured faster than 8 at K = 2048, M = 768), then 3
// (at K = 1152, 18 steps, the projector takes 9.4 us with 3 against 10.6 with 6) and 6.
template <int BM, int WN, int EPI, bool DUAL, int OCC = 1>
static int launch_tile_d4(TileArgs a, hipStream_t s) {
  if (a.K % 64 || a.splitk < 1 || (a.K / 64) % a.splitk) return PI0HIP_ERR_SHAPE;
  const int steps = a.K / 64 / a.splitk;
  if (steps % 4 == 0) return launch_tile<BM, WN, 4, EPI, DUAL, OCC>(a, s);
  if (steps % 3 == 0) return launch_tile<BM, WN, 3, EPI, DUAL, OCC>(a, s);
  if (steps % 6 == 0) return launch_tile<BM, WN, 6, EPI, DUAL, OCC>(a, s);
  if (steps % 2 == 0) return launch_tile<BM, WN, 2, EPI, DUAL, OCC>(a, s);
  return PI0HIP_ERR_SHAPE;
}

// block_gemm_kernel: K of a split a multiple of 4 steps of 32.
template <int WMC, int WNC, int FM, int FN, int EPI, bool DUAL = false>
static int launch_block(TileArgs a, hipStream_t s) {
  constexpr int BM = WMC * FM * 32, NBF = WNC * FN, OUTC = DUAL ? NBF * 16 : NBF * 32;
  if (a.splitk < 1 || a.K % (128 * a.splitk) || a.N % OUTC) return PI0HIP_ERR_SHAPE;
  if ((long long)a.K * NBF * 32 * (long long)sizeof(__bf16) > INT_MAX ||
      (long long)BM * a.lda * (long long)sizeof(__bf16) > INT_MAX)
    return PI0HIP_ERR_SHAPE;                 // 32-bit buffer offsets
  a.tiles_m = (a.M + BM - 1) / BM;
  a.tiles_n = a.N / OUTC;
  a.ksteps = a.K / 32 / a.splitk;
  a.group = tile_group(a, BM, NBF * 32);
  hipLaunchKernelGGL((block_gemm_kernel<WMC, WNC, FM, FN, EPI, DUAL>),
                     dim3(a.tiles_m * a.tiles_n * a.splitk), dim3(64 * WMC * WNC), 0, s, a);
  return (int)hipGetLastError();
}

static int launch_rows32(const TileArgs& a, hipStream_t s) {
  const int nrb = (a.M + 31) / 32, ntiles = a.N / 32, xcd_map = ntiles % 8 == 0;
  switch (a.K) {
    case 2048: hipLaunchKernelGGL(rows32_res_kernel<16>, dim3(nrb * ntiles), dim3(512), 0, s, a, nrb, xcd_map); break;
    case 4096: hipLaunchKernelGGL(rows32_res_kernel<32>, dim3(nrb * ntiles), dim3(512), 0, s, a, nrb, xcd_map); break;
    default: return PI0HIP_ERR_SHAPE;
  }
  return (int)hipGetLastError();
}

// Which tile a call takes. A launch of W workgroups runs in ceil(W / slots) rounds of about
// equal length, so a tile whose grid just overflows a round loses up to half the chip: the
// choice is the least rounds x (measured length of a full round). The lengths are single
// launches with cold weights in a graph; what matters is their ratio, which K does not change
// much. Kernels that share a CU (per_cu 2) refill it as they end, without rounds.
// A tile whose rows lie further apart than 32-bit buffer offsets reach is no choice.
static float tile_us(const TileArgs& a, int bm, int bn, float round_us, int per_cu = 1) {
  if ((long long)bm * a.lda * (long long)sizeof(__bf16) > INT_MAX) return INFINITY;
  const float w = (float)((a.M + bm - 1) / bm) * (float)((a.N + bn - 1) / bn) * (float)a.splitk;
  const float r = w / (float)(per_cu * device_cus());
  return round_us * (per_cu > 1 ? fmaxf(r, 0.8f) : ceilf(r));
}
// ... of a block_gemm_kernel tile, which needs whole column tiles and 128-deep K (launch_block)
static float block_us(const TileArgs& a, int bm, int bn, float round_us) {
  if (a.N % bn || a.K % (128 * a.splitk) || (long long)a.K * 256 * (long long)sizeof(__bf16) > INT_MAX)
    return INFINITY;
  return tile_us(a, bm, bn, round_us);
}
static int least(std::initializer_list<float> us) {
  return (int)(std::min_element(us.begin(), us.end()) - us.begin());
}

static TileArgs tile_args(const void* x, int ldx, const void* w, void* out, int ldo, int M, int N,
                          int K) {
  TileArgs a = {};
  a.a = (const __bf16*)x; a.lda = ldx; a.w0 = (const __bf16*)w;
  a.out = (__bf16*)out; a.ldo = ldo;
  a.M = M; a.N = N; a.K = K; a.splitk = 1; a.n_valid = N; a.rows_per_batch = M;
  return a;
}

static bool bad_dims(int M, int N, int K) { return M <= 0 || N <= 0 || K <= 0; }
// 16-byte vector access in the staging loads and the epilogues: row starts must be
// 16-byte aligned (leading dimension a multiple of 8 bf16, pointer 16-byte aligned).
static bool misaligned(const void* p, int ld) {
  return (reinterpret_cast<uintptr_t>(p) & 15) != 0 || (ld & 7) != 0;
}

// Plain and biased projections. Vision QKV (N = 3456, K = 1152), us before -> after: 256
// rows 8.2 -> 6.5, 1024 13.8 -> 11.9, 2048 24.7 -> 21.2.
template <int EPI>
static int linear_launch(const TileArgs& a, hipStream_t s) {
  const bool d3 = a.K % 192 == 0;
  switch (least({tile_us(a, 64, 128, 8.5f), tile_us(a, 32, 128, 6.7f),
                 d3 ? tile_us(a, 96, 128, 10.4f) : INFINITY,
                 d3 ? tile_us(a, 96, 128, 21.2f, 2) : INFINITY,
                 block_us(a, 128, 128, 12.3f), block_us(a, 256, 128, 22.f)})) {
    case 1: return launch_tile_d4<32, 32, EPI, false>(a, s);
    case 2: case 3: return launch_tile<96, 32, 3, EPI, false, 2>(a, s);
    case 4: return launch_block<4, 2, 1, 2, EPI>(a, s);
    case 5: return launch_block<4, 2, 2, 2, EPI>(a, s);
    default: return launch_tile_d4<64, 32, EPI, false>(a, s);
  }
}

// Split-K partials of a residual GEMM (round lengths at 4096 of K per split).
static int partial_launch(const TileArgs& a, hipStream_t s) {
  // small M (the encoder down of one view without a prompt): 32-row tiles, two workgroups per CU
  if (a.M <= 256) return launch_tile_auto<32, 32, 4, TE_PARTIAL, false, 2>(a, s);
  switch (least({tile_us(a, 192, 128, 57.f),
                 block_us(a, 128, 256, 62.f),
                 block_us(a, 192, 256, 92.f),
                 block_us(a, 256, 256, 112.f),
                 block_us(a, 384, 256, 155.f)})) {
    case 1: return launch_block<2, 4, 2, 2, TE_PARTIAL>(a, s);
    case 2: return launch_block<2, 4, 3, 2, TE_PARTIAL>(a, s);
    case 3: return launch_block<4, 2, 2, 4, TE_PARTIAL>(a, s);
    case 4: return launch_block<4, 2, 3, 4, TE_PARTIAL>(a, s);
    default: return launch_tile_auto<192, 32, 4, TE_PARTIAL, false>(a, s);
  }
}

extern "C" {

int pi0hip_pack_weight32(const void* w, void* packed, int K, int N, int batch, hipStream_t s) {
  if (K % 16 || N % 32) return (K <= 0 || N <= 0) ? PI0HIP_ERR_ARG : PI0HIP_ERR_SHAPE;
  return pi0hip_pack_weight32_padded(w, packed, K, N, K, N, batch, s);
}

int pi0hip_pack_weight32_padded(const void* w, void* packed, int K, int N, int K_pad, int N_pad,
                                int batch, hipStream_t s) {
  if (!w || !packed || K <= 0 || N <= 0 || batch <= 0) return PI0HIP_ERR_ARG;
  if (K_pad % 16 || N_pad % 32 || K_pad < K || N_pad < N) return PI0HIP_ERR_SHAPE;
  const long long frags = (long long)batch * (K_pad / 16) * (N_pad / 32) * 64;
  const long long blocks = (frags + 255) / 256;
  hipLaunchKernelGGL(pack_weight32_kernel, dim3((unsigned)blocks), dim3(256), 0, s,
                     (const __bf16*)w, (__bf16*)packed, K, N, K_pad, N_pad, frags);
  return (int)hipGetLastError();
}

int pi0hip_rms_norm(const void* x, int ldx, void* out, int ldo, int M, int K, hipStream_t s) {
  if (!x || !out || M <= 0 || K <= 0) return PI0HIP_ERR_ARG;
  const dim3 grid((M + 3) / 4);
  switch (K) {
    case 1024: hipLaunchKernelGGL(rms_norm_kernel<2>, grid, dim3(256), 0, s, (const __bf16*)x, ldx, (__bf16*)out, ldo, M, K); break;
    case 2048: hipLaunchKernelGGL(rms_norm_kernel<4>, grid, dim3(256), 0, s, (const __bf16*)x, ldx, (__bf16*)out, ldo, M, K); break;
    default: return PI0HIP_ERR_SHAPE;
  }
  return (int)hipGetLastError();
}

size_t pi0hip_tile_workspace_bytes(int M, int N, int splitk) {
  if (M <= 0 || N <= 0 || splitk <= 1) return 0;
  return (size_t)splitk * M * N * sizeof(float);
}

int pi0hip_tile_linear(const void* x, int ldx, const void* w_packed, const void* bias, void* out,
                       int ldo, int M, int N, int K, hipStream_t s) {
  if (!x || !w_packed || !out || bad_dims(M, N, K)) return PI0HIP_ERR_ARG;
  if (misaligned(x, ldx) || misaligned(out, ldo) || misaligned(bias, 0)) return PI0HIP_ERR_SHAPE;
  TileArgs a = tile_args(x, ldx, w_packed, out, ldo, M, N, K);
  a.bias = (const __bf16*)bias;
  return bias ? linear_launch<TE_BIAS>(a, s) : linear_launch<TE_STORE>(a, s);
}

int pi0hip_tile_linear_residual(const void* x, int ldx, const void* w_packed, void* out, int ldo,
                                int M, int N, int K, int splitk, void* ws, size_t ws_bytes,
                                hipStream_t s) {
  if (!x || !w_packed || !out || bad_dims(M, N, K) || splitk < 1) return PI0HIP_ERR_ARG;
  if (misaligned(x, ldx) || misaligned(out, ldo)) return PI0HIP_ERR_SHAPE;
  TileArgs a = tile_args(x, ldx, w_packed, out, ldo, M, N, K);
  a.splitk = splitk;
  if (splitk == 1) {
    // o-proj (N = K = 2048), us before -> after: 1632 rows 23.2 -> 20.4, 2048 33.0 -> 21.6,
    // 3264 36.5 -> 28.9, 4608 64.7 -> 43.6. A long K (ffn-down) keeps the 128 x 256 strip
    // while that grid fits one round (3264 rows 217 us against 276 for the same block of
    // block_gemm_kernel); past it 256 x 256 blocks, 6528 rows 475 -> 393.
    if (K >= 8192 && M >= 2048 && N % 256 == 0) {
      if (block_us(a, 256, 256, 393.f) < tile_us(a, 128, 256, 225.f))
        return launch_block<4, 2, 2, 4, TE_RES>(a, s);
      return launch_tile_d4<128, 64, TE_RES, false>(a, s);
    }
    // The batched decoder's o-proj and down (N = 1024, K 2048 / 4096), against 4 splits and
    // their sum: up to 256 rows, one round of them, 32 x 32 workgroups over the whole K, 204
    // rows 8.5 -> 4.9 and 11.2 -> 8.1; past it 32 x 128 strips, 408 rows 15.5 -> 8.1 and
    // 20.8 -> 14.8.
    const bool rows32 = (K == 2048 || K == 4096) && N % 128 == 0;   // whole tiles, as the others
    switch (least({tile_us(a, 64, 128, 13.3f), block_us(a, 128, 128, 20.5f),
                   block_us(a, 128, 256, 28.5f), block_us(a, 192, 256, 42.f),
                   block_us(a, 256, 256, 56.f), tile_us(a, 32, 128, 8.3f),
                   rows32 ? tile_us(a, 32, 32, 5.2f) : INFINITY})) {
      case 1: return launch_block<4, 2, 1, 2, TE_RES>(a, s);
      case 2: return launch_block<2, 4, 2, 2, TE_RES>(a, s);
      case 3: return launch_block<2, 4, 3, 2, TE_RES>(a, s);
      case 4: return launch_block<4, 2, 2, 4, TE_RES>(a, s);
      case 5: return launch_tile_d4<32, 32, TE_RES, false>(a, s);
      case 6: return launch_rows32(a, s);
      default: return launch_tile_d4<64, 32, TE_RES, false>(a, s);
    }
  }
  if (N % 4 || ldo % 4) return PI0HIP_ERR_SHAPE;
  if (!ws || ws_bytes < pi0hip_tile_workspace_bytes(M, N, splitk)) return PI0HIP_ERR_WORKSPACE;
  a.part = (float*)ws;
  if (int e = partial_launch(a, s)) return e;
  const dim3 rgrid((M * (N / 4) + 255) / 256);
  switch (splitk) {
    case 4: hipLaunchKernelGGL(tile_reduce_res_kernel<4>, rgrid, dim3(256), 0, s, a); break;
    case 8: hipLaunchKernelGGL(tile_reduce_res_kernel<8>, rgrid, dim3(256), 0, s, a); break;
    default: hipLaunchKernelGGL(tile_reduce_res_kernel<0>, rgrid, dim3(256), 0, s, a); break;
  }
  return (int)hipGetLastError();
}

int pi0hip_tile_gated_ffn(const void* x, int ldx, const void* gate_packed, const void* up_packed,
                          void* out, int ldo, int M, int N, int K, hipStream_t s) {
  if (!x || !gate_packed || !up_packed || !out || bad_dims(M, N, K)) return PI0HIP_ERR_ARG;
  if (misaligned(x, ldx) || misaligned(out, ldo)) return PI0HIP_ERR_SHAPE;
  TileArgs a = tile_args(x, ldx, gate_packed, out, ldo, M, N, K);
  a.w1 = (const __bf16*)up_packed;
  // Up to 256 rows the two-per-CU strip kernel's 128-row tiles (200 rows: 48 us against 54);
  // above, blocks of 192, 256 or 384 rows x 128 outputs. us before -> after with the encoder's
  // N = 16384, K = 2048: 269 rows 62.6 -> 48.1, 400 67 -> 59, 768 93 -> 89, 816 142 -> 108,
  // 1024 148 -> 119, 3264 396 -> 380, 6528 771 -> 730.
  if (M > 256 && std::isfinite(block_us(a, 192, 128, 50.f)))
    switch (least({block_us(a, 192, 128, 50.f), block_us(a, 256, 128, 58.f),
                   block_us(a, 384, 128, 86.f)})) {
      case 0: return launch_block<2, 4, 3, 2, TE_GATE, true>(a, s);
      case 1: return launch_block<4, 2, 2, 4, TE_GATE, true>(a, s);
      default: return launch_block<4, 2, 3, 4, TE_GATE, true>(a, s);
    }
  return launch_tile_auto<128, 64, 2, TE_GATE, true, 2>(a, s);
}

int pi0hip_tile_norm_gated_ffn(const void* x, int ldx, const void* gate_packed,
                               const void* up_packed, void* out, int ldo, int M, int N, int K,
                               hipStream_t s) {
  if (!x || !gate_packed || !up_packed || !out || bad_dims(M, N, K)) return PI0HIP_ERR_ARG;
  if (misaligned(x, ldx) || misaligned(out, ldo) || K % 128) return PI0HIP_ERR_SHAPE;
  TileArgs a = tile_args(x, ldx, gate_packed, out, ldo, M, N, K);
  a.w1 = (const __bf16*)up_packed;
  return launch_tile_auto<32, 64, 2, TE_GATE, true, 1, 1>(a, s);
}

int pi0hip_tile_qkv_rope(const void* x, int ldx, const void* w_packed, const void* rope, void* q,
                         void* k, void* v, int ldkv, int M, int K, int heads, int head_dim,
                         hipStream_t s) {
  return pi0hip_tile_qkv_rope_batched(x, ldx, w_packed, rope, q, k, v, ldkv, 0, M, M, K, heads,
                                      head_dim, s);
}

int pi0hip_tile_qkv_rope_batched(const void* x, int ldx, const void* w_packed, const void* rope,
                                 void* q, void* k, void* v, int ldkv, long long kv_bstride,
                                 int rows_per_batch, int M, int K, int heads, int head_dim,
                                 hipStream_t s) {
  if (!x || !w_packed || !rope || !q || !k || !v || M <= 0 || K <= 0 || heads <= 0 ||
      rows_per_batch <= 0)
    return PI0HIP_ERR_ARG;
  if (M % rows_per_batch || (kv_bstride & 7)) return PI0HIP_ERR_SHAPE;
  if (head_dim % 16 || misaligned(x, ldx) || misaligned(q, 0) || misaligned(k, ldkv) ||
      misaligned(v, ldkv) || misaligned(rope, head_dim))
    return PI0HIP_ERR_SHAPE;
  TileArgs a = tile_args(x, ldx, w_packed, q, heads * head_dim, M, (heads + 2) * head_dim, K);
  a.out_k = (__bf16*)k; a.out_v = (__bf16*)v; a.ldkv = ldkv;
  a.rope = (const __bf16*)rope; a.heads = heads; a.head_dim = head_dim;
  a.rows_per_batch = rows_per_batch; a.kv_bstride = kv_bstride;
  // us before -> after at N = 2560, K = 2048: 816 rows 24.3 -> 17.3 (260 workgroups of 64 x 128
  // are two rounds), 1632 29.7 -> 24.8, 3264 53.4 -> 36.9, 6528 94 -> 67
  switch (least({tile_us(a, 64, 128, 13.f), block_us(a, 128, 128, 18.f),
                 block_us(a, 128, 256, 27.f), block_us(a, 192, 256, 38.f),
                 block_us(a, 256, 256, 48.f)})) {
    case 1: return launch_block<4, 2, 1, 2, TE_QKV_ROPE>(a, s);
    case 2: return launch_block<2, 4, 2, 2, TE_QKV_ROPE>(a, s);
    case 3: return launch_block<2, 4, 3, 2, TE_QKV_ROPE>(a, s);
    case 4: return launch_block<4, 2, 2, 4, TE_QKV_ROPE>(a, s);
    default: return launch_tile_d4<64, 32, TE_QKV_ROPE, false>(a, s);
  }
}

int pi0hip_layer_norm(const void* x, int ldx, const void* w, const void* b, void* out, int ldo,
                      int M, int K, float eps, hipStream_t s) {
  if (!x || !w || !b || !out || M <= 0 || K <= 0) return PI0HIP_ERR_ARG;
  if (K % 8 || K > 2048) return PI0HIP_ERR_SHAPE;
  hipLaunchKernelGGL(layer_norm_kernel, dim3((M + 3) / 4), dim3(256), 0, s, (const __bf16*)x, ldx,
                     (const __bf16*)w, (const __bf16*)b, (__bf16*)out, ldo, M, K, eps);
  return (int)hipGetLastError();
}

static inline size_t round256_(size_t v) { return (v + 255) / 256 * 256; }

size_t pi0hip_encoder_attention_batched_workspace_bytes(int keys, int batch) {
  if (keys <= 0 || batch <= 0) return 0;
  const size_t ldvt = (size_t)(keys + 63) / 64 * 64;
  return 2 * round256_((size_t)batch * EA_HD * ldvt * sizeof(__bf16));   // packed K, packed V^T
}

size_t pi0hip_encoder_attention_workspace_bytes(int keys) {
  return pi0hip_encoder_attention_batched_workspace_bytes(keys, 1);
}

int pi0hip_encoder_attention(const void* q, int ldq, const void* k, const void* v, int ldkv,
                             void* out, int ldo, int rows, int keys, int head_dim, float scale,
                             void* ws, size_t ws_bytes, hipStream_t s) {
  return pi0hip_encoder_attention_batched(q, ldq, k, v, ldkv, 0, out, ldo, rows, keys, head_dim,
                                          scale, 1, ws, ws_bytes, s);
}

int pi0hip_encoder_attention_batched(const void* q, int ldq, const void* k, const void* v,
                                     int ldkv, long long kv_bstride, void* out, int ldo, int rows,
                                     int keys, int head_dim, float scale, int batch, void* ws,
                                     size_t ws_bytes, hipStream_t s) {
  if (!q || !k || !v || !out || rows <= 0 || keys <= 0 || batch <= 0) return PI0HIP_ERR_ARG;
  if (head_dim != EA_HD || misaligned(q, ldq) || misaligned(k, ldkv) || misaligned(v, ldkv) ||
      (ldo & 3) ||
      (reinterpret_cast<uintptr_t>(out) & 7) || (kv_bstride & 7))
    return PI0HIP_ERR_SHAPE;
  if (!ws || ws_bytes < pi0hip_encoder_attention_batched_workspace_bytes(keys, batch))
    return PI0HIP_ERR_WORKSPACE;
  const int ldvt = (keys + 63) / 64 * 64;
  __bf16* kp = reinterpret_cast<__bf16*>(ws);
  __bf16* vp = kp + round256_((size_t)batch * EA_HD * ldvt * sizeof(__bf16)) / sizeof(__bf16);
  hipLaunchKernelGGL(pack_kv_kernel, dim3(ldvt / 64, EA_HD / 64, batch), dim3(256), 0, s,
                     (const __bf16*)k, (const __bf16*)v, ldkv, kp, vp, ldvt, keys, kv_bstride);
  if (hipError_t e = hipGetLastError()) return (int)e;
  EncAttnArgs a = {};
  a.q = (const __bf16*)q; a.ldq = ldq;
  a.kp = kp; a.vp = vp; a.ldvt = ldvt;
  a.out = (__bf16*)out; a.ldo = ldo;
  a.rows = rows; a.keys = keys;
  a.scale_log2 = 1.4426950408889634f * scale;
  a.kv_bstride = kv_bstride;
  const int wide = (rows + 127) / 128;
  if (wide * batch >= 128)
    hipLaunchKernelGGL(enc_attn_wide_kernel, dim3(wide, batch), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(enc_attn_kernel, dim3((rows + 31) / 32, batch), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}

int pi0hip_tile_linear_bias_res(const void* x, int ldx, const void* w_packed, const void* bias,
                                const void* res, int ldres, int res_mod, void* out, int ldo, int M,
                                int N, int K, int N_pad, int K_pad, hipStream_t s) {
  if (!x || !w_packed || !bias || !res || !out || bad_dims(M, N, K) || res_mod < 0)
    return PI0HIP_ERR_ARG;
  if (N_pad < N || K_pad < K || N % 8 || misaligned(x, ldx) || misaligned(out, ldo) ||
      misaligned(res, ldres) || misaligned(bias, 0))
    return PI0HIP_ERR_SHAPE;
  TileArgs a = tile_args(x, ldx, w_packed, out, ldo, M, N_pad, K_pad);
  a.n_valid = N;
  a.bias = (const __bf16*)bias;
  a.res = (const __bf16*)res; a.ldres = ldres; a.res_mod = res_mod;
  // vision o-proj (K = 1152, 18 steps): a 3-deep ring, 7.1 us against 7.8-8.0 with 6 at
  // M = 768, 17.3 against 19.2 at M = 3072. Rows per tile by the rounds they make (relative
  // round lengths; o-proj at 1536 rows 11.5 -> 9.2 us, FFN-down 36.0 -> 34.2).
  const bool d3 = (K_pad / 64) % 3 == 0 && (K_pad / 64) % 4 != 0;
  switch (least({tile_us(a, 32, 128, 1.f), tile_us(a, 64, 128, 1.42f),
                 tile_us(a, 128, 128, 2.05f)})) {
    case 0: return d3 ? launch_tile<32, 32, 3, TE_BIAS_RES, false, 1>(a, s)
                      : launch_tile_auto<32, 32, 8, TE_BIAS_RES, false>(a, s);
    case 1: return d3 ? launch_tile<64, 32, 3, TE_BIAS_RES, false, 1>(a, s)
                      : launch_tile_auto<64, 32, 8, TE_BIAS_RES, false>(a, s);
    default: return d3 ? launch_tile<128, 32, 3, TE_BIAS_RES, false, 1>(a, s)
                       : launch_tile_auto<128, 32, 8, TE_BIAS_RES, false>(a, s);
  }
}

int pi0hip_tile_linear_bias_gelu(const void* x, int ldx, const void* w_packed, const void* bias,
                                 void* out, int ldo, int M, int N, int K, int N_pad, int K_pad,
                                 hipStream_t s) {
  if (!x || !w_packed || !bias || !out || bad_dims(M, N, K)) return PI0HIP_ERR_ARG;
  if (N_pad < N || K_pad < K || N % 8 || misaligned(x, ldx) || misaligned(out, ldo) ||
      misaligned(bias, 0))
    return PI0HIP_ERR_SHAPE;
  TileArgs a = tile_args(x, ldx, w_packed, out, ldo, M, N_pad, K_pad);
  a.n_valid = N;
  a.bias = (const __bf16*)bias;
  // vision FFN up (K = 1152, N = 4352): 64 x 128 strips two to a CU while the grid is small
  // (768 rows 16.3 us), then blocks by the rounds they make. us before -> after: 2048 rows
  // 39.1 -> 32.2, 3072 50.3 -> 40.3, 4096 63.8 -> 55.7, 6144 86.6 -> 78.0.
  const bool d3 = N_pad % 128 == 0 && K_pad % 192 == 0;
  switch (least({d3 ? tile_us(a, 64, 128, 17.f, 2) : INFINITY,
                 block_us(a, 128, 256, 26.5f), block_us(a, 192, 256, 33.f),
                 block_us(a, 256, 256, 40.f), block_us(a, 384, 256, 56.f),
                 1e30f})) {
    case 0: return launch_tile<64, 32, 3, TE_BIAS_GELU, false, 2>(a, s);
    case 1: return launch_block<2, 4, 2, 2, TE_BIAS_GELU>(a, s);
    case 2: return launch_block<2, 4, 3, 2, TE_BIAS_GELU>(a, s);
    case 3: return launch_block<4, 2, 2, 4, TE_BIAS_GELU>(a, s);
    case 4: return launch_block<4, 2, 3, 4, TE_BIAS_GELU>(a, s);
    default: return launch_tile_auto<64, 32, 8, TE_BIAS_GELU, false>(a, s);
  }
}

int pi0hip_im2col_patches(const void* images, int views, void* out, int ldo, hipStream_t s) {
  if (!images || !out || views <= 0) return PI0HIP_ERR_ARG;
  if (ldo < 588 || ldo % 8 || misaligned(out, ldo)) return PI0HIP_ERR_SHAPE;
  const int rows = views * 256;
  const int threads = rows * (ldo / 8);
  hipLaunchKernelGGL(im2col_patches_kernel, dim3((threads + 255) / 256), dim3(256), 0, s,
                     (const __bf16*)images, (__bf16*)out, ldo, rows);
  return (int)hipGetLastError();
}

size_t pi0hip_vision_attention_workspace_bytes(int, int) { return 0; }

int pi0hip_vision_attention(const void* qkv, int ldqkv, void* out, int ldo, int views, int tokens,
                            int heads, int head_dim, float scale, void*, size_t, hipStream_t s) {
  if (!qkv || !out || views <= 0 || heads <= 0) return PI0HIP_ERR_ARG;
  const int dim = heads * head_dim;
  if (tokens != VA_TOK || head_dim != VA_HD || ldqkv < 3 * dim || ldo < dim ||
      misaligned(qkv, ldqkv) || (ldo & 3) || (reinterpret_cast<uintptr_t>(out) & 7))
    return PI0HIP_ERR_SHAPE;
  VisAttnArgs a = {};
  a.qkv = (const __bf16*)qkv; a.ldqkv = ldqkv;
  a.out = (__bf16*)out; a.ldo = ldo;
  a.dim = dim;
  a.scale_log2 = 1.4426950408889634f * scale;
  const dim3 grid(VA_TOK / (32 * VA_QT), heads, views), block(64 * VA_QT * VA_KS);
  if ((long long)VA_TOK * ldqkv * (long long)sizeof(__bf16) > INT_MAX)
    hipLaunchKernelGGL(vision_attn_kernel<true>, grid, block, 0, s, a);
  else
    hipLaunchKernelGGL(vision_attn_kernel<false>, grid, block, 0, s, a);
  return (int)hipGetLastError();
}

int pi0hip_embed_tokens(const int* ids, int n_tok, int batch, const void* table, int vocab, int dim,
                        float scale, void* out, int ldo, int row0, int rows_per_batch,
                        hipStream_t s) {
  if (!ids || !table || !out || n_tok <= 0 || batch <= 0 || vocab <= 0 || dim <= 0)
    return PI0HIP_ERR_ARG;
  if (dim % 8 || misaligned(out, ldo) || misaligned(table, dim) || row0 + n_tok > rows_per_batch)
    return PI0HIP_ERR_SHAPE;
  const int total = n_tok * batch;
  hipLaunchKernelGGL(embed_tokens_kernel, dim3((total * (dim / 8) + 255) / 256), dim3(256), 0, s,
                     ids, n_tok, (const __bf16*)table, vocab, dim, scale, (__bf16*)out, ldo, row0,
                     rows_per_batch, total);
  return (int)hipGetLastError();
}

}  // extern "C"
