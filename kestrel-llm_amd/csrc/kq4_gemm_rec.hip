// kq4_gemm_rec.hip - prefill GEMM (int8 MFMA, gfx950) of the chains whose activation scale is
// f16-rounded, on activations laid out as the kernel's LDS tiles ("records"):
//   ASM     acc = fma(S, wd * f16r(xd), acc)                  q4 (llama_gemm_q4_0_4x4_asm.c:151-161,
//           the reference's n_batch & ~3 main segment, vllm_safetensors.c:4604-4609)
//   Q8GEMM  acc = fl(acc + fl(wd * f16r(xd) * S))             Q8_0 (gemm_q8_0_8x8_neon :4973-5050)
// bit for bit. Both scales are f16 here, so their product is exact in fp32 and comes from an f16
// MFMA, one 32 x 32 tile at a time.
#include "kq4_common.h"
#include "kq4_internal.h"
#include "../../include/kq4.h"

typedef int kq4_v4i __attribute__((ext_vector_type(4)));
typedef int kq4_v16i __attribute__((ext_vector_type(16)));
typedef float kq4_v16f __attribute__((ext_vector_type(16)));
typedef _Float16 kq4_v4h __attribute__((ext_vector_type(4)));

// Record of (64-token group g, block b): the codes at 2048 * (g * nb + b), [2 halves][64 tokens][16 B]
// (conflict-free 16-B fragment reads); after all of them the scales at 256 * (g * nb + b),
// [64 tokens] {f16r(xd), 0}.
#define KQ4_REC_A 2048
#define KQ4_REC_X 256
#define KQ4_REC_KB 2   // blocks per stage

size_t kq4_rec_bytes(int n, int cols) {
  return (size_t)((n + 63) / 64) * (cols / 32) * (KQ4_REC_A + KQ4_REC_X);
}

// ---- operands ------------------------------------------------------------------------------------

// A wave takes 16 tokens x 1 block or, lane quads over blocks, .. : quad q of a workgroup of 64 quads
// covers 16 tokens x 4 blocks (each token's 512 B read and each block's 256-B rows written whole).
struct KQ4RecAt {
  int m, b;
};
KQ4_DEV bool kq4_rec_at(int n, int nb, KQ4RecAt &at) {
  const int nbg = (nb + 3) >> 2, q = threadIdx.x >> 2;
  at.b = (int)(blockIdx.x % nbg) * 4 + (q & 3);
  at.m = (int)(blockIdx.x / nbg) * 16 + (q >> 2);
  return at.m < n && at.b < nb;
}

// Lane qq of the quad's 8 codes of (m, b), and the block's scale.
KQ4_DEV void kq4_rec_put(uint8_t *__restrict__ rec, long nrec, int nb, int m, int b, int qq,
                         uint2 c, float d) {
  const long r = (long)(m >> 6) * nb + b;
  *reinterpret_cast<uint2 *>(rec + r * KQ4_REC_A + 1024 * (qq >> 1) + 16 * (m & 63) +
                             8 * (qq & 1)) = c;
  if (qq == 0)
    *reinterpret_cast<uint32_t *>(rec + nrec * KQ4_REC_A + r * KQ4_REC_X + 4 * (m & 63)) =
        __half_as_ushort(__float2half_rn(d));
}

// kq4_quantize_kernel (the same codes and scales) into records; tokens [n_main, n) go to xq / xd
// token-major (the decode GEMV's tail).
__global__ __launch_bounds__(256) void kq4_quantize_rec_kernel(
    const float *__restrict__ x, const float *__restrict__ up, uint8_t *__restrict__ rec,
    int8_t *__restrict__ xq, float *__restrict__ xd, int n_main, int n, int cols, int nb) {
  KQ4RecAt at;
  if (!kq4_rec_at(n, nb, at)) return;   // whole quads exit together
  const int qq = threadIdx.x & 3;
  float v[8];
  kq4_load8_silu(x, up, (size_t)at.m * cols + (size_t)at.b * 32 + 8 * qq, v);
  uint32_t pk[2];
  const float d = kq4_quantize8(v, pk);
  const uint2 c = make_uint2(pk[0], pk[1]);
  if (at.m < n_main) {
    kq4_rec_put(rec, (long)((n_main + 63) >> 6) * nb, nb, at.m, at.b, qq, c, d);
  } else {
    const size_t t = at.m - n_main;
    *reinterpret_cast<uint2 *>(xq + t * cols + (size_t)at.b * 32 + 8 * qq) = c;
    if (qq == 0) xd[t * nb + at.b] = d;
  }
}

// Records from codes and scales already quantized (token-major).
__global__ __launch_bounds__(256) void kq4_rec_from_q8_kernel(const int8_t *__restrict__ xq,
                                                              const float *__restrict__ xd,
                                                              uint8_t *__restrict__ rec, int n,
                                                              int cols, int nb) {
  KQ4RecAt at;
  if (!kq4_rec_at(n, nb, at)) return;
  const int qq = threadIdx.x & 3;
  const uint2 c = *reinterpret_cast<const uint2 *>(xq + (size_t)at.m * cols + (size_t)at.b * 32 +
                                                   8 * qq);
  kq4_rec_put(rec, (long)((n + 63) >> 6) * nb, nb, at.m, at.b, qq, c,
              xd[(size_t)at.m * nb + at.b]);
}

static unsigned rec_grid(int n, int nb) { return (unsigned)(((n + 15) / 16) * ((nb + 3) / 4)); }

int kq4_launch_quantize_rec(const float *x, const float *up, uint8_t *rec, int8_t *xq, float *xd,
                            int n_main, int n, int cols, hipStream_t s) {
  const int nb = cols / 32;
  hipLaunchKernelGGL(kq4_quantize_rec_kernel, dim3(rec_grid(n, nb)), dim3(256), 0, s, x, up, rec, xq,
                     xd, n_main, n, cols, nb);
  return (int)hipGetLastError();
}

int kq4_launch_rec_from_q8(const int8_t *xq, const float *xd, uint8_t *rec, int n, int cols,
                           hipStream_t s) {
  const int nb = cols / 32;
  hipLaunchKernelGGL(kq4_rec_from_q8_kernel, dim3(rec_grid(n, nb)), dim3(256), 0, s, xq, xd, rec, n,
                     cols, nb);
  return (int)hipGetLastError();
}

// ---- the GEMM ------------------------------------------------------------------------------------
// Workgroup = WN waves = 32*TM tokens x 32*WN rows; a wave owns one 32-row set against every token of
// the tile (TM tiles of v_mfma_i32_32x32x32_i8, one block's sum each), so each weight is unpacked once
// per workgroup, in the lane that multiplies it: the stream layout's lane (row, half) is the MFMA's B
// operand. Per tile and block: the block sum (32 matrix-core cycles), the scale product from
// v_mfma_f32_32x32x8_f16 (32) and a convert and an fma per output.
// Everything a stage needs (KB = 2 blocks) goes from global memory straight to LDS, raw: the codes and
// scales as the record holds them, shared by the waves (one barrier a stage), and each wave's weights,
// read back by that wave only. The ring holds three stages; a slot is refilled for the third stage
// ahead as soon as the barrier has freed it, so a load has two stages to arrive, and no vector register
// holds one. Software-pipelined over the tiles as the token-major kernel: the block sum of tile q+1 is
// issued before tile q's epilogue, its scale product after it, its fragments one tile earlier.
// Against kq4_gemm_kernel (128 x 128, the ASM chain): 16 registers of scale products instead of 64
// (f16 tiles instead of f32 outer products of two tiles) and none of staged loads, 149 instead of 239,
// so three workgroups share a CU instead of two (2.7 waves resident per SIMD instead of 1.9). Qwen3-8B gate
// 12288 x 4096 at M = 2048: 158 SIMD cycles per tile and block instead of 196 (GRBM_GUI_ACTIVE, both at
// 2.0 GHz), with the quantizer 228-234 instead of 263-268 us in graph replays (0.18 of int8 peak). What
// bounds it: VALU issue. A wave issues 38 VALU instructions per tile and block, 32 of them the convert
// and the fma per output; the SIMD issues one every 4.2 cycles, the matrix unit beside it is busy 40 %.
// Operands of fp6 digits, whose MFMA gives the sum in fp32 without a convert, measured 6 % slower: 42
// VALU per block to unpack the weights' signs and magnitudes, 1.5 times the operand bytes, a lower clock.

template <int TM, int WN, int WF, int NW>
__global__ __launch_bounds__(64 * WN, NW) void kq4_gemm_rec_kernel(
    float *__restrict__ out, const float *__restrict__ res, const uint8_t *__restrict__ w,
    const uint8_t *__restrict__ rec, int rows, int n_tok, int nbt, int nst, int mtiles, int ntiles,
    uint32_t wbytes, int ksplit, int ks, float *__restrict__ part, long pstride, int prio) {
  constexpr int BM = 32 * TM, BN = 32 * WN, KB = KQ4_REC_KB, GB = BM / 64;
  constexpr int NQ = KB * TM;                       // tiles of a stage
  constexpr int CBK = WF ? KQ8_STREAM_CB : KQ4_STREAM_CB;
  constexpr int CHK = WF ? KQ8_STREAM_CHUNK : KQ4_STREAM_CHUNK;
  constexpr int AP = GB * KB * 2 / WN;              // 1-KB code planes each wave brings in (1 or 2)
  static_assert(AP == 2 || (AP == 1 && WF == 0), "kq4_gemm_rec_kernel: a record or (q4) half of one per wave");
  // a wave's part of a stage in LDS: codes, their scales, its row set's scales and weights
  constexpr int XO = AP * 1024, SO = XO + KQ4_REC_X, WO = SO + 128, RW = WO + (WF ? 2048 : 1024);
  constexpr int SB = WN * RW, OPS = AP + (WF ? 4 : 3);   // a stage; its loads per wave
  __shared__ __align__(16) uint8_t ring[3 * SB];

  // XCD-aware tile order (kq4_gemm_kernel)
  const int ntile = mtiles * ntiles * ksplit;
  const int wg = blockIdx.x;
  const int xcd = wg & 7, q8 = ntile >> 3, r8 = ntile & 7;
  const int vtile = xcd * q8 + (xcd < r8 ? xcd : r8) + (wg >> 3);
  const int tile = vtile % (mtiles * ntiles);
  const int m0 = (tile % mtiles) * BM;
  const int n0 = (tile / mtiles) * BN;
  int k0 = 0, nb = nbt;
  if (ksplit > 1) {
    const int sl = vtile / (mtiles * ntiles);
    k0 = sl * ks;
    nb = min(ks, nbt - k0);
    if (sl > 0) {
      out = part + (size_t)(sl - 1) * pstride;
      res = nullptr;
    }
  }
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, half = lane >> 5;

  const int ngrp = (n_tok + 63) >> 6;
  const uint32_t nrec = (uint32_t)(ngrp * nbt);
  const kq4_rsrc4 ra = kq4_rsrc_at(rec, nrec * KQ4_REC_A, 0);
  const kq4_rsrc4 rx = kq4_rsrc_at(rec + (size_t)nrec * KQ4_REC_A, nrec * KQ4_REC_X, XO);
  const kq4_rsrc4 rw = kq4_rsrc_at(w, wbytes, WO);
  const uint32_t v16 = 16u * lane, v4 = 4u * lane;
  // this wave's row set (past the matrix: the last one again, computed on and not stored) and record
  // (AP = 2: record `wave`, AP = 1: plane wave % 2 of record wave / 2; group-major, KB blocks each)
  const uint32_t sb = (uint32_t)min((n0 >> 5) + wave, ((rows + 31) >> 5) - 1) * (uint32_t)nst * CHK;
  const int rr = AP == 2 ? wave : wave >> 1, rbl = rr % KB;
  const uint32_t r0 = (uint32_t)(min((m0 >> 6) + rr / KB, ngrp - 1) * nbt + k0);
  const uint32_t a0 = r0 * KQ4_REC_A + (AP == 2 ? 0u : (wave & 1) * 1024u), x0 = r0 * KQ4_REC_X;
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t *)&ring[0];
  const uint32_t ldw = lds0 + wave * RW;

  float acc[TM][16];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;

  // This wave's loads of the stage of blocks b0, b0 + 1 into ring slot `slot`, straight to LDS (a
  // block past the slice: its last one again, against zero weights). The scales' 128 B go by lanes
  // 0-31 (through the exec mask, all set here: a branch in the pipelined loop costs its schedule).
  auto load = [&](uint32_t slot, int b0) {
    const int b = k0 + b0, ba = min(b0 + rbl, nb - 1);
    const uint32_t sc = sb + (uint32_t)((b / CBK) * CHK);
    const uint32_t sw = sc + (uint32_t)(WF ? 1024 * (b & 7) : 1024 * ((b & 15) >> 1));
    const uint32_t ss = sc + (uint32_t)(8192 + (WF ? 2 * (b & 7) : 512 * ((b & 15) >> 3) + 2 * (b & 7))) +
                        (uint32_t)(WO - SO);
    const uint32_t sa = a0 + (uint32_t)ba * KQ4_REC_A, sx = x0 + (uint32_t)ba * KQ4_REC_X;
    const uint32_t l = ldw + slot;
#define KQ4_REC_TAIL                                                     \
  "buffer_load_dword %2, %4, %6 offen offset:%9 lds\n\t"                 \
  "buffer_load_dwordx4 %1, %5, %7 offen offset:%10 lds\n\t"
#define KQ4_REC_SC                                                       \
  "s_mov_b32 exec_hi, 0\n\t"                                             \
  "buffer_load_dword %1, %5, %8 offen offset:%11 lds\n\t"                \
  "s_mov_b32 exec_hi, -1"
#define KQ4_REC_ARGS                                                                            \
  ::"s"(l), "v"(v16), "v"(v4), "s"(ra), "s"(rx), "s"(rw), "s"(sx), "s"(sw), "s"(ss), "n"(XO),   \
      "n"(WO), "n"(SO), "s"(sa), "n"(WO + 1024) : "memory", "m0"
    if constexpr (AP == 1)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                   "buffer_load_dwordx4 %1, %3, %12 offen lds\n\t" KQ4_REC_TAIL
                   KQ4_REC_SC KQ4_REC_ARGS);
    else if constexpr (WF == 0)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                   "buffer_load_dwordx4 %1, %3, %12 offen lds\n\t"
                   "buffer_load_dwordx4 %1, %3, %12 offen offset:1024 lds\n\t" KQ4_REC_TAIL
                   KQ4_REC_SC KQ4_REC_ARGS);
    else
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                   "buffer_load_dwordx4 %1, %3, %12 offen lds\n\t"
                   "buffer_load_dwordx4 %1, %3, %12 offen offset:1024 lds\n\t" KQ4_REC_TAIL
                   "buffer_load_dwordx4 %1, %5, %7 offen offset:%13 lds\n\t" KQ4_REC_SC KQ4_REC_ARGS);
#undef KQ4_REC_TAIL
#undef KQ4_REC_SC
#undef KQ4_REC_ARGS
  };

  const kq4_v16i zi = {0};
  const kq4_v16f zf = {0};
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  typedef const volatile __attribute__((address_space(3))) kq4_v4i *lds16;
  typedef const volatile __attribute__((address_space(3))) v2u *lds8;
  typedef const volatile __attribute__((address_space(3))) uint32_t *lds4;
  const uint32_t la = lds0 + (AP == 2 ? half * 1024u : half * (uint32_t)RW) + l32 * 16u;
  const uint32_t lx = lds0 + XO + l32 * 4u;
  const uint32_t lw = ldw + WO + v16, ls = ldw + SO + l32 * 4u;
  kq4_v4i af[2], bf[2];
  kq4_v4h xv, wd;
  kq4_v16i S[2];
  kq4_v16f sc;
  uint32_t ws;    // the two row scales of the stage whose weights come next
  // tile q of a stage: block q / TM, token tile q % TM of the record of its group
  auto rslot = [](int q) { return (uint32_t)((((q % TM) >> 1) * KB + q / TM) * (AP == 2 ? 1 : 2) * RW); };
  auto ld_a = [&](int q, uint32_t base) {
    af[q & 1] = *(lds16)(base + rslot(q) + (uint32_t)((q & 1) * 512));
  };
  auto ld_x = [&](int q, uint32_t base) {
    const v2u u = {*(lds4)(base + rslot(q) + (uint32_t)((q & 1) * 128)), 0u};
    xv = __builtin_bit_cast(kq4_v4h, u);
  };
  v2u wr;
  auto ld_w = [&](int bl, uint32_t base) {
    if constexpr (WF) bf[bl] = *(lds16)(base + (uint32_t)(1024 * bl));
    else wr = *(lds8)(base + (uint32_t)(8 * bl));
  };
  auto unpack = [&](int bl) {
    if constexpr (WF == 0) {
      uint32_t o[4];
      kq4_unpack_half(wr[0], wr[1], o);
      bf[bl] = kq4_v4i{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
    }
  };
  auto set_wd = [&](uint32_t s) {
    const v2u u = {s, 0u};
    wd = __builtin_bit_cast(kq4_v4h, u);
  };
  auto issue_s = [&](int q) {
    S[q & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[q & 1], bf[(q / TM) & 1], zi, 0, 0, 0);
  };
  // 2 * wd * f16r(xd), exact: both lane halves (K slots 0 and 4) hold the same two scales, so the
  // product is added to itself; the accumulators are kept scaled by that 2 and by the 16 of the q4
  // block sums (both powers of two, so every rounding is the chain's), and scaled back at the end
  auto issue_sc = [&] { sc = __builtin_amdgcn_mfma_f32_32x32x8f16(xv, wd, zf, 0, 0, 0); };
  constexpr float OSC = WF ? 0.5f : 0.03125f;

  const int lastb = (nb - 1) / KB * KB;
  uint32_t sl0 = 0, sl1 = SB, sl2 = 2 * SB;   // ring slots of the current, next, second next stage

  load(sl0, 0);
  load(sl1, min(KB, lastb));
  load(sl2, min(2 * KB, lastb));
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * OPS) : "memory");
  ld_w(0, lw);
  ws = *(lds4)ls;
  unpack(0);
  set_wd(ws & 0xFFFFu);
  ld_a(0, la);
  ld_x(0, lx);
  ld_w(1, lw);
  issue_s(0);
  issue_sc();
  ld_a(1, la);
  ld_x(1, lx);
  for (int b0 = 0; b0 < nb; b0 += KB) {
    if (prio && (b0 & 7) == 0) kq4_prio_by_progress(8 * b0 / nb);
    const uint32_t ca = la + sl0, cx = lx + sl0, na = la + sl1, nx = lx + sl1;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int bl = q / TM, i = q % TM;
      __builtin_amdgcn_sched_barrier(0);
      issue_s(q + 1);
      if (q == NQ - 2) {   // every wave is done with this stage's slot; the next stage's is full
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        load(sl0, min(b0 + 3 * KB, lastb));
      }
      if (q + 2 < NQ) ld_a(q + 2, ca);
      else ld_a(q + 2 - NQ, na);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        if constexpr (WF) acc[i][v] = acc[i][v] + sc[v] * (float)S[q & 1][v];
        else acc[i][v] = fmaf((float)S[q & 1][v], sc[v], acc[i][v]);
      }
      __builtin_amdgcn_sched_barrier(0);
      issue_sc();
      if (q + 2 < NQ) ld_x(q + 2, cx);
      else ld_x(q + 2 - NQ, nx);
      if (i == TM - 2) set_wd(bl == 0 ? ws >> 16 : ws & 0xFFFFu);
      __builtin_amdgcn_sched_barrier(0);
      if (i == 0) unpack(1 - bl);   // the next block's weights
      if (bl == 0 && i == TM - 2) {
        // this wave's loads of the next stage are in LDS (the second next's may be under way)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(OPS) : "memory");
        ws = *(lds4)(ls + sl1);
      }
      // the codes of the block after the next (q8: bf[bl]'s last use is issued)
      if (i == TM - 1) ld_w(bl, lw + sl1);
    }
    const uint32_t x = sl0;
    sl0 = sl1;
    sl1 = sl2;
    sl2 = x;
  }

  const int row = n0 + 32 * wave + l32;
  if (row >= rows) return;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int tok = m0 + 32 * i + 8 * (v >> 2) + 4 * half + (v & 3);
      if (tok >= n_tok) continue;
      const size_t o = (size_t)tok * rows + row;
      const float r = acc[i][v] * OSC;
      out[o] = res ? res[o] + r : r;
    }
}

template <int TM, int WN, int WF, int NW>
static hipError_t rec_launch(float *out, const float *res, const uint8_t *w, const uint8_t *rec,
                             int rows, int cols, int n_tok, int ksplit, int ks, float *part,
                             int prio, hipStream_t s) {
  const int cb = WF ? KQ8_STREAM_CB : KQ4_STREAM_CB;
  const int nb = cols / 32, nst = (nb + cb - 1) / cb;
  const int mtiles = (n_tok + 32 * TM - 1) / (32 * TM), ntiles = (rows + 32 * WN - 1) / (32 * WN);
  hipLaunchKernelGGL((kq4_gemm_rec_kernel<TM, WN, WF, NW>),
                     dim3((unsigned)(mtiles * ntiles * ksplit)), dim3(64 * WN), 0, s, out,
                     ksplit > 1 ? nullptr : res, w, rec, rows, n_tok, nb, nst, mtiles, ntiles,
                     (uint32_t)(WF ? kq8_stream_bytes(rows, cols) : kq4_stream_bytes(rows, cols)),
                     ksplit, ks, part, (long)n_tok * rows, prio);
  return hipGetLastError();
}

int kq4_rec_has_tile(int tile, int wf) { return tile == 1 || (tile == 2 && !wf); }

int kq4_gemm_rec_ok(int rows, int cols, int n_tok, int wf) {
  return kq4_rec_bytes(n_tok, cols) < KQ4_OOB - 4096 &&
         (wf ? kq8_stream_bytes(rows, cols) : kq4_stream_bytes(rows, cols)) < KQ4_OOB - 4096;
}

// The rule, from graph replays with the quantizer (us, token-major form / this one). A launch runs in
// rounds of three 128 x 128 (q4, q8) or four 64 x 128 (q4) workgroups per CU, a 64 x 128 round taking
// 0.71 of a 128 x 128 one's time:
//   * q4, 64 x 64 plans (one token tile, or short K): token-major (Qwen3-8B QKV 6144 x 4096 at M = 24
//     17.5 / 19.8, Qwen3-VL-2B gate 6144 x 2048 at M = 128 19.6 / 25.0: this form's ring takes longer
//     to fill);
//   * q4, K-split plans: the plan's tile (8B down 4096 x 12288 at M = 96 / 256 / 768 32.2 / 30.6,
//     49.1 / 44.7, 116.0 / 105.8);
//   * q4, unsplit: the tile of fewer rounds (8B gate 12288 x 4096 at M = 512, 64 x 128: 75.9 / 68.4;
//     M = 768 and 2048, 128 x 128: 118.1 / 107.7, 267.8 / 232.3; QKV M = 2048 150.9 / 120.0);
//   * q8: 128 x 128 only, split or from two tiles per CU (8B gate M = 768 / 1000 / 2048 137.2 / 127.5,
//     162.7 / 143.3, 330.6 / 280.3; at M = 512, 384 tiles, 85.2 / 95.6; there is no 64 x 128 form:
//     at twice the weight bytes it was slower throughout).
int kq4_rec_tile(int n_tok, int rows, int wf, int ncu, const KQ4GemmPlan &plan) {
  const long cu = ncu < 1 ? 1 : ncu;
  const long t1 = (long)((n_tok + 127) / 128) * ((rows + 127) / 128);
  const long t2 = (long)((n_tok + 63) / 64) * ((rows + 127) / 128);
  if (wf) return plan.ksplit > 1 ? plan.tile == 1 : t1 >= 2 * cu;
  if (plan.tile == 3) return 0;
  if (plan.ksplit > 1) return kq4_rec_has_tile(plan.tile, wf) ? plan.tile : 0;
  const long r1 = (t1 + 3 * cu - 1) / (3 * cu), r2 = (t2 + 4 * cu - 1) / (4 * cu);
  return 100 * r1 <= 71 * r2 ? 1 : 2;
}

int kq4_launch_gemm_rec(float *out, const float *res, const uint8_t *w, const uint8_t *rec, int rows,
                        int cols, int n_tok, int wf, hipStream_t s, int tile, int ksplit,
                        float *part, int prio) {
  if (n_tok <= 0 || rows <= 0) return 0;
  const int ks = kq4_split_len(cols / 32, wf ? KQ8_STREAM_CB : KQ4_STREAM_CB, ksplit);
  if (!kq4_gemm_rec_ok(rows, cols, n_tok, wf) || !kq4_rec_has_tile(tile, wf) || ksplit < 1 ||
      ksplit > KQ4_GEMM_SPLIT_MAX || !ks || (ksplit > 1 && !part))
    return (int)hipErrorInvalidValue;
  const hipError_t e =
      wf          ? rec_launch<4, 4, 1, 3>(out, res, w, rec, rows, cols, n_tok, ksplit, ks, part, prio, s)
      : tile == 1 ? rec_launch<4, 4, 0, 3>(out, res, w, rec, rows, cols, n_tok, ksplit, ks, part, prio, s)
                  : rec_launch<2, 4, 0, 4>(out, res, w, rec, rows, cols, n_tok, ksplit, ks, part, prio, s);
  if (e != hipSuccess || ksplit < 2) return (int)e;
  return kq4_launch_split_reduce(out, res, part, ksplit - 1, (long)n_tok * rows, s);
}
