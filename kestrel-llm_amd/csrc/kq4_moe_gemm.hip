// kq4_moe_gemm.hip - the expert projections of the MoE FFN as a grouped GEMM (int8 MFMA, gfx950), for
// launches with enough (token, rank) pairs per expert. The same chains as kq4_moe.hip, bit for bit:
//   gate/up  acc = fl(acc + fl(fl(sc*xd) * S)) over blocks ascending (vllm_safetensors.c:11861-11924),
//            av = fl(fl(g / fl(1 + exp(-g))) * u) re-quantized per 32 rows (:12671-12675)
//   down     the same chain over the expert's column band, unweighted partials (:14799-14840)
#include "kq4_common.h"
#include "kq4_internal.h"

typedef int kq4_v4i __attribute__((ext_vector_type(4)));
typedef int kq4_v16i __attribute__((ext_vector_type(16)));
typedef float kq4_v32f __attribute__((ext_vector_type(32)));

struct KQ4MoeGemmArgs {
  const uint8_t *w0, *w1;   // the two matrices whose row sets a wave takes (G, U; D, D)
  const int8_t *aq;         // activation codes, row-major (X per token; av per pair)
  const float *ad;          // their scales
  const int *tiles;         // [1 + 4 * k]: count, then per tile expert, offset in ex_pair, pairs (<= 32)
  const int *ex_pair;       // (t*tk+j) grouped by expert
  int8_t *avq;              // gate/up: outputs
  float *avd, *g_out, *u_out, *av_out;
  float *P;                 // down: output [pair][d]
  uint32_t wbytes0, wbytes1, abytes, dbytes;
  int nst;                  // stream-layout stages of a weight row set
  int nb;                   // blocks of K (even)
  int tk;                   // gate/up: pairs per token
  int ef, d;
  int nrg;                  // workgroups per tile (4 row sets, or 4 pairs of them, each)
  int nsets;                // row sets: ef/32 (gate/up), d/32 (down)
};

// Workgroup = 4 waves, one tile of up to 32 pairs of one expert; wave w takes the row set rg*4 + w of G and
// of U (gate/up) or the row sets 2*(rg*4 + w) and + 1 of D (down): two MFMA tiles, whose scale products
// fl(wd*xd) come from one v_mfma_f32_32x32x1_2b_f32 (its two blocks are the two row sets).
// Loads go straight to LDS through a three-stage ring as in kq4_gemm_rec_kernel; a pair's activation
// row is gathered there by its lane's address, so nothing is copied into expert order first.
// Bound by the VALU work of the chain (a conversion, a multiply and an add per block, row and pair: a VALU
// instruction every 4.6 SIMD cycles with 2.8 waves resident, the matrix unit busy 20 %), with a fifth of
// the tiles' pairs padding at 64 pairs per expert on average. 32-pair tiles, not 64: with four accumulator tiles
// and the scale products a wave needs more than 128 VGPRs and spills. Rings of 4 and 5 stages
// (3 and 2 workgroups per CU) were 4% and 17% slower. Qwen3-30B-A3B's FFN at 1024 tokens (8192 pairs, kernel
// trace of the layer): gate/up 482 us -> 157 us (164 TMAC/s) and down 148 us -> 84 us against
// kq4_moe.hip's kernels, which unpack an expert's weights again for every 4 to 8 of its pairs and contract on v_dot4.
template <int DOWN>
__global__ __launch_bounds__(256, 4) void kq4_moe_gemm_kernel(KQ4MoeGemmArgs a) {
  constexpr int KB = 2, NQ = 2 * KB;
  constexpr int ST = 3;   // stages of the ring
  // a wave's part of a stage in LDS: 32 rows' half codes of a block, 32 scales of a block, its row
  // sets' scales and weights
  constexpr int XO = 512, SO0 = XO + 128, SO1 = SO0 + 128, WO0 = SO1 + 128, WO1 = WO0 + 1024;
  constexpr int RW = WO1 + 1024, SB = 4 * RW, OPS = 6;
  __shared__ __align__(16) uint8_t ring[ST * SB];
  __shared__ int sp[32];
  // XCD-aware order over the tiles there are: an XCD takes consecutive (tile, row group) items, so a
  // tile's activations and an expert's weights are shared in its L2
  const int n = a.tiles[0] * a.nrg, wg = blockIdx.x;
  if (wg >= n) return;
  const int xcd = wg & 7, q8 = n >> 3, r8 = n & 7;
  const int it = xcd * q8 + (xcd < r8 ? xcd : r8) + (wg >> 3);
  const int k = it / a.nrg, rg = it - k * a.nrg;
  const int e = __builtin_amdgcn_readfirstlane(a.tiles[1 + 4 * k]);
  const int off = __builtin_amdgcn_readfirstlane(a.tiles[2 + 4 * k]);
  const int cnt = __builtin_amdgcn_readfirstlane(a.tiles[3 + 4 * k]);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int nb = a.nb;

  const int su = rg * 4 + wave;   // row set (gate/up) or pair of row sets (down)
  const int s0 = DOWN ? min(2 * su, a.nsets - 1) : min(su, a.nsets - 1);
  const int s1 = DOWN ? min(2 * su + 1, a.nsets - 1) : s0;
  const int kb0 = DOWN ? e * nb : 0;                       // first block of the weights' band
  const int r0 = DOWN ? 0 : e * a.nsets;                   // first row set of the expert
  const uint32_t b0w = (uint32_t)((r0 + s0) * a.nst) * KQ4_STREAM_CHUNK;
  const uint32_t b1w = (uint32_t)((r0 + s1) * a.nst) * KQ4_STREAM_CHUNK;
  const kq4_rsrc4 ra = kq4_rsrc_at(a.aq, a.abytes, 0);
  const kq4_rsrc4 rx = kq4_rsrc_at(a.ad, a.dbytes, XO);
  const kq4_rsrc4 rw0 = kq4_rsrc_at(a.w0, a.wbytes0, WO0), rw1 = kq4_rsrc_at(a.w1, a.wbytes1, WO1);
  const uint32_t v16 = 16u * lane;
  // the lane's pair (past the tile: its last one again, computed on and not stored)
  const int pr = a.ex_pair[off + min(l32, cnt - 1)];
  if (threadIdx.x < 32) sp[threadIdx.x] = pr;
  const uint32_t row = (uint32_t)(DOWN ? pr : pr / a.tk);
  const uint32_t va = row * (uint32_t)(32 * nb), vx = row * (uint32_t)(4 * nb);
  const uint32_t lds0 =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t *)ring;
  const uint32_t ldw = lds0 + wave * RW;
  const int pbl = wave >> 1, phf = wave & 1;   // the block and half of the codes this wave brings in

  float acc[2][16];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[g][v] = 0.0f;

  auto load = [&](uint32_t slot, int b0) {
    const int b = kb0 + b0;
    const uint32_t c = (uint32_t)((b >> 4) * KQ4_STREAM_CHUNK);
    const uint32_t cu = c + (uint32_t)(1024 * ((b & 15) >> 1));
    const uint32_t cs = c + (uint32_t)(8192 + 512 * ((b & 15) >> 3) + 2 * (b & 7));
    const uint32_t sa = (uint32_t)(32 * (b0 + pbl) + 16 * phf), sx = (uint32_t)(4 * (b0 + pbl));
    asm volatile(
        "s_mov_b32 m0, %0\n\ts_nop 0\n\t"
        "buffer_load_dwordx4 %3, %6, %10 offen offset:%15 lds\n\t"
        "buffer_load_dwordx4 %3, %7, %11 offen offset:%16 lds\n\t"
        "s_mov_b32 exec_hi, 0\n\t"
        "buffer_load_dwordx4 %1, %4, %8 offen lds\n\t"
        "buffer_load_dword %2, %5, %9 offen offset:%14 lds\n\t"
        "buffer_load_dword %3, %6, %12 offen offset:%17 lds\n\t"
        "buffer_load_dword %3, %7, %13 offen offset:%18 lds\n\t"
        "s_mov_b32 exec_hi, -1"
        ::"s"(ldw + slot), "v"(va), "v"(vx), "v"(v16), "s"(ra), "s"(rx), "s"(rw0), "s"(rw1), "s"(sa),
        "s"(sx), "s"(b0w + cu), "s"(b1w + cu), "s"(b0w + cs + (WO0 - SO0)),
        "s"(b1w + cs + (WO1 - SO1)), "n"(XO), "n"(WO0), "n"(WO1), "n"(SO0), "n"(SO1)
        : "memory", "m0");
  };

  const kq4_v16i zi = {0};
  const kq4_v32f z32 = {0};
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  typedef const volatile __attribute__((address_space(3))) kq4_v4i *lds16;
  typedef const volatile __attribute__((address_space(3))) v2u *lds8;
  typedef const volatile __attribute__((address_space(3))) uint32_t *lds4;
  typedef const volatile __attribute__((address_space(3))) float *ldsf;
  const uint32_t la = lds0 + half * (uint32_t)RW + l32 * 16u, lx = lds0 + XO + l32 * 4u;
  const uint32_t lw = ldw + WO0 + v16, ls = ldw + SO0 + half * 128u + l32 * 4u;
  kq4_v4i af[2], bf[2];
  kq4_v16i S[2];
  kq4_v32f sc;
  v2u wr[2];
  uint32_t ws;
  float xv, wv;
  // block t's codes are in the waves 2t, 2t + 1's parts, its scales in 2t's
  auto ld_a = [&](int t, uint32_t base) { af[t & 1] = *(lds16)(base + (uint32_t)((t & 1) * 2 * RW)); };
  auto ld_x = [&](int t, uint32_t base) { xv = *(ldsf)(base + (uint32_t)((t & 1) * 2 * RW)); };
  auto ld_w = [&](int bl, uint32_t base) {
    wr[0] = *(lds8)(base + (uint32_t)(8 * bl));
    wr[1] = *(lds8)(base + (uint32_t)(WO1 - WO0 + 8 * bl));
  };
  auto unpack = [&] {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      uint32_t o[4];
      kq4_unpack_half(wr[g][0], wr[g][1], o);
      bf[g] = kq4_v4i{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
    }
  };
  // lanes 0-31: the first row set's scales, 32-63: the second's. S comes as 16*S, so wd / 16: every
  // step is scaled by a power of two far from underflow (wd >= 2^-24, xd >= 1e-10/127). (Where wd * xd
  // itself overflows, activations beyond 6e35, a zero S gives 0 here and NaN in the chain.)
  auto set_w = [&](uint32_t s) { wv = kq4_h2f(s) * 0.0625f; };
  auto issue_s = [&](int q) {
    S[q & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[(q >> 1) & 1], bf[q & 1], zi, 0, 0, 0);
  };
  auto issue_sc = [&] { sc = __builtin_amdgcn_mfma_f32_32x32x1f32(xv, wv, z32, 0, 0, 0); };

  const int lastb = nb - KB;
  uint32_t sl[ST];
#pragma unroll
  for (int i = 0; i < ST; ++i) {
    sl[i] = (uint32_t)(i * SB);
    load(sl[i], min(i * KB, lastb));
  }
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 1) * OPS) : "memory");
  ld_w(0, lw);
  ws = *(lds4)ls;
  unpack();
  set_w(ws);
  ld_a(0, la);
  ld_x(0, lx);
  ld_w(1, lw);
  issue_s(0);
  issue_sc();
  set_w(ws >> 16);
  ld_a(1, la);
  ld_x(1, lx);
  for (int b0 = 0; b0 < nb; b0 += KB) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int t = q >> 1, g = q & 1;   // block of the stage, row set
      __builtin_amdgcn_sched_barrier(0);
      issue_s(q + 1);
      if (q == 1) {        // every wave is done with this stage's slot; the next stage's is full
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        load(sl[0], min(b0 + ST * KB, lastb));
      }
      if (g == 1) ld_a(t, la + sl[1]);   // block t + 1's products take the other fragments
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[g][v] = acc[g][v] + sc[16 * g + v] * (float)S[g][v];
      __builtin_amdgcn_sched_barrier(0);
      if (g == 1) {
        issue_sc();        // block t + 1's
        ld_x(t, lx + sl[1]);
        set_w(t ? ws >> 16 : ws);
        ld_w(t, lw + sl[1]);
      } else {
        // the next block's weights (this block's products are issued)
        __builtin_amdgcn_sched_barrier(0);
        unpack();
        if (t == 0) {
          // this wave's loads of the next stage are in LDS (the second next's may be under way)
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * OPS) : "memory");
          ws = *(lds4)(ls + sl[1]);
        }
      }
    }
    const uint32_t x = sl[0];
#pragma unroll
    for (int i = 1; i < ST; ++i) sl[i - 1] = sl[i];
    sl[ST - 1] = x;
  }

  if (DOWN) {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int s = 2 * su + g;
      if (s >= a.nsets) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = 8 * (v >> 2) + 4 * half + (v & 3);
        if (r < cnt) a.P[(size_t)sp[r] * a.d + 32 * s + l32] = acc[g][v];
      }
    }
  } else if (su < a.nsets) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = 8 * (v >> 2) + 4 * half + (v & 3);
      const float gt = acc[0][v], up = acc[1][v];
      const float av = (gt / (1.0f + (float)exp((double)-gt))) * up;
      const float amax = kq4_max32(fmaxf(fabsf(av), 1e-10f));   // the set's 32 rows: one av block
      const float dq = amax / 127.0f;
      int qv = (int)(av / dq + 0.5f);
      qv = qv > 127 ? 127 : (qv < -127 ? -127 : qv);
      if (r < cnt) {
        const int p = sp[r];
        const size_t o = (size_t)p * a.ef + 32 * su + l32;
        a.avq[o] = (int8_t)qv;
        if (l32 == 0) a.avd[(size_t)p * a.nsets + su] = dq;
        if (a.g_out) { a.g_out[o] = gt; a.u_out[o] = up; }
        if (a.av_out) a.av_out[o] = av;
      }
    }
  }
}

// The projections as grouped GEMMs from 6 pairs per expert slot on average, or 10 where the gate/up
// tiles (at least one per slot) leave CUs without a workgroup: the kernel's time is nearly flat up
// to 32 pairs (a tile is a tile), kq4_moe_gu_kernel's and the down kernels' grow with the pairs. A
// whole FFN at 4 / 6 / 8 pairs on average, this form against those, in us: d 2048, ef 768, 128
// experts 99 / 100 / 99 against 92 / 106 / 131; d 2048, ef 1024, 64 experts 63 / 63 / 65 against
// 69 / 86 / 109; d 1024, ef 512, 32 experts (128 tiles) 33.2 / 33.8 / 34.3 against 23.4 / 31.1 /
// 32.0, and at 12 pairs 35.2 against 38.5. Even block counts (a stage is two blocks).
int kq4_moe_gemm_ok(int T, int tk, int ne, int d, int ef) {
  const long np_ = (long)T * tk, slots = ne < np_ ? ne : np_, wgs = slots * ((ef / 32 + 3) / 4);
  return (d / 32) % 2 == 0 && (ef / 32) % 2 == 0 && np_ >= slots * (wgs >= 256 ? 6 : 10) &&
         (size_t)T * d < KQ4_OOB - 4096 && (size_t)np_ * ef < KQ4_OOB - 4096 &&
         kq4_stream_bytes(ne * ef, d) < KQ4_OOB - 4096 && kq4_stream_bytes(d, ne * ef) < KQ4_OOB - 4096;
}

int kq4_launch_moe_gemm(int down, const uint8_t *w0, const uint8_t *w1, const KQ4MoeWs &ws, int T,
                        int tk, int ne, int d, int ef, float *g_out, float *u_out, float *av_out,
                        hipStream_t s) {
  const int np_ = T * tk, slots = ne < np_ ? ne : np_;
  KQ4MoeGemmArgs a = {};
  a.w0 = w0;
  a.w1 = w1;
  a.aq = down ? ws.avq : ws.xq;
  a.ad = down ? ws.avd : ws.xd;
  a.tiles = ws.tiles;
  a.ex_pair = ws.ex_pair;
  a.avq = ws.avq;
  a.avd = ws.avd;
  a.g_out = g_out;
  a.u_out = u_out;
  a.av_out = av_out;
  a.P = ws.P;
  a.wbytes0 = a.wbytes1 = (uint32_t)(down ? kq4_stream_bytes(d, ne * ef) : kq4_stream_bytes(ne * ef, d));
  const int rows = down ? np_ : T, cols = down ? ef : d;
  a.abytes = (uint32_t)((size_t)rows * cols);
  a.dbytes = (uint32_t)((size_t)rows * (cols / 32) * 4);
  a.nb = cols / 32;
  a.nst = ((down ? ne * ef : d) / 32 + KQ4_STREAM_CB - 1) / KQ4_STREAM_CB;
  a.tk = tk;
  a.ef = ef;
  a.d = d;
  a.nsets = (down ? d : ef) / 32;
  a.nrg = (a.nsets + (down ? 7 : 3)) / (down ? 8 : 4);
  const unsigned grid = (unsigned)((np_ / 32 + slots) * a.nrg);
  auto k = down ? kq4_moe_gemm_kernel<1> : kq4_moe_gemm_kernel<0>;
  hipLaunchKernelGGL(k, dim3(grid), dim3(256), 0, s, a);
  return (int)hipGetLastError();
}
