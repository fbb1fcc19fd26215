// Grouped expert GEMMs on MFMA for batched decode and prefill (gfx950).
//
// After dispatch (pairs sorted by expert), every expert's tokens form a dense
// [tokens x K] operand, so the SwiGLU up+gate projection and the down
// projection become per-expert GEMMs: y = W_e (rows x K) . X_e^T (K x tokens).
//
// Forms, by pairs per expert and by K:
//  * decode batches (few pairs): 16-pair tiles whose rows lie in LDS for all of
//    K, up to 4096 values (gd), else K split over the waves with operands in
//    registers (ks), each stage by its own K;
//  * prefill: tiles of 64 or 32 pairs x 256 rows, K in steps through LDS (gp).
// gd and gp multiply on the scaled 8-bit matrix instructions: codes as FP4,
// activations as mx rows (mx.h).  ks multiplies in bf16: each lane expands its
// packed words with expand_word (common.h) into bf16x2 dwords of 1 + c/f --
// exactly the dword order of the bf16 x' pairs, an (arbitrary but shared)
// permutation of K inside each word -- against x' = f * x pairs; the MFMA then
// accumulates sum (f + c) x, and subtracting C_t = sum (f + 1) x per token
// leaves sum (c - 1) x, the ternary product (float32 accumulation).
//
// v_mfma_f32_16x16x32_bf16 lane layout (checked on the device):
//   A: lane l holds row l%16, k 8(l/16)..+8;  B: col l%16, k 8(l/16)..+8;
//   C: lane l holds col l%16, rows 4(l/16)..+4.
//
// Stage 1 computes h (each wave holds up rows and the matching gate rows, so
// SwiGLU is applied in registers), rounded to bf16 like the reference's x.dtype
// store (ternary_expert.py:441), in the layout the down stage reads and
// optionally in the plain [slot, I] layout.  Stage 2 writes each pair's down
// output rounded to bf16 (ternary_expert.py:208); a gather kernel then forms
// y[t] = sum_j w[t,j] out[pair(t,j)] (+ residual) in float32
// (fused_norm.py:83-96).
#include <mutex>

#include "mfma.h"
#include "mx.h"

namespace ma {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));


__device__ __forceinline__ f32x4_t mfma_bf16(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// Tile `tile` of a grouped launch with NT pairs per tile -> expert e, first
// sorted position pos0 and pair count np.  Each wave computes it (no LDS).
// Returns false for tiles past the end (the grid is an upper bound).
__device__ __forceinline__ bool decode_tile(const int32_t* __restrict__ offsets, int n_exp,
                                            int64_t tile, int nt, int& e, int& pos0, int& np) {
  const int lane = threadIdx.x & 63;
  int run = 0;  // tiles of the experts before this 64-expert slice
  // The first 256 experts' offsets in one round trip (indices past the end read
  // the last one: no tiles); a load per slice was a round trip each.
  constexpr int kAhead = 4;
  int a0[kAhead], a1[kAhead];
#pragma unroll
  for (int i = 0; i < kAhead; ++i) {
    const int ee = 64 * i + lane;
    a0[i] = offsets[ee < n_exp ? ee : n_exp];
    a1[i] = offsets[ee + 1 < n_exp ? ee + 1 : n_exp];
  }
  // the slice of the tile, by the slices' totals (side by side, where a scan of
  // one slice after the other is a chain of lane exchanges each)
  int first = 0;
  if (n_exp > 64) {
    int total[kAhead - 1];
#pragma unroll
    for (int i = 0; i < kAhead - 1; ++i)
      total[i] = static_cast<int>(group_sum<64>(static_cast<float>((a1[i] - a0[i] + nt - 1) / nt)));
#pragma unroll
    for (int i = 0; i < kAhead - 1; ++i)
      if (first == 64 * i && 64 * (i + 1) < n_exp && tile >= run + total[i]) {
        run += total[i];
        first = 64 * (i + 1);
      }
  }
  for (int base = first; base < n_exp; base += 64) {
    const int ee = base + lane;
    int o0 = base == 0 ? a0[0] : base == 64 ? a0[1] : base == 128 ? a0[2] : a0[3];
    int o1 = base == 0 ? a1[0] : base == 64 ? a1[1] : base == 128 ? a1[2] : a1[3];
    if (base >= 64 * kAhead) {
      o0 = offsets[ee < n_exp ? ee : n_exp];
      o1 = offsets[ee + 1 < n_exp ? ee + 1 : n_exp];
    }
    const int tiles = (o1 - o0 + nt - 1) / nt;
    int incl = tiles;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    const int excl = incl - tiles;
    const bool mine = ee < n_exp && tile >= run + excl && tile < run + incl;
    const uint64_t m = __ballot(mine);
    if (m) {
      const int src = __ffsll(static_cast<unsigned long long>(m)) - 1;
      e = __shfl(ee, src, 64);
      const int t_in = static_cast<int>(tile) - run - __shfl(excl, src, 64);
      const int start = __shfl(o0, src, 64);
      const int end = __shfl(o1, src, 64);
      pos0 = start + t_in * nt;
      np = min(nt, end - pos0);
      return true;
    }
    run += __shfl(incl, 63, 64);
  }
  return false;
}

// sum (f + 1)/f * (lo + hi) over 8 x' pair dwords (recovers sum (f + 1) x).
__device__ __forceinline__ float pairs_cst(const uint32_t pr[8]) {
  float c = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float f = pair_scale(j);
    c += ((f + 1.0f) / f) * (__uint_as_float(pr[j] << 16) + __uint_as_float(pr[j] & 0xffff0000u));
  }
  return c;
}

// ---------------------------------------------------------------------------
// Decode form of rows past 4096 values: 16-pair tiles, K split over the KW waves
// of a workgroup, each wave's operands loaded and built in registers (no LDS
// staging) and the partial tiles added in wave order through LDS; with a
// handful of tokens per expert, a K walk per workgroup left the chip idle.
// Same per-word arithmetic as the kernels above; every sum has a fixed order.
// ---------------------------------------------------------------------------

// SwiGLU stage: a workgroup takes 16 MBH intermediate rows (MBH 16-row blocks
// of up rows and the matching gate rows) of one 16-pair tile; wave w takes the
// 16-word chunks w, w + KW, ... of K.  PAIRS: the activations arrive as x'
// pairs with their per-token correction (x_pairs, x_corr: built once per
// token upstream) and are loaded as B operands directly; otherwise each lane
// builds its B operands from x.  MX: h goes out as mx rows (hp, scale words hs)
// for the tile-resident down stage, with a correction part per 32 outputs
// (hcorr); otherwise as x' pairs for the K-split one.
template <int MBH, int ADT, int KW, bool PAIRS, bool MX>
__global__ __launch_bounds__(64 * KW) void k_grouped_swiglu_ks(
    const uint16_t* __restrict__ x, int64_t ldx, const uint32_t* __restrict__ x_pairs,
    const float* __restrict__ x_corr, int64_t topk,
    const uint32_t* __restrict__ w, int64_t n_half, int64_t nwords,
    const void* __restrict__ alpha, const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ pair_ids, int n_exp,
    uint16_t* __restrict__ hp, uint32_t* __restrict__ hs, float* __restrict__ hcorr,
    uint16_t* __restrict__ h, int64_t ldh) {
  constexpr int MB = 2 * MBH;  // row blocks: up 0 .. MBH-1, gate MBH .. MB-1
  static_assert(KW >= MBH, "the epilogue takes 64 threads per up block");
  static_assert(!MX || MBH == 2, "a workgroup's outputs are one scale block");
  __shared__ float red[KW][MB][4][64];
  __shared__ float red_c[KW][4][16];
  int e, pos0, np;
  if (!decode_tile(offsets, n_exp, blockIdx.y, 16, e, pos0, np)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int64_t i0 = static_cast<int64_t>(blockIdx.x) * 16 * MBH;
  const uint32_t* we = w + static_cast<int64_t>(e) * (2 * n_half) * nwords;
  const uint32_t* rowp[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    int64_t i = i0 + 16 * (mb % MBH) + r16;
    i = i < n_half ? i : n_half - 1;
    rowp[mb] = we + (i + (mb / MBH) * n_half) * nwords + 4 * g;
  }
  // this lane's B column: pair pos0 + r16 (token row of x), zero past np
  const bool valid = r16 < np;
  const int64_t tok = valid ? pair_ids[pos0 + r16] / topk : 0;
  const uint16_t* xrow = x + tok * ldx + 64 * g;
  const uint32_t* prow = x_pairs + (tok * nwords + 4 * g) * 8;
  f32x4d_t acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4d_t{0.f, 0.f, 0.f, 0.f};
  float cp = 0.f;
  const ExpandConsts kc;
  for (int64_t c0 = 16 * wv; c0 < nwords; c0 += 16 * KW) {
    u32x4v_t wq[MB], xv[4][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) wq[mb] = *reinterpret_cast<const u32x4v_t*>(rowp[mb] + c0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x4v_t* src = PAIRS ? reinterpret_cast<const u32x4v_t*>(prow + (c0 + q) * 8)
                                  : reinterpret_cast<const u32x4v_t*>(xrow + (c0 + q) * 16);
      xv[q][0] = src[0];
      xv[q][1] = src[1];
    }
    MA_ISSUE_FENCE();  // every load of the chunk in flight before the first use
#pragma unroll
    for (int qh = 0; qh < 4; qh += 2) {  // two words per step (operand registers)
      u32x4v_t av[2][MB][2], bv[2][2];
#pragma unroll
      for (int qi = 0; qi < 2; ++qi) {
        const int q = qh + qi;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          uint32_t ex[8];
          expand_word(wq[mb][q], ex, kc);
          av[qi][mb][0] = u32x4v_t{ex[0], ex[1], ex[2], ex[3]};
          av[qi][mb][1] = u32x4v_t{ex[4], ex[5], ex[6], ex[7]};
        }
        if constexpr (PAIRS) {
          bv[qi][0] = valid ? xv[q][0] : u32x4v_t{0u, 0u, 0u, 0u};
          bv[qi][1] = valid ? xv[q][1] : u32x4v_t{0u, 0u, 0u, 0u};
        } else {
          uint32_t pr[8];
          const float c = x16_to_pairs(make_uint4(xv[q][0].x, xv[q][0].y, xv[q][0].z, xv[q][0].w),
                                       make_uint4(xv[q][1].x, xv[q][1].y, xv[q][1].z, xv[q][1].w), pr);
          cp += valid ? c : 0.f;
          bv[qi][0] = valid ? u32x4v_t{pr[0], pr[1], pr[2], pr[3]} : u32x4v_t{0u, 0u, 0u, 0u};
          bv[qi][1] = valid ? u32x4v_t{pr[4], pr[5], pr[6], pr[7]} : u32x4v_t{0u, 0u, 0u, 0u};
        }
      }
      pin(cp);
      mfma_block_begin();
#pragma unroll
      for (int qi = 0; qi < 2; ++qi)
#pragma unroll
        for (int hf = 0; hf < 2; ++hf)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) mfma_acc(acc[mb], av[qi][mb][hf], bv[qi][hf]);
      mfma_block_end();
      keep_b(av, acc);
      keep_b(bv, acc);
    }
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv][mb][r][lane] = acc[mb][r];
  if constexpr (!PAIRS) red_c[wv][g][r16] = cp;
  __syncthreads();
  // Thread t < 64 MBH: pair column col = t % 16, rows 4 rq .. +3 of up block mbu.
  const int col = tid & 15, rq = (tid >> 4) & 3, mbu = tid >> 6;
  if (tid >= 64 * MBH) return;  // (a later barrier waits for the waves that are left)
  const bool live = col < np;
  if (!MX && !live) return;
  const int64_t nwh = n_half / 16;
  float hv[4] = {0.f, 0.f, 0.f, 0.f}, hsum = 0.f;
  uint32_t ex = 0;
  if (live) {
    const int pid = pair_ids[pos0 + col];
    float c = 0.f;
    if constexpr (PAIRS) {
      c = x_corr[pid / topk];
    } else {
#pragma unroll
      for (int k = 0; k < KW; ++k)
#pragma unroll
        for (int gg = 0; gg < 4; ++gg) c += red_c[k][gg][col];
    }
    const int ln = col + 16 * rq;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t i = i0 + 16 * mbu + 4 * rq + r;
      if (i >= n_half) continue;
      float su = 0.f, sg = 0.f;
#pragma unroll
      for (int k = 0; k < KW; ++k) {
        su += red[k][mbu][r][ln];
        sg += red[k][mbu + MBH][r][ln];
      }
      const float au = ld_t<ADT>(alpha, static_cast<int64_t>(e) * 2 * n_half + i);
      const float ag = ld_t<ADT>(alpha, static_cast<int64_t>(e) * 2 * n_half + n_half + i);
      const uint16_t hb = f32_to_bf16(swiglu_act(au * (su - c), ag * (sg - c)));
      if constexpr (MX) {
        hv[r] = bf16_to_f32(hb);
        hsum += hv[r];
        ex = mx_exponent(ex, hv[r]);
      } else {
        const int pos = static_cast<int>(i & 15), j = pos & 7, hh = pos >> 3;
        const float hx = bf16_to_f32(hb) * pair_scale(j);  // exact: power-of-two scale
        hp[((static_cast<int64_t>(pos0 + col) * nwh + (i >> 4)) * 8 + j) * 2 + hh] =
            static_cast<uint16_t>(bf16_bits_exact(hx));
      }
      if (h) h[static_cast<int64_t>(pid) * ldh + i] = hb;
    }
  }
  if constexpr (MX) {
    // the 32 outputs' exponent and sum: over a wave's lane groups, then its two waves
    __shared__ uint32_t s_ex[MBH][16];
    __shared__ float s_sum[MBH][16];
    uint32_t eo = __shfl_xor(ex, 16, 64);
    ex = ex > eo ? ex : eo;
    eo = __shfl_xor(ex, 32, 64);
    ex = ex > eo ? ex : eo;
    hsum += __shfl_xor(hsum, 16, 64);
    hsum += __shfl_xor(hsum, 32, 64);
    if (rq == 0) {
      s_ex[mbu][col] = ex;
      s_sum[mbu][col] = hsum;
    }
    // s_barrier leaves out waves that have ended (the other six, whose slots the
    // next workgroup's waves take meanwhile: 59.9 us with them held here, 54.2 now,
    // for 256 pairs of 64 experts, 5120 -> 768)
    __syncthreads();
    if (!live) return;
    ex = s_ex[0][col] > s_ex[1][col] ? s_ex[0][col] : s_ex[1][col];
    // word wd of the row: block pos / 2 of its step, word pos of the step's 8 (launch_mx_prep_wide's order)
    const int64_t wd = i0 / 16 + mbu, row = pos0 + col;
    const int64_t step = wd / 16 * 2 + (wd >> 1 & 1), nsteps = n_half / kMxStep;
    const int pos = static_cast<int>((wd >> 2 & 3) * 2 + (wd & 1));
    const float f = mx_factor(ex);
    float v[4] = {hv[0] * f, hv[2] * f, hv[1] * f, hv[3] * f};
    uint16_t* dst = hp + (row * nsteps + step) * kMxStep + 8 * pos + rq;  // even values, then the odd ones
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const uint32_t w4 = mx_piece4(v);
      dst[64 * p] = static_cast<uint16_t>(w4);
      dst[64 * p + 4] = static_cast<uint16_t>(w4 >> 16);
    }
    if (mbu == 0 && rq == 0) {
      reinterpret_cast<uint8_t*>(hs + row * nsteps + step)[pos / 2] = static_cast<uint8_t>(mx_scale_byte(ex));
      hcorr[row * (n_half / 32) + i0 / 32] = s_sum[0][col] + s_sum[1][col];
    }
  }
}

// Down stage: a workgroup takes 16 MB output rows of one 16-pair tile; wave w
// takes the 4 QW-word chunks w, w + KW, ... of K (QW words per lane), reading
// h's x' pairs straight from the pair-format buffer.
template <int MB, int ADT, int KW, int QW>
__global__ __launch_bounds__(64 * KW) void k_grouped_down_ks(
    const uint32_t* __restrict__ hp, const uint32_t* __restrict__ w, int64_t n_out,
    int64_t nwk, const void* __restrict__ alpha, const int32_t* __restrict__ offsets,
    int n_exp, uint16_t* __restrict__ out) {
  constexpr int CW = 4 * QW;  // words per chunk
  static_assert(KW >= MB, "the epilogue takes 64 threads per row block");
  __shared__ float red[KW][MB][4][64];
  __shared__ float red_c[KW][4][16];
  int e, pos0, np;
  if (!decode_tile(offsets, n_exp, blockIdx.y, 16, e, pos0, np)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int64_t n0 = static_cast<int64_t>(blockIdx.x) * 16 * MB;
  const uint32_t* we = w + static_cast<int64_t>(e) * n_out * nwk;
  const uint32_t* rowp[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    int64_t n = n0 + 16 * mb + r16;
    n = n < n_out ? n : n_out - 1;
    rowp[mb] = we + n * nwk + QW * g;
  }
  const bool valid = r16 < np;
  const uint32_t* hrow = hp + static_cast<int64_t>(pos0 + (valid ? r16 : 0)) * nwk * 8 + QW * g * 8;
  f32x4d_t acc[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb] = f32x4d_t{0.f, 0.f, 0.f, 0.f};
  float cp = 0.f;
  const ExpandConsts kc;
  for (int64_t c0 = CW * wv; c0 < nwk; c0 += CW * KW) {
    uint32_t wq[MB][QW];
    u32x4v_t bv[QW][2];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      if constexpr (QW == 2) {
        const uint2 v2 = *reinterpret_cast<const uint2*>(rowp[mb] + c0);
        wq[mb][0] = v2.x;
        wq[mb][1] = v2.y;
      } else {
#pragma unroll
        for (int q = 0; q < QW; ++q) wq[mb][q] = rowp[mb][c0 + q];
      }
    }
#pragma unroll
    for (int q = 0; q < QW; ++q) {
      const u32x4v_t* src = reinterpret_cast<const u32x4v_t*>(hrow + (c0 + q) * 8);
      bv[q][0] = src[0];
      bv[q][1] = src[1];
    }
    MA_ISSUE_FENCE();  // every load of the chunk in flight before the first use
#pragma unroll
    for (int q = 0; q < QW; ++q) {  // one word per step (operand registers)
      u32x4v_t av[MB][2];
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        uint32_t ex[8];
        expand_word(wq[mb][q], ex, kc);
        av[mb][0] = u32x4v_t{ex[0], ex[1], ex[2], ex[3]};
        av[mb][1] = u32x4v_t{ex[4], ex[5], ex[6], ex[7]};
      }
      if (!valid) bv[q][0] = bv[q][1] = u32x4v_t{0u, 0u, 0u, 0u};
      const uint32_t pr[8] = {bv[q][0].x, bv[q][0].y, bv[q][0].z, bv[q][0].w,
                              bv[q][1].x, bv[q][1].y, bv[q][1].z, bv[q][1].w};
      cp += pairs_cst(pr);
      pin(cp);
      mfma_block_begin();
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) mfma_acc(acc[mb], av[mb][hf], bv[q][hf]);
      mfma_block_end();
      keep_b(av, acc);
      keep_b(bv[q], acc);
    }
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv][mb][r][lane] = acc[mb][r];
  red_c[wv][g][r16] = cp;
  __syncthreads();
  // Thread t < 64 MB: pair column col = t % 16, rows 4 rq .. +3 of block mb.
  if (tid >= 64 * MB) return;
  const int col = tid & 15, rq = (tid >> 4) & 3, mb = tid >> 6;
  if (col >= np) return;
  float c = 0.f;
#pragma unroll
  for (int k = 0; k < KW; ++k)
#pragma unroll
    for (int gg = 0; gg < 4; ++gg) c += red_c[k][gg][col];
  const int ln = col + 16 * rq;
  const int64_t nb0 = n0 + 16 * mb + 4 * rq;
  float o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < KW; ++k) s += red[k][mb][r][ln];
    const int64_t n = nb0 + r < n_out ? nb0 + r : n_out - 1;
    o[r] = ld_t<ADT>(alpha, static_cast<int64_t>(e) * n_out + n) * (s - c);
  }
  uint16_t* orow = out + static_cast<int64_t>(pos0 + col) * n_out;
  if (nb0 + 3 < n_out) {
    uint2 rr;
    rr.x = pack_bf16x2_rn(o[0], o[1]);
    rr.y = pack_bf16x2_rn(o[2], o[3]);
    *reinterpret_cast<uint2*>(orow + nb0) = rr;
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (nb0 + r < n_out) orow[nb0 + r] = f32_to_bf16(o[r]);
  }
}

// ---------------------------------------------------------------------------
// Decode form (few pairs per expert): tiles of 16 pairs whose mx rows (two FP8
// pieces, mx.h) lie in LDS for all of K, staged once; then each wave takes two
// blocks of 16 rows over all of K, weights kAhead chunks of 16 words ahead in
// registers, with no barrier and no reduction across waves.  The codes go in as
// FP4: three instructions a word where the bf16 operands took twelve, and the
// products need no spacing by hand.  The SwiGLU stage writes the tile's mx rows
// of x itself (with every pair's sum), so it needs x alone, and h's like the
// prefill form; both stages' operands hold the bf16 values to 2^-20 of their
// block's largest (mx.h), so a row differs from its float64 value by its bf16
// rounding and little else.  The down stage issues its loads of h and of the
// first weights unconditionally up front, a lane past the tile's end reading its
// last pair again: under a branch the compiler moved them next to their uses and
// waited there, one round trip a row (256 experts, 32 tokens x 8: 27 us that way).
// (The SwiGLU stage's x rows are under a wave's own branch and are issued
// together all the same; scales and sums are one load a thread.)  Bound by the
// weights' bytes and a few such round trips.  Hidden 2048: a block of 64 experts
// (inter 768) 24 us at 4 tokens x 8 and 38 at 32 (30 and 41 with bf16 operands),
// of 256 (inter 512) 53 at 32 and 66 at 64 (57 and 74).
// NCH: chunks of 256 values of K (0: at run time, up to 16; the others unroll).
// The run-time instances reserve LDS for 16 chunks, so one workgroup runs on a
// CU whatever K is; they are still no slower than the bf16 kernels at any size
// tried (32 tokens x 8, us a block, bf16 / now: hidden 1024, inter 512, 64 experts
// 37 / 25; 3072, 768, 32 44 / 36; 4096, 1024, 32 68 / 50; 2048, 256, 64 37 / 30).
// ---------------------------------------------------------------------------
namespace gd {
constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kMaxChunks = 16;
// Weight chunks in flight ahead of the products.  (All of a wave's share at
// once kept the tile's x loads waiting behind the other workgroups' weights.)
constexpr int kAhead = 3, kRing = 4;
constexpr int kRow = 272;  // bytes of a staged row of h: 256 and padding (banks)

template <int NCH>
struct Shared {
  static constexpr int kSteps = 2 * (NCH ? NCH : kMaxChunks);
  // step s, chunk c of pair p at (p * nsteps + s) * 16 + (c ^ p)
  __align__(16) uint4 x[16 * kSteps * 16];
  uint32_t scale[16][kSteps + 1];
};

// Rows r16 of the wave's two blocks from rp[j] (+ 4 g), nch chunks, against the
// tile: acc[j][p] of piece p.
template <int NCH>
__device__ __forceinline__ void load(const uint32_t* const (&rp)[2], int c, uint4 (&w)[2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j) w[j] = *reinterpret_cast<const uint4*>(rp[j] + 16 * c);
}

__device__ __forceinline__ void chunk(const uint4 (&w)[2], const uint4* x, const uint32_t* scale, int g, int r16,
                                      mx_f32x4_t (&acc)[2][2]) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int sb = reinterpret_cast<const uint8_t*>(scale + s)[g];
    const i32x8_t b0 = mx_operand(x[16 * s + (g ^ r16)], x[16 * s + ((4 + g) ^ r16)]);
    const i32x8_t b1 = mx_operand(x[16 * s + ((8 + g) ^ r16)], x[16 * s + ((12 + g) ^ r16)]);
    uint32_t a[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j) mx_expand2(s ? make_uint2(w[j].z, w[j].w) : make_uint2(w[j].x, w[j].y), a[j]);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      acc[j][0] = mx_mfma_fp4(a[j], b0, acc[j][0], mx_piece_scale(0), sb);
      acc[j][1] = mx_mfma_fp4(a[j], b1, acc[j][1], mx_piece_scale(1), sb);
    }
  }
}

template <int NCH>
__device__ __forceinline__ void kloop(const uint32_t* const (&rp)[2], int nch, uint4 (&ring)[kRing][2],
                                      const Shared<NCH>& sh, int g, int r16, mx_f32x4_t (&acc)[2][2]) {
  const uint4* x = sh.x + r16 * (2 * nch) * 16;
  const uint32_t* scale = sh.scale[r16];
  if constexpr (NCH > 0) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      if (c + kAhead < NCH) load<NCH>(rp, c + kAhead, ring[(c + kAhead) % kRing]);
      MA_ISSUE_FENCE();
      chunk(ring[c % kRing], x + 32 * c, scale + 2 * c, g, r16, acc);
      mx_pin(acc[0][0], acc[0][1], acc[1][0], acc[1][1]);
    }
  } else {
    for (int c0 = 0; c0 < nch; c0 += kRing) {
#pragma unroll
      for (int s = 0; s < kRing; ++s) {
        const int c = c0 + s;
        if (c >= nch) break;
        load<NCH>(rp, c + kAhead < nch ? c + kAhead : nch - 1, ring[(s + kAhead) % kRing]);
        MA_ISSUE_FENCE();
        chunk(ring[s], x + 32 * c, scale + 2 * c, g, r16, acc);
        mx_pin(acc[0][0], acc[0][1], acc[1][0], acc[1][1]);
      }
    }
  }
}
}  // namespace gd

// SwiGLU: 128 outputs (8 up blocks and the matching gate blocks, one of each a
// wave) of a tile of 16 pairs.  PAIRS: h goes out as x' pairs, for the K-split
// down stage.
template <int ADT, int NCH, bool PAIRS>
__global__ __launch_bounds__(gd::kThreads) void k_gd_swiglu(
    const uint16_t* __restrict__ x, int64_t ldx, int64_t topk, const uint32_t* __restrict__ w, int64_t n_half,
    int nch_arg, const void* __restrict__ alpha, const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ pair_ids, int n_exp, uint16_t* __restrict__ hp, uint32_t* __restrict__ hs,
    float* __restrict__ hcorr, uint16_t* __restrict__ h, int64_t ldh) {
  using namespace gd;
  constexpr int MAXCH = NCH ? NCH : kMaxChunks;
  constexpr int kPer = (16 * MAXCH + 63) / 64;  // words of a pair per lane
  __shared__ Shared<NCH> sh;
  __shared__ int32_t s_pid[16], s_tok[16];
  __shared__ float s_c[16], s_sum[kWaves][16];
  __shared__ uint32_t s_ex[kWaves][16], s_hsc[16];
  int e, pos0, np;
  if (!decode_tile(offsets, n_exp, blockIdx.y, 16, e, pos0, np)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  pos0 = __builtin_amdgcn_readfirstlane(pos0);
  np = __builtin_amdgcn_readfirstlane(np);
  const int nch = NCH ? NCH : nch_arg, nwords = 16 * nch, nsteps = 2 * nch;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int n_rtiles = static_cast<int>(n_half / 128), rtile = static_cast<int>(blockIdx.x);
  // Issue order matters (memory counters complete in issue order): the pair
  // ids, then the tile's rows of x, then the weights, so that staging x waits
  // for nothing behind it and the weights stream while it happens.
  if (tid < np) {
    const int p = pair_ids[pos0 + tid];
    s_pid[tid] = p;
    s_tok[tid] = p / static_cast<int>(topk);
  }
  __syncthreads();
  uint4 xv[2][kPer][2];  // pairs wv and wv + 8
#pragma unroll
  for (int ci = 0; ci < 2; ++ci) {
    const int col = wv + 8 * ci;
    if (col < np) {
      const uint4* src = reinterpret_cast<const uint4*>(x + s_tok[col] * ldx);
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int wd = lane + 64 * k < nwords ? lane + 64 * k : nwords - 1;
        xv[ci][k][0] = src[2 * wd];
        xv[ci][k][1] = src[2 * wd + 1];
      }
    }
  }
  MA_ISSUE_FENCE();
  const int64_t blk = static_cast<int64_t>(rtile) * kWaves + wv;
  const uint32_t* we = w + static_cast<int64_t>(e) * (2 * n_half) * nwords;
  const uint32_t* rp[2] = {we + (blk * 16 + r16) * nwords + 4 * g, we + (n_half + blk * 16 + r16) * nwords + 4 * g};
  uint4 ring[kRing][2];
#pragma unroll
  for (int c = 0; c < kAhead; ++c)
    if (NCH == 0 || c < NCH) load<NCH>(rp, c < nch ? c : nch - 1, ring[c]);
  MA_ISSUE_FENCE();
#pragma unroll
  for (int ci = 0; ci < 2; ++ci) {
    const int col = wv + 8 * ci;
    if (col >= np) continue;  // (a column past np keeps what is there: its products are dropped)
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int wd = lane + 64 * k;
      if (wd >= nwords) break;  // a word pair's two lanes together
      const uint4 a = xv[ci][k][0], b = xv[ci][k][1];
      const uint32_t u[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      float v[16];
      uint32_t ex = 0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        v[2 * q] = __uint_as_float(u[q] << 16);
        v[2 * q + 1] = __uint_as_float(u[q] & 0xffff0000u);
        sum += v[2 * q];
        sum += v[2 * q + 1];
        ex = mx_exponent(mx_exponent(ex, v[2 * q]), v[2 * q + 1]);
      }
      const uint32_t eo = __shfl_xor(ex, 1, 64);
      ex = ex > eo ? ex : eo;
      uint4 out[2];
      mx_word<2>(v, mx_factor(ex), out);
      const int step = wd / 16 * 2 + (wd >> 1 & 1), pos = (wd >> 2 & 3) * 2 + (wd & 1);
#pragma unroll
      for (int p = 0; p < 2; ++p) sh.x[(col * nsteps + step) * 16 + ((8 * p + pos) ^ col)] = out[p];
      if ((wd & 1) == 0)
        reinterpret_cast<uint8_t*>(&sh.scale[col][step])[pos / 2] = static_cast<uint8_t>(mx_scale_byte(ex));
    }
    sum = group_sum<64>(sum);
    if (lane == 0) s_c[col] = sum;
  }
  __syncthreads();
  mx_f32x4_t acc[2][2];  // up, gate by piece
#pragma unroll
  for (int j = 0; j < 2; ++j) acc[j][0] = acc[j][1] = mx_f32x4_t{0.f, 0.f, 0.f, 0.f};
  kloop<NCH>(rp, nch, ring, sh, g, r16, acc);
  // Epilogue: lane holds pair r16, outputs i0 + r of its 16-output word (word wv
  // of the tile's 8).  Two waves' words share a scale block, so the exponents
  // meet in LDS first; then as the prefill form: h's bytes staged as [pair][two
  // half steps], out in 16-byte pieces.
  const int64_t i0 = blk * 16 + 4 * g;
  const float cc = s_c[r16];
  float hv[4], hsum = 0.f;
  uint32_t ex = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float au = ld_t<ADT>(alpha, static_cast<int64_t>(e) * 2 * n_half + i0 + r);
    const float ag = ld_t<ADT>(alpha, static_cast<int64_t>(e) * 2 * n_half + n_half + i0 + r);
    const uint16_t hb = f32_to_bf16(
        swiglu_act(au * (acc[0][0][r] + acc[0][1][r] - cc), ag * (acc[1][0][r] + acc[1][1][r] - cc)));
    hv[r] = bf16_to_f32(hb);
    hsum += hv[r];
    ex = mx_exponent(ex, hv[r]);
    if (h && r16 < np) h[static_cast<int64_t>(s_pid[r16]) * ldh + i0 + r] = hb;
    if (PAIRS && r16 < np) {
      const int pos = 4 * g + r, j = pos & 7;
      hp[((static_cast<int64_t>(pos0 + r16) * (n_half / 16) + blk) * 8 + j) * 2 + (pos >> 3)] =
          static_cast<uint16_t>(bf16_bits_exact(hv[r] * pair_scale(j)));  // exact: power-of-two scale
    }
  }
  if constexpr (PAIRS) return;
  uint32_t eo = __shfl_xor(ex, 16, 64);
  ex = ex > eo ? ex : eo;
  eo = __shfl_xor(ex, 32, 64);
  ex = ex > eo ? ex : eo;
  hsum += __shfl_xor(hsum, 16, 64);
  hsum += __shfl_xor(hsum, 32, 64);
  if (g == 0) {
    s_ex[wv][r16] = ex;
    s_sum[wv][r16] = hsum;
  }
  __syncthreads();  // (and every wave is done with the tile's rows)
  eo = s_ex[wv ^ 1][r16];
  ex = ex > eo ? ex : eo;
  const int b = wv / 2;  // block of 32 outputs: step b & 1, half b / 2 of the tile's part
  uint8_t* hst = reinterpret_cast<uint8_t*>(sh.x);
  const float f = mx_factor(ex);
  float v[4] = {hv[0] * f, hv[2] * f, hv[1] * f, hv[3] * f};
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const uint32_t w4 = mx_piece4(v);
    uint16_t* dst =
        reinterpret_cast<uint16_t*>(hst + r16 * kRow + 128 * (b & 1) + 64 * p + 32 * (b / 2) + 16 * (wv & 1) + 2 * g);
    dst[0] = static_cast<uint16_t>(w4);
    dst[4] = static_cast<uint16_t>(w4 >> 16);
  }
  if (g == 0 && (wv & 1) == 0)
    reinterpret_cast<uint8_t*>(s_hsc + r16)[(b & 1) * 2 + b / 2] = static_cast<uint8_t>(mx_scale_byte(ex));
  __syncthreads();
  if (tid < np) {
    float c = 0.f;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) c += s_sum[k][tid];
    hcorr[static_cast<int64_t>(pos0 + tid) * n_rtiles + rtile] = c;
  }
  if (tid < 2 * np) {  // the scale bytes of the tile's two blocks of each step
    const int col = tid >> 1, st = tid & 1;
    reinterpret_cast<uint16_t*>(hs + static_cast<int64_t>(pos0 + col) * n_rtiles + (rtile & ~1) + st)[rtile & 1] =
        reinterpret_cast<const uint16_t*>(s_hsc + col)[st];
  }
  if (tid < 16 * np) {
    const int col = tid / 16, part = tid % 16;
    *reinterpret_cast<uint4*>(hp + (static_cast<int64_t>(pos0 + col) * n_rtiles + (rtile & ~1) + part / 8) * kMxStep +
                              64 * (part / 4 & 1) + 32 * (rtile & 1) + 8 * (part & 3)) =
        *reinterpret_cast<const uint4*>(hst + col * kRow + part * 16);
  }
}

// Down: 256 output rows (two blocks a wave) of a tile of 16 pairs, whose mx rows
// of h, scale words and correction parts (CP to each 128 values) the SwiGLU stage
// wrote.
template <int ADT, int NCH, int CP>
__global__ __launch_bounds__(gd::kThreads) void k_gd_down(const uint32_t* __restrict__ hp,
                                                          const uint32_t* __restrict__ hs,
                                                          const float* __restrict__ hcorr,
                                                          const uint32_t* __restrict__ w, int64_t n_out, int nch_arg,
                                                          const void* __restrict__ alpha,
                                                          const int32_t* __restrict__ offsets, int n_exp,
                                                          uint16_t* __restrict__ out) {
  using namespace gd;
  constexpr int MAXCH = NCH ? NCH : kMaxChunks;
  constexpr int kPer = (2 * MAXCH * 16 + 63) / 64;  // 16-byte chunks of a pair per lane
  __shared__ Shared<NCH> sh;
  __shared__ float s_cp[16][2 * MAXCH + 1];
  int e, pos0, np;
  if (!decode_tile(offsets, n_exp, blockIdx.y, 16, e, pos0, np)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  pos0 = __builtin_amdgcn_readfirstlane(pos0);
  np = __builtin_amdgcn_readfirstlane(np);
  const int nch = NCH ? NCH : nch_arg, nwk = 16 * nch, nsteps = 2 * nch;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  // the rows' loads go out before the weights' (memory counters complete in
  // issue order), so staging does not wait for the weight stream
  uint4 hv[2][kPer];  // pairs wv and wv + 8 (past np: the last one's, not stored)
#pragma unroll
  for (int ci = 0; ci < 2; ++ci) {
    const int col = wv + 8 * ci < np ? wv + 8 * ci : np - 1;
    const uint4* src = reinterpret_cast<const uint4*>(hp) + static_cast<int64_t>(pos0 + col) * nsteps * 16;
#pragma unroll
    for (int k = 0; k < kPer; ++k) hv[ci][k] = src[lane + 64 * k < nsteps * 16 ? lane + 64 * k : 0];
  }
  uint32_t sw = 0;
  float cp[CP] = {};  // (added up where they are stored: an addition here waits for its load)
  const int sc = tid / nsteps, ss = tid % nsteps;  // 16 nsteps <= 512
  if (sc < np) {
    sw = hs[static_cast<int64_t>(pos0 + sc) * nsteps + ss];
    if constexpr (CP == 1) {
      cp[0] = hcorr[static_cast<int64_t>(pos0 + sc) * nsteps + ss];
    } else {
      const float* const parts = hcorr + (static_cast<int64_t>(pos0 + sc) * nsteps + ss) * CP;
#pragma unroll
      for (int q = 0; q < CP; ++q) cp[q] = parts[q];
    }
  }
  MA_ISSUE_FENCE();
  const uint32_t* we = w + static_cast<int64_t>(e) * n_out * nwk;
  const int64_t n0 = (static_cast<int64_t>(blockIdx.x) * kWaves + wv) * 32;  // n_out % 256 == 0
  const uint32_t* rp[2] = {we + (n0 + r16) * nwk + 4 * g, we + (n0 + 16 + r16) * nwk + 4 * g};
  uint4 ring[kRing][2];
#pragma unroll
  for (int c = 0; c < kAhead; ++c)
    if (NCH == 0 || c < NCH) load<NCH>(rp, c < nch ? c : nch - 1, ring[c]);
  MA_ISSUE_FENCE();
#pragma unroll
  for (int ci = 0; ci < 2; ++ci) {
    const int col = wv + 8 * ci;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int i = lane + 64 * k;
      if (col < np && i < nsteps * 16) sh.x[(col * nsteps + i / 16) * 16 + (i % 16 ^ col)] = hv[ci][k];
    }
  }
  if (sc < np) {
    sh.scale[sc][ss] = sw;
    float c = cp[0];
#pragma unroll
    for (int q = 1; q < CP; ++q) c += cp[q];
    s_cp[sc][ss] = c;
  }
  __syncthreads();
  mx_f32x4_t acc[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j) acc[j][0] = acc[j][1] = mx_f32x4_t{0.f, 0.f, 0.f, 0.f};
  kloop<NCH>(rp, nch, ring, sh, g, r16, acc);
  if (r16 >= np) return;
  float cc = 0.f;  // the correction parts in order
  for (int k = 0; k < nsteps; ++k) cc += s_cp[r16][k];
  uint16_t* orow = out + static_cast<int64_t>(pos0 + r16) * n_out;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int64_t n = n0 + 16 * j + 4 * g;
    float o[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      o[r] = ld_t<ADT>(alpha, static_cast<int64_t>(e) * n_out + n + r) * (acc[j][0][r] + acc[j][1][r] - cc);
    uint2 rr;
    rr.x = pack_bf16x2_rn(o[0], o[1]);
    rr.y = pack_bf16x2_rn(o[2], o[3]);
    *reinterpret_cast<uint2*>(orow + n) = rr;
  }
}

// y[t, n] = sum_j w[t, j] * out[inverse[t*k + j], n] (+ residual), float32 sum.
__global__ __launch_bounds__(256) void k_combine(const uint16_t* __restrict__ out,
                                                 const int32_t* __restrict__ inverse,
                                                 const float* __restrict__ wts, int64_t topk,
                                                 int64_t n, const void* __restrict__ res,
                                                 int res_dt, uint16_t* __restrict__ y) {
  const int64_t t = blockIdx.y;
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 2;
  if (i >= n) return;
  float a0 = 0.f, a1 = 0.f;
  for (int64_t j = 0; j < topk; ++j) {
    const float wj = wts[t * topk + j];
    const uint32_t v = *reinterpret_cast<const uint32_t*>(out + static_cast<int64_t>(inverse[t * topk + j]) * n + i);
    a0 += wj * __uint_as_float(v << 16);
    a1 += wj * __uint_as_float(v & 0xffff0000u);
  }
  if (res) {
    a0 += ld_f(res, res_dt, t * n + i);
    a1 += ld_f(res, res_dt, t * n + i + 1);
  }
  *reinterpret_cast<uint32_t*>(y + t * n + i) =
      static_cast<uint32_t>(f32_to_bf16(a0)) | (static_cast<uint32_t>(f32_to_bf16(a1)) << 16);
}

// The same combine for top-k <= K, bf16 rows, 8 outputs per thread: the
// token's k (position, weight) pairs are wave-uniform scalar loads, then every
// slot's 16-byte load and the residual's are issued before the sums (the
// arithmetic and its order are k_combine's).
template <int K>
__global__ __launch_bounds__(256) void k_combine8(const uint16_t* __restrict__ out,
                                                  const int32_t* __restrict__ inverse,
                                                  const float* __restrict__ wts, int topk,
                                                  int64_t n, const uint16_t* __restrict__ res,
                                                  uint16_t* __restrict__ y) {
  const int64_t t = blockIdx.y;
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  static_assert(K == 8, "slot pairs");
  int64_t row[8];
  float wj[8];
  slot_pairs8(inverse, wts, t, topk, row, wj);
  if (i >= n) return;
  uint4 v[K], r = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
  for (int j = 0; j < K; ++j) v[j] = *reinterpret_cast<const uint4*>(out + row[j] * n + i);
  if (res) r = *reinterpret_cast<const uint4*>(res + t * n + i);
  float a[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) a[e] = 0.f;
#pragma unroll
  for (int j = 0; j < K; ++j) {
    if (j >= topk) break;
    const uint32_t u[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a[2 * q] += wj[j] * __uint_as_float(u[q] << 16);
      a[2 * q + 1] += wj[j] * __uint_as_float(u[q] & 0xffff0000u);
    }
  }
  if (res) {
    const uint32_t u[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      a[2 * q] += __uint_as_float(u[q] << 16);
      a[2 * q + 1] += __uint_as_float(u[q] & 0xffff0000u);
    }
  }
  uint4 o;
  o.x = pack_bf16x2_rn(a[0], a[1]);
  o.y = pack_bf16x2_rn(a[2], a[3]);
  o.z = pack_bf16x2_rn(a[4], a[5]);
  o.w = pack_bf16x2_rn(a[6], a[7]);
  *reinterpret_cast<uint4*>(y + t * n + i) = o;
}

// ---------------------------------------------------------------------------
// Prefill form (many pairs per expert): tiles of 64 or 32 pairs x 256 weight
// rows, four waves of 64 rows, K walked in steps of 8 words (128 codes) on
// v_mfma_scale_f32_16x16x128_f8f6f4: the codes as FP4, the activations as mx
// rows of two FP8 pieces (mx.h), which hold bf16 values to 2^-20 of their block's
// largest.  A step's mx
// rows of the pairs are copied into LDS by the LDS DMA
// (global_load_lds_dwordx4: no staging registers), one step ahead with the
// step's weights, one barrier per step; three workgroups run on a CU (two steps
// ahead was no faster: 194 against 189 us a block of 2048 tokens).  The
// tokens' mx rows are written once (launch_mx_prep_wide) and h's by the SwiGLU
// epilogue, so staging is a copy.  Each lane expands its own weight words with
// two ANDs and a shift a word: words 4g .. 4g+3 of two steps' 16 for lane group
// g, loaded at once (64 bytes of a row), the first two in the even step.  Tiles
// go to workgroups so that the row tiles of one pair tile share an XCD (workgroups are placed on the 8 XCDs round-robin), which keeps that
// tile's rows in one L2.
//
// 2048 tokens x 8 on 64 experts (103 GFLOP SwiGLU, 52 down): 104 and 60 us with
// 32 bytes of a row at a time, 121 and 69 as bf16 tiles of 128 pairs, whose
// matrix units waited for the expansion (12 instructions a word) and multiplied
// a quarter of padding; with 64 bytes at a time the whole block went from 189 to
// 176 us (237 as bf16).  Bound by issue: the matrix units work 58 % of the time,
// the epilogue and the addresses take most of the rest.
// ---------------------------------------------------------------------------
namespace gp {
constexpr int kRows = 256;   // weight rows per tile (SwiGLU: 128 up + the 128 matching gate rows)
constexpr int kWords = 8;    // packed words of K per step
constexpr int kPieces = 2;
constexpr int kChunks = 8 * kPieces;  // 16-byte chunks of an mx row per step
constexpr int kXcds = 8;
// After the K loop a buffer stages the output tile for coalesced stores: h as
// [pair][one step of an mx row] (256 bytes padded to 272), the down outputs as
// [pair][256 rows] (rows padded to 264 bf16); the padding keeps the 16 pair
// columns of a lane group on different banks and every row 16-byte aligned.
constexpr int kHRow = 272, kORow = 264;
// Tiles of TOK pairs: 4 waves of 64 rows each over all of the pairs.
template <int TOK>
struct Tile {
  static constexpr int kRb = 4, kNb = TOK / 16;  // blocks of 16 rows and of 16 pairs a wave
  static constexpr int kThreads = 256;
  static constexpr int kWaves = TOK == 64 ? 3 : 4;          // per SIMD, at most
  static constexpr int kCopies = TOK * kChunks / kThreads;  // per thread and step
  // One step's mx rows in LDS: 16-byte slot p * 16 + (c ^ (p % 16)) holds
  // chunk c (piece c / 8, bytes 16 (c % 8) ..+15) of pair p -- each pair's 256
  // bytes in one run, the chunks XOR-swizzled so that the B reads (16 pairs of
  // one chunk) hit 16 different bank groups; the DMA fills slots in order, so
  // each copy's source is chosen to match.
  static constexpr int kXsDwords = TOK * kChunks * 4;
  // Buffer A also stages the output tile: all of h, or half of the down tile's
  // pairs at a time.
  static constexpr int kOut = TOK / 2 * kORow / 2, kH = TOK * kHRow / 4;
  static constexpr int kXaDwords = kH > kOut ? (kH > kXsDwords ? kH : kXsDwords) : (kOut > kXsDwords ? kOut : kXsDwords);
};
}  // namespace gp

// Tile of workgroup L (workgroups go to the 8 XCDs round-robin: L on XCD
// L % 8, the XCD's slot L / 8).  The M x n_rtiles tiles (pair tiles with their
// experts in order, the row tiles of a pair tile together) are cut into 8
// contiguous ranges of equal length, one per XCD: so an expert's pair tiles run
// on one XCD (two at a range boundary) and read its codes through one L2, the
// row tiles of a pair tile share its mx rows, and no XCD has more than one tile
// above its share.  M is counted from the dispatch offsets (the grid is sized
// for the most tiles T k / TOK + E).  Returns false for the workgroups past the
// XCD's range.
template <int TOK>
__device__ __forceinline__ bool gp_tile(const int32_t* __restrict__ offsets, int n_exp, int n_rtiles, int& mtile,
                                        int& rtile) {
  const int lane = threadIdx.x & 63;
  int m = 0;  // pair tiles of every expert
#pragma unroll 4
  for (int base = 0; base < n_exp; base += 64) {
    const int ee = base + lane;
    m += (offsets[ee + 1 < n_exp ? ee + 1 : n_exp] - offsets[ee < n_exp ? ee : n_exp] + TOK - 1) / TOK;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m += __shfl_xor(m, off, 64);
  m = __builtin_amdgcn_readfirstlane(m);
  const int L = blockIdx.x, xcd = L % gp::kXcds, slot = L / gp::kXcds;
  const int per = (m * n_rtiles + gp::kXcds - 1) / gp::kXcds;
  const int idx = xcd * per + slot;
  mtile = idx / n_rtiles;
  rtile = idx % n_rtiles;
  return slot < per && mtile < m;
}

// One K step of a wave: RB row blocks x NB pair blocks x 2 pieces of
// v_mfma_scale_f32_16x16x128_f8f6f4.  a: the lane's two words of its row
// blocks, expanded; xsb, ssb: the step's mx rows in the swizzled layout (pair
// 16 nb + r16 has p % 16 == r16) and their scale words.
// send issues the next step's copies and loads, behind the first products: the
// matrix unit works while their addresses are formed.
template <int RB, int NB, typename F>
__device__ __forceinline__ void gp_step(const uint32_t (&a)[RB][4], const uint32_t* __restrict__ xsb,
                                        const uint32_t* __restrict__ ssb, int g, int r16,
                                        mx_f32x4_t (&acc)[RB][NB], F&& send) {
  // byte offset of chunk g of column r16: chunk c + g of the same column
  // is at that offset ^ 16 c (c a multiple of 4), 16 columns on 4 KB further.
  // (Recomputed each step: hoisted out of the loop, the sixteen addresses cost
  // the registers the products need.)
  uint32_t off = static_cast<uint32_t>(r16 * gp::kChunks + (g ^ r16)) * 16;
  uint32_t soff = static_cast<uint32_t>(r16) * 4 + g;
  asm volatile("" : "+v"(off), "+v"(soff));
  auto read = [&](int i) {  // piece i % 2 of pair block i / 2
    const char* xc = reinterpret_cast<const char*>(xsb) + 4096 * (i / 2);
    return mx_operand(*reinterpret_cast<const uint4*>(xc + (off ^ (128 * (i % 2)))),
                      *reinterpret_cast<const uint4*>(xc + (off ^ (128 * (i % 2) + 64))));
  };
  // One block's reads go out ahead of the previous one's products, and no
  // further: hoisted to the top of the step, all of them need more registers
  // than there are.
  int sb = reinterpret_cast<const uint8_t*>(ssb)[soff];
  i32x8_t b = read(0);
#pragma unroll
  for (int i = 0; i < NB * gp::kPieces; ++i) {
    const int nb = i / 2, p = i % 2;
    i32x8_t bn = b;
    int sn = sb;
    if (i + 1 < NB * gp::kPieces) bn = read(i + 1);
    if (p == 1 && nb + 1 < NB) sn = reinterpret_cast<const uint8_t*>(ssb)[soff + 64 * (nb + 1)];
    MA_ISSUE_FENCE();
#pragma unroll
    for (int mb = 0; mb < RB; ++mb) acc[mb][nb] = mx_mfma_fp4(a[mb], b, acc[mb][nb], mx_piece_scale(p), sb);
#pragma unroll
    for (int mb = 0; mb < RB; mb += 4) mx_pin(acc[mb][nb], acc[mb + 1][nb], acc[mb + 2][nb], acc[mb + 3][nb]);
    if (i == 0) {
      MA_ISSUE_FENCE();
      send();
      MA_ISSUE_FENCE();
    }
    b = bn;
    sb = sn;
  }
}

// A step's copies: copy i of thread tid fills slot S = tid + threads * i (so
// each wave's copy i fills 64 consecutive slots, as the LDS DMA writes them)
// with chunk c = (S % 16) ^ (p % 16) of pair p = S / 16; then the pairs' scale
// words, one by each of the first TOK threads.  rows[p] is pair p's row in
// base (16 nsteps chunks a row, nsteps scale words a row).
typedef __attribute__((address_space(3))) void* lds_void_t;
template <int TOK>
struct GpDma {
  using T = gp::Tile<TOK>;
  const uint4* base;        // the same in every lane
  uint32_t off[T::kCopies];  // copy i's source at step 0, in chunks from base (< 2^32: checked by the host)
  const uint32_t* scale;    // this thread's scale word of step 0 (threads below TOK)

  __device__ __forceinline__ GpDma(const uint32_t* b, const uint32_t* scales, int64_t nsteps, const int32_t* rows)
      : base(reinterpret_cast<const uint4*>(b)),
        scale(scales + static_cast<int64_t>(rows[threadIdx.x % TOK]) * nsteps) {
#pragma unroll
    for (int i = 0; i < T::kCopies; ++i) {
      const int S = threadIdx.x + T::kThreads * i, p = S / 16, c = (S % 16) ^ (p % 16);
      off[i] = static_cast<uint32_t>(static_cast<int64_t>(rows[p]) * nsteps * gp::kChunks + c);
    }
  }

  // The copies of step k into the LDS buffers (in flight until the issuing
  // wave's vector memory counter drains).
  __device__ __forceinline__ void copy(int64_t k, uint32_t* xsb, uint32_t* ssb) const {
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int i = 0; i < T::kCopies; ++i)
      __builtin_amdgcn_global_load_lds(base + k * gp::kChunks + off[i],
                                       (lds_void_t)(xsb + 4 * (64 * wv + T::kThreads * i)), 16, 0, 0);
    if (64 * wv < TOK && threadIdx.x < TOK)
      __builtin_amdgcn_global_load_lds(scale + k, (lds_void_t)(ssb + 64 * wv), 4, 0, 0);
  }
};
// s_waitcnt immediate (gfx9 encoding): vmcnt(n) and lgkmcnt(0), expcnt left open.
constexpr int gp_vmcnt(int n) { return n | (0x7 << 4); }

// One step of the K loop: expand this step's weights, issue the next step's
// copies into the other buffers (if there is a next step) and, in an odd step,
// the next two steps' weights into w, with this step's MFMAs, then wait for the
// copies and meet at the barrier.
template <int TOK, bool ODD>
__device__ __forceinline__ void gp_kstep(const uint32_t* rp, uint32_t loff, const int64_t (&moff)[gp::Tile<TOK>::kRb],
                                         int64_t k, int64_t nsteps, const GpDma<TOK>& d, const uint32_t* cur,
                                         const uint32_t* cur_s, uint32_t* nxt, uint32_t* nxt_s,
                                         uint4 (&w)[gp::Tile<TOK>::kRb], int g, int r16,
                                         mx_f32x4_t (&acc)[gp::Tile<TOK>::kRb][gp::Tile<TOK>::kNb]) {
  using namespace gp;
  constexpr int RB = Tile<TOK>::kRb;
  // This step's weights are in (an even step's were loaded during the last):
  // nothing else is outstanding, so the copies and loads below are all this
  // wave has in flight during the MFMAs.
  __builtin_amdgcn_s_waitcnt(0);
  MA_ISSUE_FENCE();
  uint32_t a[RB][4];
#pragma unroll
  for (int mb = 0; mb < RB; ++mb) mx_expand2(ODD ? make_uint2(w[mb].z, w[mb].w) : make_uint2(w[mb].x, w[mb].y), a[mb]);
  MA_ISSUE_FENCE();
  gp_step<RB, Tile<TOK>::kNb>(a, cur, cur_s, g, r16, acc, [&]() {
    if (!ODD || k + 1 < nsteps) d.copy(k + 1, nxt, nxt_s);
    if constexpr (ODD) {
      MA_ISSUE_FENCE();  // the copies are issued before the weights
      const int64_t kn = k + 1 < nsteps ? k + 1 : k - 1;
#pragma unroll
      for (int mb = 0; mb < RB; ++mb) w[mb] = *reinterpret_cast<const uint4*>(rp + moff[mb] + kn * kWords + loff);
    }
  });
  // This wave's copies have landed: at most the weight loads issued after
  // them are outstanding (vector memory completes in issue order); those
  // are waited for where the next step uses them.
  __builtin_amdgcn_s_waitcnt(gp_vmcnt(ODD ? RB : 0));
  // The next buffer is in and this one is free to refill once every wave is
  // here.  A plain barrier: __syncthreads' fence would also wait for the
  // weight loads just issued (it drains every outstanding write to LDS, and
  // the LDS DMA counts in the same counter as those loads).
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // Register copies the loop needs between steps stay here, after the
  // barrier, where the next step's first wait covers their loads.
  MA_ISSUE_FENCE();
}

// The K loop shared by both stages: acc += W x, the lane's weight row of
// block mb at rp + moff[mb] + loff (rp and moff the same in every lane; nwk
// words), the pairs' mx rows in d; weights one step ahead in registers, mx rows
// one step ahead by DMA into the other LDS buffer.  The two buffers are
// distinct arrays and the loop is unrolled by two, so the compiler sees that a
// step's LDS reads and the copies in flight into the other buffer do not
// overlap (it would otherwise wait for the copies before the reads).
template <int TOK>
__device__ __forceinline__ void gp_kloop(const uint32_t* rp, uint32_t loff, const int64_t (&moff)[gp::Tile<TOK>::kRb],
                                         int64_t nwk, const GpDma<TOK>& d, uint32_t* xa, uint32_t* xb, uint32_t* sa,
                                         uint32_t* sb, int g, int r16,
                                         mx_f32x4_t (&acc)[gp::Tile<TOK>::kRb][gp::Tile<TOK>::kNb]) {
  using namespace gp;
  constexpr int RB = Tile<TOK>::kRb;
  const int64_t nsteps = nwk / kWords;
  uint4 w[RB];
#pragma unroll
  for (int mb = 0; mb < RB; ++mb) w[mb] = *reinterpret_cast<const uint4*>(rp + moff[mb] + loff);
  d.copy(0, xa, sa);
  __builtin_amdgcn_s_waitcnt(0);  // this wave's copies have landed
  __syncthreads();                // and every other wave's
  for (int64_t k = 0; k < nsteps; k += 2) {  // K is a multiple of 256: nsteps is even
    gp_kstep<TOK, false>(rp, loff, moff, k, nsteps, d, xa, sa, xb, sb, w, g, r16, acc);
    gp_kstep<TOK, true>(rp, loff, moff, k + 1, nsteps, d, xb, sb, xa, sa, w, g, r16, acc);
  }
}

// SwiGLU stage: h = SwiGLU(up, gate) of 128 outputs (rows [o, o+128) of the
// up half and the matching gate rows) for a tile of TOK pairs of expert e,
// rounded to bf16 and written as half of steps 2 (rtile / 2) and 2 (rtile / 2)
// + 1 of the pair's mx row (hp, scale words hs) and optionally in slot order (h); hcorr[pos * n_rtiles + rtile]
// gets the tile's part of the down stage's correction sum h.
template <int ADT, int TOK>
__global__ __launch_bounds__(gp::Tile<TOK>::kThreads) __attribute__((amdgpu_waves_per_eu(gp::Tile<TOK>::kWaves, gp::Tile<TOK>::kWaves))) void k_gp_swiglu(
    const uint32_t* __restrict__ xq, const uint32_t* __restrict__ xs, const float2* __restrict__ xc, int64_t topk,
    const uint32_t* __restrict__ w, int64_t n_half, int64_t nwords,
    const void* __restrict__ alpha, const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ pair_ids, int n_exp, uint16_t* __restrict__ hp, uint32_t* __restrict__ hs,
    float* __restrict__ hcorr, uint16_t* __restrict__ h, int64_t ldh) {
  using namespace gp;
  using T = Tile<TOK>;
  constexpr int kTok = TOK, kThreads = T::kThreads, RB = T::kRb, NB = T::kNb;
  __shared__ __align__(16) uint32_t xa[T::kXaDwords];
  __shared__ __align__(16) uint32_t xb[T::kXsDwords];
  __shared__ uint32_t sa[kTok], sb[kTok], hsc[kTok];
  __shared__ float cst[kTok], hcp[4][kTok];
  __shared__ int32_t tokrow[kTok], pid[kTok];
  const int n_rtiles = static_cast<int>((n_half + kRows / 2 - 1) / (kRows / 2));
  int mtile, rtile;
  if (!gp_tile<TOK>(offsets, n_exp, n_rtiles, mtile, rtile)) return;
  int e, pos0, np;
  if (!decode_tile(offsets, n_exp, mtile, kTok, e, pos0, np)) return;
  e = __builtin_amdgcn_readfirstlane(e);  // the same in every lane: the weights' addresses stay scalar
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  if (tid < kTok) {
    const int p = tid < np ? pair_ids[pos0 + tid] : -1;
    pid[tid] = p;
    const int t = p >= 0 ? static_cast<int>(p / topk) : 0;
    tokrow[tid] = t;
    cst[tid] = p >= 0 ? xc[t].x : 0.f;
  }
  const int64_t o0 = static_cast<int64_t>(rtile) * (kRows / 2) + wv * 8 * RB;  // this wave's first output
  const uint32_t* we = w + static_cast<int64_t>(e) * 2 * n_half * nwords;
  // (n_half % 128 == 0: every row of the tile exists)
  const uint32_t* rp = we + o0 * nwords;
  const uint32_t loff = static_cast<uint32_t>(r16 * nwords + 4 * g);
  int64_t moff[RB];
#pragma unroll
  for (int mb = 0; mb < RB; ++mb) moff[mb] = (16 * (mb % (RB / 2)) + (mb / (RB / 2)) * n_half) * nwords;
  __syncthreads();  // tokrow
  const GpDma<TOK> xsrc(xq, xs, nwords / kWords, tokrow);
  mx_f32x4_t acc[RB][NB];
#pragma unroll
  for (int mb = 0; mb < RB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = mx_f32x4_t{0.f, 0.f, 0.f, 0.f};
  gp_kloop<TOK>(rp, loff, moff, nwords, xsrc, xa, xb, sa, sb, g, r16, acc);
  // Epilogue: lane (r16, g) of row block mb holds rows 4g..4g+3 of the block
  // for pair column 16 nb + r16.  h goes to LDS as its parts of two steps of
  // its mx row (the loop's last barrier has freed the LDS), then out in 16-byte
  // pieces, each pair's in runs of 64 bytes.  Output i = o0 + 16 mb + 4 g + r
  // (< n_half: n_half % 128 == 0) is value 4 g + r of a word: byte 2 g + r / 2
  // of its 16 bytes, + 8 for odd r.  The wave's 32 outputs are words 2 wv and
  // 2 wv + 1 of the tile's 8, so block 2 (rtile & 1) + wv / 2 of step wv & 1 of
  // the two: in LDS byte 128 (wv & 1) + 64 piece + 32 (wv / 2) of the pair's row.
  uint8_t* hst = reinterpret_cast<uint8_t*>(xa);
  const int64_t abase = static_cast<int64_t>(e) * 2 * n_half;
#pragma unroll
  for (int q = 0; q < RB / 4; ++q) {
    const int blk = (wv & 1) * 2 + wv / 2;
    float au[2][4], ag[2][4];
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t i = o0 + 32 * q + 16 * m + 4 * g + r;
        au[m][r] = ld_t<ADT>(alpha, abase + i);
        ag[m][r] = ld_t<ADT>(alpha, abase + n_half + i);
      }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int col = nb * 16 + r16;
      const float cc = cst[col];
      float hv[2][4], hsum = 0.f;
      uint32_t ex = 0;
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float up = au[m][r] * (acc[2 * q + m][nb][r] - cc);
          const float gt = ag[m][r] * (acc[RB / 2 + 2 * q + m][nb][r] - cc);
          const uint16_t hb = f32_to_bf16(swiglu_act(up, gt));
          hv[m][r] = bf16_to_f32(hb);
          hsum += hv[m][r];
          ex = mx_exponent(ex, hv[m][r]);
          if (h) {
            if (col < np) h[static_cast<int64_t>(pid[col]) * ldh + o0 + 32 * q + 16 * m + 4 * g + r] = hb;
          }
        }
      // over the lane groups: the block's exponent and sum
      uint32_t eo = __shfl_xor(ex, 16, 64);
      ex = ex > eo ? ex : eo;
      eo = __shfl_xor(ex, 32, 64);
      ex = ex > eo ? ex : eo;
      hsum += __shfl_xor(hsum, 16, 64);
      hsum += __shfl_xor(hsum, 32, 64);
      const float f = mx_factor(ex);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        float v[4] = {hv[m][0] * f, hv[m][2] * f, hv[m][1] * f, hv[m][3] * f};
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
          const uint32_t w4 = mx_piece4(v);
          uint16_t* dst = reinterpret_cast<uint16_t*>(hst + col * kHRow + 128 * (wv & 1) + 64 * p + 32 * (wv / 2) + 16 * m + 2 * g);
          dst[0] = static_cast<uint16_t>(w4);
          dst[4] = static_cast<uint16_t>(w4 >> 16);
        }
      }
      if (g == 0) {
        hcp[blk][col] = hsum;
        reinterpret_cast<uint8_t*>(hsc + col)[blk] = static_cast<uint8_t>(mx_scale_byte(ex));
      }
    }
  }
  __syncthreads();
  // the tile's correction part per pair: blocks in order
  if (tid < np) {
    const float v = ((hcp[0][tid] + hcp[1][tid]) + hcp[2][tid]) + hcp[3][tid];
    hcorr[static_cast<int64_t>(pos0 + tid) * n_rtiles + rtile] = v;
  }
  // the scale bytes of the tile's two blocks of each step
  if (tid < 2 * np) {
    const int col = tid >> 1, st = tid & 1;
    reinterpret_cast<uint16_t*>(hs + static_cast<int64_t>(pos0 + col) * n_rtiles + (rtile & ~1) + st)[rtile & 1] =
        reinterpret_cast<const uint16_t*>(hsc + col)[st];
  }
  // the tile's h (n_half % 256 == 0: whole pairs of steps), 16 B per copy
#pragma unroll
  for (int k = 0; k < kTok * 16 / kThreads; ++k) {
    const int c = tid + kThreads * k, col = c / 16, part = c % 16;
    if (col < np)
      *reinterpret_cast<uint4*>(hp + (static_cast<int64_t>(pos0 + col) * n_rtiles + (rtile & ~1) + part / 8) * kMxStep +
                                64 * (part / 4 & 1) + 32 * (rtile & 1) + 8 * (part & 3)) =
          *reinterpret_cast<const uint4*>(hst + col * kHRow + part * 16);
  }
}

// Down stage: out[pos, n] = bf16(alpha[e, n] * sum_k (c - 1) h) for a tile of
// TOK pairs and 256 output rows; the correction is the sum of the SwiGLU
// stage's n_ctiles parts, added in tile order.
template <int ADT, int TOK>
__global__ __launch_bounds__(gp::Tile<TOK>::kThreads) __attribute__((amdgpu_waves_per_eu(gp::Tile<TOK>::kWaves, gp::Tile<TOK>::kWaves))) void k_gp_down(
    const uint32_t* __restrict__ hp, const uint32_t* __restrict__ hs, const float* __restrict__ hcorr, int n_ctiles,
    const uint32_t* __restrict__ w, int64_t n_out, int64_t nwk, const void* __restrict__ alpha,
    const int32_t* __restrict__ offsets, int n_exp, uint16_t* __restrict__ out) {
  using namespace gp;
  using T = Tile<TOK>;
  constexpr int kTok = TOK, kThreads = T::kThreads, RB = T::kRb, NB = T::kNb;
  __shared__ __align__(16) uint32_t xa[T::kXaDwords];
  __shared__ __align__(16) uint32_t xb[T::kXsDwords];
  __shared__ uint32_t sa[kTok], sb[kTok];
  __shared__ float cst[kTok];
  __shared__ int32_t prow[kTok];
  const int n_rtiles = static_cast<int>((n_out + kRows - 1) / kRows);
  int mtile, rtile;
  if (!gp_tile<TOK>(offsets, n_exp, n_rtiles, mtile, rtile)) return;
  int e, pos0, np;
  if (!decode_tile(offsets, n_exp, mtile, kTok, e, pos0, np)) return;
  e = __builtin_amdgcn_readfirstlane(e);  // the same in every lane: the weights' addresses stay scalar
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  if (tid < kTok) {
    float c = 0.f;
    if (tid < np)
      for (int ct = 0; ct < n_ctiles; ++ct) c += hcorr[static_cast<int64_t>(pos0 + tid) * n_ctiles + ct];
    cst[tid] = c;
    prow[tid] = pos0 + (tid < np ? tid : np - 1);
  }
  const int64_t n0 = static_cast<int64_t>(rtile) * kRows + wv * 16 * RB;
  const uint32_t* we = w + static_cast<int64_t>(e) * n_out * nwk;
  // (n_out % 256 == 0: every row of the tile exists)
  const uint32_t* rp = we + n0 * nwk;
  const uint32_t loff = static_cast<uint32_t>(r16 * nwk + 4 * g);
  int64_t moff[RB];
#pragma unroll
  for (int mb = 0; mb < RB; ++mb) moff[mb] = 16 * mb * nwk;
  __syncthreads();  // prow
  const GpDma<TOK> xsrc(hp, hs, nwk / kWords, prow);
  mx_f32x4_t acc[RB][NB];
#pragma unroll
  for (int mb = 0; mb < RB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = mx_f32x4_t{0.f, 0.f, 0.f, 0.f};
  gp_kloop<TOK>(rp, loff, moff, nwk, xsrc, xa, xb, sa, sb, g, r16, acc);
  // The tile goes out through LDS buffer A as [pair][256 rows], half of the
  // pairs at a time (every wave writes its rows, then every thread copies them
  // out in 16-byte pieces, each pair's 512 bytes contiguous; n_out % 256 == 0).
  // The loop's last barrier has freed the buffer.
  uint2 v[RB][NB];
#pragma unroll
  for (int mb = 0; mb < RB; ++mb) {
    const int64_t n = n0 + 16 * mb + 4 * g;
    float a[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = ld_t<ADT>(alpha, static_cast<int64_t>(e) * n_out + (n + r < n_out ? n + r : n_out - 1));
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const float c = cst[nb * 16 + r16];
      v[mb][nb].x = pack_bf16x2_rn(a[0] * (acc[mb][nb][0] - c), a[1] * (acc[mb][nb][1] - c));
      v[mb][nb].y = pack_bf16x2_rn(a[2] * (acc[mb][nb][2] - c), a[3] * (acc[mb][nb][3] - c));
    }
  }
  uint16_t* ost = reinterpret_cast<uint16_t*>(xa);
  const int64_t ntile0 = static_cast<int64_t>(rtile) * kRows;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
#pragma unroll
    for (int mb = 0; mb < RB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB / 2; ++nb)
        *reinterpret_cast<uint2*>(ost + (nb * 16 + r16) * kORow + wv * 16 * RB + 16 * mb + 4 * g) =
            v[mb][half * (NB / 2) + nb];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTok / 2 * 32 / kThreads; ++k) {
      const int c = tid + kThreads * k, colh = c / 32, part = c % 32, col = half * (kTok / 2) + colh;
      if (col < np)
        *reinterpret_cast<uint4*>(out + static_cast<int64_t>(pos0 + col) * n_out + ntile0 + part * 8) =
            *reinterpret_cast<const uint4*>(ost + colh * kORow + part * 8);
    }
    __syncthreads();  // the buffer is free for the next half
  }
}

}  // namespace ma

using namespace ma;

// Up to this many pairs per expert on average (decode batches) 16-pair tiles
// run, above it (prefill) tiles of 32 and 64 pairs: at 16 an expert (256
// experts, inter 512, 509 tokens x 8) 103 us a block against 104, at 16 of 64
// experts (128 tokens) 52 against 53, at 1 of 256 53
// against 71.
constexpr int64_t kKsMaxPairsPerExpert = 16;
// Up to this many the prefill form's tiles hold 32 pairs instead of 64 (64
// experts: at 64 pairs an expert 94 against 97 us a block, at 96 104 against
// 121; 256 experts at 64 209 against 243).
constexpr int64_t kSmallTilePairsPerExpert = 48;

static size_t align256(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }

// Workspace of one call: h [P, inter] in 16 bits a value (pairs, or mx rows),
// per-pair down outputs [P, hidden] bf16, h's scale words and the SwiGLU tiles'
// correction parts [P, inter / 128]; in the prefill form also the mx rows of the
// tokens (2 bytes a value), their sums and scale words.
static bool grouped_prefill_form(int64_t n_pairs, int64_t n_experts) {
  return n_pairs > kKsMaxPairsPerExpert * n_experts;
}
static size_t grouped_bytes(int64_t n_pairs, int64_t tokens, int64_t inter, int64_t hidden, bool prefill) {
  size_t b = align256(static_cast<size_t>(n_pairs) * inter * 2) + align256(static_cast<size_t>(n_pairs) * hidden * 2) +
             2 * align256(static_cast<size_t>(n_pairs) * (inter / kMxStep) * 4);
  if (prefill)
    b += align256(static_cast<size_t>(tokens) * hidden * 2) + align256(static_cast<size_t>(tokens) * 8) +
         align256(static_cast<size_t>(tokens) * (hidden / kMxStep) * 4);
  else if (hidden > 256 * gd::kMaxChunks && inter <= 256 * gd::kMaxChunks)
    b += align256(3 * static_cast<size_t>(n_pairs) * (inter / kMxStep) * 4);  // four correction parts instead of one
  return b;
}

extern "C" size_t ma_grouped_workspace_bytes(int64_t n_pairs, int64_t inter, int64_t hidden) {
  // an upper bound over both forms (tokens <= pairs)
  return grouped_bytes(n_pairs, n_pairs, inter, hidden, true);
}

// Argument checks shared by ma_moe_grouped and ma_moe_grouped_noalloc.
static int grouped_check(const void* x, int64_t ldx, int64_t tokens, int64_t top_k,
                         int alpha_dtype, int64_t n_experts, int64_t hidden, int64_t inter,
                         const char* what) {
  if (tokens < 0 || top_k < 1 || n_experts < 1 || n_experts > 1024)
    return fail(MA_EVALUE, "%s: bad sizes", what);
  if (hidden % 256 || inter % 256)
    return fail(MA_EVALUE, "%s: hidden (%lld) and intermediate (%lld) must be multiples of 256", what,
                (long long)hidden, (long long)inter);
  if (alpha_dtype != MA_BF16 && alpha_dtype != MA_F32)
    return fail(MA_ETYPE, "%s: row_alpha must be bfloat16 or float32", what);
  if ((reinterpret_cast<uintptr_t>(x) & 15u) || (ldx % 8))
    return fail(MA_EVALUE, "%s: x rows must be 16-byte aligned", what);
  return MA_OK;
}

// The launches of one grouped MoE call; workspace holds
// ma_grouped_workspace_bytes(tokens * top_k, inter, hidden) bytes.
static int grouped_launch(const void* x, int64_t ldx, const uint32_t* x_pairs, const float* x_corr,
                          int64_t tokens, int64_t top_k, const uint32_t* up_gate,
                          const void* up_gate_alpha, const uint32_t* down, const void* down_alpha,
                          int alpha_dtype, int64_t n_experts, int64_t hidden, int64_t inter,
                          const int32_t* offsets, const int32_t* pair_ids, const int32_t* inverse,
                          const float* topk_weight, const void* residual, int residual_dtype,
                          void* h_out, int64_t ldh, void* y, void* workspace, void* stream) {
  const int64_t n_pairs = tokens * top_k;
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* wsb = static_cast<char*>(workspace);
  uint16_t* hp = reinterpret_cast<uint16_t*>(wsb);
  uint16_t* out = reinterpret_cast<uint16_t*>(wsb + align256(static_cast<size_t>(n_pairs) * inter * 2));
  const int ne = static_cast<int>(n_experts);
  const auto* xb = static_cast<const uint16_t*>(x);
  auto* hb = static_cast<uint16_t*>(h_out);
  if (!grouped_prefill_form(n_pairs, n_experts)) {
    // decode: 16-pair tiles
    const unsigned max_tiles = static_cast<unsigned>(n_pairs / 16 + n_experts);
    // Each stage by its own K: tiles in LDS up to 256 * gd::kMaxChunks values, K
    // split over the waves past that; h goes between them as the down stage reads
    // it (mx rows, or x' pairs).  One rule over both stages cost the one that
    // fits: hidden 2048, intermediate 4352, 8 experts, 8 tokens x 8 44.9 us a block for 32.8,
    // hidden 5120, intermediate 768, 64 experts, 8 tokens x 8 70.3 for 55.9.
    const bool up_tile = hidden <= 256 * gd::kMaxChunks, down_tile = inter <= 256 * gd::kMaxChunks;
    const int64_t hsteps = inter / kMxStep;
    const int uch = static_cast<int>(hidden / 256), dch = static_cast<int>(inter / 256);
    uint32_t* hs = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(out) +
                                               align256(static_cast<size_t>(n_pairs) * hidden * 2));
    float* hcorr = reinterpret_cast<float*>(reinterpret_cast<char*>(hs) +
                                            align256(static_cast<size_t>(n_pairs) * hsteps * 4));
#define MA_GD_UP(ADT, NCH, PAIRS)                                                                                    \
  hipLaunchKernelGGL((k_gd_swiglu<ADT, NCH, PAIRS>), dim3(static_cast<unsigned>(hsteps), max_tiles),                  \
                     dim3(gd::kThreads), 0, s, xb, ldx, top_k, up_gate, inter, uch, up_gate_alpha, offsets, pair_ids, \
                     ne, hp, hs, hcorr, hb, ldh)
#define MA_KS_UP(ADT, XP, MX)                                                                                        \
  hipLaunchKernelGGL((k_grouped_swiglu_ks<2, ADT, 8, XP, MX>), dim3(static_cast<unsigned>(cdiv(inter, 32)), max_tiles), \
                     dim3(512), 0, s, xb, ldx, x_pairs, x_corr, top_k, up_gate, inter, hidden / 16, up_gate_alpha,    \
                     offsets, pair_ids, ne, hp, hs, hcorr, hb, ldh)
#define MA_GD_DOWN(ADT, NCH, CP)                                                                                     \
  hipLaunchKernelGGL((k_gd_down<ADT, NCH, CP>), dim3(static_cast<unsigned>(hidden / 256), max_tiles),                 \
                     dim3(gd::kThreads), 0, s, reinterpret_cast<const uint32_t*>(hp), hs, hcorr, down, hidden, dch,   \
                     down_alpha, offsets, ne, out)
#define MA_GD_DOWNS(ADT, CP) \
  if (dch == 2) MA_GD_DOWN(ADT, 2, CP); else if (dch == 3) MA_GD_DOWN(ADT, 3, CP); else MA_GD_DOWN(ADT, 0, CP);
#define MA_DECODE(ADT)                                                                                              \
  if (up_tile && down_tile) {                                                                                        \
    if (uch == 8) MA_GD_UP(ADT, 8, false); else MA_GD_UP(ADT, 0, false);                                             \
  } else if (up_tile) {                                                                                              \
    if (uch == 8) MA_GD_UP(ADT, 8, true); else MA_GD_UP(ADT, 0, true);                                               \
  } else if (down_tile) {                                                                                            \
    if (x_pairs) MA_KS_UP(ADT, true, true); else MA_KS_UP(ADT, false, true);                                         \
  } else {                                                                                                           \
    if (x_pairs) MA_KS_UP(ADT, true, false); else MA_KS_UP(ADT, false, false);                                       \
  }                                                                                                                  \
  if (!down_tile) {                                                                                                  \
    hipLaunchKernelGGL((k_grouped_down_ks<4, ADT, 8, 2>), dim3(static_cast<unsigned>(cdiv(hidden, 64)), max_tiles),   \
                       dim3(512), 0, s, reinterpret_cast<const uint32_t*>(hp), down, hidden, inter / 16, down_alpha,  \
                       offsets, ne, out);                                                                            \
  } else if (up_tile) {                                                                                              \
    MA_GD_DOWNS(ADT, 1)                                                                                              \
  } else {                                                                                                           \
    MA_GD_DOWNS(ADT, 4)                                                                                              \
  }
    if (alpha_dtype == MA_BF16) { MA_DECODE(MA_BF16) } else { MA_DECODE(MA_F32) }
#undef MA_DECODE
#undef MA_GD_DOWNS
#undef MA_GD_DOWN
#undef MA_KS_UP
#undef MA_GD_UP
  } else {
    // prefill: the tokens' mx rows once (x_pairs are the K-split form's), then
    // tiles of 64 or 32 pairs x 256 weight rows.  The tiles' copy sources are
    // 32-bit offsets in 16-byte chunks into the mx rows of x and h.
    if (static_cast<uint64_t>(tokens) * hidden / 2 >= (uint64_t{1} << 32) ||
        static_cast<uint64_t>(n_pairs) * inter / 2 >= (uint64_t{1} << 32))
      return fail(MA_EVALUE, "moe_grouped: %lld tokens x hidden %lld (or their pairs x intermediate %lld) "
                  "exceed the 16 GiB the batched kernels address; split the batch",
                  (long long)tokens, (long long)hidden, (long long)inter);
    char* p = reinterpret_cast<char*>(out) + align256(static_cast<size_t>(n_pairs) * hidden * 2);
    auto take = [&p](size_t bytes) {
      char* q = p;
      p += align256(bytes);
      return q;
    };
    const int64_t xsteps = hidden / kMxStep, hsteps = cdiv(inter, gp::kRows / 2);
    uint32_t* xq = reinterpret_cast<uint32_t*>(take(static_cast<size_t>(tokens) * hidden * 2));
    float2* xc = reinterpret_cast<float2*>(take(static_cast<size_t>(tokens) * 8));
    uint32_t* xs = reinterpret_cast<uint32_t*>(take(static_cast<size_t>(tokens) * xsteps * 4));
    uint32_t* hs = reinterpret_cast<uint32_t*>(take(static_cast<size_t>(n_pairs) * hsteps * 4));
    float* hcorr = reinterpret_cast<float*>(take(static_cast<size_t>(n_pairs) * hsteps * 4));
    launch_mx_prep_wide(xb, ldx, tokens, hidden / 16, xq, xs, xc, s);
    const int64_t tok = n_pairs > kSmallTilePairsPerExpert * n_experts ? 64 : 32;
    const int64_t mtiles = cdiv(n_pairs, tok) + n_experts;  // an upper bound
    const int64_t mt8 = cdiv(mtiles, gp::kXcds) * gp::kXcds;
    const int rt1 = static_cast<int>(cdiv(inter, gp::kRows / 2)), rt2 = static_cast<int>(cdiv(hidden, gp::kRows));
    const dim3 g1(static_cast<unsigned>(mt8 * rt1)), g2(static_cast<unsigned>(mt8 * rt2));
#define MA_GP(ADT, TOK)                                                                            \
  hipLaunchKernelGGL((k_gp_swiglu<ADT, TOK>), g1, dim3(gp::Tile<TOK>::kThreads), 0, s, xq, xs, xc, top_k, up_gate, \
                     inter, hidden / 16, up_gate_alpha, offsets, pair_ids, ne, hp, hs, hcorr, hb, ldh);  \
  hipLaunchKernelGGL((k_gp_down<ADT, TOK>), g2, dim3(gp::Tile<TOK>::kThreads), 0, s,               \
                     reinterpret_cast<const uint32_t*>(hp), hs, hcorr, rt1, down, hidden, inter / 16, \
                     down_alpha, offsets, ne, out);
    if (alpha_dtype == MA_BF16) {
      if (tok == 64) { MA_GP(MA_BF16, 64) } else { MA_GP(MA_BF16, 32) }
    } else {
      if (tok == 64) { MA_GP(MA_F32, 64) } else { MA_GP(MA_F32, 32) }
    }
#undef MA_GP
  }
  if (y) {
    auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    if (top_k <= 8 && (!residual || (residual_dtype == MA_BF16 && a16(residual))) && a16(y) &&
        hidden % 8 == 0) {
      dim3 g3(static_cast<unsigned>(cdiv(hidden, 256 * 8)), static_cast<unsigned>(tokens));
      hipLaunchKernelGGL(k_combine8<8>, g3, dim3(256), 0, s, out, inverse, topk_weight,
                         static_cast<int>(top_k), hidden, static_cast<const uint16_t*>(residual),
                         static_cast<uint16_t*>(y));
    } else {
      dim3 g3(static_cast<unsigned>(cdiv(hidden, 512)), static_cast<unsigned>(tokens));
      hipLaunchKernelGGL(k_combine, g3, dim3(256), 0, s, out, inverse, topk_weight, top_k, hidden,
                         residual, residual_dtype, static_cast<uint16_t*>(y));
    }
  }
  return check_launch("moe_grouped");
}

extern "C" int ma_moe_grouped(const void* x, int64_t ldx, const uint32_t* x_pairs,
                              const float* x_corr, int64_t tokens, int64_t top_k,
                              const uint32_t* up_gate, const void* up_gate_alpha,
                              const uint32_t* down, const void* down_alpha, int alpha_dtype,
                              int64_t n_experts, int64_t hidden, int64_t inter,
                              const int32_t* offsets, const int32_t* pair_ids,
                              const int32_t* inverse, const float* topk_weight,
                              const void* residual, int residual_dtype, void* h_out, int64_t ldh,
                              void* y, void* workspace, size_t workspace_bytes, void* stream) {
  if (int rc = grouped_check(x, ldx, tokens, top_k, alpha_dtype, n_experts, hidden, inter, "moe_grouped"))
    return rc;
  const int64_t n_pairs = tokens * top_k;
  if (n_pairs == 0) return MA_OK;
  if (!workspace || workspace_bytes < grouped_bytes(n_pairs, tokens, inter, hidden,
                                                    grouped_prefill_form(n_pairs, n_experts)))
    return fail(MA_EVALUE, "moe_grouped: workspace too small");
  return grouped_launch(x, ldx, x_pairs, x_corr, tokens, top_k, up_gate, up_gate_alpha, down,
                        down_alpha, alpha_dtype, n_experts, hidden, inter, offsets, pair_ids,
                        inverse, topk_weight, residual, residual_dtype, h_out, ldh, y, workspace,
                        stream);
}

// ---------------------------------------------------------------------------
// ma_moe_grouped without a workspace argument and without any allocation:
// the staging buffer is this file-scope device array, one per GPU, held until
// the process ends.  In host code `scratch` names a host-side stand-in, so
// kernels get the device address from hipGetSymbolAddress, taken once per
// device on that device's first call.
// ---------------------------------------------------------------------------
constexpr size_t kGroupedScratchBytes = size_t{16} << 20;
// Scale words and the tokens' sums have room of their own: a call counts its
// rows, outputs and correction parts (grouped_counted_bytes) against the 16
// MiB.  What the whole layout takes beyond that count is at most 1/32 of it
// (4 bytes beside each 256 of a row or a pair's h) and some alignment.
constexpr size_t kGroupedScratchExtra = size_t{1} << 20;
static __device__ __align__(256) uint8_t scratch[kGroupedScratchBytes + kGroupedScratchExtra];

static void* grouped_scratch_ptr() {
  static std::mutex mu;
  static void* ptrs[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    fail(MA_ERUNTIME, "moe_grouped_noalloc: no current HIP device");
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      fail(MA_ERUNTIME, "moe_grouped_noalloc: device address of the scratch array unavailable");
      return nullptr;
    }
    ptrs[dev] = p;
  }
  return ptrs[dev];
}

static size_t grouped_counted_bytes(int64_t n_pairs, int64_t tokens, int64_t inter, int64_t hidden, bool prefill) {
  size_t b = align256(static_cast<size_t>(n_pairs) * inter * 2) + align256(static_cast<size_t>(n_pairs) * hidden * 2);
  if (prefill)
    b += align256(static_cast<size_t>(tokens) * hidden * 2) + align256(static_cast<size_t>(tokens) * 4) +
         align256(static_cast<size_t>(n_pairs) * cdiv(inter, gp::kRows / 2) * 4);
  return b;
}

extern "C" size_t ma_moe_grouped_noalloc_max_bytes(void) { return kGroupedScratchBytes; }

extern "C" int ma_moe_grouped_noalloc(const void* x, int64_t ldx, const uint32_t* x_pairs,
                                      const float* x_corr, int64_t tokens, int64_t top_k,
                                      const uint32_t* up_gate, const void* up_gate_alpha,
                                      const uint32_t* down, const void* down_alpha,
                                      int alpha_dtype, int64_t n_experts, int64_t hidden,
                                      int64_t inter, const int32_t* offsets,
                                      const int32_t* pair_ids, const int32_t* inverse,
                                      const float* topk_weight, const void* residual,
                                      int residual_dtype, void* h_out, int64_t ldh, void* y,
                                      void* stream) {
  const char* what = "moe_grouped_noalloc";
  if (int rc = grouped_check(x, ldx, tokens, top_k, alpha_dtype, n_experts, hidden, inter, what))
    return rc;
  if (!y)
    return fail(MA_EVALUE, "%s: y is required (the per-pair outputs stay in the internal scratch)", what);
  const int64_t n_pairs = tokens * top_k;
  if (n_pairs == 0) return MA_OK;
  const bool prefill = grouped_prefill_form(n_pairs, n_experts);
  const size_t need = grouped_counted_bytes(n_pairs, tokens, inter, hidden, prefill);
  if (need > kGroupedScratchBytes ||
      grouped_bytes(n_pairs, tokens, inter, hidden, prefill) > sizeof(scratch))
    return fail(MA_EVALUE,
                "%s: %lld (token, expert) pairs need %zu bytes of staging; the built-in scratch holds %zu "
                "(use ma_moe_grouped with a workspace)",
                what, static_cast<long long>(n_pairs), need, kGroupedScratchBytes);
  void* ws = grouped_scratch_ptr();
  if (!ws) return MA_ERUNTIME;
  return grouped_launch(x, ldx, x_pairs, x_corr, tokens, top_k, up_gate, up_gate_alpha, down,
                        down_alpha, alpha_dtype, n_experts, hidden, inter, offsets, pair_ids,
                        inverse, topk_weight, residual, residual_dtype, h_out, ldh, y, ws, stream);
}
