// Ternary projection of many tokens on the scaled 8-bit matrix instructions
// (gfx950): y = alpha (.) (T x_hat) [* rsqrt(mean(x^2) + eps)], the semantics
// of reference src/maple_run/kernels/ternary_gemv.py:156-258.  One launch
// writes every token as an mx row (mx.h), its sum and its RMS factor; the
// second is a tiled GEMM whose operands need no arithmetic but two ANDs a word.
#include "mx.h"
#include "mfma.h"

namespace ma {

namespace mx {
constexpr int kThreads = 256;  // 2 waves along the rows x 2 along the tokens
constexpr int kRows = 128;     // weight rows per tile, 64 a wave
constexpr int kWords = 8;      // packed words per step
}  // namespace mx

constexpr int kMxTok = 64;  // tokens of the larger tile; the workspace's rows are padded to it

// One token per workgroup: x (times w_rms) as an mx row of NP pieces, xs[t *
// s_row + step * s_step] its scale bytes, xc[t] = (sum x_hat, RMS factor) with the sums in a
// fixed order.  Two pieces hold bf16 x (mx.h); the RMS-folded product is float32
// and takes four, which hold it to 2^-19 of itself or 2^-29 of its block's
// largest (the two bf16 numbers of the smaller batches' operands: 2^-17 of
// itself).  Latency: about 5 us for 2048
// x 2048 with two pieces and 8 with four (16 MB written).  XCD x takes the
// tokens of its eighth, whose tiles it multiplies too (k_mx_gemm), and a step's
// scale word is one store: with tokens dealt to the XCDs in turn and a byte a
// block, a line of scale words was written by all eight (both launches for 2048
// tokens at K = 2048: 27.2 -> 23.9 us to 2048 rows, with the RMSNorm 49.4 -> 43.0
// to 2560 and 31.5 -> 26.1 to 1024).  (WIDE rows are gathered
// by expert from every XCD: in order.)  With a MoE combine in front (cb.slot_out
// set, NP 4) the rows are combined first instead of read from x.
template <int NP, bool WIDE>
__global__ __launch_bounds__(128) void k_mx_prep(const uint16_t* __restrict__ x, int64_t ldx, int64_t nwords,
                                                 const void* __restrict__ rms_w, int rms_dt, float rms_eps,
                                                 int64_t s_row, int64_t s_step, uint4* __restrict__ xq,
                                                 uint32_t* __restrict__ xs, float2* __restrict__ xc, int64_t tokens,
                                                 CombineIn cb) {
  __shared__ float red_c[2], red_s[2];
  const int64_t t = WIDE ? static_cast<int64_t>(blockIdx.x)
                         : static_cast<int64_t>(blockIdx.x % kXcds) * (gridDim.x / kXcds) + blockIdx.x / kXcds;
  if (t >= tokens) return;
  const int tid = threadIdx.x;
  const int64_t nsteps = nwords / mx::kWords;
  float c = 0.f, ss = 0.f;
  int64_t crow[8];
  float cw[8];
  if (NP == 4 && cb.slot_out) slot_pairs8(cb.inverse, cb.wts, t, cb.topk, crow, cw);
  for (int64_t wd = tid; wd < nwords; wd += 128) {  // nwords % 16 == 0: a step's 8 lanes stay together
    float v[16];
    if (NP == 4 && cb.slot_out) {
      combine_word16(cb, crow, cw, t, wd, nwords * 16, v);
    } else {
      const uint4* src = reinterpret_cast<const uint4*>(x + t * ldx + wd * 16);
      const uint4 a = src[0], b = src[1];
      const uint32_t u[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        v[2 * q] = __uint_as_float(u[q] << 16);
        v[2 * q + 1] = __uint_as_float(u[q] & 0xffff0000u);
      }
    }
    if (rms_w) {
      float r[16];
      load_rms16(rms_w, rms_dt, wd, r);
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        ss += v[q] * v[q];
        v[q] *= r[q];
      }
    }
    uint32_t e = 0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      c += v[q];
      e = mx_exponent(e, v[q]);
    }
    const uint32_t eo = __shfl_xor(e, 1, 64);  // the block's other word
    e = e > eo ? e : eo;
    uint4 out[NP];
    mx_word<NP>(v, mx_factor(e), out);
    // the word's step and its place among that step's 8
    const int64_t step = WIDE ? wd / 16 * 2 + (wd >> 1 & 1) : wd / mx::kWords;
    const int pos = static_cast<int>(WIDE ? (wd >> 2 & 3) * 2 + (wd & 1) : wd % mx::kWords);
    uint4* dst = xq + (t * nsteps + step) * (8 * NP) + pos;
#pragma unroll
    for (int p = 0; p < NP; ++p) dst[8 * p] = out[p];
    // the step's scale word: its first lane takes the other blocks' bytes
    constexpr int kStepBit = WIDE ? 4 : 2;
    uint32_t sw = mx_scale_byte(e) << (8 * (pos / 2));
    sw |= __shfl_xor(sw, kStepBit, 64);
    sw |= __shfl_xor(sw, 2 * kStepBit, 64);
    if (pos == 0) xs[t * s_row + step * s_step] = sw;
  }
  c = group_sum<64>(c);
  ss = group_sum<64>(ss);
  if ((tid & 63) == 0) {
    red_c[tid >> 6] = c;
    red_s[tid >> 6] = ss;
  }
  __syncthreads();
  if (tid == 0) {
    const float f = rms_w ? rsqrtf((red_s[0] + red_s[1]) / static_cast<float>(nwords * 16) + rms_eps) : 1.f;
    xc[t] = make_float2(red_c[0] + red_c[1], f);
  }
}

typedef __attribute__((address_space(3))) void* mx_lds_t;
constexpr int mx_vmcnt(int n) { return (n & 0xF) | (0x7 << 4) | ((n >> 4) << 14); }  // and lgkmcnt(0)

// Tiles of 128 rows x TOK tokens, waves of 64 x TOK / 2; a step's token rows,
// scale words and weight words all come by the LDS DMA, NBUF - 1 steps ahead (a
// step's copies come mostly from memory that another XCD wrote: a call of 64
// tokens at K = 2048 took 20 us with one step ahead, 16.7 with two).  The
// operands need two ANDs and a shift a word, so a tile is bound by the matrix
// instructions and the steps' fixed parts: both launches for 2048 tokens x 2048
// -> 2560 take 28.4 us (208 as bf16 MFMAs of 16-row tiles, which read each
// token's operands 160 times), 43.1 with the RMSNorm (149), 777 x 2048 -> 2048
// 17.4 (68).
template <int NP, int TOK, int NBUF>
struct MxTile {
  // (a wave's lanes copy 64 scale words; those past a tile of 32 tokens are the
  // next tokens' or, past the last step's rows, the sums that follow them)
  static_assert(TOK == 64 || TOK == 32, "tokens");
  static constexpr int kNb = TOK / 32, kCh = 8 * NP;
  static constexpr int kXDwords = TOK * kCh * 4, kWDwords = mx::kRows * mx::kWords;
  static constexpr int kBuf = kXDwords + kWDwords + 4 * 64;  // one step: rows, weights, each wave's scale words
  static constexpr int kPer = mx::kThreads / kCh;
  static constexpr int kCopies = TOK / kPer + 2;  // per wave and step

  const uint4* xq;  // the tile's first token
  int64_t ld;       // 16-byte chunks of a token
  const uint32_t* xs;
  int64_t srows;  // words between steps
  const uint32_t* w;
  uint32_t woff;  // this thread's weight copy: 4 words of row tid / 2

  // Step k into a buffer: token p's chunk c at slot p kCh + (c ^ p % 16), so
  // that the 16 rows of one chunk lie on different banks; weights row by row.
  __device__ __forceinline__ void copy(int64_t k, uint32_t* buf) const {
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p0 = tid / kCh;
#pragma unroll
    for (int i = 0; i < TOK / kPer; ++i) {
      const int c = (tid % kCh) ^ ((p0 + kPer * i) % 16);
      const uint4* base = xq + kPer * i * ld + k * kCh;  // the same in every lane
      __builtin_amdgcn_global_load_lds(base + static_cast<uint32_t>(p0 * static_cast<int>(ld) + c),
                                       (mx_lds_t)(buf + 4 * (64 * wv + mx::kThreads * i)), 16, 0, 0);
    }
    __builtin_amdgcn_global_load_lds(w + k * mx::kWords + woff, (mx_lds_t)(buf + kXDwords + 256 * wv), 16, 0, 0);
    // (by every wave for itself: all have as many copies to wait for, with no branch between them)
    __builtin_amdgcn_global_load_lds(xs + k * srows + (tid & 63), (mx_lds_t)(buf + kXDwords + kWDwords + 64 * wv), 4, 0,
                                     0);
  }

  // One step of a wave: 4 row blocks x kNb token blocks x NP pieces.  send
  // issues a later step's copies, behind the first products: the matrix unit
  // works while their addresses are formed.
  template <typename F>
  static __device__ __forceinline__ void multiply(const uint32_t* buf, int wv, int wr, int wm, int g, int r16,
                                                  mx_f32x4_t (&acc)[4][kNb], F&& send) {
    const uint32_t* wp = buf + kXDwords + (64 * wr + r16) * mx::kWords + 2 * g;
    uint32_t a[4][4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
      mx_expand2(*reinterpret_cast<const uint2*>(wp + 16 * mb * mx::kWords), a[mb]);
    // byte offset of chunk g of the wave's column r16: chunk c + g of the same
    // column is at that offset ^ 16 c (c a multiple of 4).  (Recomputed each
    // step: hoisted out of the loop, the addresses cost more registers than a
    // XOR each.)
    const int col = wm * (TOK / 2) + r16;
    uint32_t off = static_cast<uint32_t>(col * kCh + (g ^ r16)) * 16;
    uint32_t soff = static_cast<uint32_t>(kXDwords + kWDwords + 64 * wv + col) * 4 + g;
    asm volatile("" : "+v"(off), "+v"(soff));
    const char* const b8 = reinterpret_cast<const char*>(buf);
    auto read = [&](int i) {  // piece i % NP of token block i / NP
      const char* xc = b8 + 16 * (i / NP) * kCh * 16;
      return mx_operand(*reinterpret_cast<const uint4*>(xc + (off ^ (128 * (i % NP)))),
                        *reinterpret_cast<const uint4*>(xc + (off ^ (128 * (i % NP) + 64))));
    };
    // one block's reads go out ahead of the previous one's products
    int sb = reinterpret_cast<const uint8_t*>(b8)[soff];
    i32x8_t b = read(0);
#pragma unroll
    for (int i = 0; i < kNb * NP; ++i) {
      const int nb = i / NP, p = i % NP;
      i32x8_t bn = b;
      int sn = sb;
      if (i + 1 < kNb * NP) bn = read(i + 1);
      if (p == NP - 1 && nb + 1 < kNb) sn = reinterpret_cast<const uint8_t*>(b8)[soff + 64 * (nb + 1)];
      MA_ISSUE_FENCE();
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) acc[mb][nb] = mx_mfma_fp4(a[mb], b, acc[mb][nb], mx_piece_scale(p), sb);
      mx_pin(acc[0][nb], acc[1][nb], acc[2][nb], acc[3][nb]);
      if (i == 0) {
        MA_ISSUE_FENCE();
        send();
        MA_ISSUE_FENCE();
      }
      b = bn;
      sb = sn;
    }
  }

  // Wait for step k's copies (those of the NBUF - 2 steps after it may be in
  // flight), meet the other waves, which also frees the buffer of step k - 1,
  // send the copies of step k + NBUF - 1 there, and multiply.  TAIL: the last
  // steps, whose later copies there are none of.
  template <bool TAIL>
  __device__ __forceinline__ void step(int64_t k, int64_t nsteps, const uint32_t* cur, uint32_t* prev, int wv, int wr,
                                       int wm, int g, int r16, mx_f32x4_t (&acc)[4][kNb]) const {
    if (!TAIL || k + NBUF - 1 < nsteps) __builtin_amdgcn_s_waitcnt(mx_vmcnt((NBUF - 2) * kCopies));
    else __builtin_amdgcn_s_waitcnt(mx_vmcnt(0));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    multiply(cur, wv, wr, wm, g, r16, acc, [&]() {
      if (!TAIL || k + NBUF - 1 < nsteps) copy(k + NBUF - 1, prev);
    });
    MA_ISSUE_FENCE();
  }
};

// Tile order: workgroup L runs on XCD L % 8 and takes that XCD's next tile of
// a contiguous eighth of the token-major list, so an XCD's L2 holds its tokens
// once and the packed weights whole.
template <int NP, int TOK, int NBUF, int ADT>
__global__ __launch_bounds__(mx::kThreads) __attribute__((amdgpu_waves_per_eu(2, 4))) void k_mx_gemm(
    const uint4* __restrict__ xq, const uint32_t* __restrict__ xs, const float2* __restrict__ xc, int64_t batch,
    int64_t rows, const uint32_t* __restrict__ w, int64_t n_out, int64_t nwords, const void* __restrict__ alpha,
    uint16_t* __restrict__ y, int64_t ldy, int n_rtiles, int n_tiles) {
  using T = MxTile<NP, TOK, NBUF>;
  static_assert(NBUF == 2 || NBUF == 3, "buffers");
  // (distinct arrays: the compiler then sees that a step's reads and the
  // copies in flight into the other buffers do not overlap)
  __shared__ __align__(16) uint32_t b0[T::kBuf], b1[T::kBuf], b2[NBUF == 3 ? T::kBuf : 4];
  const int per = (n_tiles + kXcds - 1) / kXcds;
  const int local = static_cast<int>(blockIdx.x) / kXcds;
  const int idx = (static_cast<int>(blockIdx.x) % kXcds) * per + local;
  if (local >= per || idx >= n_tiles) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wv & 1, wm = wv >> 1, r16 = lane & 15, g = lane >> 4;
  const int64_t t0 = static_cast<int64_t>(idx / n_rtiles) * TOK;
  const int64_t n0 = static_cast<int64_t>(idx % n_rtiles) * mx::kRows;
  const int64_t nsteps = nwords / mx::kWords;
  const int wrow = n0 + tid / 2 < n_out ? tid / 2 : static_cast<int>(n_out - 1 - n0);  // past n_out: its last row
  const T t{xq + t0 * nsteps * T::kCh, nsteps * T::kCh, xs + t0, rows, w + n0 * nwords,
            static_cast<uint32_t>(wrow * nwords + 4 * (tid & 1))};
  mx_f32x4_t acc[4][T::kNb];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb)
#pragma unroll
    for (int nb = 0; nb < T::kNb; ++nb) acc[mb][nb] = mx_f32x4_t{0.f, 0.f, 0.f, 0.f};
  // step 0's copies before step 1's: the counted wait for them goes by issue
  // order, and nothing else ties copies into distinct arrays together
  MA_ISSUE_FENCE();
  t.copy(0, b0);
  MA_ISSUE_FENCE();
  if constexpr (NBUF == 3) t.copy(1, b1);  // nsteps is even
  MA_ISSUE_FENCE();
  // The loop's copies are unconditional: past a branch around them the compiler
  // counts on fewer being in flight, and waits for all of them.
  int64_t k = 0;
  for (; k + 2 * NBUF - 1 <= nsteps; k += NBUF) {
    t.template step<false>(k, nsteps, b0, NBUF == 2 ? b1 : b2, wv, wr, wm, g, r16, acc);
    t.template step<false>(k + 1, nsteps, b1, b0, wv, wr, wm, g, r16, acc);
    if constexpr (NBUF == 3) t.template step<false>(k + 2, nsteps, b2, b1, wv, wr, wm, g, r16, acc);
  }
  // at most 2 NBUF - 2 steps are left
  if (k < nsteps) t.template step<true>(k, nsteps, b0, NBUF == 2 ? b1 : b2, wv, wr, wm, g, r16, acc);
  if (k + 1 < nsteps) t.template step<true>(k + 1, nsteps, b1, b0, wv, wr, wm, g, r16, acc);
  if constexpr (NBUF == 3) {
    if (k + 2 < nsteps) t.template step<true>(k + 2, nsteps, b2, b1, wv, wr, wm, g, r16, acc);
    if (k + 3 < nsteps) t.template step<true>(k + 3, nsteps, b0, b2, wv, wr, wm, g, r16, acc);
  }
#pragma unroll
  for (int nb = 0; nb < T::kNb; ++nb) {
    const int64_t tok = t0 + wm * (TOK / 2) + 16 * nb + r16;
    if (tok >= batch) continue;
    const float2 c = xc[tok];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const int64_t n = n0 + 64 * wr + 16 * mb + 4 * g;
      float o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i] = ld_t<ADT>(alpha, n + i < n_out ? n + i : n_out - 1) * (acc[mb][nb][i] - c.x) * c.y;
      if (n + 3 < n_out && (ldy % 4) == 0) {
        uint2 r;
        r.x = pack_bf16x2_rn(o[0], o[1]);
        r.y = pack_bf16x2_rn(o[2], o[3]);
        *reinterpret_cast<uint2*>(y + tok * ldy + n) = r;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < n_out) y[tok * ldy + n + i] = f32_to_bf16(o[i]);
      }
    }
  }
}

void launch_mx_prep_wide(const uint16_t* x, int64_t ldx, int64_t tokens, int64_t nwords, uint32_t* xq, uint32_t* xs,
                         float2* xc, hipStream_t s) {
  hipLaunchKernelGGL((k_mx_prep<2, true>), dim3(static_cast<unsigned>(tokens)), dim3(128), 0, s, x, ldx, nwords, nullptr,
                     0, 0.f, nwords / mx::kWords, int64_t{1}, reinterpret_cast<uint4*>(xq),
                     xs, xc, tokens, CombineIn{});
}

}  // namespace ma

using namespace ma;

static int64_t mx_rows(int64_t batch) { return cdiv(batch, kMxTok) * kMxTok; }

// Workspace: mx rows, scale words, (sum, factor) per token.
size_t tgemm_mx_bytes(int64_t batch, int64_t nwords, bool rms) {
  const int64_t rows = mx_rows(batch), nsteps = nwords / mx::kWords;
  return static_cast<size_t>(rows) * (nwords * 16 * (rms ? 4 : 2) + nsteps * 4 + 8);
}

int launch_tgemm_mx(const uint16_t* x, int64_t batch, int64_t ldx, const uint32_t* w, int64_t n_out, int64_t nwords,
                    const void* alpha, int alpha_dt, const void* rms_w, int rms_dt, float rms_eps, uint16_t* y,
                    int64_t ldy, void* workspace, hipStream_t s, const CombineIn& cb) {
  const int64_t rows = mx_rows(batch), nsteps = nwords / mx::kWords;
  const int np = rms_w ? 4 : 2;
  uint4* xq = static_cast<uint4*>(workspace);
  uint32_t* xs = reinterpret_cast<uint32_t*>(xq + rows * nwords * np);
  float2* xc = reinterpret_cast<float2*>(xs + rows * nsteps);
  const int64_t n_rtiles = cdiv(n_out, mx::kRows);
  const dim3 grid(static_cast<unsigned>(cdiv(batch, kXcds) * kXcds));
  const int64_t n64 = n_rtiles * cdiv(batch, 64), n32 = n_rtiles * cdiv(batch, 32);
#define MA_MX1(NP, TOK, NBUF, ADT)                                                                                   \
  hipLaunchKernelGGL((k_mx_gemm<NP, TOK, NBUF, ADT>),                                                                \
                     dim3(static_cast<unsigned>(cdiv(TOK == 64 ? n64 : n32, kXcds) * kXcds)), dim3(mx::kThreads), 0, \
                     s, xq, xs, xc, batch, rows, w, n_out, nwords, alpha, y, ldy, static_cast<int>(n_rtiles),        \
                     static_cast<int>(TOK == 64 ? n64 : n32))
#define MA_MX(NP, TOK, NBUF) \
  if (alpha_dt == MA_F32) MA_MX1(NP, TOK, NBUF, MA_F32); else MA_MX1(NP, TOK, NBUF, MA_BF16)
  // Tiles of 32 tokens instead of 64 take about 0.6 of the time each and more of
  // them fit on a CU, so they win wherever that saves a pass over the chip or
  // spreads a small call over more of it.
  if (rms_w) {
    hipLaunchKernelGGL((k_mx_prep<4, false>), grid, dim3(128), 0, s, x, ldx, nwords, rms_w, rms_dt, rms_eps,
                       int64_t{1}, rows, xq, xs, xc, batch, cb);
    // 32 tokens with three buffers (two a CU) in one pass, with two buffers (three
    // a CU) as long as that takes no more passes than 64 tokens (two a CU).  K =
    // 2048, us: 256 x 2560 16.6 / 18.4 / 24.3 in that order, 777 x 2560 25.3 / 26.0
    // / 36.2, 1024 x 2560 34.2 / 30.2 / 36.3, 1344 x 2560 41.5 / 41.1 / 39.2, 2048
    // x 2560 52.4 / 49.3 / 54.7, 1536 x 5120 69.1 / 67.7 / 65.9, 2048 x 5120 86.4 /
    // 84.1 / 79.2; at K = 4096 alike (1024 x 2560 - / 49.0 / 58.9, 2048 x 5120 - /
    // 151 / 141).
    if (n32 <= 512) {
      MA_MX(4, 32, 3);
    } else if (cdiv(n32, 768) <= cdiv(n64, 512)) {
      MA_MX(4, 32, 2);
    } else {
      MA_MX(4, 64, 2);
    }
  } else {
    hipLaunchKernelGGL((k_mx_prep<2, false>), grid, dim3(128), 0, s, x, ldx, nwords, nullptr, 0, 0.f,
                       int64_t{1}, rows, xq, xs, xc, batch, CombineIn{});
    // 32 tokens with three buffers (four a CU) in one pass, else 64 with two
    // (three a CU).  K = 2048, us: 128 x 2560 12.8 / 16.4, 777 x 2048 16.9 / 19.3,
    // 777 x 5120 26.4 / 30.3, 1536 x 2560 26.5 / 25.8, 2048 x 2048 27.7 / 28.5, past
    // it 1664 x 2560 31.7 / 30.4, 2048 x 5120 55.6 / 49.9.
    if (n32 <= 1024) {
      MA_MX(2, 32, 3);
    } else {
      MA_MX(2, 64, 2);
    }
  }
#undef MA_MX1
#undef MA_MX
  return check_launch("ternary_gemv (mx)");
}
