// 4-bit RTN GEMM on the scaled 8-bit matrix instructions (gfx950): y[t, n] =
// sum_g s[n, g] (sum_{k in g} q x) + b[n, g] sum_{k in g} x, the factored form
// of reference src/maple_run/kernels/rtn4.py:170-282.
//
// A code 0..15 as the bits of an E4M3 number reads as code / 512, exactly, so
// eight codes become operand bytes with two ANDs and a shift, and x goes in as
// two FP8 pieces (mx.h).  v_mfma_scale_f32_32x32x64_f8f6f4 takes 64 values of
// K, the smaller RTN group.  Tokens are its rows and table rows its columns:
// a lane then folds a group with one scale and one bias of its own, and the 16
// token sums it needs are the same for every table row.  The bias half, sum_g b
// X, is itself a small product over the groups: with bf16 biases it runs on
// v_mfma_f32_32x32x16_bf16 ahead of the K loop, X as three bf16 numbers that
// add up to it exactly, instead of one FMA per output and group.
//
// Lane layout of 32x32x64 (checked on the device): A and B: lane l holds row /
// column l % 32 and the same 32 of the 64 values of K on both sides (here: half
// l / 32 of the group's words, 4 of 8); C: lane l holds column l % 32, register
// i row 8 (i / 4) + 4 (l / 32) + i % 4.
#include "mx.h"

namespace ma {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __bf16 mh_bf16x8_t __attribute__((ext_vector_type(8)));

namespace mh {
constexpr int kGroup = 64;       // values of K per instruction
constexpr int kGroupWords = 8;   // packed words of a group
constexpr int kGroupChunks = 8;  // 16-byte chunks of a group in an x row: piece p, half h at 4 p + 2 h
constexpr int kPad = 128;        // x rows are padded to the largest tile
}  // namespace mh

// x as FP8 rows: token t's group gi at xq + (t ng + gi) * 8, the scale byte of
// (gi, t) at xs[gi * rows + t], the sum over RTN group r (gw words) at
// xg[r * rows + t] and as three bf16 numbers at x3[(3 t + i) n_groups + r].
// One token per workgroup, a word per lane and pass.
__global__ __launch_bounds__(256) void k_mx_head_prep(const uint16_t* __restrict__ x, int64_t ldx, int64_t nwords,
                                                      int gw, int64_t rows, uint4* __restrict__ xq,
                                                      uint8_t* __restrict__ xs, float* __restrict__ xg,
                                                      uint16_t* __restrict__ x3) {
  const int64_t t = blockIdx.x;
  const int64_t ng = nwords / mh::kGroupWords;
  for (int64_t wd = threadIdx.x; wd < nwords; wd += 256) {  // nwords % 16 == 0: a group's lanes stay together
    const uint4 u4 = *reinterpret_cast<const uint4*>(x + t * ldx + wd * 8);
    const uint32_t u[4] = {u4.x, u4.y, u4.z, u4.w};
    float v[8], sum = 0.f;
    uint32_t e = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[2 * q] = __uint_as_float(u[q] << 16);
      v[2 * q + 1] = __uint_as_float(u[q] & 0xffff0000u);
      sum += v[2 * q] + v[2 * q + 1];
      e = mx_exponent(mx_exponent(e, v[2 * q]), v[2 * q + 1]);
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) {
      const uint32_t eo = __shfl_xor(e, off, 64);
      e = e > eo ? e : eo;
      sum += __shfl_xor(sum, off, 64);
    }
    if (gw == 16) sum += __shfl_xor(sum, 8, 64);
    const float f = mx_factor(e);
    float a[4] = {v[0] * f, v[2] * f, v[4] * f, v[6] * f}, b[4] = {v[1] * f, v[3] * f, v[5] * f, v[7] * f};
    const int64_t gi = wd / mh::kGroupWords;
    const int w8 = static_cast<int>(wd % mh::kGroupWords);
    uint2* dst = reinterpret_cast<uint2*>(xq + (t * ng + gi) * mh::kGroupChunks) + w8;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const uint32_t qa = mx_piece4(a), qb = mx_piece4(b);
      dst[8 * p] = make_uint2(qa, qb);
    }
    if (w8 == 0) xs[gi * rows + t] = static_cast<uint8_t>(mx_scale_byte(e));
    if (wd % gw == 0) {
      const int64_t r = wd / gw, n_groups = nwords / gw;
      xg[r * rows + t] = sum;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const uint16_t h = f32_to_bf16(sum);
        x3[(3 * t + i) * n_groups + r] = h;
        sum -= bf16_to_f32(h);
      }
    }
  }
}

typedef __attribute__((address_space(3))) void* mh_lds_t;
constexpr int mh_vmcnt(int n) { return (n & 0xF) | (0x7 << 4) | ((n >> 4) << 14); }  // and lgkmcnt(0)

// N consecutive row scales or biases as loaded (N SDT values, N * size bytes
// aligned), and element i of them.
template <int N, int SDT>
struct MhRaw {
  static constexpr int kWords = SDT == MA_F32 ? N : (N + 1) / 2;
  uint32_t w[kWords];
  __device__ __forceinline__ void load(const void* p, int64_t i) {
    if constexpr (SDT != MA_F32 && N == 1) {
      w[0] = static_cast<const uint16_t*>(p)[i];
    } else {
      const char* q = static_cast<const char*>(p) + i * (SDT == MA_F32 ? 4 : 2);
      if constexpr (kWords == 4) {
        const uint4 v = *reinterpret_cast<const uint4*>(q);
        w[0] = v.x, w[1] = v.y, w[2] = v.z, w[3] = v.w;
      } else if constexpr (kWords == 2) {
        const uint2 v = *reinterpret_cast<const uint2*>(q);
        w[0] = v.x, w[1] = v.y;
      } else {
        w[0] = *reinterpret_cast<const uint32_t*>(q);
      }
    }
  }
  __device__ __forceinline__ float get(int i) const {
    if constexpr (SDT == MA_F32) return __uint_as_float(w[i]);
    else return __uint_as_float((i & 1) ? (w[i / 2] & 0xffff0000u) : (w[i / 2] << 16));
  }
};

// The FP8 operand of four packed words.
__device__ __forceinline__ i32x8_t mh_expand(uint4 w) {
  return i32x8_t{static_cast<int>(w.x & 0x0F0F0F0Fu), static_cast<int>((w.x >> 4) & 0x0F0F0F0Fu),
                 static_cast<int>(w.y & 0x0F0F0F0Fu), static_cast<int>((w.y >> 4) & 0x0F0F0F0Fu),
                 static_cast<int>(w.z & 0x0F0F0F0Fu), static_cast<int>((w.z >> 4) & 0x0F0F0F0Fu),
                 static_cast<int>(w.w & 0x0F0F0F0Fu), static_cast<int>((w.w >> 4) & 0x0F0F0F0Fu)};
}

// out += sum_g b X for MB x NB blocks of 32 tokens from t0 and the lane's rows:
// n_groups % 16 == 0; lane half h holds groups 8 h ..+7 of each 16 on both sides.
template <int MB, int NB>
__device__ __forceinline__ void mh_bias(const uint16_t* x3, int64_t t0, const uint16_t* biases, const int64_t (&row)[NB],
                                        int64_t n_groups, f32x16_t (&out)[MB][NB]) {
  const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
  for (int64_t g0 = 8 * h; g0 < n_groups; g0 += 16) {
    uint4 b[NB], xp[MB][3];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) b[nb] = *reinterpret_cast<const uint4*>(biases + row[nb] * n_groups + g0);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < 3; ++i)
        xp[mb][i] = *reinterpret_cast<const uint4*>(x3 + (3 * (t0 + mb * 32 + r32) + i) * n_groups + g0);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          out[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mh_bf16x8_t, xp[mb][i]),
                                                                __builtin_bit_cast(mh_bf16x8_t, b[nb]), out[mb][nb], 0,
                                                                0, 0);
  }
}

// Rows 2j and 2j + 1 of a lane pair's two columns: the even lane stores the
// first row's two values, the odd lane the second's.
template <int MB, int NB>
__device__ __forceinline__ void mh_store(const f32x16_t (&out)[MB][NB], int64_t t0, int64_t n0, int64_t batch,
                                         int64_t n_out, uint16_t* y, int64_t ldy) {
  const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
  const bool packed = (ldy % 2) == 0;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = out[mb][nb][2 * j], b = out[mb][nb][2 * j + 1];
        const float o = __shfl_xor((lane & 1) ? a : b, 1, 64);
        const int i = 2 * j + (lane & 1);
        const int64_t t = t0 + mb * 32 + 8 * (i / 4) + 4 * h + i % 4;
        const int64_t n = n0 + 32 * nb + (r32 & ~1);
        const float v0 = (lane & 1) ? o : a, v1 = (lane & 1) ? b : o;
        if (t < batch && n < n_out) {
          uint16_t* dst = y + t * ldy + n;
          if (packed && n + 1 < n_out) {
            *reinterpret_cast<uint32_t*>(dst) = pack_bf16x2_rn(v0, v1);
          } else {
            dst[0] = f32_to_bf16(v0);
            if (n + 1 < n_out) dst[1] = f32_to_bf16(v1);
          }
        }
      }
}

// Bound by the table's bytes up to 64 tokens (151,936 x 2048 in groups of 64:
// 57 us both launches at 24 tokens for 175 MB, 90 as bf16 MFMAs), above by the
// matrix instructions and the folds between them (k_mx_head_ring, and this form
// where the bias half cannot go to the matrix units).
//
// Tiles of 32 MB WT tokens x 32 NB WN table rows, KS groups of 64 per stage;
// BM: the bias half on the matrix units.  Per stage:
// the stage's x rows, scale bytes and group sums come by the LDS DMA, the
// table words and row scales of the wave's own rows in registers, all one
// stage ahead; one barrier per stage.
template <int MB, int NB, int WT, int WN, int KS, int GW, int SDT, bool BM>
struct MxHead {
  static constexpr int kTok = 32 * MB * WT, kRows = 32 * NB * WN, kThreads = 64 * WT * WN;
  static constexpr int kRowChunks = mh::kGroupChunks * KS;  // of a token per stage
  static constexpr int kXDwords = kTok * kRowChunks * 4;
  static constexpr int kSums = KS * mh::kGroupWords / GW;  // RTN groups per stage
  static constexpr int kLoads = NB * (KS + (BM ? 1 : 2));             // register loads per stage

  struct Buf {
    uint32_t* x;
    uint32_t* s;
    float* g;
  };
  struct Src {
    const uint4* xq;  // the tile's first token
    const uint8_t* xs;
    const float* xg;
    int64_t ld, rows;  // chunks per token; tokens (padded)
  };
  struct Regs {
    uint4 w[NB][KS];
    MhRaw<kSums, SDT> s[NB], b[NB];
  };

  // slot p * kRowChunks + (c ^ (p % 16)) holds chunk c of token p: 16 tokens'
  // reads of one chunk fall on different banks
  static __device__ __forceinline__ void dma(const Src& d, int64_t st, const Buf& o) {
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int PER = kThreads / kRowChunks;
    const int p0 = tid / kRowChunks;
#pragma unroll
    for (int i = 0; i < kTok / PER; ++i) {
      const int c = (tid % kRowChunks) ^ ((p0 + PER * i) % 16);
      const uint4* base = d.xq + PER * i * d.ld + st * kRowChunks;  // the same in every lane
      __builtin_amdgcn_global_load_lds(base + static_cast<uint32_t>(p0 * static_cast<int>(d.ld) + c),
                                       (mh_lds_t)(o.x + 4 * (64 * wv + kThreads * i)), 16, 0, 0);
    }
    // scale bytes [KS][kTok], 4 a lane
    constexpr int SW = KS * kTok / 4;
    static_assert(SW % 32 == 0 && SW <= kThreads, "scale words");
    if (64 * wv < SW && tid < SW)
      __builtin_amdgcn_global_load_lds(
          reinterpret_cast<const uint32_t*>(d.xs + (st * KS + tid / (kTok / 4)) * d.rows) + tid % (kTok / 4),
          (mh_lds_t)(o.s + 64 * wv), 4, 0, 0);
    // group sums [kSums][kTok]
    constexpr int GWD = kSums * kTok;
    static_assert(GWD <= kThreads, "group sums");
    if (64 * wv < GWD && tid < GWD)
      __builtin_amdgcn_global_load_lds(d.xg + (st * kSums + tid / kTok) * d.rows + tid % kTok,
                                       (mh_lds_t)(o.g + 64 * wv), 4, 0, 0);
  }

  static __device__ __forceinline__ void load(Regs& r, const uint32_t* const (&wp)[NB], const int64_t (&row)[NB],
                                              const void* scales, const void* biases, int64_t n_groups, int64_t st) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
      for (int gi = 0; gi < KS; ++gi)
        r.w[nb][gi] = *reinterpret_cast<const uint4*>(wp[nb] + (st * KS + gi) * mh::kGroupWords);
      r.s[nb].load(scales, row[nb] * n_groups + st * kSums);
      if constexpr (!BM) r.b[nb].load(biases, row[nb] * n_groups + st * kSums);
    }
  }

  // send issues the next stage's copies and loads, behind the first products.
  template <typename F>
  static __device__ __forceinline__ void stage(const Regs& r, const Buf& in, int wt, f32x16_t (&out)[MB][NB], F&& send) {
    const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5;
    uint32_t off[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int p = (wt * MB + mb) * 32 + r32;
      off[mb] = static_cast<uint32_t>(p * kRowChunks + ((2 * h) ^ (p % 16))) * 16;
      asm volatile("" : "+v"(off[mb]));  // recomputed per stage: hoisted, every read's address takes a register
    }
    const char* const xb = reinterpret_cast<const char*>(in.x);
    constexpr int GPR = GW / mh::kGroupWords;  // 64-value groups per RTN group
    constexpr int U = kSums * MB;              // units: an RTN group of a token block
    auto scale = [&](int u, int g2) {
      return static_cast<int>(
          reinterpret_cast<const uint8_t*>(in.s)[((u / MB) * GPR + g2) * kTok + (wt * MB + u % MB) * 32 + r32]);
    };
    auto read = [&](int j) {  // piece j % 2 of group j / 2 % GPR of unit j / 2 / GPR
      const int u = j / 2 / GPR;
      const uint32_t c = (((u / MB) * GPR + j / 2 % GPR) * 8 + (j % 2) * 4) * 16;
      return mx_operand(*reinterpret_cast<const uint4*>(xb + (off[u % MB] ^ c)),
                        *reinterpret_cast<const uint4*>(xb + (off[u % MB] ^ (c + 16))));
    };
    // A unit's products go out, then the previous unit's fold runs behind
    // them (its products have finished; folding a unit right after its own
    // products waited for the last of them, with the matrix unit idle).
    f32x16_t acc[2][NB];
    i32x8_t bv[GPR][NB];
    auto fold = [&](int u) {
      const int rg = u / MB, mb = u % MB;
      float4 X[4];
      if constexpr (!BM) {
        const float* xg = in.g + rg * kTok + (wt * MB + mb) * 32 + 4 * h;
#pragma unroll
        for (int q = 0; q < 4; ++q) X[q] = *reinterpret_cast<const float4*>(xg + 8 * q);
      }
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const float s = r.s[nb].get(rg);
        f32x16_t& o = out[mb][nb];
        if constexpr (!BM) {
          const float b = r.b[nb].get(rg);
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float xv[4] = {X[q].x, X[q].y, X[q].z, X[q].w};
#pragma unroll
            for (int i = 0; i < 4; ++i) o[4 * q + i] = __builtin_fmaf(b, xv[i], o[4 * q + i]);
          }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i)  // explicit FMAs: every build rounds the fold alike
          o[i] = __builtin_fmaf(s, acc[u & 1][nb][i], o[i]);
        asm volatile("" : "+v"(o)::"memory");
      }
    };
    int sa = scale(0, 0);
    i32x8_t av = read(0);
#pragma unroll
    for (int j = 0; j < 2 * GPR * U; ++j) {
      const int u = j / 2 / GPR, g2 = j / 2 % GPR, p = j % 2;
      if (p == 0 && u % MB == 0) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          bv[g2][nb] = mh_expand(r.w[nb][(u / MB) * GPR + g2]);
        }
      }
      i32x8_t an = av;  // the next operand's reads go out ahead of these products
      int sn = sa;
      if (j + 1 < 2 * GPR * U) {
        an = read(j + 1);
        if (p == 1) sn = scale((j + 1) / 2 / GPR, (j + 1) / 2 % GPR);
      }
      MA_ISSUE_FENCE();
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if (g2 == 0 && p == 0) {
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[u & 1][nb][i] = 0.f;
        }
        // codes / 512 against piece p / 16^p
        acc[u & 1][nb] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv[g2][nb], acc[u & 1][nb], 0, 0, 0, sa, 0,
                                                                         136 - 4 * p);
        asm volatile("" : "+v"(acc[u & 1][nb])::"memory");  // one operand's reads at a time (mx_pin)
      }
      if (j == 0) {
        MA_ISSUE_FENCE();
        send();
        MA_ISSUE_FENCE();
      }
      av = an;
      sa = sn;
      if (g2 == GPR - 1 && p == 1 && u > 0) fold(u - 1);
    }
    fold(U - 1);
  }

  static __device__ __forceinline__ void run(const uint4* __restrict__ xq, const uint8_t* __restrict__ xs,
                                             const float* __restrict__ xg, const uint16_t* __restrict__ x3, int64_t batch,
                                             int64_t rows, const uint32_t* __restrict__ w, int64_t n_out, int64_t nwords,
                                             const void* __restrict__ scales, const void* __restrict__ biases,
                                             uint16_t* __restrict__ y, int64_t ldy, int n_ttiles, int n_tiles,
                                             const Buf& ba, const Buf& bb) {
    // workgroup L runs on XCD L % 8: the token tiles of a row tile one after
    // the other on one XCD, so that its L2 has the table's words once
    const int per = (n_tiles + kXcds - 1) / kXcds;
    const int local = static_cast<int>(blockIdx.x) / kXcds;
    const int idx = (static_cast<int>(blockIdx.x) % kXcds) * per + local;
    if (local >= per || idx >= n_tiles) return;
    const int tid = threadIdx.x, lane = tid & 63, r32 = lane & 31, h = lane >> 5;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wt = wv % WT, wn = wv / WT;
    const int64_t t0 = static_cast<int64_t>(idx % n_ttiles) * kTok;
    const int64_t n0 = static_cast<int64_t>(idx / n_ttiles) * kRows + 32 * NB * wn;
    const int64_t nst = nwords / (mh::kGroupWords * KS), n_groups = nwords / GW;
    const int64_t ld = nwords / mh::kGroupWords * mh::kGroupChunks;
    const Src d{xq + t0 * ld, xs + t0, xg + t0, ld, rows};
    int64_t row[NB];
    const uint32_t* wp[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      row[nb] = n0 + 32 * nb + r32;
      row[nb] = row[nb] < n_out ? row[nb] : n_out - 1;
      wp[nb] = w + row[nb] * nwords + 4 * h;
    }
    f32x16_t out[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) out[mb][nb][i] = 0.f;
    Regs nx;
    load(nx, wp, row, scales, biases, n_groups, 0);
    dma(d, 0, ba);
    if constexpr (BM)
      mh_bias<MB, NB>(x3, t0 + wt * MB * 32, static_cast<const uint16_t*>(biases), row, n_groups, out);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    auto step = [&](int64_t st, const Buf& cur, const Buf& nxt) {
      __builtin_amdgcn_s_waitcnt(0);  // this stage's registers (loaded during the last) are in
      MA_ISSUE_FENCE();
      const Regs r = nx;
      MA_ISSUE_FENCE();
      stage(r, cur, wt, out, [&]() {
        const bool more = st + 1 < nst;
        if (more) dma(d, st + 1, nxt);
        MA_ISSUE_FENCE();  // the copies are issued before the register loads
        load(nx, wp, row, scales, biases, n_groups, more ? st + 1 : st);
      });
      __builtin_amdgcn_s_waitcnt(mh_vmcnt(kLoads));  // the copies have landed
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      MA_ISSUE_FENCE();
    };
    for (int64_t st = 0; st < nst; st += 2) {
      step(st, ba, bb);
      if (st + 1 < nst) step(st + 1, bb, ba);
    }
    mh_store<MB, NB>(out, t0 + wt * MB * 32, n0, batch, n_out, y, ldy);
  }
};

template <int MB, int NB, int WT, int WN, int KS, int GW, int SDT, bool BM, int WPE>
__global__ __launch_bounds__(64 * WT * WN) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void k_mx_head(
    const uint4* __restrict__ xq, const uint8_t* __restrict__ xs, const float* __restrict__ xg,
    const uint16_t* __restrict__ x3, int64_t batch, int64_t rows, const uint32_t* __restrict__ w, int64_t n_out,
    int64_t nwords, const void* __restrict__ scales, const void* __restrict__ biases, uint16_t* __restrict__ y,
    int64_t ldy, int n_ttiles, int n_tiles) {
  using H = MxHead<MB, NB, WT, WN, KS, GW, SDT, BM>;
  // (distinct arrays: the compiler then sees that a stage's reads and the
  // copies in flight into the other buffer do not overlap)
  __shared__ __align__(16) uint32_t xa[H::kXDwords], xb[H::kXDwords];
  __shared__ __align__(16) uint32_t sa[KS * H::kTok / 4], sb[KS * H::kTok / 4];
  __shared__ __align__(16) float ga[H::kSums * H::kTok], gb[H::kSums * H::kTok];
  H::run(xq, xs, xg, x3, batch, rows, w, n_out, nwords, scales, biases, y, ldy, n_ttiles, n_tiles,
         typename H::Buf{xa, sa, ga}, typename H::Buf{xb, sb, gb});
}

// The tile of many tokens, 128 x 256 table rows on 8 waves (2 along the tokens,
// 64 x 64 each): everything a stage of 128 values of K needs -- x rows, table
// words, row scales, scale bytes -- comes by the LDS DMA two stages ahead, into
// three buffers (156 KB: one workgroup a CU).  A stage multiplies for about 1 us
// and its copies take 1 to 2; with one stage ahead the waves waited for them at
// every barrier.  bf16 scales and biases, the bias half on the matrix units.
// Both launches, 151,936 x 2048 in groups of 128 (64): 182 us at 256 tokens
// (201), 350 (551) as bf16 MFMAs, 203 in MxHead's tile of the same size, 194
// with a unit's fold in one piece; 104 (122) at 96, 124 in MxHead's tile.  The
// matrix units work 51 % of the time; the vector unit's 9 instructions a product
// hide behind them in part, and 4.6 tiles a CU leave the last round half empty.
template <int GW>
struct MxRing {
  static constexpr int MB = 2, NB = 2, WT = 2, WN = 4;
  static constexpr int kTok = 128, kRows = 256, kThreads = 512, KS = 2, NBUF = 3;
  static constexpr int kSums = KS * mh::kGroupWords / GW, GPR = GW / mh::kGroupWords;
  static constexpr int kCh = mh::kGroupChunks * KS;  // of a token per stage
  // dwords of a buffer: x rows, table words, then each wave's own scale bytes
  // (64 words, all tokens) and row scales (64 rows)
  static constexpr int kX = kTok * kCh * 4, kW = kRows * 16, kS = 8 * 64, kBuf = kX + kW + 2 * kS;
  static constexpr int kCopies = 4 + 2 + 1 + 1;  // per wave and stage

  const uint4* xq;
  int64_t ld, rows;
  const uint8_t* xs;
  const uint32_t* w;
  uint32_t woff[2];  // this thread's table copies
  const uint16_t* sc;  // scales of the lane's row of the wave's 64

  // x: token p's chunk c at slot p kCh + (c ^ p % 16); table row r's chunk c (4
  // words) at slot 4 r + (c ^ r / 4 % 4): a wave's reads of one chunk fall on
  // different banks
  __device__ __forceinline__ void copy(int64_t st, uint32_t* buf) const {
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int PER = kThreads / kCh;
    const int p0 = tid / kCh;
#pragma unroll
    for (int i = 0; i < kTok / PER; ++i) {
      const int c = (tid % kCh) ^ ((p0 + PER * i) % 16);
      const uint4* base = xq + PER * i * ld + st * kCh;  // the same in every lane
      __builtin_amdgcn_global_load_lds(base + static_cast<uint32_t>(p0 * static_cast<int>(ld) + c),
                                       (mh_lds_t)(buf + 4 * (64 * wv + kThreads * i)), 16, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
      __builtin_amdgcn_global_load_lds(w + st * 16 + woff[i], (mh_lds_t)(buf + kX + 4 * (64 * wv + kThreads * i)), 16, 0,
                                       0);
    __builtin_amdgcn_global_load_lds(
        reinterpret_cast<const uint32_t*>(xs + (st * KS + (lane >> 5)) * rows) + (lane & 31),
        (mh_lds_t)(buf + kX + kW + 64 * wv), 4, 0, 0);
    // the word that holds the stage's scales (n_groups is even)
    __builtin_amdgcn_global_load_lds(reinterpret_cast<const uint32_t*>(sc + (st * kSums & ~int64_t{1})),
                                     (mh_lds_t)(buf + kX + kW + kS + 64 * wv), 4, 0, 0);
  }

  // A stage's products, each unit's (an RTN group of a token block) followed by
  // a part of the unit before's fold: the vector unit folds while the matrix
  // unit multiplies (folding a unit in one piece, the two took turns).  acc[1]
  // and sp (its scales) carry the last unit over to the next stage.
  template <typename F>
  static __device__ __forceinline__ void multiply(const uint32_t* buf, int64_t st, int wv, f32x16_t (&out)[MB][NB],
                                                  f32x16_t (&acc)[2][NB], float (&sp)[NB], F&& send) {
    const int lane = threadIdx.x & 63, r32 = lane & 31, h = lane >> 5, wt = wv % WT, wn = wv / WT;
    const char* const b8 = reinterpret_cast<const char*>(buf);
    uint32_t off[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int p = (wt * MB + mb) * 32 + r32;
      off[mb] = static_cast<uint32_t>(p * kCh + ((2 * h) ^ (p % 16))) * 16;
      asm volatile("" : "+v"(off[mb]));  // recomputed per stage: hoisted, every read's address takes a register
    }
    uint4 w[KS][NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int r = wn * 64 + 32 * nb + r32;
#pragma unroll
      for (int gi = 0; gi < KS; ++gi)
        w[gi][nb] = *reinterpret_cast<const uint4*>(buf + kX + 4 * (4 * r + ((2 * gi + h) ^ (r / 4 % 4))));
    }
    uint32_t sw[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) sw[nb] = buf[kX + kW + kS + 64 * wv + 32 * nb + r32];
    constexpr int U = kSums * MB;
    const uint8_t* const s8 = reinterpret_cast<const uint8_t*>(buf + kX + kW + 64 * wv);
    auto scale = [&](int u, int g2) {
      return static_cast<int>(s8[((u / MB) * GPR + g2) * kTok + (wt * MB + u % MB) * 32 + r32]);
    };
    auto read = [&](int j) {  // piece j % 2 of group j / 2 % GPR of unit j / 2 / GPR
      const int u = j / 2 / GPR;
      const uint32_t c = (((u / MB) * GPR + j / 2 % GPR) * 8 + (j % 2) * 4) * 16;
      return mx_operand(*reinterpret_cast<const uint4*>(b8 + (off[u % MB] ^ c)),
                        *reinterpret_cast<const uint4*>(b8 + (off[u % MB] ^ (c + 16))));
    };
    i32x8_t bv[GPR][NB];
    float s[kSums][NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if constexpr (kSums == 2) {
        s[0][nb] = __uint_as_float(sw[nb] << 16);
        s[kSums - 1][nb] = __uint_as_float(sw[nb] & 0xffff0000u);
      } else {
        s[0][nb] = __uint_as_float((st & 1) ? (sw[nb] & 0xffff0000u) : (sw[nb] << 16));
      }
    }
    // part q of kParts of the fold of the unit before unit u
    constexpr int kParts = 2 * GPR * NB, kPer = 16 * NB / kParts;
    auto fold = [&](int u, int q) {
      const int up = u == 0 ? U - 1 : u - 1, mb = up % MB, nb = q * kPer / 16;
      const float f = u == 0 ? sp[nb] : s[up / MB][nb];
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int e = q * kPer % 16 + i;
        out[mb][nb][e] = __builtin_fmaf(f, acc[up & 1][nb][e], out[mb][nb][e]);
      }
    };
    int sa = scale(0, 0);
    i32x8_t av = read(0);
#pragma unroll
    for (int j = 0; j < 2 * GPR * U; ++j) {
      const int u = j / 2 / GPR, g2 = j / 2 % GPR, p = j % 2;
      if (p == 0 && u % MB == 0) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) bv[g2][nb] = mh_expand(w[(u / MB) * GPR + g2][nb]);
      }
      i32x8_t an = av;  // the next operand's reads go out ahead of these products
      int sn = sa;
      if (j + 1 < 2 * GPR * U) {
        an = read(j + 1);
        if (p == 1) sn = scale((j + 1) / 2 / GPR, (j + 1) / 2 % GPR);
      }
      MA_ISSUE_FENCE();
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if (g2 == 0 && p == 0) {
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[u & 1][nb][i] = 0.f;
        }
        acc[u & 1][nb] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv[g2][nb], acc[u & 1][nb], 0, 0, 0, sa, 0,
                                                                         136 - 4 * p);
        asm volatile("" : "+v"(acc[u & 1][nb])::"memory");  // one operand's reads at a time (mx_pin)
        fold(u, (g2 * 2 + p) * NB + nb);
        MA_ISSUE_FENCE();
      }
      if (j == 0) {
        MA_ISSUE_FENCE();
        send();
        MA_ISSUE_FENCE();
      }
      av = an;
      sa = sn;
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) sp[nb] = s[kSums - 1][nb];
  }

  // As MxTile::step (mx_gemm.hip): wait for stage st's copies, meet, send a
  // later stage's into the buffer just freed, multiply.
  template <bool TAIL>
  __device__ __forceinline__ void step(int64_t st, int64_t nst, const uint32_t* cur, uint32_t* prev, int wv,
                                       f32x16_t (&out)[MB][NB], f32x16_t (&acc)[2][NB], float (&sp)[NB]) const {
    if (!TAIL || st + NBUF - 1 < nst) __builtin_amdgcn_s_waitcnt(mh_vmcnt((NBUF - 2) * kCopies));
    else __builtin_amdgcn_s_waitcnt(mh_vmcnt(0));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    multiply(cur, st, wv, out, acc, sp, [&]() {
      if (!TAIL || st + NBUF - 1 < nst) copy(st + NBUF - 1, prev);
    });
    MA_ISSUE_FENCE();
  }
};

template <int GW>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_mx_head_ring(
    const uint4* __restrict__ xq, const uint8_t* __restrict__ xs, const uint16_t* __restrict__ x3, int64_t batch,
    int64_t rows, const uint32_t* __restrict__ w, int64_t n_out, int64_t nwords, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, uint16_t* __restrict__ y, int64_t ldy, int n_ttiles, int n_tiles) {
  using R = MxRing<GW>;
  __shared__ __align__(16) uint32_t b0[R::kBuf], b1[R::kBuf], b2[R::kBuf];
  const int per = (n_tiles + kXcds - 1) / kXcds;
  const int local = static_cast<int>(blockIdx.x) / kXcds;
  const int idx = (static_cast<int>(blockIdx.x) % kXcds) * per + local;
  if (local >= per || idx >= n_tiles) return;
  const int tid = threadIdx.x, lane = tid & 63, r32 = lane & 31, h = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wt = wv % R::WT, wn = wv / R::WT;
  const int64_t t0 = static_cast<int64_t>(idx % n_ttiles) * R::kTok;
  const int64_t r0 = static_cast<int64_t>(idx / n_ttiles) * R::kRows, n0 = r0 + 64 * wn;
  const int64_t nst = nwords / 16, n_groups = nwords / GW;
  const int64_t ld = nwords / mh::kGroupWords * mh::kGroupChunks;
  R t{xq + t0 * ld, ld, rows, xs + t0, w + r0 * nwords, {0u, 0u}, nullptr};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (tid + 512 * i) / 4, c = (tid % 4) ^ (r / 4 % 4);
    const int rc = r0 + r < n_out ? r : static_cast<int>(n_out - 1 - r0);  // past n_out: its last row
    t.woff[i] = static_cast<uint32_t>(rc * nwords + 4 * c);
  }
  t.sc = scales + (n0 + lane < n_out ? n0 + lane : n_out - 1) * n_groups;
  f32x16_t out[R::MB][R::NB];
#pragma unroll
  for (int mb = 0; mb < R::MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < R::NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) out[mb][nb][i] = 0.f;
  int64_t row[R::NB];
#pragma unroll
  for (int nb = 0; nb < R::NB; ++nb) row[nb] = n0 + 32 * nb + r32 < n_out ? n0 + 32 * nb + r32 : n_out - 1;
  mh_bias<R::MB, R::NB>(x3, t0 + wt * 64, biases, row, n_groups, out);
  MA_ISSUE_FENCE();
  t.copy(0, b0);
  MA_ISSUE_FENCE();
  t.copy(1, b1);  // nst is even
  MA_ISSUE_FENCE();
  // (no unit before the first: its fold adds 0 x 0)
  f32x16_t acc[2][R::NB];
  float sp[R::NB];
#pragma unroll
  for (int nb = 0; nb < R::NB; ++nb) {
    sp[nb] = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[1][nb][i] = 0.f;
  }
  int64_t st = 0;
  for (; st + 5 <= nst; st += 3) {
    t.template step<false>(st, nst, b0, b2, wv, out, acc, sp);
    t.template step<false>(st + 1, nst, b1, b0, wv, out, acc, sp);
    t.template step<false>(st + 2, nst, b2, b1, wv, out, acc, sp);
  }
  if (st < nst) t.template step<true>(st, nst, b0, b2, wv, out, acc, sp);
  if (st + 1 < nst) t.template step<true>(st + 1, nst, b1, b0, wv, out, acc, sp);
  if (st + 2 < nst) t.template step<true>(st + 2, nst, b2, b1, wv, out, acc, sp);
  if (st + 3 < nst) t.template step<true>(st + 3, nst, b0, b2, wv, out, acc, sp);
#pragma unroll
  for (int nb = 0; nb < R::NB; ++nb)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      out[R::MB - 1][nb][i] = __builtin_fmaf(sp[nb], acc[1][nb][i], out[R::MB - 1][nb][i]);
  mh_store<R::MB, R::NB>(out, t0 + wt * 64, n0, batch, n_out, y, ldy);
}

static int64_t mx_head_rows(int64_t batch) { return cdiv(batch, mh::kPad) * mh::kPad; }

// x rows, group sums (float32, then three bf16 parts), scale bytes.
size_t rtn4_mx_bytes(int64_t batch, int64_t nwords, int64_t group) {
  const int64_t rows = mx_head_rows(batch);
  return static_cast<size_t>(rows) * (nwords * 16 + nwords / mh::kGroupWords + nwords * 8 / group * 10);
}

}  // namespace ma

using namespace ma;

int launch_rtn4_mx(const uint16_t* x, int64_t batch, int64_t ldx, const uint32_t* w, int64_t n_out, int64_t nwords,
                   int64_t group, const void* scales, const void* biases, int s_dt, uint16_t* y, int64_t ldy,
                   void* workspace, hipStream_t s) {
  const int64_t rows = mx_head_rows(batch), gw = group / 8;
  uint4* xq = static_cast<uint4*>(workspace);
  float* xg = reinterpret_cast<float*>(xq + rows * nwords);
  uint16_t* x3 = reinterpret_cast<uint16_t*>(xg + rows * (nwords / gw));
  uint8_t* xs = reinterpret_cast<uint8_t*>(x3 + 3 * rows * (nwords / gw));
  hipLaunchKernelGGL(k_mx_head_prep, dim3(static_cast<unsigned>(batch)), dim3(256), 0, s, x, ldx, nwords,
                     static_cast<int>(gw), rows, xq, xs, xg, x3);
#define MA_MH(MB, NB, WT, WN, KS, GW, SDT, BM, WPE)                                                                  \
  do {                                                                                                               \
    using H = MxHead<MB, NB, WT, WN, KS, GW, SDT, BM>;                                                               \
    const int64_t tt = cdiv(batch, H::kTok), tiles = tt * cdiv(n_out, H::kRows);                                     \
    hipLaunchKernelGGL((k_mx_head<MB, NB, WT, WN, KS, GW, SDT, BM, WPE>),                                            \
                       dim3(static_cast<unsigned>(cdiv(tiles, kXcds) * kXcds)), dim3(H::kThreads), 0, s, xq, xs, xg, \
                       x3, batch, rows, w, n_out, nwords, scales, biases, y, ldy, static_cast<int>(tt),              \
                       static_cast<int>(tiles));                                                                     \
  } while (0)
// Tile by the number of tiles, so that a table of any height fills the chip.
// 32 tokens x 128 rows while that is one token tile or at most 512 tiles, two a
// CU (a wave's chain through K is the shorter one: 8,192 rows at 128 tokens, us,
// groups of 128: 17 against 22 with 64 tokens and 34 in the ring; 16,384 at 64
// 16 / 21; past it 50,000 at 64 35 / 26).  Above, 64 tokens x 128 rows, and from
// 768 of those the ring's 128 x 256 (one workgroup a CU), unless that pads the
// tokens by more than an eighth (groups of 128 (64): 32,000 rows at 128 27 (29)
// against 35 (38), at 192 37 (40) / 38 (42), at 256 49 (52) / 39 (42); 151,936
// at 128 99 (108) / 98 (106), at 192 136 (148) / 160 (173), at 256 179 (198) /
// 161 (175)).  The ring needs the bias half's product, whole steps of 16 bf16
// groups; float32 scales and other K keep to the small tiles (one of 128 x 128
// took 106 us for 94 at 100,003 rows, 128 tokens, groups of 64).
  const int64_t rtiles = cdiv(n_out, 128);
  const int64_t t32 = cdiv(batch, 32) * rtiles, t64 = cdiv(batch, 64) * rtiles;
  const int64_t tring = cdiv(batch, 128) * cdiv(n_out, 256);
  const bool bias_mm = s_dt == MA_BF16 && nwords / gw % 16 == 0;
#define MA_MH_T(GW, SDT, BM)              \
  if (batch <= 32 || t32 <= 2 * 256)      \
    MA_MH(1, 1, 1, 4, 4, GW, SDT, BM, 3); \
  else                                    \
    MA_MH(2, 1, 1, 4, 2, GW, SDT, BM, 3);
#define MA_MH_G(SDT, BM) \
  if (group == 64) { MA_MH_T(8, SDT, BM) } else { MA_MH_T(16, SDT, BM) }
  if (bias_mm && t64 > 3 * 256 && 32 * tring <= 9 * t64) {
    const int64_t tt = cdiv(batch, 128);
    auto* const kernel = group == 64 ? &k_mx_head_ring<8> : &k_mx_head_ring<16>;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(cdiv(tring, kXcds) * kXcds)), dim3(512), 0, s, xq, xs, x3,
                       batch, rows, w, n_out, nwords, static_cast<const uint16_t*>(scales),
                       static_cast<const uint16_t*>(biases), y, ldy, static_cast<int>(tt), static_cast<int>(tring));
  } else if (s_dt == MA_F32) {
    MA_MH_G(MA_F32, false)
  } else if (bias_mm) {
    MA_MH_G(MA_BF16, true)
  } else {
    MA_MH_G(MA_BF16, false)
  }
#undef MA_MH_G
#undef MA_MH_T
#undef MA_MH
  return check_launch("rtn4_gemv (mx)");
}
