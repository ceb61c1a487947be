// Products of many rows (prompts, drafter contexts) with affine group-64 codes: y[m] = x[m] . W^T for
// bf16 x [M, K], any M, on the tiled weights of w8.hip.
//
// Arithmetic, as the skinny GEMM's: w = s * q + b per group of 64 columns, so
//   y[m][n] = sum_g s[n][g] * (x . q)[m][n][g] + sum_g b[n][g] * X[m][g],   X[m][g] = sum of x over g.
// The codes are exact in bf16, their products accumulate in fp32 in the MFMA, and each group's sum is
// scaled in fp32. The second term is a product over K / 64 group sums: X as three bf16 terms (within
// 2^-26) against the bf16 biases, in the same MFMA accumulators (5 % more MFMA work, where X from a
// ones operand and four more fmas per tile and group would take 25 % and as many VALU slots as the
// scaling).
//
// dsk_rows_prep forms what a product needs of its input in one pass over the rows: the residual add
// that precedes it (with the sandwich norm), the RMSNorm, the X terms, and x in the order the product's
// loads take it (rows_index): one wave-wide load of an MFMA operand is 1 KiB of consecutive bytes. Read
// from row-major rows the 64 lanes of a load touch 64 separate pieces of 16 bytes (lanes next to each
// other hold different rows), and the product took 1.8 times as long (24576 x 4096, 2048 rows).
#include "common.h"
#include "wfrag.h"

namespace dsk {

// Element (m, k) of an operand with G 64-column groups: [m / 16][k / 64][half][lane][8], lane = m % 16 +
// 16 * ((k % 64) / 16), half = (k % 16) / 8. Rows past the last of a tile hold arbitrary values; they
// only reach their own columns of the product, which are not stored.
__device__ __forceinline__ int64_t rows_index(int64_t m, int64_t k, int64_t G) {
  return ((((m >> 4) * G + (k >> 6)) * 2 + ((k >> 3) & 1)) * 64 + (m & 15) + 16 * ((k >> 4) & 3)) * 8 + (k & 7);
}

// =====================================================================================
// rows_prep: one workgroup per row, the row held in registers
// =====================================================================================
constexpr int kPrepThreads = 512;
constexpr int kPrepMaxChunks = 6;  // 8-column chunks per thread: K <= 24576

struct PrepArgs {
  uint16_t* h;              // [M, K] bf16 rows, stride ldh; written back when y is added
  int64_t ldh;
  const uint16_t* y;        // projection output to add (bf16 [M, K], stride ldy), or null
  int64_t ldy;
  const uint16_t* y_norm;   // RMSNorm of y before the add, or null
  uint16_t* copy;           // h after the add (tap), or null
  int64_t ldc;
  int64_t K, G, Gp;         // G = K / 64 groups, Gp = G rounded up to 64
  int M;
  const uint16_t* norm_w;   // RMSNorm weight of the product's input, or null (x = h)
  int later;                // norm_w: x = bf16(h * w), row scale in rsc; else x = bf16(h * r * w)
  float eps;
  uint16_t* x;              // the product's input (rows_index), or null: no product follows
  uint16_t* xt;             // three terms of the group sums of x, each [M, Gp] as rows_index
  int64_t plane;            // elements of one term
  float* rsc;               // [M] row scales (later)
};

template <int NV>
__global__ __launch_bounds__(kPrepThreads) void rows_prep_kernel(PrepArgs a) {
  __shared__ float red[kPrepThreads / 64];
  // the 16 rows of a tile go to one XCD (workgroups go round robin to the eight): their 16-byte pieces
  // of the operand order share cache lines, which that XCD's L2 then writes whole (2048 rows of 20480:
  // 87 -> 52 us; 1027 of 15360: 34 -> 17.5)
  const int64_t m = (((int64_t)blockIdx.x / 128) * 8 + blockIdx.x % 8) * 16 + (blockIdx.x / 8) % 16;
  if (m >= a.M) return;
  const int tid = threadIdx.x;
  const int64_t nchunk = a.K / 8;
  u32x4 hv[NV], yv[NV], yw[NV], wv[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) {  // every load in flight at once; chunks past the row re-read its last
    const int64_t c = min(tid + (int64_t)i * kPrepThreads, nchunk - 1) * 8;
    hv[i] = *reinterpret_cast<const u32x4*>(a.h + m * a.ldh + c);
    if (a.y) yv[i] = *reinterpret_cast<const u32x4*>(a.y + m * a.ldy + c);
    if (a.y_norm) yw[i] = *reinterpret_cast<const u32x4*>(a.y_norm + c);
    if (a.norm_w) wv[i] = *reinterpret_cast<const u32x4*>(a.norm_w + c);
  }
  auto block_sum = [&](float s) {
    s = wave_sum(s);
    __syncthreads();
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int i = 0; i < kPrepThreads / 64; ++i) t += red[i];
    return t;
  };
  auto sumsq = [&](const u32x4 (&v)[NV]) {
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      if (tid + (int64_t)i * kPrepThreads >= nchunk) continue;
      const uint16_t* e16 = reinterpret_cast<const uint16_t*>(&v[i]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = bf16_to_f32(e16[e]);
        ss = fmaf(f, f, ss);
      }
    }
    return block_sum(ss);
  };
  if (a.y) {
    const float r1 = a.y_norm ? rsqrtf(sumsq(yv) / (float)a.K + a.eps) : 1.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const uint16_t* hh = reinterpret_cast<const uint16_t*>(&hv[i]);
      const uint16_t* yy = reinterpret_cast<const uint16_t*>(&yv[i]);
      const uint16_t* gg = reinterpret_cast<const uint16_t*>(&yw[i]);
      uint16_t o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float f = bf16_to_f32(yy[e]);
        if (a.y_norm) f = round_bf16((f * r1) * bf16_to_f32(gg[e]));
        o[e] = f32_to_bf16(bf16_to_f32(hh[e]) + f);
      }
      hv[i] = *reinterpret_cast<const u32x4*>(o);
    }
  }
  float r = 1.0f;
  if (a.norm_w) {
    r = rsqrtf(sumsq(hv) / (float)a.K + a.eps);
    if (a.later) {
      if (tid == 0) a.rsc[m] = r;
      r = 1.0f;
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = tid + (int64_t)i * kPrepThreads, g = c / 8;
    const bool live = c < nchunk;
    u32x4 xv = hv[i];
    if (a.norm_w) {
      const uint16_t* hh = reinterpret_cast<const uint16_t*>(&hv[i]);
      const uint16_t* gg = reinterpret_cast<const uint16_t*>(&wv[i]);
      uint16_t o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = f32_to_bf16((bf16_to_f32(hh[e]) * r) * bf16_to_f32(gg[e]));
      xv = *reinterpret_cast<const u32x4*>(o);
    }
    if (live) {
      if (a.y) *reinterpret_cast<u32x4*>(a.h + m * a.ldh + c * 8) = hv[i];
      if (a.copy) *reinterpret_cast<u32x4*>(a.copy + m * a.ldc + c * 8) = hv[i];
      if (a.x) *reinterpret_cast<u32x4*>(a.x + rows_index(m, c * 8, a.G)) = xv;
    }
    if (!a.x) continue;
    const uint16_t* e16 = reinterpret_cast<const uint16_t*>(&xv);
    float s = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) s += bf16_to_f32(e16[e]);
    s += __shfl_xor(s, 1, 64);  // 8 neighbouring threads hold one group
    s += __shfl_xor(s, 2, 64);
    s += __shfl_xor(s, 4, 64);
    if ((tid & 7) == 0 && g < a.Gp) {  // the NV kPrepThreads chunks cover Gp: padding groups get zero
      const Bf16x2Terms t = split3_bf16x2(live ? s : 0.0f, 0.0f);
      const int64_t o = rows_index(m, g, a.Gp / 64);
      a.xt[o] = (uint16_t)(t.hi & 0xffffu);
      a.xt[a.plane + o] = (uint16_t)(t.mid & 0xffffu);
      a.xt[2 * a.plane + o] = (uint16_t)(t.lo & 0xffffu);
    }
  }
}

// =====================================================================================
// the product
// =====================================================================================
struct RowsArgs {
  const u32x4* x;      // bf16 [M, K] as rows_index
  const u32x4* xt;     // three terms, [M, Gp] each
  const void* wt;      // tiled codes
  const uint32_t* sb;
  int M;
  int64_t N, K, G, Gp;
  int mblocks, nblocks;
  const float* rsc;    // row scales, or null
  int epi;
  uint16_t* y;         // bf16 output, row stride ldy (gated: [M, N / 2])
  int64_t ldy;
  uint16_t* h;         // DSK_EPI_RESIDUAL: h[m][n] = bf16(h[m][n] + y) in place, copy = h
  int64_t ldh;
  uint16_t* copy;
  int64_t ldc;
};

// 16 4-bit codes -> two bf16 x 8 holding the codes themselves (exact), so that the scales and biases
// enter as stored
__device__ __forceinline__ void codes_to_bf16(const u32x4 w, bf16x8& lo, bf16x8& hi) { u8x16_to_bf16(w, lo, hi); }
__device__ __forceinline__ void codes_to_bf16(const u32x2 w, bf16x8& lo, bf16x8& hi) {
  u32x4 c;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const uint32_t even = w[h] & 0x0f0f0f0fu, odd = (w[h] >> 4) & 0x0f0f0f0fu;
    c[2 * h] = __builtin_amdgcn_perm(odd, even, 0x05010400u);
    c[2 * h + 1] = __builtin_amdgcn_perm(odd, even, 0x07030602u);
  }
  u8x16_to_bf16(c, lo, hi);
}

// A workgroup computes 64 MTW rows x 16 NTW columns: its four waves own 16 MTW rows each and share
// every code, which one of them converts to bf16 and leaves in LDS (two buffers, one barrier per U
// 64-column groups; codes are loaded two steps ahead, the rows of x one, straight into the registers
// that feed the MFMA). KS > 1: KS such sets of four waves take a slice of the groups each. The weights are
// the A operand, so a lane ends with four consecutive columns of one row. Workgroup ids: a column block's
// row blocks run one after the other on one XCD, whose L2 then holds the column block's codes.
//
// What bounds it: with 256 x 64 tiles the 24576 x 4096 gate_up over 2048 rows takes 485 us = 849 TFLOP/s
// (stored without its activation 473; o 4096 x 4096 89 us, 771). Working copies of the 473 us without the
// loads of x or the scaling took 0.71 and 0.84 of it, without the conversion of the codes as long, without
// all three 0.58: the matrix pipe alone would reach 1.5 PFLOP/s behind the barriers, and the L2 traffic of x
// (6.4 GB) and the scaling's VALU work each add to it. Sharing x between two column halves of eight waves,
// 256 x 128 tiles or more steps in flight measured no faster at 2048 rows; at 1027, where 128-row tiles run,
// two column halves of them took 271 against 288 us (not built).
template <int MTW, int NTW, int U, int KS, int BITS, int EK>
__global__ __launch_bounds__(256 * KS) __attribute__((amdgpu_waves_per_eu(KS < 2 ? 2 : KS))) void w8_rows_kernel(RowsArgs a) {
  using WT = typename WeightChunk<BITS>::type;
  constexpr int CW = NTW * U / 4;  // tile-groups a wave converts per step
  static_assert(CW * 4 == NTW * U, "whole tile-groups per wave");
  __shared__ u32x4 bs_all[KS][2][U][NTW][2][64];
  __shared__ __attribute__((aligned(16))) float ss_all[KS][2][U][NTW][16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wv = wave & 3, ks = wave >> 2;
  auto& bs = bs_all[ks];
  auto& ss = ss_all[ks];
  const int i = blockIdx.x >> 3, nb = (i / a.mblocks) * 8 + (blockIdx.x & 7), mb = i % a.mblocks;
  if (nb >= a.nblocks) return;
  const int64_t t0 = (int64_t)nb * NTW;
  const int m0 = (mb * 4 + wv) * MTW * 16;
  const int G = (int)a.G, steps = G / (U * KS), first = ks * steps;  // the slice's steps
  const WT* wt = reinterpret_cast<const WT*>(a.wt);

  WT cw[2][CW];
  uint32_t cs[2][CW];
  auto load_codes = [&](int st, WT (&cw)[CW], uint32_t (&cs)[CW]) {
    st = first + min(st, steps - 1);
#pragma unroll
    for (int k = 0; k < CW; ++k) {
      const int it = wv + 4 * k, u = it / NTW, j = it % NTW;
      const int64_t tg = (t0 + j) * a.G + st * U + u;
      cw[k] = wt[tg * 64 + lane];
      cs[k] = a.sb[tg * 16 + (lane & 15)];
    }
  };
  auto convert = [&](int buf, const WT (&cw)[CW], const uint32_t (&cs)[CW]) {
#pragma unroll
    for (int k = 0; k < CW; ++k) {
      const int it = wv + 4 * k, u = it / NTW, j = it % NTW;
      bf16x8 lo, hi;
      codes_to_bf16(cw[k], lo, hi);
      bs[buf][u][j][0][lane] = __builtin_bit_cast(u32x4, lo);
      bs[buf][u][j][1][lane] = __builtin_bit_cast(u32x4, hi);
      ss[buf][u][j][lane & 15] = bf16_to_f32((uint16_t)(cs[k] & 0xffffu));  // four lanes, one value
    }
  };
  load_codes(0, cw[0], cs[0]);
  load_codes(1, cw[1], cs[1]);
  const bool live = m0 < a.M;
  if (!live) {  // a wave past the last row converts its codes only (its own loop, so that the
                // compiler counts the loads in flight of the other one exactly)
    convert(0, cw[0], cs[0]);
    load_codes(2, cw[0], cs[0]);
    for (int st0 = 0; st0 < steps; st0 += 2) {
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int st = st0 + k;
        if (st >= steps) break;
        __syncthreads();
        convert((st + 1) & 1, cw[1 - k], cs[1 - k]);
        load_codes(st + 3, cw[1 - k], cs[1 - k]);
      }
    }
    if constexpr (KS == 1) return;
  }
  f32x4 acc[MTW][NTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) acc[mt][nt] = f32x4{0, 0, 0, 0};
  const int last = (a.M - 1) / 16;  // row tiles past it re-read it and are not stored
  auto load_x = [&](int st, u32x4 (&d)[U][MTW][2]) {
    st = first + min(st, steps - 1);
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
        for (int f = 0; f < 2; ++f)
          d[u][mt][f] = a.x[(((int64_t)min(m0 / 16 + mt, last) * G + st * U + u) * 2 + f) * 64 + lane];
  };

  if (live) {
  // ---- the bias term: sum over groups of b * X, 64 groups per step (the first slice adds it)
  for (int gb = 0; gb < (ks == 0 ? G : 0); gb += 64) {
    bf16x8 bf[NTW][2];
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      uint32_t w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int g = gb + 16 * (lane >> 4) + 2 * e;
        const uint32_t* p = a.sb + ((t0 + nt) * a.G + min(g, G - 1)) * 16 + (lane & 15);
        const uint32_t w0 = p[0], w1 = p[g + 1 < G ? 16 : 0];
        w[e] = (g < G ? w0 >> 16 : 0u) | (g + 1 < G ? w1 & 0xffff0000u : 0u);
      }
      bf[nt][0] = __builtin_bit_cast(bf16x8, (u32x4{w[0], w[1], w[2], w[3]}));
      bf[nt][1] = __builtin_bit_cast(bf16x8, (u32x4{w[4], w[5], w[6], w[7]}));
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt) {
        const int64_t row = (int64_t)min(m0 / 16 + mt, last) * (a.Gp / 64) + gb / 64;
        const u32x4* px = a.xt + p * ((int64_t)(last + 1) * 16 * a.Gp / 8) + row * 128 + lane;
#pragma unroll
        for (int f = 0; f < 2; ++f) {
          const bf16x8 xf = __builtin_bit_cast(bf16x8, px[f * 64]);
#pragma unroll
          for (int nt = 0; nt < NTW; ++nt)
            acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[nt][f], xf, acc[mt][nt], 0, 0, 0);
        }
      }
  }
  convert(0, cw[0], cs[0]);
  load_codes(2, cw[0], cs[0]);
  u32x4 xs[2][U][MTW][2];
  load_x(0, xs[0]);

  // step st: the barrier publishes buffer st & 1 and retires every read of the other one. Column tile
  // i's operands are read from LDS while tile i - 1 is multiplied, the first ones before the next
  // step's codes are converted.
  constexpr int NI = U * NTW;
  struct Frag {
    u32x4 w[2];
    f32x4 s;
  };
  auto frag = [&](int buf, int i) {
    Frag f;
    const int u = i / NTW, j = i % NTW;
    f.w[0] = bs[buf][u][j][0][lane];
    f.w[1] = bs[buf][u][j][1][lane];
    f.s = *reinterpret_cast<const f32x4*>(&ss[buf][u][j][4 * (lane >> 4)]);
    return f;
  };
  for (int st0 = 0; st0 < steps; st0 += 2) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int st = st0 + k;
      if (st >= steps) break;
      __syncthreads();
      Frag f[2];
      f[0] = frag(st & 1, 0);
      load_x(st + 1, xs[1 - k]);
      __builtin_amdgcn_sched_barrier(0);
      convert((st + 1) & 1, cw[1 - k], cs[1 - k]);
      load_codes(st + 3, cw[1 - k], cs[1 - k]);
      // column tile i's products are issued ahead of the scaling of tile i - 1's, so that the matrix
      // pipe runs through the scaling
      f32x4 t[2][MTW];
      auto scale = [&](int i) {
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            acc[mt][i % NTW][q] = fmaf(f[i & 1].s[q], t[i & 1][mt][q], acc[mt][i % NTW][q]);
      };
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int u = i / NTW;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int mt = 0; mt < MTW; ++mt)
            t[i & 1][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                __builtin_bit_cast(bf16x8, f[i & 1].w[h]), __builtin_bit_cast(bf16x8, xs[k][u][mt][h]),
                h == 0 ? f32x4{0, 0, 0, 0} : t[i & 1][mt], 0, 0, 0);
        if (i > 0) scale(i - 1);
        if (i + 1 < NI) f[(i + 1) & 1] = frag(st & 1, i + 1);
        if (i > 0) {
#pragma unroll
          for (int g = 0; g < 2 * MTW; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA,
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two of the 4 MTW fmas
          }
          __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);    // the next tile's LDS reads
        }
      }
      scale(NI - 1);
    }
  }
  }  // live

  // ---- the K slices' sums, added in slice order by the first one, a column tile at a time
  if constexpr (KS > 1) {
    f32x4(&red)[KS - 1][4][MTW][64] = reinterpret_cast<f32x4(&)[KS - 1][4][MTW][64]>(bs_all);
    static_assert(sizeof(red) <= sizeof(bs_all), "the slices' sums fit the code buffers");
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      __syncthreads();
      if (ks > 0 && live)
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt) red[ks > 0 ? ks - 1 : 0][wv][mt][lane] = acc[mt][nt];
      __syncthreads();
      if (ks == 0 && live)
#pragma unroll
        for (int q = 0; q < KS - 1; ++q)
#pragma unroll
          for (int mt = 0; mt < MTW; ++mt) acc[mt][nt] += red[q][wv][mt][lane];
    }
    if (ks > 0 || !live) return;
  }

  // ---- epilogue: lane holds columns n .. n + 3 of row m
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    const int64_t m = m0 + 16 * mt + (lane & 15);
    if (m >= a.M) continue;
    const float r = a.rsc ? a.rsc[m] : 1.0f;
#pragma unroll
    for (int nt = 0; nt < NTW; ++nt) {
      if (EK == 1 && (nt & 1)) continue;
      f32x4 v = acc[mt][nt] * r;
      const int64_t n = (t0 + nt) * 16 + 4 * (lane >> 4);
      if constexpr (EK == 1) {
        const f32x4 u = acc[mt][nt + 1 < NTW ? nt + 1 : nt] * r;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float gb = round_bf16(v[q]);
          v[q] = round_bf16(a.epi == DSK_EPI_SWIGLU ? silu_f(gb) : gelu_tanh_f(gb)) * round_bf16(u[q]);
        }
        const int64_t col = ((t0 + nt) >> 1) * 16 + 4 * (lane >> 4);
        *reinterpret_cast<uint2*>(a.y + m * a.ldy + col) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      } else if constexpr (EK == 3) {
        const uint2 hw = *reinterpret_cast<const uint2*>(a.h + m * a.ldh + n);
        const uint2 o = uint2{pack_bf16x2(bits_f32(hw.x << 16) + v[0], bits_f32(hw.x & 0xffff0000u) + v[1]),
                              pack_bf16x2(bits_f32(hw.y << 16) + v[2], bits_f32(hw.y & 0xffff0000u) + v[3])};
        *reinterpret_cast<uint2*>(a.h + m * a.ldh + n) = o;
        if (a.copy) *reinterpret_cast<uint2*>(a.copy + m * a.ldc + n) = o;
      } else {
        *reinterpret_cast<uint2*>(a.y + m * a.ldy + n) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
    }
  }
}

// =====================================================================================
// host side
// =====================================================================================
struct RowsPlan {
  int mt, nt, u, ks;  // workgroup tile in 64 rows and 16 columns, groups per step, K slices
};

// A sweep on MI355X over the Qwen3-8B and Gemma-style 12B projections (and the 4-bit DFlash context's)
// at M = 65, 130, 203, 300, 700, 1027 and 2048 (times in us):
//  - 256 x 64 where that gives every CU two workgroups (gate_up 24576 x 4096 at M = 2048: 496 against
//    537 for 128 x 64; its four waves read 8 KB of x per group for 32 MFMAs each) and its last row
//    block pads the rows by no more than the 128-row one would by a tenth;
//  - else 128 x 64 with the groups in one slice from 512 workgroups (o 4096 x 4096 at M = 1027: 62),
//    two from 256 (o at M = 700: 43 against 48 in one slice), four above 128 (qkv 6144 x 4096 at
//    M = 203: 28 against 38): the slices keep two to four waves on every SIMD;
//  - else 64 x 64 in four slices (down 4096 x 12288 at M = 203: 52 against 69 for 128 x 64 in four);
//  - and 64 x 32 in four slices when that leaves most of the chip idle (o at M = 65: 14 against 20).
// Before, such rows ran as passes of 64 (o at M = 203: four launches, 74; gate_up: 215 against 70).
static RowsPlan plan_rows(int M, int64_t N, int64_t G) {
  const int64_t tiles = N / 16;
  if (tiles % 2) return {1, 1, 4, 1};
  if (tiles % 4 == 0) {
    const int64_t cols = tiles / 4, b4 = ceil_div(M, 256), b2 = ceil_div(M, 128);
    if (b4 * cols >= 512 && 20 * b4 <= 11 * b2) return {4, 4, 1, 1};
    if (b2 * cols >= 512) return {2, 4, 1, 1};
    if (b2 * cols >= 256) return {2, 4, 1, 2};
    if (b2 * cols > 128) return {2, 4, 1, 4};
    if (ceil_div(M, 64) * cols >= 160) return {1, 4, 1, 4};
  }
  return {1, 2, 2, G % 8 == 0 ? 4 : 2};
}

template <int MTW, int NTW, int U, int KS, int BITS>
static bool launch_rows_t(const RowsArgs& a, dim3 grid, hipStream_t st) {
  const dim3 blk(256 * KS);
  if (a.epi == DSK_EPI_STORE) {
    hipLaunchKernelGGL((w8_rows_kernel<MTW, NTW, U, KS, BITS, 0>), grid, blk, 0, st, a);
  } else if (a.epi == DSK_EPI_RESIDUAL) {
    hipLaunchKernelGGL((w8_rows_kernel<MTW, NTW, U, KS, BITS, 3>), grid, blk, 0, st, a);
  } else {
    if constexpr (NTW % 2 != 0) return false;
    else hipLaunchKernelGGL((w8_rows_kernel<MTW, NTW, U, KS, BITS, 1>), grid, blk, 0, st, a);
  }
  return true;
}

template <int BITS>
static bool launch_rows(const RowsArgs& a, const RowsPlan& p, hipStream_t st) {
  const dim3 grid((unsigned)(ceil_div(a.nblocks, 8) * 8 * a.mblocks));
#define DSK_ROWS_CASE(M_, N_, U_, S_) \
  if (p.mt == M_ && p.nt == N_ && p.u == U_ && p.ks == S_) return launch_rows_t<M_, N_, U_, S_, BITS>(a, grid, st);
  DSK_ROWS_CASE(4, 4, 1, 1) DSK_ROWS_CASE(2, 4, 1, 1) DSK_ROWS_CASE(2, 4, 1, 2) DSK_ROWS_CASE(2, 4, 1, 4)
  DSK_ROWS_CASE(1, 4, 1, 4) DSK_ROWS_CASE(1, 2, 2, 4) DSK_ROWS_CASE(1, 2, 2, 2) DSK_ROWS_CASE(1, 1, 4, 1)
#undef DSK_ROWS_CASE
  return false;
}

}  // namespace dsk

using namespace dsk;

extern "C" int dsk_rows_prep(uint16_t* h, int64_t ldh, const uint16_t* y, int64_t ldy, const uint16_t* y_norm_w,
                             uint16_t* copy, int64_t ldc, int M, int64_t K, const uint16_t* norm_w, int later,
                             float eps, uint16_t* x, uint16_t* xt, float* rsc, dsk_stream_t stream) {
  DSK_REQUIRE(h && M > 0, "dsk_rows_prep: no rows");
  DSK_REQUIRE(K > 0 && K % 64 == 0 && K <= 8 * kPrepThreads * kPrepMaxChunks,
              "dsk_rows_prep: K=%lld must be a multiple of 64 <= %d", (long long)K, 8 * kPrepThreads * kPrepMaxChunks);
  DSK_REQUIRE(ldh >= K && ldh % 8 == 0 && (!y || (ldy >= K && ldy % 8 == 0)) && (!copy || (ldc >= K && ldc % 8 == 0)),
              "dsk_rows_prep: bad row stride");
  DSK_REQUIRE(!y_norm_w || y, "dsk_rows_prep: y_norm_w needs y");
  DSK_REQUIRE(!norm_w || !later || rsc, "dsk_rows_prep: a norm applied later needs rsc");
  DSK_REQUIRE(!x == !xt && (!norm_w || x), "dsk_rows_prep: x and xt come together, normed rows with them");
  DSK_REQUIRE(((((uintptr_t)h | (uintptr_t)y | (uintptr_t)y_norm_w | (uintptr_t)copy) | (uintptr_t)norm_w |
                (uintptr_t)x | (uintptr_t)xt) & 15) == 0,
              "dsk_rows_prep: pointers must be 16-byte aligned");
  const int64_t G = K / 64;
  PrepArgs a{h, ldh, y, ldy, y_norm_w, copy, ldc, K, G, (G + 63) / 64 * 64, M, norm_w, later, eps, x, xt,
             (int64_t)((M + 15) / 16 * 16) * ((G + 63) / 64 * 64), rsc};
  const dim3 grid((unsigned)(ceil_div(M, 128) * 128)), blk(kPrepThreads);
  const hipStream_t st = as_stream(stream);
  switch (ceil_div(K / 8, kPrepThreads)) {
    case 1: hipLaunchKernelGGL(rows_prep_kernel<1>, grid, blk, 0, st, a); break;
    case 2: hipLaunchKernelGGL(rows_prep_kernel<2>, grid, blk, 0, st, a); break;
    case 3: hipLaunchKernelGGL(rows_prep_kernel<3>, grid, blk, 0, st, a); break;
    case 4: hipLaunchKernelGGL(rows_prep_kernel<4>, grid, blk, 0, st, a); break;
    case 5: hipLaunchKernelGGL(rows_prep_kernel<5>, grid, blk, 0, st, a); break;
    default: hipLaunchKernelGGL(rows_prep_kernel<6>, grid, blk, 0, st, a); break;
  }
  DSK_LAUNCH_CHECK("dsk_rows_prep");
  return DSK_OK;
}

extern "C" int dsk_w8_rows(const uint16_t* x, const uint16_t* xt, const uint8_t* wt, const uint32_t* sb,
                           int bits, int M, int64_t N, int64_t K, int epi, const float* rsc, uint16_t* y, int64_t ldy,
                           uint16_t* h, int64_t ldh, uint16_t* copy, int64_t ldc, dsk_stream_t stream) {
  DSK_REQUIRE(x && xt && wt && sb, "dsk_w8_rows: null pointer");
  DSK_REQUIRE(bits == 8 || bits == 4, "dsk_w8_rows: bits=%d (8 or 4)", bits);
  DSK_REQUIRE(M > 0 && N > 0 && N % 16 == 0 && K > 0 && K % 256 == 0, "dsk_w8_rows: bad shape M=%d N=%lld K=%lld", M,
              (long long)N, (long long)K);
  DSK_REQUIRE((((uintptr_t)x | (uintptr_t)xt | (uintptr_t)wt) & 15) == 0,
              "dsk_w8_rows: x and the weights must be 16-byte aligned");
  const bool gated = epi == DSK_EPI_SWIGLU || epi == DSK_EPI_GEGLU;
  if (epi == DSK_EPI_RESIDUAL) {
    DSK_REQUIRE(h && ldh >= N && ldh % 4 == 0 && ((uintptr_t)h & 7) == 0, "dsk_w8_rows: bad h");
    DSK_REQUIRE(!copy || (ldc >= N && ldc % 4 == 0 && ((uintptr_t)copy & 7) == 0), "dsk_w8_rows: bad copy");
  } else {
    DSK_REQUIRE(epi == DSK_EPI_STORE || gated, "dsk_w8_rows: bad epilogue %d", epi);
    DSK_REQUIRE(!gated || N % 32 == 0, "dsk_w8_rows: gated weights come in tile pairs");
    DSK_REQUIRE(y && ldy >= (gated ? N / 2 : N) && ldy % 4 == 0 && ((uintptr_t)y & 7) == 0, "dsk_w8_rows: bad y");
  }
  const RowsPlan p = plan_rows(M, N, K / 64);
  RowsArgs a{};
  a.x = reinterpret_cast<const u32x4*>(x);
  a.xt = reinterpret_cast<const u32x4*>(xt);
  a.wt = wt;
  a.sb = sb;
  a.M = M;
  a.N = N;
  a.K = K;
  a.G = K / 64;
  a.Gp = (a.G + 63) / 64 * 64;
  a.mblocks = (int)ceil_div(M, 64 * p.mt);
  a.nblocks = (int)(N / 16 / p.nt);
  a.rsc = rsc;
  a.epi = epi;
  a.y = y;
  a.ldy = ldy;
  a.h = h;
  a.ldh = ldh;
  a.copy = copy;
  a.ldc = ldc;
  const bool ok = bits == 8 ? launch_rows<8>(a, p, as_stream(stream)) : launch_rows<4>(a, p, as_stream(stream));
  DSK_REQUIRE(ok, "dsk_w8_rows: no kernel for M=%d N=%lld K=%lld", M, (long long)N, (long long)K);
  DSK_LAUNCH_CHECK("dsk_w8_rows");
  return DSK_OK;
}
