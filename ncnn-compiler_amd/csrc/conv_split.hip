// fp32 Convolution (reference ConvertConvolution fp32 path,
// NCNNToTosa.cpp:1316-1529) as an implicit GEMM on the bf16 matrix
// instructions with every fp32 operand as three bf16 pieces.  (Short reductions
// are faster in fp32: conv_igemm.hip, conv_smallk.hip.)
//
// v_mfma_f32_32x32x16_bf16 does 16 times the work of v_mfma_f32_32x32x2_f32
// in a cycle.  x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0),
// x2 = bf16(x - x0 - x1), each rounded to nearest even, loses nothing while x2 is
// a normal number or 0 (|x| from 2^-102 on, or fewer bits): three 8-bit
// significands cover fp32's 24 bits, the differences are exact in fp32, and bf16
// has fp32's exponent range.  Of the nine products of two such sums
// the six of order 2^-16 and above are formed (x0 w0, x0 w1, x1 w0, x0 w2,
// x1 w1, x2 w0); the three dropped (x1 w2, x2 w1, x2 w2) are below 2^-23 of |x w|
// (on 40 million random pairs at most 2^-24.1, 2.7% above 2^-26).  Sums stay in
// fp32 accumulators, and a matrix instruction adds 16 products before it rounds
// where the fp32 one adds two.  So from two products on a sum is nearer to 64
// bits than a chain of fp32 (normwise 2.6e-8 against 3.1e-8 at two, 3.1e-8 against
// 7.4e-8 at 16, emulated); one product alone is not (2.60e-8 against 2.53e-8, up
// to 1.7 half ulps against one) and is formed in fp32.
//
// Where the pieces do not stand for the number: an infinity or NaN (or a value
// that rounds to bf16's infinity) turns the pieces below it into NaN, x0 w0 may
// overflow where x w does not, and a last piece below fp32's normal numbers may be
// rounded (an input of 1e-36 would keep 15 bits).  A wave that met such an input,
// or whose block holds such a sum or one that is not finite, forms its block again on
// v_mfma_f32_32x32x2_f32, so what the caller sees is fp32 arithmetic, with its
// infinities and NaNs.  (32 x 64 -> 128 below, 47 us: 96 with every value NaN, 69
// with one; 69 on the fp32 kernel that it replaced, 6070 and 2650 where each such
// output was summed by one lane.)  Weights that small are scaled by the plan.
//
// GEMM view: D[i][j] = sum_k A[i][k] B[k][j], i an output channel, j an output
// pixel over the whole batch.  The reduction runs over octets of eight input
// channels of one kernel tap, taps outermost, so that an octet's bounds check
// and address are found once and its eight loads differ by a scalar offset;
// inputs of few channels (network stems) keep the (c, kh, kw) order and the
// table of taps instead.  The weights come split and in fragment order from
// the plan, [m/32][step of 16 k][piece][64 lanes][8].
//
// A wave owns 32 TM x 32 outputs (its lanes a pixel and half of a step's k) and
// streams both operands into registers, two steps ahead: the weights as whole
// fragments, the input as eight gathered values that it splits itself (5.5
// vector operations a value, in the shadow of its 6 TM matrix instructions).
// No LDS and no barrier in the loop.  A workgroup's waves are pixel blocks
// that share the weights through the L1 cache, and parts of the reduction,
// added through LDS in wave order at the end; long reductions of few outputs
// are also cut over workgroups and added by a second launch.  With operand
// tiles shared through LDS instead (64 x 128 outputs, stages of 32 k, a barrier
// each) 3x3 stride 2, 64 -> 128 at 56x56 x 32 took the same 40 us and every
// smaller launch more (one wave in flight per SIMD to cover the loads).
//
// What bounds it: large launches the operand stream from L2 (a step brings 5
// or 8 KB for 6 or 12 matrix instructions: 36 steps, 1568 workgroups, 41 us at
// 64 -> 128 above, 70 us on fp32 matrix instructions and LDS tiles), small ones
// the chain of load round trips (9 x 40 -> 24 at 21x21: 6.6 us).  Before ->
// now: 3x3 stride 2, 128 -> 256 at 28x28 x 32: 79 -> 41 us; 8 x 64 -> 128 at
// 56x56: 29 -> 16; 5x5 stride 2, 4 x 256 -> 32 at 103x103: 237 -> 78; 1 x 168 ->
// 24 at 80x80: 27 -> 14; 1x1, 576 -> 96 at 14x14: 17 -> 7.4; stem 7x7 at 224x224
// x 32: 107 -> 100.  Error against 64 bits, normwise: 4.3e-7 -> 1.4e-7 (576
// terms), 2.8e-7 -> 0.95e-7 (3384 terms), 1.5e-7 -> 0.7e-7 (1x1, 232 terms).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>

#include "nhip_internal.h"

namespace nhip {
namespace {

constexpr int kXcds = 8;
constexpr int kPieces = 3;
constexpr int kFrag = 1024;  // bytes of one 32 x 16 bf16 operand fragment (64 lanes x 16)

typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Reduction order: the table of (c, kh, kw); channels per tap, a multiple of
// 16; channels per tap in octets, the last one possibly ragged.
enum { kTable, kTaps, kTapsRagged };

// 2 |x| - 1 in bits for |x| = 2^-102: below it the last piece may be subnormal.
constexpr uint32_t kSmall = 25u << 24;

struct SplitArgs {
  const uint16_t* a;     // split weights in fragment order
  int nk;                // steps of 16 k
  int m;                 // output channels
  const float* x;        // input NCHW
  uint32_t x_bytes;      // < 2^31
  int npix;              // output pixels of the batch
  int C, c_pad, khw, KW, H, W, OW, OHW, sh, sw, pt, pl, dh, dw;
  const int* ktab;       // (c, kh, kw) order: c << 16 | dy << 8 | dx
  int kred;
  const float* unscale;  // [m_pad] powers of two that undo the scaling of the weights' rows, or null
  FastDiv ohw_div, ow_div, oct_div, kw_div;  // by OHW, OW, steps (kTaps) or octets per tap, KW
  float* d;              // out NCHW, or partial sums [split][m][npix]
  const float* bias;
  const float* residual;
  int act, splits;       // splits: parts of the reduction in separate workgroups (grid z)
  int wn, kparts;        // a workgroup's waves: pixel blocks x parts of its reduction
};

__device__ __forceinline__ float split_act(float v, int act) {
  if (act == NHIP_ACT_RELU) return v < 0.0f ? 0.0f : v;
  if (act == NHIP_ACT_SIGMOID) return 1.0f / (1.0f + __expf(-v));
  return v;
}

// The three pieces of two values, one word (low half: a) per piece.
__device__ __forceinline__ void split2(float a, float b, uint32_t (&p)[kPieces]) {
#pragma unroll
  for (int i = 0; i < kPieces; ++i) {
    const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f{a, b}), bf16x2));
    p[i] = u;
    a -= __uint_as_float(u << 16);
    b -= __uint_as_float(u & 0xffff0000u);
  }
}

template <int TM, int ORDER>
__global__ __launch_bounds__(TM == 1 ? 1024 : 512) void conv_split_kernel(SplitArgs g) {
  constexpr int BM = 32 * TM;
  const int BN = 32 * g.wn;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, lh = lane >> 5;
  const int kpart = wave / g.wn, wn = wave - kpart * g.wn;
  // consecutive blocks on one XCD (workgroups go round-robin over the XCDs):
  // the blocks of one pixel range share its input, all share the weights
  int bx, by, bz;
  {
    const int nbx = gridDim.x, nby = gridDim.y, total = nbx * nby * gridDim.z;
    const int L = blockIdx.x + nbx * (blockIdx.y + nby * blockIdx.z);
    const int x = L % kXcds, q = L / kXcds;
    const int logical = x * (total / kXcds) + min(x, total % kXcds) + q;
    by = logical % nby;
    bx = (logical / nby) % nbx;
    bz = logical / (nbx * nby);
  }
  const int j0 = bx * BN, i0 = by * BM;
  // the launch's part of the reduction, and this wave's
  const int zper = (g.nk + g.splits - 1) / g.splits, z_begin = min(g.nk, bz * zper), z_end = min(g.nk, z_begin + zper);
  const int per = (z_end - z_begin + g.kparts - 1) / g.kparts;
  const int k_begin = min(z_end, z_begin + kpart * per), k_end = min(z_end, k_begin + per);

  const __amdgpu_buffer_rsrc_t xr = make_rsrc(g.x, g.x_bytes);
  const int plane = g.H * g.W;
  int iy0, ix0, pbase;
  bool pix_ok;
  {
    const int p = j0 + 32 * wn + li;
    pix_ok = p < g.npix;
    const int pp = pix_ok ? p : 0;
    const int img = fdiv(pp, g.ohw_div), rem = pp - img * g.OHW;
    const int oh = fdiv(rem, g.ow_div), ow = rem - oh * g.OW;
    iy0 = oh * g.sh - g.pt;
    ix0 = ow * g.sw - g.pl;
    pbase = img * g.C * plane + (ORDER == kTaps ? 8 * lh * plane : 0);
  }
  struct Step {
    v4i a[TM][kPieces];
    float b[8];
  };
  const char* abase = reinterpret_cast<const char*>(g.a) + (int64_t)(i0 / 32) * g.nk * (kPieces * kFrag) + lane * 16;
  // the lane's value u of step k, in the table's order
  auto gather = [&](int k, int u) {
    const int ka = min(k, g.nk - 1), t0 = g.ktab[ka * 16 + u], t1 = g.ktab[ka * 16 + 8 + u], e = lh ? t1 : t0;
    const int c = e >> 16, kk = k * 16 + lh * 8 + u;
    const int y = iy0 + ((e >> 8) & 255), x = ix0 + (e & 255);
    const bool in = pix_ok && k < k_end && kk < g.kred && (unsigned)y < (unsigned)g.H && (unsigned)x < (unsigned)g.W;
    return buf_load_f32(xr, in ? (uint32_t)(pbase + (c * g.H + y) * g.W + x) * 4u : kBufOOB);
  };
  auto load = [&](Step& st, int k) {  // past the end: the input reads zero
    const int ka = min(k, g.nk - 1);
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int p = 0; p < kPieces; ++p)
        st.a[a][p] = *reinterpret_cast<const v4i*>(abase + ((int64_t)a * g.nk + ka) * (kPieces * kFrag) + p * kFrag);
    if constexpr (ORDER == kTable) {
#pragma unroll
      for (int u = 0; u < 8; ++u) st.b[u] = gather(k, u);
    } else {
      const int o = ORDER == kTaps ? k : 2 * k + lh, per_tap = ORDER == kTaps ? g.c_pad / 16 : g.c_pad / 8;
      const int tap = fdiv(o, g.oct_div), c0 = (o - tap * per_tap) * (ORDER == kTaps ? 16 : 8);
      const int ky = fdiv(tap, g.kw_div), kx = tap - ky * g.KW;
      const int y = iy0 + ky * g.dh, x = ix0 + kx * g.dw;
      const bool in = pix_ok && k < k_end && tap < g.khw && (unsigned)y < (unsigned)g.H && (unsigned)x < (unsigned)g.W;
      const int at = pbase + (ORDER == kTaps ? 0 : c0 * plane) + y * g.W + x;
      const uint32_t off = in ? (uint32_t)at * 4u : kBufOOB;
#pragma unroll
      for (int u = 0; u < 8; ++u) {  // channels past the last one (the weights are zero there) read zero
        // (the scalar offset stays inside the tensor, also where it has fewer
        // than eight channels in all: the range check subtracts it from the size)
        const int soff =
            __builtin_amdgcn_readfirstlane((ORDER == kTaps ? c0 + u : ORDER == kTapsRagged && u >= g.C ? 0 : u) * plane * 4);
        st.b[u] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(xr, ORDER == kTaps || c0 + u < g.C ? off : kBufOOB, soff, 0));
      }
    }
  };
  // x0 w0 on its own: its sum is rounded once per 16 products, the other
  // five (2^-8 and below of it) add into theirs
  v16f acc[TM], low[TM];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[a][r] = low[a][r] = 0.f;
  // The smallest magnitude met but 0, as 2 |x| - 1 in bits (0: the largest): 1.5
  // operations a value.  Left to the compiler they wait at the loop's end, sixteen
  // registers and a wave per SIMD more (up to 11% of a launch), so they are tied
  // to the values before the split (few registers to spare there) or closed after it.
  // (A sum of one product is formed in fp32 whatever its values.)
  uint32_t least = g.kred > 1 ? 0xffffffffu : 0u;
  auto track = [&](float a, float b) {
    least = min(least, min((__float_as_uint(a) << 1) - 1, (__float_as_uint(b) << 1) - 1));
  };
  auto mul = [&](const Step& st) {
    uint32_t w[4][kPieces];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float x0 = st.b[2 * u], x1 = st.b[2 * u + 1];
      if constexpr (ORDER == kTable) {
        track(x0, x1);
        asm("" : "+v"(least), "+v"(x0), "+v"(x1));
      }
      split2(x0, x1, w[u]);
    }
    bf16x8 f[kPieces];
#pragma unroll
    for (int p = 0; p < kPieces; ++p)
      f[p] = __builtin_bit_cast(bf16x8, (v4i{(int)w[0][p], (int)w[1][p], (int)w[2][p], (int)w[3][p]}));
    if constexpr (ORDER != kTable) {
#pragma unroll
      for (int u = 0; u < 4; ++u) track(st.b[2 * u], st.b[2 * u + 1]);
      asm volatile("" : "+v"(least));
    }
    constexpr int kProd[6][2] = {{0, 0}, {1, 0}, {0, 1}, {1, 1}, {2, 0}, {0, 2}};
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        v16f& c = q == 0 ? acc[a] : low[a];
        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, st.a[a][kProd[q][0]]), f[kProd[q][1]], c,
                                                    0, 0, 0);
      }
  };
  // The same steps in fp32, into acc: a lane's weights put together again (a sum
  // of their pieces is exact), value u of its eight the k of one instruction.
  float un[TM];  // what undoes the scaling of the lane's rows
#pragma unroll
  for (int a = 0; a < TM; ++a) un[a] = 1.f;
  auto mul32 = [&](const Step& st) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        float w[kPieces];
#pragma unroll
        for (int p = 0; p < kPieces; ++p) {
          const uint32_t two = (uint32_t)st.a[a][p][u >> 1];
          w[p] = __uint_as_float(u & 1 ? two & 0xffff0000u : two << 16);
        }
        acc[a] = __builtin_amdgcn_mfma_f32_32x32x2f32((w[0] + w[1] + w[2]) * un[a], st.b[u], acc[a], 0, 0, 0);
      }
  };
  {
    Step s0, s1;
    load(s0, k_begin);
    load(s1, k_begin + 1);
    for (int k = k_begin; k < k_end; k += 2) {
      mul(s0);
      load(s0, k + 2);
      mul(s1);  // (zero where the range has ended)
      load(s1, k + 3);
    }
  }
  float chk = 0.f;
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[a][r] += low[a][r];
      chk = __builtin_fmaf(acc[a][r], 0.f, chk);  // 0, or NaN from the first one that is not finite
      if (r & 1) track(acc[a][r - 1], acc[a][r]);  // (sums near the subnormal numbers: two roundings there are more than one)
    }
  if (__builtin_expect(__ballot(least < kSmall || chk != chk) != 0, 0)) {
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      if (g.unscale) un[a] = g.unscale[i0 + 32 * a + li];
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][r] = 0.f;
    }
#pragma unroll 1
    for (int k = k_begin; k < k_end; ++k) {
      if constexpr (ORDER == kTable) {  // one value at a time: eight would take a wave per SIMD's registers
#pragma unroll 1
        for (int u = 0; u < 8; ++u) {
          const float x = gather(k, u);
#pragma unroll
          for (int a = 0; a < TM; ++a) {
            float w = 0.f;
#pragma unroll
            for (int p = 0; p < kPieces; ++p)
              w += __uint_as_float((uint32_t)*reinterpret_cast<const uint16_t*>(
                       abase + ((int64_t)a * g.nk + k) * (kPieces * kFrag) + p * kFrag + 2 * u) << 16);
            acc[a] = __builtin_amdgcn_mfma_f32_32x32x2f32(w * un[a], x, acc[a], 0, 0, 0);
          }
        }
      } else {
        Step st;
        load(st, k);
        mul32(st);
      }
    }
  } else if (g.unscale) {
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][r] *= g.unscale[i0 + 32 * a + (r & 3) + 8 * (r >> 2) + 4 * lh];
  }
  // partial blocks, [kpart][row][pixel] with the row pitch padded
  const int TS = BN + 4;
  float* mine = lds + kpart * BM * TS + wn * 32 + li;
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int r = 0; r < 16; ++r) mine[(a * 32 + (r & 3) + 8 * (r >> 2) + 4 * lh) * TS] = acc[a][r];
  __syncthreads();
  const int ohw = g.OHW;
  const bool raw = g.splits > 1, vec = (ohw & 3) == 0;
  float* part = g.d + (int64_t)bz * g.m * g.npix;
  for (int q = tid; q < BM * (8 * g.wn); q += blockDim.x) {
    const int row = q / (8 * g.wn), lc = (q - row * (8 * g.wn)) * 4, i = i0 + row, j = j0 + lc;
    if (i >= g.m || j >= g.npix) continue;
    v4f v = *reinterpret_cast<const v4f*>(&lds[row * TS + lc]);
    for (int w = 1; w < g.kparts; ++w) v += *reinterpret_cast<const v4f*>(&lds[(w * BM + row) * TS + lc]);
    if (raw) {
      float* dst = part + (int64_t)i * g.npix + j;
      if (vec) {
        *reinterpret_cast<v4f*>(dst) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (j + e < g.npix) dst[e] = v[e];
      }
      continue;
    }
    const float bi = g.bias[i];
    const int img = fdiv(j, g.ohw_div), o = (img * g.m + i) * ohw + (j - img * ohw);
    if (vec) {
      v += bi;
      if (g.residual) v += *reinterpret_cast<const v4f*>(g.residual + o);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = split_act(v[e], g.act);
      *reinterpret_cast<v4f*>(g.d + o) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int je = j + e, ie = fdiv(je, g.ohw_div), oe = (ie * g.m + i) * ohw + (je - ie * ohw);
        if (je >= g.npix) break;
        float t = v[e] + bi;
        if (g.residual) t += g.residual[oe];
        g.d[oe] = split_act(t, g.act);
      }
    }
  }
}

struct SplitCfg {
  int tm, wn, kparts, splits;
};

// Work split, by the workgroups it gives.  64-row waves (each input value
// multiplied twice as often) where 64-row blocks still give three workgroups
// per four CUs, with four pixel blocks a workgroup, then two with the
// reduction in two parts, then one in four (8 x 64 -> 128, 3x3 stride 2 at
// 56x56: 25 / 15.5 / 16 us; 32 x 384 -> 64 at 14x14: 17 / 10.7 / 7.5); else
// 32-row waves, four or (few workgroups, 32+ steps) eight parts, and long
// reductions in parts over the launch up to two workgroups per CU (512 ->
// 512, 3x3 stride 2, one 14x14 image, 288 steps: 28 us in one launch part,
// 15 in four; 128 -> 256 at 28x28, 72 steps: 10.7 and 9.2; 1x1, one 7x7
// image, 960 -> 160, 60 steps, 10 workgroups, weights not in L2: 9.1 and 7.3).
SplitCfg split_config(const nhip_conv_plan* p, int64_t npix) {
  const int64_t cus = cu_count();
  auto wgs = [&](int tm, int wn) { return ceil_div(npix, 32 * wn) * ceil_div(p->g.k, 32 * tm); };
  const int nk = p->split_nk;
  SplitCfg c{1, 1, 4, 1};
  if (p->g.k > 32 && 2 * wgs(2, 4) >= 3 * cus) {
    c = {2, 4, 1, 1};
  } else if (p->g.k > 32 && 4 * wgs(2, 2) >= 3 * cus) {
    c = {2, 2, 2, 1};
  } else if (p->g.k > 32 && 4 * wgs(2, 1) >= 3 * cus) {
    c = {2, 1, 4, 1};
  } else if (2 * wgs(1, 4) >= 3 * cus) {
    c = {1, 4, 1, 1};
  } else {
    if (nk >= 32 && nk < 64 && 8 * wgs(1, 1) <= cus)
      c.splits = 4;
    else if (nk >= 64)
      while (c.splits < 8 && nk / (8 * c.splits) >= 4 && wgs(1, 1) * c.splits <= 2 * cus) c.splits *= 2;
    if (c.splits == 1 && nk >= 32 && 4 * wgs(1, 1) <= cus) c.kparts = 8;
  }
  // tuning override "row blocks, pixel blocks, waves per pixel block, launch parts"
  if (const char* env = setting("NHIP_SPLIT_CFG")) {
    int tm = 0, wn = 0, kp = 0, z = 0;
    if (std::sscanf(env, "%d,%d,%d,%d", &tm, &wn, &kp, &z) == 4 && (tm == 1 || tm == 2) && wn >= 1 && kp >= 1 &&
        wn * kp <= (tm == 1 ? 16 : 8) && z >= 1 && z <= 16)
      c = {tm, wn, kp, z};
  }
  return c;
}

template <int TM>
int launch_tm(const nhip_conv_plan* p, const SplitArgs& g, hipStream_t s) {
  const dim3 grid((unsigned)ceil_div(g.npix, 32 * g.wn), (unsigned)ceil_div(g.m, 32 * TM), (unsigned)g.splits);
  const dim3 block(64 * g.wn * g.kparts);
  const int lds = g.kparts * 32 * TM * (32 * g.wn + 4) * 4;
#define NHIP_SPLIT(ORDER_)                                                                                   \
  {                                                                                                          \
    const auto kernel = conv_split_kernel<TM, ORDER_>;                                                       \
    if (lds > 64 * 1024) NHIP_TRY(ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), 160 * 1024));    \
    NHIP_LAUNCH("conv_split_f32", kernel, grid, block, (unsigned)lds, s, g);                                 \
  }
  if (!p->split_taps)
    NHIP_SPLIT(kTable)
  else if (p->g.c % 16 == 0)
    NHIP_SPLIT(kTaps)
  else
    NHIP_SPLIT(kTapsRagged)
#undef NHIP_SPLIT
  return check_launch("conv_split_f32");
}

// Eight values' pieces, each piece's eight 16-bit words at out[piece * stride]
// (fixed-length loops without branches: the compiler vectorizes them).  Their sum
// is the value, whatever it is: with LARGE, the first piece of an infinity or NaN
// is that and the others 0, and a number never rounds up to infinity; without,
// for numbers below kLarge.
constexpr uint32_t kLarge = 0x7f7f8000u;  // (bits; it and what follows would round to bf16's infinity)

template <bool LARGE>
void split_octet(const float (&x)[8], uint16_t* out, size_t stride) {
  float v[8];
  for (int e = 0; e < 8; ++e) v[e] = x[e];
  for (int q = 0; q < kPieces; ++q) {
    uint32_t u[8], rest[8];
    std::memcpy(u, v, sizeof(u));
    for (int e = 0; e < 8; ++e) {
      if (LARGE) {
        const uint32_t mag = u[e] & 0x7fffffffu;
        const uint32_t special = mag >= 0x7f800000u ? 0xffffffffu : 0u, nan = mag > 0x7f800000u ? 0x400000u : 0u;
        const uint32_t up = mag < kLarge ? 0x7fffu + ((u[e] >> 16) & 1) : 0u;  // to nearest even
        u[e] = (((u[e] + up) & ~special) | ((u[e] | nan) & special)) & 0xffff0000u;
        rest[e] = ~special;
      } else {
        u[e] = (u[e] + 0x7fffu + ((u[e] >> 16) & 1)) & 0xffff0000u;
      }
    }
    float h[8];
    std::memcpy(h, u, sizeof(h));
    for (int e = 0; e < 8; ++e) v[e] -= h[e];
    if (LARGE) {
      uint32_t w[8];
      std::memcpy(w, v, sizeof(w));
      for (int e = 0; e < 8; ++e) rest[e] &= w[e];
      std::memcpy(v, rest, sizeof(v));
    }
    uint16_t words[8];
    for (int e = 0; e < 8; ++e) words[e] = (uint16_t)(u[e] >> 16);
    std::memcpy(out + q * stride, words, sizeof(words));
  }
}

// Split-K reduction: part [S][m][npix] -> out NCHW = act(sum_s part + bias
// (+ residual)), the parts in order, eight loads in flight.
__global__ void conv_splitk_reduce(const float* __restrict__ part, int splits, int m, int npix, FastDiv npix_div,
                                   FastDiv ohw_div, int ohw, const float* __restrict__ bias,
                                   const float* __restrict__ residual, float* __restrict__ out, int act) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;  // < 2^31 (the parts' size is checked on the host)
  const int stride = m * npix;
  if (idx >= stride) return;
  const int i = fdiv(idx, npix_div), j = idx - i * npix;
  const int img = fdiv(j, ohw_div), o = (img * m + i) * ohw + (j - img * ohw);
  const float b = bias[i], r = residual ? residual[o] : 0.f;
  float acc = 0.f;
  for (int s = 0; s < splits; s += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = s + u < splits ? part[(int64_t)(s + u) * stride + idx] : 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = s + u == 0 ? v[0] : s + u < splits ? acc + v[u] : acc;
  }
  float v = acc + b;
  if (residual) v += r;
  out[o] = split_act(v, act);
}

}  // namespace

// One buffer: the weights [K][C][kh][kw] split into bf16 pieces, in fragment
// order, and the table of taps where the reduction runs in (c, kh, kw) order.
// Nothing that the kernel reads belongs to another part of the plan: a Winograd
// plan has no table of its own.
//
// Rows with weights too small for their pieces (below 2^-100, as the channels that
// training leaves dead have them) are stored times a power of two that lifts the
// smallest there, as far as the largest stays finite (it does where they span less
// than 2^226), and their sums are scaled back: [m_pad] factors after the table.
int conv_split_prepack(nhip_conv_plan* p, const float* weight) {
  const int K = p->g.k, C = p->g.c, khw = p->g.kh * p->g.kw;
  const int c8 = (int)round_up(C, 8);
  // taps order pads the channels to eight: not where that adds over a third
  p->split_taps = 3 * c8 <= 4 * C;
  p->split_c_pad = c8;
  p->split_nk = (int)ceil_div(p->split_taps ? (int64_t)c8 * khw : (int64_t)C * khw, 16);
  const int nk = p->split_nk;
  std::vector<float> unscale;
  bool large = false;
  for (int i = 0; i < K; ++i) {
    // (in integers, which the compiler vectorizes)
    int32_t least = 0x7fffffff, most = 0, top = 0;  // magnitudes of finite numbers but 0; of all
    const float* wi = weight + (size_t)i * C * khw;
    for (int j = 0; j < C * khw; ++j) {
      int32_t mag;
      std::memcpy(&mag, wi + j, 4);
      mag &= 0x7fffffff;
      const int32_t num = mag < 0x7f800000 ? mag : 0, low = num != 0 ? num : 0x7fffffff;
      least = low < least ? low : least;
      most = num > most ? num : most;
      top = mag > top ? mag : top;
    }
    large |= top >= (int32_t)kLarge;
    if (most == 0) continue;
    float lo, hi;
    std::memcpy(&lo, &least, 4);
    std::memcpy(&hi, &most, 4);
    const int up = std::min(-100 - std::ilogb(lo), 126 - std::ilogb(hi));
    if (up <= 0) continue;
    large = true;  // (scaled, the largest may come near the largest number)
    unscale.resize((size_t)p->m_pad, 1.f);
    unscale[i] = std::ldexp(1.f, -up);
  }
  const size_t frag = kFrag / 2, pieces = (size_t)(p->m_pad / 32) * nk * kPieces * frag;
  const size_t factors = pieces + (p->split_taps ? 0 : (size_t)2 * nk * 16);  // 16-bit words ahead of them
  std::vector<uint16_t> out(factors + 2 * unscale.size(), 0);
  // 32 rows together, so that a fragment's lines are written once (1280 x 320: 2.6
  // ms with a row at a time and the general octets, 0.9 so)
  const int kend = p->split_taps ? c8 * khw : C * khw;
  for (int i0 = 0; i0 < K; i0 += 32)
    for (int k = 0; k < kend; k += 8) {
      uint16_t* at = out.data() + ((size_t)(i0 / 32) * nk + k / 16) * kPieces * frag + (size_t)(k % 16 / 8) * 256;
      const int r = p->split_taps ? k / c8 : 0, c0 = p->split_taps ? k - r * c8 : k;
      const int left = (p->split_taps ? C : kend) - c0, step = p->split_taps ? khw : 1;
      for (int i = i0; i < std::min(K, i0 + 32); ++i, at += 8) {
        const float* from = weight + (size_t)i * C * khw + (size_t)c0 * step + r;
        float x[8];
        if (left >= 8 && step == 1)
          for (int e = 0; e < 8; ++e) x[e] = from[e];
        else
          for (int e = 0; e < 8; ++e) x[e] = e < left ? from[(size_t)e * step] : 0.f;
        if (!unscale.empty() && unscale[i] != 1.f)
          for (int e = 0; e < 8; ++e) x[e] *= 1.f / unscale[i];
        if (large)
          split_octet<true>(x, at, frag);
        else
          split_octet<false>(x, at, frag);
      }
    }
  if (!p->split_taps) {
    std::vector<int32_t> kt((size_t)nk * 16, 0x7fff << 16);
    for (int k = 0; k < C * khw; ++k) {
      const int c = k / khw, r = k % khw;
      kt[k] = (c << 16) | ((r / p->g.kw * p->g.dh) << 8) | (r % p->g.kw * p->g.dw);
    }
    std::memcpy(out.data() + pieces, kt.data(), kt.size() * 4);
  }
  if (!unscale.empty()) std::memcpy(out.data() + factors, unscale.data(), unscale.size() * 4);
  NHIP_TRY(check_hip(hipMalloc(&p->weight_split, out.size() * 2), "hipMalloc(split conv weight)"));
  NHIP_TRY(check_hip(hipMemcpy(p->weight_split, out.data(), out.size() * 2, hipMemcpyHostToDevice),
                     "hipMemcpy(split conv weight)"));
  p->split_unscale = unscale.empty() ? nullptr : reinterpret_cast<float*>(p->weight_split + factors);
  p->split_ktab = p->split_taps ? nullptr : reinterpret_cast<int32_t*>(p->weight_split + pieces);
  return ok();
}

uint64_t conv_split_workspace(const nhip_conv_plan* p, int n, int oh, int ow) {
  const int64_t npix = (int64_t)n * oh * ow;
  const SplitCfg c = split_config(p, npix);
  return c.splits > 1 ? (uint64_t)c.splits * p->g.k * npix * sizeof(float) : 0;
}

int launch_conv_split(const nhip_conv_plan* p, const float* in, const float* residual, float* out, int n, int h,
                      int w, int oh, int ow, void* ws, uint64_t ws_bytes, hipStream_t s) {
  SplitArgs g{};
  g.a = p->weight_split;
  g.nk = p->split_nk;
  g.m = p->g.k;
  g.x = in;
  g.x_bytes = (uint32_t)((size_t)n * p->g.c * h * w * sizeof(float));
  g.npix = n * oh * ow;
  g.C = p->g.c;
  g.c_pad = p->split_c_pad;
  g.khw = p->g.kh * p->g.kw;
  g.KW = p->g.kw;
  g.H = h;
  g.W = w;
  g.OW = ow;
  g.OHW = oh * ow;
  g.sh = p->g.sh;
  g.sw = p->g.sw;
  g.pt = p->g.pt;
  g.pl = p->g.pl;
  g.dh = p->g.dh;
  g.dw = p->g.dw;
  g.ktab = p->split_ktab;
  g.kred = p->g.c * g.khw;
  g.unscale = p->split_unscale;
  g.ohw_div = fast_div((uint32_t)g.OHW);
  g.ow_div = fast_div((uint32_t)g.OW);
  g.oct_div = fast_div((uint32_t)std::max(1, p->g.c % 16 == 0 ? g.c_pad / 16 : g.c_pad / 8));
  g.kw_div = fast_div((uint32_t)g.KW);
  g.d = out;
  g.bias = p->bias;
  g.residual = residual;
  g.act = p->g.act;
  SplitCfg c = split_config(p, g.npix);
  // A workspace of another batch may be smaller than this one's parts (a small
  // launch has parts where a large one has none): one part then, which needs none.
  if (c.splits > 1 && (ws == nullptr || ws_bytes < conv_split_workspace(p, n, oh, ow))) c.splits = 1;
  g.splits = c.splits;
  g.wn = c.wn;
  g.kparts = c.kparts;
  if (c.splits > 1) g.d = static_cast<float*>(ws);
  if (c.tm == 2)
    NHIP_TRY(launch_tm<2>(p, g, s));
  else
    NHIP_TRY(launch_tm<1>(p, g, s));
  if (c.splits == 1) return ok();
  const int64_t total = (int64_t)p->g.k * g.npix;
  NHIP_LAUNCH("conv_splitk_reduce", conv_splitk_reduce, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, s,
              static_cast<const float*>(ws), c.splits, p->g.k, g.npix, fast_div((uint32_t)g.npix), g.ohw_div, g.OHW,
              p->bias, residual, out, p->g.act);
  return check_launch("conv_splitk_reduce");
}

}  // namespace nhip
