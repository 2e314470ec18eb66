// int8 Convolution with requantize (reference ConvertConvolution int8 path,
// NCNNToTosa.cpp:1136-1315) in one launch: the workgroup's input window goes
// from the NCHW tensor (int8, or fp32 quantized on the way) into LDS as NHWC,
// and the weights stream from their fragment-order copy into registers.  Same
// arithmetic as conv_int8.hip's kernels, bit for bit: exact integer sums in any
// order, then the separately rounded fp32 steps of the epilogue.
//
// What bounds it: at the sizes quantized networks have, the launches and the
// chain of latencies, not the 5 POP/s of the matrix instructions.  The other
// kernels read an NHWC copy of the whole input that a pass of its own writes
// to memory first (5 us at 32 x 128 x 28 x 28, 3 at the least), and stream the
// weights through LDS with a barrier per stage.  Here
//   - a workgroup owns R output rows, whole or CW columns of them, of one image
//     (at most 128 pixels; a stride-1 1x1 layer's image is one row) and MBW
//     blocks of 32 output channels (of 1x1 planes, an InnerProduct's rows: the
//     images are the pixels of one row, channels contiguous on both sides; 335 x
//     2081 -> 1783 84.6 us with an image per workgroup, 18.9 us so); an item of its fill is four channels by four pixels: four
//     loads, a 4 x 4 byte transpose (or sixteen quantizations), four LDS words;
//   - a wave holds one channel block and one of KP parts of the reduction, its
//     weights four steps ahead in registers (the first requested before the
//     fill), the window's pixels from LDS: no barrier in the loop;
//   - one part: the results leave from the registers, for int8 output with
//     the pixels as the matrix instruction's rows, so that a lane holds sixteen
//     consecutive pixels of one channel (16-byte stores), for fp32 output with
//     the channels as rows (32 lanes store 128 consecutive bytes).  More parts
//     meet in LDS (integer adds, any order) and leave as runs of four pixels.
// Against the kernels that read an NHWC copy (a second launch, and one that kept
// window and streamed weights in LDS for the middle sizes): 32 x 128 x 28 x 28 ->
// 256 at 1x1, int8, 14.2 -> 9.1 us; 2 to 20 images of 20 to 120 channels at 7 x 7
// to 43 x 43 11.7 to 14.8 -> 5.5 to 7.7 us; 7 x 235 x 21 x 21 -> 121 at 5x5 stride 2
// 46.4 -> 12.1 us; 32 x 256 x 14 x 14 3x3 25.6 -> 12.9 us; 16 x
// 48 x 95 x 95 -> 360 at 1x1 to fp32 261 -> 92 us; to int8 69 -> 39 us, where the
// eleven vector instructions of a requantized result take about half the time.
#include <algorithm>
#include <cstdio>

#include "nhip_internal.h"

namespace nhip {
namespace {

constexpr int kMaxLds = 64 * 1024;

struct WinArgs {
  const void* x;
  const int8_t* w;     // fragment order [m_pad/32][steps][64 lanes][16]
  const float* recip;  // [m_pad]
  const float* bias;   // [m_pad]
  void* out;
  float is, os;
  int relu, qlo;
  int C, H, W, M, OH, OW, c_pad, KW, sh, sw, pt, pl, dh, dw;
  int steps, kred;     // steps of 32 bytes; reduction bytes (kh, kw, c_pad)
  int mblocks;         // 32-channel blocks of the layer
  int mbw, kp;         // channel blocks and reduction parts of a workgroup
  int R, CW;           // output rows and columns of a workgroup (CW a multiple of 16 where CW < OW, but any for vecs)
  int rgs, segs;       // row groups of an image, column segments of a row
  int FH, FW, FS;      // window rows, columns, bytes per pixel
  int rstep, wsh;      // input rows per window row; window rows per output row
  int xg;              // groups of four columns in a window row's fill
  int tab;             // LDS byte offset of the chunk offsets
  int vecs;            // 1x1 planes (an InnerProduct): the images are the pixels of one row, channels contiguous
  FastDiv xg_div, c4_div, rg_div, seg_div;
};

__device__ __forceinline__ float rescale(int sum, float recip, float bias) {
#pragma clang fp contract(off)
  const float f = (float)sum * recip;
  return f + bias;
}

template <int TN, bool IN8, bool OUT8>
__global__ __launch_bounds__(512, 4) void conv_int8_win_kernel(WinArgs g) {
  extern __shared__ __attribute__((aligned(16))) int8_t dsm[];
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, li = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kpart = wave / g.mbw, mb = blockIdx.y * g.mbw + (wave - kpart * g.mbw);
  const int rowb = fdiv(blockIdx.x, g.seg_div), ox0 = (blockIdx.x - rowb * g.segs) * g.CW;
  const int img = fdiv(rowb, g.rg_div), oy0 = (rowb - img * g.rgs) * g.R;
  const int ncol = min(g.CW, g.OW - ox0), nrow = min(g.R, g.OH - oy0);
  const bool live = mb < g.mblocks;
  const int per = (g.steps + g.kp - 1) / g.kp;
  const int s0 = min(g.steps, kpart * per), s1 = live ? min(g.steps, s0 + per) : s0;

  // weights: four steps ahead (past the end: the last step again, unused)
  constexpr int kAhead = 4;
  const int8_t* wp = g.w + (int64_t)min(mb, g.mblocks - 1) * g.steps * 1024 + lane * 16;
  v4i wr[kAhead];
#pragma unroll
  for (int d = 0; d < kAhead; ++d) wr[d] = *reinterpret_cast<const v4i*>(wp + (int64_t)min(s0 + d, g.steps - 1) * 1024);

  // ---- fill
  int* koff = reinterpret_cast<int*>(dsm + g.tab);
  const int iy0 = oy0 * g.sh - g.pt, ix0 = ox0 * g.sw - g.pl;
  {
    const int all16 = (g.FH * g.FW * g.FS) >> 4;  // FS is a multiple of 16
    for (int i = tid; i < all16; i += nt) reinterpret_cast<v4i*>(dsm)[i] = v4i{0, 0, 0, 0};
    // byte offset in the window of each 16-byte chunk of the reduction
    // (kh, kw, c); past its end (the weights are zero there) any window byte
    for (int q = tid; q < 2 * g.steps; q += nt) {
      const int k = q * 16, r = k / g.c_pad, c0 = k - r * g.c_pad, kh = r / g.KW, kw = r - kh * g.KW;
      koff[q] = k < g.kred ? (kh * g.dh * g.FW + kw * g.dw) * g.FS + c0 : 0;
    }
  }
  __syncthreads();
  if (g.vecs) {
    // items: sixteen channels of one pixel
    const int groups = g.c_pad >> 4, items = ncol * groups;
    for (int i = tid; i < items; i += nt) {
      const int px = i / groups, c0 = 16 * (i - px * groups);
      const int64_t e = (int64_t)(ox0 + px) * g.C + c0;
      v4i v = {0, 0, 0, 0};
      if constexpr (IN8) {
        const int8_t* src = static_cast<const int8_t*>(g.x) + e;
        if (c0 + 16 <= g.C) {
          __builtin_memcpy(&v, src, 16);
        } else {
#pragma unroll
          for (int u = 0; u < 16; ++u)
            if (c0 + u < g.C) v[u >> 2] |= (int)((uint32_t)(uint8_t)src[u] << (8 * (u & 3)));
        }
      } else {
        const float* src = static_cast<const float*>(g.x) + e;
        v4f f[4];
        if (c0 + 16 <= g.C) {
          __builtin_memcpy(f, src, 64);
        } else {
#pragma unroll
          for (int u = 0; u < 16; ++u) f[u >> 2][u & 3] = c0 + u < g.C ? src[u] : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
          v[q] = (int)pack_i8x4(quantize_q(f[q][0], g.is), quantize_q(f[q][1], g.is), quantize_q(f[q][2], g.is),
                                quantize_q(f[q][3], g.is));
      }
      *reinterpret_cast<v4i*>(dsm + px * g.FS + c0) = v;
    }
  } else {
    // items: window row, four channels, four pixels (x fastest).  Groups past
    // a row's end start at W - 4 and the last channel group repeats the last
    // channel (the weights of the padding channels are zero).
    const int c4n = (g.C + 3) >> 2, items = g.FH * c4n * g.xg, xs = max(0, ix0);
    const int64_t plane = (int64_t)g.H * g.W;
    constexpr int kBatch = IN8 ? 4 : 2;
    for (int i0 = tid; i0 < items; i0 += kBatch * nt) {
      int d8[kBatch][4];
      v4f df[kBatch][4];
      int dst[kBatch], col[kBatch];
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const int i = i0 + b * nt;
        dst[b] = -1;
        if (i >= items) continue;
        const int rest = fdiv(i, g.xg_div), x = max(0, min(xs + 4 * (i - rest * g.xg), g.W - 4));
        const int fy = fdiv(rest, g.c4_div), c4 = rest - fy * c4n, iy = iy0 + fy * g.rstep;
        if (iy < 0 || iy >= g.H) continue;
        const int64_t at = ((int64_t)img * g.C * g.H + iy) * g.W + x;
        col[b] = x - ix0;
        dst[b] = fy * g.FW * g.FS + 4 * c4;
        if (g.W >= 4) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int64_t e = at + min(4 * c4 + j, g.C - 1) * plane;
            if constexpr (IN8)
              __builtin_memcpy(&d8[b][j], static_cast<const int8_t*>(g.x) + e, 4);
            else
              __builtin_memcpy(&df[b][j], static_cast<const float*>(g.x) + e, 16);
          }
        } else {  // (rows shorter than a group: the last pixel again)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int64_t e = at + min(4 * c4 + j, g.C - 1) * plane;
            if constexpr (IN8) d8[b][j] = 0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const int64_t eu = e + min(u, g.W - 1);
              if constexpr (IN8)
                d8[b][j] |= (int)((uint32_t)(uint8_t)static_cast<const int8_t*>(g.x)[eu] << (8 * u));
              else
                df[b][j][u] = static_cast<const float*>(g.x)[eu];
            }
          }
        }
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        if (dst[b] < 0) continue;
        uint32_t px[4];
        if constexpr (IN8) {
          const uint32_t a0 = (uint32_t)d8[b][0], a1 = (uint32_t)d8[b][1], a2 = (uint32_t)d8[b][2], a3 = (uint32_t)d8[b][3];
          const uint32_t l01 = __builtin_amdgcn_perm(a1, a0, 0x05010400u), h01 = __builtin_amdgcn_perm(a1, a0, 0x07030602u);
          const uint32_t l23 = __builtin_amdgcn_perm(a3, a2, 0x05010400u), h23 = __builtin_amdgcn_perm(a3, a2, 0x07030602u);
          px[0] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
          px[1] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
          px[2] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
          px[3] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            px[e] = pack_i8x4(quantize_q(df[b][0][e], g.is), quantize_q(df[b][1][e], g.is), quantize_q(df[b][2][e], g.is),
                              quantize_q(df[b][3][e], g.is));
        }
        // (columns outside the window are read by no output; those past the
        // row's end stay zero)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if ((unsigned)(col[b] + e) < (unsigned)g.FW && col[b] + e < g.W - ix0)
            *reinterpret_cast<uint32_t*>(dsm + dst[b] + (col[b] + e) * g.FS) = px[e];
      }
    }
  }
  // int8 output: operand row li is the pixel whose sums lane half (li >> 2 & 1)
  // gets in register (li & 3) + 4 * (li >> 3)
  const int pli = OUT8 ? 16 * (li >> 2 & 1) + (li & 3) + 4 * (li >> 3) : li;
  int fbase[TN];
#pragma unroll
  for (int b = 0; b < TN; ++b) {
    const int pc = b * 32 + pli, pr = pc / g.CW, py = min(pr, nrow - 1), px = min(pc - pr * g.CW, ncol - 1);
    fbase[b] = (py * g.wsh * g.FW + px * g.sw) * g.FS;
  }
  __syncthreads();

  // ---- D[channel][pixel], or [pixel][channel] for int8 output
  v16i acc[TN];
#pragma unroll
  for (int b = 0; b < TN; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = 0;
  int ko[kAhead];
#pragma unroll
  for (int d = 0; d < kAhead; ++d) ko[d] = koff[2 * min(s0 + d, g.steps - 1) + lh];
  for (int s = s0; s < s1; s += kAhead) {
#pragma unroll
    for (int d = 0; d < kAhead; ++d) {
      const v4i a = wr[d];
      const int k = ko[d], ahead = min(s + d + kAhead, g.steps - 1);
      wr[d] = *reinterpret_cast<const v4i*>(wp + (int64_t)ahead * 1024);
      ko[d] = koff[2 * ahead + lh];
      if (s + d < s1) {
        v4i xv[TN];
#pragma unroll
        for (int b = 0; b < TN; ++b) xv[b] = *reinterpret_cast<const v4i*>(dsm + fbase[b] + k);
#pragma unroll
        for (int b = 0; b < TN; ++b)
          acc[b] = OUT8 ? __builtin_amdgcn_mfma_i32_32x32x32_i8(xv[b], a, acc[b], 0, 0, 0)
                        : __builtin_amdgcn_mfma_i32_32x32x32_i8(a, xv[b], acc[b], 0, 0, 0);
      }
    }
  }
  const int64_t plane_out = (int64_t)g.OH * g.OW, out0 = (int64_t)img * g.M * plane_out + (int64_t)oy0 * g.OW + ox0;
  // where a run of at most 16 pixels from p on goes, and how many of the
  // workgroup's pixels are left there (whole rows are one run; a run of a
  // column segment ends with its row)
  auto place = [&](int p, int64_t& at) {
    if (g.segs == 1) {
      at = p;
      return nrow * g.CW - p;
    }
    const int py = p / g.CW, px = p - py * g.CW;
    at = (int64_t)py * g.OW + px;
    return py < nrow ? ncol - px : 0;
  };
  if (g.kp == 1 && !g.vecs) {
    if constexpr (OUT8) {
      __syncthreads();  // (every wave is past its reads of the window)
      if (!live) return;
      // through the wave's own LDS rows, so that a store instruction covers
      // TN * 32 consecutive bytes of a channel
      constexpr int RS = TN * 32 + 16, kRunsPer = TN * 2;
      int8_t* stage = dsm + wave * 32 * RS;
      {
        const float rc = g.recip[mb * 32 + li], bs = g.bias[mb * 32 + li];
#pragma unroll
        for (int b = 0; b < TN; ++b) {
          v4i y;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            int f[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = quantize_q(rescale(acc[b][4 * j + e], rc, bs), g.os, g.qlo);
            y[j] = (int)pack_i8x4(f[0], f[1], f[2], f[3]);
          }
          *reinterpret_cast<v4i*>(stage + li * RS + b * 32 + 16 * lh) = y;
        }
      }
      // the rows read back are other lanes' of this wave
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int run = lane % kRunsPer, row0 = lane / kRunsPer;
      int64_t p;
      const int left = place(run * 16, p);
      int8_t* dst = static_cast<int8_t*>(g.out) + out0 + p;
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        const int row = row0 + i * (64 / kRunsPer), ch = mb * 32 + row;
        if (ch >= g.M) continue;
        const v4i y = *reinterpret_cast<const v4i*>(stage + row * RS + run * 16);
        if (left >= 16) {
          __builtin_memcpy(dst + ch * plane_out, &y, 16);
        } else {
#pragma unroll
          for (int j = 0; j < 16; ++j)
            if (j < left) dst[ch * plane_out + j] = (int8_t)((uint32_t)y[j >> 2] >> (8 * (j & 3)));
        }
      }
    } else {
      if (!live) return;
      int64_t at[TN];
      bool ok[TN];
#pragma unroll
      for (int b = 0; b < TN; ++b) ok[b] = place(b * 32 + li, at[b]) > 0;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int ch = mb * 32 + (j & 3) + 8 * (j >> 2) + 4 * lh;
        if (ch >= g.M) continue;
        const float rc = g.recip[ch], bs = g.bias[ch];
        float* row = static_cast<float*>(g.out) + out0 + ch * plane_out;
#pragma unroll
        for (int b = 0; b < TN; ++b) {
          const float f = rescale(acc[b][j], rc, bs);
          if (ok[b]) row[at[b]] = g.relu && f < 0.0f ? 0.0f : f;
        }
      }
    }
    return;
  }
  // ---- sums [channel][pixel] in LDS over the window, one part after another
  constexpr int TS = TN * 32 + 4;
  int* sums = reinterpret_cast<int*>(dsm);
  int* mine = sums + (wave - kpart * g.mbw) * 32 * TS;
  for (int k = 0; k < g.kp; ++k) {
    __syncthreads();
    if (k != kpart) continue;
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      if constexpr (OUT8) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v4i* at = reinterpret_cast<v4i*>(mine + li * TS + b * 32 + 16 * lh + 4 * j);
          v4i v = {acc[b][4 * j], acc[b][4 * j + 1], acc[b][4 * j + 2], acc[b][4 * j + 3]};
          if (k != 0) v += *at;
          *at = v;
        }
      } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          int* at = mine + ((j & 3) + 8 * (j >> 2) + 4 * lh) * TS + b * 32 + li;
          *at = k == 0 ? acc[b][j] : *at + acc[b][j];
        }
      }
    }
  }
  __syncthreads();
  const int rows = g.mbw * 32;
  if (g.vecs) {  // channels fastest, one result per thread
    for (int q = tid; q < rows * ncol; q += nt) {
      const int px = q / rows, row = q - px * rows, ch = blockIdx.y * rows + row;
      if (ch >= g.M) continue;
      const float f = rescale(sums[row * TS + px], g.recip[ch], g.bias[ch]);
      const int64_t o = (int64_t)(ox0 + px) * g.M + ch;
      if constexpr (OUT8)
        static_cast<int8_t*>(g.out)[o] = (int8_t)quantize_q(f, g.os, g.qlo);
      else
        static_cast<float*>(g.out)[o] = g.relu && f < 0.0f ? 0.0f : f;
    }
    return;
  }
  // ---- epilogue: four pixels of a channel per thread, TN * 8 threads per channel
  for (int q = tid; q < rows * TN * 8; q += nt) {
    const int row = q / (TN * 8), p = (q - row * TN * 8) * 4, ch = blockIdx.y * rows + row;
    int64_t at;
    const int left = place(p, at);
    if (ch >= g.M || left <= 0) continue;
    const float rc = g.recip[ch], bs = g.bias[ch];
    const v4i v = *reinterpret_cast<const v4i*>(&sums[row * TS + p]);
    float f[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = rescale(v[e], rc, bs);
    const int64_t o = out0 + ch * plane_out + at;
    if constexpr (OUT8) {
      const uint32_t y = pack_i8x4(quantize_q(f[0], g.os, g.qlo), quantize_q(f[1], g.os, g.qlo),
                                   quantize_q(f[2], g.os, g.qlo), quantize_q(f[3], g.os, g.qlo));
      int8_t* dst = static_cast<int8_t*>(g.out) + o;
      if (left >= 4) {
        __builtin_memcpy(dst, &y, 4);
      } else {
        for (int e = 0; e < left; ++e) dst[e] = (int8_t)(y >> (8 * e));
      }
    } else {
      v4f y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = g.relu && f[e] < 0.0f ? 0.0f : f[e];
      float* dst = static_cast<float*>(g.out) + o;
      if (left >= 4) {
        __builtin_memcpy(dst, &y, 16);
      } else {
        for (int e = 0; e < left; ++e) dst[e] = y[e];
      }
    }
  }
}

template <int TN>
int launch_tn(const WinArgs& a, dim3 grid, dim3 block, int lds, bool in8, bool out8, hipStream_t s) {
#define NHIP_WIN(IN8_, OUT8_)                                                                              \
  {                                                                                                        \
    const auto kernel = conv_int8_win_kernel<TN, IN8_, OUT8_>;                                             \
    NHIP_LAUNCH("conv_int8_win", kernel, grid, block, (unsigned)lds, s, a);                                \
  }
  if (in8 && out8) NHIP_WIN(true, true)
  else if (in8) NHIP_WIN(true, false)
  else if (out8) NHIP_WIN(false, true)
  else NHIP_WIN(false, false)
#undef NHIP_WIN
  return check_launch("conv_int8_win");
}

struct WinCfg {
  int n, h, w, oh, ow;  // the images as the kernel sees them
  bool vecs;            // n images of one pixel as one row
  int R, CW, mbw, kp, tn, FH, FW, FS, rstep, wsh, tab, lds;  // R 0: no window fits
};

WinCfg win_config(const nhip_conv_plan* p, int in_is_i8, int n, int h, int w, int oh, int ow) {
  const ConvGeom& g = p->g;
  WinCfg c{n, h, w, oh, ow};
  // a 1x1 layer with stride 1 and no padding: one row of h * w pixels
  if (g.kh == 1 && g.kw == 1 && g.sh == 1 && g.sw == 1 && oh == h && ow == w && g.pt == 0 && g.pl == 0 &&
      (int64_t)h * w < (1 << 30)) {
    c.vecs = h * w == 1;
    c.w = c.ow = c.vecs ? n : h * w;
    c.h = c.oh = 1;
    if (c.vecs) c.n = 1;
  }
  const int mblocks = (int)ceil_div(g.k, 32), steps = p->kred_pad / 32;
  // an odd number of 16-byte chunks, so that sixteen pixels' reads fall into
  // different banks (2 x 109 -> 368, 7x7 stride 2 at 67x67: 52.7 us with 128 bytes per
  // pixel, 21.8 with 112)
  c.FS = p->c_pad / 16 % 2 ? p->c_pad : p->c_pad + 16;
  c.rstep = g.kh == 1 ? g.sh : 1;  // a one-row kernel's window leaves the rows between out
  c.wsh = g.kh == 1 ? 1 : g.sh;
  auto fh = [&](int R) { return (R - 1) * c.wsh + (g.kh - 1) * g.dh + 1; };
  auto fw = [&](int CW) { return (CW - 1) * g.sw + (g.kw - 1) * g.dw + 1; };
  auto tn = [&](int R, int CW) {
    const int t = (int)ceil_div(R * CW, 32);
    return t > 2 ? 4 : t;
  };
  auto window = [&](int R, int CW) {
    return (int)std::min<int64_t>(round_up((int64_t)fh(R) * fw(CW) * c.FS, 16), 1 << 24);
  };
  auto lds_of = [&](int R, int CW, int mbw, int kp) {
    const int t = tn(R, CW) * 32;
    return std::max(window(R, CW) + 8 * steps, mbw * 32 * (kp > 1 || c.vecs ? (t + 4) * 4 : t + 16));
  };
  // Tile, channel blocks and parts with the least estimated clocks on a CU: the
  // larger of what its workgroups keep busy together (fill items, matrix
  // instructions or the weights' way from L2, epilogue, the parts' exchange) and
  // the chain of latencies of those that follow one another, and half of the
  // smaller.  The constants are fitted to the times of 4500 launches over 60
  // layers (1 to 64 images, 3 to 504 channels, 7 x 7 to 224 x 224); the choice
  // was 4% from the best of a layer's launches on average, 41% at the worst
  // (16 x 64 x 111 x 113 fp32, 66 against 47 us; 87 us with the most whole rows
  // per workgroup, 95 us from an NHWC copy).
  int R = 0, CW = 0, mbw = 0, kp = 0;
  float best = 0.0f;
  const int cus = cu_count();
  auto consider = [&](int r, int cw) {
    const int win = window(r, cw);
    if (r < 1 || win + 8 * steps > kMaxLds) return;
    const int t = tn(r, cw), tiles = c.n * (int)ceil_div(c.oh, r) * (int)ceil_div(c.ow, cw);
    const int items = fh(r) * ((std::min(c.w, fw(cw)) + 3) / 4) * ((g.c + 3) / 4);
    int m = 1;
    for (bool last = false; !last; m = std::min(2 * m, mblocks)) {
      last = m == 8 || m == mblocks || 2 * m > 8;
      const int per_cu = (tiles * ((mblocks + m - 1) / m) + cus - 1) / cus;
      for (int k = 1; m * k <= 8 && (k == 1 || steps >= 2 * k); k *= 2) {
        const int lds = lds_of(r, cw, m, k);
        if (lds > kMaxLds) break;
        const int together = std::max(1, std::min(160 * 1024 / lds, 16 / (m * k)));
        const int rounds = (per_cu + together - 1) / together, nt = 64 * m * k * (in_is_i8 ? 4 : 2);
        const float busy = per_cu * (1000.0f + items * (in_is_i8 ? 1.7f : 5.2f) + m * steps * std::max(20.0f * t, 27.0f) +
                                     m * t * 1024 * (0.3f + (k > 1 ? 0.07f * k : 0.0f)));
        const float chain = rounds * (4100.0f + 2700.0f * ((items + nt - 1) / nt) +
                                      (float)steps / k * 157.0f * std::max(1.0f, 0.5f * t));
        float cost = std::max(busy, chain) + 0.5f * std::min(busy, chain);
        if (cw < c.ow && cw < 64 && !c.vecs) cost *= 1.05f;  // shorter runs to store
        if (R == 0 || cost < best) {
          best = cost;
          R = r;
          CW = cw;
          mbw = m;
          kp = k;
        }
      }
    }
  };
  if (c.ow <= 128)
    for (int r = std::min(128 / c.ow, c.oh);; r = (r + 1) / 2) {
      consider(r, c.ow);
      if (r <= 1) break;
    }
  constexpr int kSegments[] = {128, 112, 96, 64, 32};
  for (int cw : kSegments) {
    if (cw >= c.ow) continue;
    const int r = std::min(128 / cw, c.oh);
    consider(r, cw);
    if (r > 1) consider((r + 1) / 2, cw);
  }
  if (R == 0 && c.ow > 16) consider(1, 16);
  if (c.vecs)  // (any width: no runs along a row)
    for (int cw : {16, 8, 4})
      if (cw < c.ow) consider(1, cw);
  // Not where only sixteen columns fit and a CU gets many such workgroups: each
  // fills a window for half a matrix operand, and the gather kernel's 128 pixels,
  // with the pass that quantizes the image, take less.  load: workgroups and a
  // quarter of their channel blocks, per CU.  Window / gather: fp32 input, which is
  // quantized once per window, below 5 0.7 to 1.1, above 5.25 0.99 to 2.3 (29 x 635 -> 14,
  // 3x3 at 64x64: 396 / 183 us); int8 with two or more blocks per workgroup, below 10
  // 0.8 to 1.0, above 11 1.26 to 1.75 (29 x 629 -> 62 at 33x33: 98 / 56 us), with one 0.7 to
  // 1.1 up to 27.  1x1 windows have no rows to fill twice (15 x 594 -> 422 stride 2: 126
  // / 174).
  if (R > 0 && R * CW <= 16 && CW < c.ow && g.kh * g.kw > 1 && (!in_is_i8 || mbw > 1)) {
    const int64_t tiles = (int64_t)c.n * ceil_div(c.oh, R) * ceil_div(c.ow, CW);
    const int64_t load4 = tiles * (4 * ceil_div(mblocks, mbw) + mblocks);
    if (load4 >= (in_is_i8 ? 40LL : 21LL) * cus) R = 0;
  }
  if (R == 0) return c;
  if (const char* env = setting("NHIP_INT8_WIN_CFG")) {  // tuning: rows, columns, channel blocks, parts
    int r = 0, w4 = 0, m = 0, k = 0;
    if (std::sscanf(env, "%d,%d,%d,%d", &r, &w4, &m, &k) == 4 && r >= 1 && r <= c.oh && w4 >= 1 && w4 <= c.ow &&
        (w4 == c.ow || w4 % 16 == 0) && (int64_t)r * w4 <= 128 && m >= 1 && k >= 1 && m * k <= 8 &&
        lds_of(r, w4, m, k) <= kMaxLds) {
      R = r;
      CW = w4;
      mbw = m;
      kp = k;
    }
  }
  c.R = R;
  c.CW = CW;
  c.mbw = mbw;
  c.kp = kp;
  c.FH = fh(R);
  c.FW = fw(CW);
  c.tab = (int)window(R, CW);
  c.tn = tn(R, CW);
  c.lds = (int)lds_of(R, CW, mbw, kp);
  return c;
}

}  // namespace

int launch_conv_int8_win(const nhip_conv_plan* p, const void* in, int in_is_i8, void* out, int n, int h, int w, int oh,
                         int ow, hipStream_t s, bool* taken) {
  const WinCfg c = win_config(p, in_is_i8, n, h, w, oh, ow);
  *taken = c.R > 0;
  if (!*taken) return NHIP_STATUS_SUCCESS;
  WinArgs a{};
  a.x = in;
  a.w = p->weight_i8_frag;
  a.recip = p->recip;
  a.bias = p->bias;
  a.out = out;
  a.is = p->input_scale;
  a.os = p->output_scale;
  a.relu = p->g.act == NHIP_ACT_RELU;
  a.qlo = a.relu ? 0 : -127;
  a.C = p->g.c;
  a.H = c.h;
  a.W = c.w;
  a.M = p->g.k;
  a.OH = c.oh;
  a.OW = c.ow;
  a.c_pad = p->c_pad;
  a.KW = p->g.kw;
  a.sh = p->g.sh;
  a.sw = p->g.sw;
  a.pt = p->g.pt;
  a.pl = p->g.pl;
  a.dh = p->g.dh;
  a.dw = p->g.dw;
  a.steps = p->kred_pad / 32;
  a.kred = p->kred;
  a.mblocks = (int)ceil_div(p->g.k, 32);
  a.mbw = c.mbw;
  a.kp = c.kp;
  a.R = c.R;
  a.CW = c.CW;
  a.rgs = (int)ceil_div(c.oh, c.R);
  a.segs = (int)ceil_div(c.ow, c.CW);
  a.FH = c.FH;
  a.FW = c.FW;
  a.FS = c.FS;
  a.rstep = c.rstep;
  a.wsh = c.wsh;
  a.xg = (int)ceil_div(std::min(c.w, c.FW), 4);
  a.tab = c.tab;
  a.vecs = c.vecs;
  a.xg_div = fast_div((uint32_t)a.xg);
  a.c4_div = fast_div((uint32_t)ceil_div(a.C, 4));
  a.rg_div = fast_div((uint32_t)a.rgs);
  a.seg_div = fast_div((uint32_t)a.segs);
  const dim3 grid((unsigned)(c.n * a.rgs * a.segs), (unsigned)ceil_div(a.mblocks, c.mbw)), block(64 * c.mbw * c.kp);
  const bool in8 = in_is_i8 != 0, out8 = p->scale_term > 100;
  if (c.tn == 1) return launch_tn<1>(a, grid, block, c.lds, in8, out8, s);
  if (c.tn == 2) return launch_tn<2>(a, grid, block, c.lds, in8, out8, s);
  return launch_tn<4>(a, grid, block, c.lds, in8, out8, s);
}

}  // namespace nhip
