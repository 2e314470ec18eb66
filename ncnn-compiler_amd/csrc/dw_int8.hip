// int8 ConvolutionDepthWise (NCNNToTosa.cpp:3257-3376) for square 3x3 and 5x5
// kernels, stride 1 or 2, dilation 1, any padding up to 12 columns: the input
// is brought into LDS as it lies and every thread forms 4 x 4 outputs with
// v_dot4_i32_i8.  Same arithmetic as dwconv_int8_kernel, bit for bit: exact
// int32 window sums, then (float)acc * r[c], + bias[c], requantize when
// term > 100, relu last, every fp32 step rounded on its own.
//
// What bounds it: a byte per element of input and output is little traffic,
// so the per-element instruction count decides.  The general kernel stages
// one byte per load and forms one output per lane with a load and a multiply
// per tap (15 x 116 x 57 x 43 -> int8: 31 us for 8.5 MB).  Here
//   - whole planes, or a band of rows of one plane, are one contiguous run of
//     the NCHW input, copied with 16-byte loads and no re-pitching (fp32
//     input: four values per load, quantized on the way into one LDS word);
//   - a thread takes four neighbouring outputs of four rows.  It reads each
//     of its input rows once as aligned LDS words, shifts them to the
//     window's byte offset (v_alignbyte_b32), zeroes the bytes left and right
//     of the image with a mask formed once, and one dot4 adds up to four taps
//     of a row (the weights of a row padded with zeros to whole words), for
//     every output row that the input row belongs to;
//   - four int8 results leave as one word, four fp32 ones as 16 bytes.
// 15 x 116 x 57 x 43 int8 -> int8, 3x3 stride 1: 31 -> 8.3 us in the kernel
// trace; 32 x 96 x 74 x 74 fp32 -> int8, stride 2: 66 -> 9.3 us a call;
// 15 x 144 x 22 x 22 fp32 -> fp32, 5x5 stride 2: 17 -> 8.1 us a call.
// Launches that were bound by the call itself (8 us) stay there.
#include <algorithm>

#include "nhip_internal.h"

namespace nhip {
namespace {

constexpr int kThreads = 256;
constexpr int kRows = 4;      // output rows per thread
constexpr int kFront = 16;    // LDS bytes ahead of the staged run (window columns left of the image)
constexpr int kBack = 32;     // and past it
constexpr int kMaxStage = 48 * 1024;
constexpr int kMaxPadLeft = 12;

struct DwI8RunArgs {
  const void* x;
  void* y;
  const int* w;        // [C][K][words of a row]: the taps as bytes, zero padded
  const float* bias;   // [C]
  const float* recip;  // [C]
  float is, os;
  int relu, qlo;
  int C, H, W, OH, OW, pt, pl;
  int planes, ppb;     // planes per workgroup (1 when a plane is cut into bands)
  int bands, ob;       // bands per plane, output rows per band
  int quads, rgs;      // groups of 4 output columns, groups of kRows output rows (of a band)
  FastDiv item_div, quad_div, band_div;  // rgs * quads, quads, bands
};

// Bytes [lo, hi) of word d of a row segment kept, the others zeroed.
__device__ __forceinline__ uint32_t byte_mask(int d, int lo, int hi) {
  const int a = min(max(lo - 4 * d, 0), 4), b = min(max(hi - 4 * d, 0), 4);
  const uint64_t below_b = (uint64_t(1) << (8 * b)) - 1, below_a = (uint64_t(1) << (8 * a)) - 1;
  return (uint32_t)(below_b & ~below_a);
}

template <int K, int S, bool IN8, bool OUT8>
__global__ __launch_bounds__(kThreads) void dw_int8_runs_kernel(DwI8RunArgs g) {
  constexpr int KW = (K + 3) / 4;                    // words of one row of taps
  constexpr int ND = (3 * S + 4 * KW + 3) / 4;       // words of a row segment: 4 outputs' taps
  constexpr int IR = (kRows - 1) * S + K;            // input rows of a thread
  extern __shared__ __attribute__((aligned(16))) int8_t lds8[];
  const int tid = threadIdx.x;
  const int grp = fdiv(blockIdx.x, g.band_div), band = blockIdx.x - grp * g.bands;
  const int plane0 = grp * g.ppb, np = min(g.ppb, g.planes - plane0);
  const int oy0 = band * g.ob, rows = min(g.ob, g.OH - oy0);
  const int hw = g.H * g.W;
  // staged input rows [ylo, yhi) of each plane (the whole plane unless banded)
  int ylo = 0, yhi = g.H;
  if (g.bands > 1) {
    ylo = max(0, oy0 * S - g.pt);
    yhi = max(ylo, min(g.H, (oy0 + rows - 1) * S - g.pt + K));
  }
  const int count = g.bands > 1 ? (yhi - ylo) * g.W : np * hw;
  const int64_t src0 = (int64_t)plane0 * hw + (int64_t)ylo * g.W;
  int8_t* st = lds8 + kFront;
  if constexpr (IN8) {
    const int8_t* xs = static_cast<const int8_t*>(g.x) + src0;
    const int n16 = count >> 4;
    for (int i0 = tid; i0 < n16; i0 += 4 * kThreads) {
      v4i v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + u * kThreads < n16) __builtin_memcpy(&v[u], xs + 16 * (i0 + u * kThreads), 16);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (i0 + u * kThreads < n16) reinterpret_cast<v4i*>(st)[i0 + u * kThreads] = v[u];
    }
    for (int e = (n16 << 4) + tid; e < count; e += kThreads) st[e] = xs[e];
  } else {
    const float* xs = static_cast<const float*>(g.x) + src0;
    const int n4 = count >> 2;
    for (int i0 = tid; i0 < n4; i0 += 8 * kThreads) {
      v4f v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (i0 + u * kThreads < n4) __builtin_memcpy(&v[u], xs + 4 * (i0 + u * kThreads), 16);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (i0 + u * kThreads < n4)
          reinterpret_cast<uint32_t*>(st)[i0 + u * kThreads] =
              pack_i8x4(quantize_q(v[u].x, g.is), quantize_q(v[u].y, g.is), quantize_q(v[u].z, g.is),
                        quantize_q(v[u].w, g.is));
    }
    for (int e = (n4 << 2) + tid; e < count; e += kThreads) st[e] = quantize_i8(xs[e], g.is);
  }
  __syncthreads();
  const int per = g.rgs * g.quads, total = np * per;
  for (int item = tid; item < total; item += kThreads) {
    const int pi = fdiv(item, g.item_div), rest = item - pi * per;
    const int rg = fdiv(rest, g.quad_div), q = rest - rg * g.quads;
    const int plane = plane0 + pi, c = plane % g.C;
    const int oy = oy0 + rg * kRows, nrow = min(kRows, oy0 + rows - oy);
    if (nrow <= 0) continue;
    int w[K][KW];
#pragma unroll
    for (int i = 0; i < K; ++i)
#pragma unroll
      for (int j = 0; j < KW; ++j) w[i][j] = g.w[(c * K + i) * KW + j];
    const float rc = g.recip[c], bs = g.bias[c];
    const int x0 = 4 * q * S - g.pl, xc = min(x0, g.W);  // past the image: every byte masked
    uint32_t m[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) m[d] = byte_mask(d, -x0, g.W - x0);
    int acc[kRows][4];
#pragma unroll
    for (int r = 0; r < kRows; ++r)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[r][u] = 0;
    const int y0 = oy * S - g.pt, base = kFront + (g.bands > 1 ? 0 : pi * hw) + xc;
#pragma unroll
    for (int i = 0; i < IR; ++i) {
      const int y = y0 + i;
      const bool ok = y >= ylo && y < yhi;
      const int a = base + (ok ? y - ylo : 0) * g.W;
      const uint32_t* p = reinterpret_cast<const uint32_t*>(lds8 + (a & ~3));
      uint32_t raw[ND + 1], d[ND + 1];
#pragma unroll
      for (int j = 0; j <= ND; ++j) raw[j] = p[j];
#pragma unroll
      for (int j = 0; j < ND; ++j)
        d[j] = __builtin_amdgcn_alignbyte(raw[j + 1], raw[j], (uint32_t)a) & (ok ? m[j] : 0u);
      d[ND] = 0;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int t = 0; t < KW; ++t) {
          constexpr int kWord = 4;
          const int off = u * S + kWord * t;  // byte offset of these taps in the segment
          const uint32_t taps = off % 4 == 0 ? d[off / 4]
                                             : __builtin_amdgcn_alignbyte(d[off / 4 + 1], d[off / 4], off % 4);
#pragma unroll
          for (int r = 0; r < kRows; ++r)
            if (i - r * S >= 0 && i - r * S < K)
              acc[r][u] = __builtin_amdgcn_sdot4((int)taps, w[i - r * S][t], acc[r][u], false);
        }
      }
    }
    const int nx = min(4, g.OW - 4 * q);
    const int64_t o0 = ((int64_t)plane * g.OH + oy) * g.OW + 4 * q;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      if (r >= nrow) break;
      float f[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma clang fp contract(off)
        f[u] = (float)acc[r][u];
        f[u] = f[u] * rc;
        f[u] = f[u] + bs;
      }
      const int64_t o = o0 + (int64_t)r * g.OW;
      if constexpr (OUT8) {
        const uint32_t v = pack_i8x4(quantize_q(f[0], g.os, g.qlo), quantize_q(f[1], g.os, g.qlo),
                                     quantize_q(f[2], g.os, g.qlo), quantize_q(f[3], g.os, g.qlo));
        int8_t* dst = static_cast<int8_t*>(g.y) + o;
        if (nx == 4) {
          __builtin_memcpy(dst, &v, 4);
        } else {
          for (int u = 0; u < nx; ++u) dst[u] = (int8_t)(v >> (8 * u));
        }
      } else {
        v4f v;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = g.relu && f[u] < 0.f ? 0.f : f[u];
        float* dst = static_cast<float*>(g.y) + o;
        if (nx == 4) {
          __builtin_memcpy(dst, &v, 16);
        } else {
          for (int u = 0; u < nx; ++u) dst[u] = v[u];
        }
      }
    }
  }
}

template <int K, int S>
int launch_ks(const DwI8RunArgs& a, int64_t blocks, size_t lds, bool in8, bool out8, hipStream_t s) {
  const dim3 grid((unsigned)blocks), block(kThreads);
  if (in8 && out8)
    NHIP_LAUNCH("dwconv_int8_runs", (dw_int8_runs_kernel<K, S, true, true>), grid, block, lds, s, a);
  else if (in8)
    NHIP_LAUNCH("dwconv_int8_runs", (dw_int8_runs_kernel<K, S, true, false>), grid, block, lds, s, a);
  else if (out8)
    NHIP_LAUNCH("dwconv_int8_runs", (dw_int8_runs_kernel<K, S, false, true>), grid, block, lds, s, a);
  else
    NHIP_LAUNCH("dwconv_int8_runs", (dw_int8_runs_kernel<K, S, false, false>), grid, block, lds, s, a);
  return check_launch("dwconv_int8_runs");
}

// Rows of a band: whole planes where a plane fits LDS and there are planes
// enough for two workgroups per CU, else bands of whole thread rows.  0: not
// even kRows output rows' input fits.
int band_rows(const nhip_conv_plan* p, int64_t planes, int h, int w, int oh) {
  const int s = p->g.sh, k = p->g.kh;
  const int64_t want = 2LL * cu_count();
  int64_t bands = planes >= want ? 1 : std::min<int64_t>(ceil_div(want, planes), ceil_div(oh, 2 * kRows));
  if (bands <= 1 && (int64_t)h * w <= kMaxStage) return oh;
  int ob = (int)round_up(ceil_div(oh, std::max<int64_t>(bands, 2)), kRows);
  while (ob > kRows && (int64_t)((ob - 1) * s + k) * w > kMaxStage) ob = (int)round_up(ob / 2, kRows);
  return (int64_t)((ob - 1) * s + k) * w <= kMaxStage ? ob : 0;
}

}  // namespace

// The [C][K][words] copy of the taps for a plan this kernel can take (empty
// otherwise).
std::vector<int32_t> dw_int8_pack(const nhip_conv_plan* p, const int8_t* wq) {
  std::vector<int32_t> out;
  const ConvGeom& g = p->g;
  if (g.kh != g.kw || (g.kh != 3 && g.kh != 5) || g.sh != g.sw || (g.sh != 1 && g.sh != 2) || g.dh != 1 || g.dw != 1 ||
      g.pl > kMaxPadLeft)
    return out;
  const int K = g.kh, KW = (K + 3) / 4;
  out.assign((size_t)g.c * K * KW, 0);
  for (int c = 0; c < g.c; ++c)
    for (int i = 0; i < K; ++i)
      for (int j = 0; j < K; ++j)
        out[((size_t)c * K + i) * KW + j / 4] |=
            (int32_t)((uint32_t)(uint8_t)wq[((size_t)c * K + i) * K + j] << (8 * (j % 4)));
  return out;
}

bool dw_int8_runs_supported(const nhip_conv_plan* p, int n, int h, int w, int oh) {
  if (p->weight_dw_pack == nullptr || setting_int("NHIP_DW_INT8_RUNS", 1) == 0) return false;
  return band_rows(p, (int64_t)n * p->g.c, h, w, oh) > 0;
}

int launch_dw_int8_runs(const nhip_conv_plan* p, const void* in, int in_is_i8, void* out, int n, int h, int w, int oh,
                        int ow, hipStream_t s) {
  DwI8RunArgs a{};
  a.x = in;
  a.y = out;
  a.w = p->weight_dw_pack;
  a.bias = p->bias;
  a.recip = p->recip;
  a.is = p->input_scale;
  a.os = p->output_scale;
  a.relu = p->g.act == NHIP_ACT_RELU;
  a.qlo = a.relu ? 0 : -127;
  a.C = p->g.c;
  a.H = h;
  a.W = w;
  a.OH = oh;
  a.OW = ow;
  a.pt = p->g.pt;
  a.pl = p->g.pl;
  a.planes = n * p->g.c;
  a.quads = (int)ceil_div(ow, 4);
  a.ob = band_rows(p, a.planes, h, w, oh);
  if (a.ob <= 0) return fail(NHIP_STATUS_UNSUPPORTED, "int8 depthwise: input rows too wide for LDS staging");
  a.bands = (int)ceil_div(oh, a.ob);
  a.rgs = (int)ceil_div(std::min(a.ob, oh), kRows);
  // several small planes per workgroup: one item (4 x 4 outputs) per thread,
  // two workgroups per CU first
  a.ppb = 1;
  if (a.bands == 1) {
    const int64_t items = (int64_t)a.rgs * a.quads;
    int64_t ppb = std::max<int64_t>(1, kThreads / items);
    ppb = std::min<int64_t>(ppb, std::max<int64_t>(1, a.planes / (2LL * cu_count())));
    a.ppb = (int)std::min<int64_t>(ppb, std::max<int64_t>(1, kMaxStage / std::max(1, h * w)));
  }
  const int64_t staged = a.bands == 1 ? (int64_t)a.ppb * h * w : (int64_t)((a.ob - 1) * p->g.sh + p->g.kh) * w;
  const size_t lds = (size_t)round_up(kFront + staged + kBack, 16);
  a.item_div = fast_div((uint32_t)(a.rgs * a.quads));
  a.quad_div = fast_div((uint32_t)a.quads);
  a.band_div = fast_div((uint32_t)a.bands);
  const int64_t blocks = ceil_div(a.planes, a.ppb) * a.bands;
  const bool in8 = in_is_i8 != 0, out8 = p->scale_term > 100;
  if (p->g.kh == 3)
    return p->g.sh == 1 ? launch_ks<3, 1>(a, blocks, lds, in8, out8, s) : launch_ks<3, 2>(a, blocks, lds, in8, out8, s);
  return p->g.sh == 1 ? launch_ks<5, 1>(a, blocks, lds, in8, out8, s) : launch_ks<5, 2>(a, blocks, lds, in8, out8, s);
}

}  // namespace nhip
