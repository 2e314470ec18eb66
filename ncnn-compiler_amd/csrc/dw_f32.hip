// fp32 ConvolutionDepthWise (NCNNToTosa.cpp:3376-3503) for square 3x3 and 5x5
// kernels, stride 1 or 2, dilation 1, any padding, with rows of any width and
// alignment: whole planes or bands of rows in LDS, a column run of outputs per
// thread.  Same operation order as the CPU loop nest, so bit-identical to the
// other depthwise kernels: acc = 0, += x * w over (kh, kw) with every multiply
// and add rounded on its own, then + bias, then the activation.
//
// What bounds it: HBM, and close behind it the arithmetic (two operations a
// tap without fused multiply-adds: 50 for 5x5, which 25 TB/s of LDS and 8 of
// HBM would allow 60 of).  So the loads and the LDS traffic per output are what
// the layout saves:
//   - a workgroup's input is one contiguous run of the NCHW tensor (several
//     planes, a plane, or a band), read with 16-byte loads, eight in flight per
//     thread, whatever the row width; it goes into LDS re-pitched to rows of
//     the window's width with the zero padding around them, so the inner loop
//     has no bounds check;
//   - lanes take neighbouring columns (consecutive LDS words, consecutive
//     output addresses) and each forms kRun outputs of its column, reading every
//     input row once: (kRun - 1 + K) K words for kRun outputs instead of K K
//     each (5x5 stride 1: 7.5 an output instead of 25).
// 5x5 stride 1: 29 x 57 @ 79x94 (98 MB) 150 -> 40 us, 32 x 240 @ 28x28 67 -> 18.5,
// 32 x 960 @ 7x7 22 -> 7.1; stride 2: 32 x 672 @ 14x14 28 -> 9.3 (before: the
// general kernel, a bounds-checked load per staged element and a window read
// per output).  3x3 stride 1, rows not 16-byte vectors: 16 x 24 @ 94x94 16.2 ->
// 11.3, 1 x 64 @ 75x75 10.7 -> 5.4 (before: six 4-byte loads a row per thread,
// 16 bytes apart between lanes).
#include <algorithm>

#include "nhip_internal.h"

namespace nhip {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxLds = 40 * 1024;  // four workgroups per CU

struct DwRunArgs {
  const float* x;
  float* y;
  const float* w;     // [C][K*K]
  const float* bias;  // [C]
  int act;
  int C, H, W, OH, OW, pt, pl;
  int planes, ppb;    // planes per workgroup (1 when a plane is cut into bands)
  int bands, ob;      // bands per plane, output rows per band
  int rgs, ir, lw;    // column runs per column (of a band), LDS rows and row pitch of a plane
  FastDiv w_div, h_div, item_div, ow_div, band_div;  // W, H, rgs * OW, OW, bands
};

template <int K, int S>
__global__ __launch_bounds__(kThreads) void dw_f32_runs_kernel(DwRunArgs g) {
  constexpr int kRun = S == 1 ? 8 : 4;
  constexpr int IR = (kRun - 1) * S + K;
  constexpr int kLoads = 8;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int tid = threadIdx.x;
  const int grp = fdiv(blockIdx.x, g.band_div), band = blockIdx.x - grp * g.bands;
  const int plane0 = grp * g.ppb, np = min(g.ppb, g.planes - plane0);
  const int oy0 = band * g.ob, rows = min(g.ob, g.OH - oy0);
  const int ytop = oy0 * S - g.pt;  // image row of LDS row 0
  const int hw = g.H * g.W, per_lds = g.ir * g.lw;
  // image rows [ylo, yhi) staged (whole planes unless banded)
  int ylo = 0, yhi = g.H;
  if (g.bands > 1) {
    ylo = max(0, ytop);
    yhi = max(ylo, min(g.H, ytop + g.ir));
  }
  const int count = g.bands > 1 ? (yhi - ylo) * g.W : np * hw, n4 = count >> 2;
  const float* xs = g.x + (int64_t)plane0 * hw + (int64_t)ylo * g.W;
  // element e of the run (e = 0 in row ylo): its image row, counted over planes, and column
  auto put = [&](int e, const float* v, int m) {
    int gr = fdiv(e, g.w_div), col = e - gr * g.W;
    gr += ylo;
    int pi = g.bands > 1 ? 0 : fdiv(gr, g.h_div), y = gr - pi * g.H;
    for (int u = 0; u < m; ++u) {
      const int ly = y - ytop, lx = col + g.pl;
      if (ly < g.ir && lx < g.lw) lds[pi * per_lds + ly * g.lw + lx] = v[u];
      if (++col == g.W) {
        col = 0;
        if (++y == g.H) {
          y = 0;
          ++pi;
        }
      }
    }
  };
  for (int base = 0; base < n4 || base == 0; base += kLoads * kThreads) {
    v4f v[kLoads];
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int i = base + u * kThreads + tid;
      if (i < n4) __builtin_memcpy(&v[u], xs + 4 * i, 16);
    }
    if (base == 0) {  // the zero padding, while the loads are on their way
      const int all4 = (g.ppb * per_lds + 3) >> 2;
      for (int i = tid; i < all4; i += kThreads) reinterpret_cast<v4f*>(lds)[i] = v4f{0.f, 0.f, 0.f, 0.f};
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int i = base + u * kThreads + tid;
      if (i < n4) {
        const float f[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
        put(4 * i, f, 4);
      }
    }
  }
  if (tid < (count & 3)) {
    const float f = xs[4 * n4 + tid];
    put(4 * n4 + tid, &f, 1);
  }
  __syncthreads();
  const int per = g.rgs * g.OW, total = np * per;
  for (int item = tid; item < total; item += kThreads) {
    const int pi = fdiv(item, g.item_div), rest = item - pi * per;
    const int rg = fdiv(rest, g.ow_div), x = rest - rg * g.OW;
    const int plane = plane0 + pi, c = plane % g.C;
    float w[K * K];
#pragma unroll
    for (int t = 0; t < K * K; ++t) w[t] = g.w[c * (K * K) + t];
    const float b = g.bias[c];
    const float* src = lds + pi * per_lds + rg * kRun * S * g.lw + x * S;
    float acc[kRun];
#pragma unroll
    for (int r = 0; r < kRun; ++r) acc[r] = 0.f;
#pragma unroll
    for (int i = 0; i < IR; ++i) {
      float v[K];
#pragma unroll
      for (int j = 0; j < K; ++j) v[j] = src[i * g.lw + j];
#pragma unroll
      for (int r = 0; r < kRun; ++r)
        if (i - r * S >= 0 && i - r * S < K) {
#pragma unroll
          for (int j = 0; j < K; ++j) acc[r] = acc[r] + v[j] * w[(i - r * S) * K + j];
        }
    }
    const int oy = oy0 + rg * kRun, nrow = oy0 + rows - oy;
    float* dst = g.y + ((int64_t)plane * g.OH + oy) * g.OW + x;
#pragma unroll
    for (int r = 0; r < kRun; ++r) {
      float o = acc[r] + b;
      if (g.act == NHIP_ACT_RELU) o = o < 0.f ? 0.f : o;
      if (r < nrow) dst[(int64_t)r * g.OW] = o;
    }
  }
}

template <int K, int S>
int launch_ks(const DwRunArgs& a, int64_t blocks, size_t lds, hipStream_t s) {
  NHIP_LAUNCH("dw_f32_runs", (dw_f32_runs_kernel<K, S>), dim3((unsigned)blocks), dim3(kThreads), lds, s, a);
  return check_launch("dw_f32_runs");
}

struct DwRunCfg {
  int ob, ppb, rgs, ir, lw;  // ob 0: one column run's rows do not fit LDS
};

// Whole planes where they fit LDS and give two workgroups per CU, several
// small ones per workgroup while that holds; else bands of whole column runs.
DwRunCfg run_config(const nhip_conv_plan* p, int64_t planes, int oh, int ow) {
  const int s = p->g.sh, k = p->g.kh, run = s == 1 ? 8 : 4;
  const int64_t want = 2LL * cu_count();
  DwRunCfg c{};
  c.lw = (ow - 1) * s + k;
  auto ir_of = [&](int ob) { return (int)(round_up(ob, run) - 1) * s + k; };
  auto fits = [&](int ob) { return (int64_t)ir_of(ob) * c.lw * 4 <= kMaxLds; };
  const int64_t bands = planes >= want ? 1 : std::min<int64_t>(ceil_div(want, planes), ceil_div(oh, run));
  c.ob = bands <= 1 && fits(oh) ? oh : (int)round_up(ceil_div(oh, std::max<int64_t>(bands, 2)), run);
  while (c.ob > run && !fits(c.ob)) c.ob = (int)round_up(c.ob / 2, run);
  if (!fits(c.ob)) {
    c.ob = 0;
    return c;
  }
  c.ob = std::min(c.ob, oh);
  c.rgs = (int)ceil_div(c.ob, run);
  c.ir = ir_of(c.ob);
  c.ppb = 1;
  if (c.ob >= oh) {
    int64_t ppb = std::max<int64_t>(1, kThreads / ((int64_t)c.rgs * ow));
    ppb = std::min<int64_t>(ppb, std::max<int64_t>(1, planes / want));
    c.ppb = (int)std::min<int64_t>(ppb, std::max<int64_t>(1, kMaxLds / ((int64_t)c.ir * c.lw * 4)));
  }
  return c;
}

}  // namespace

bool dw_f32_runs_supported(const nhip_conv_plan* p, int n, int oh, int ow) {
  const ConvGeom& g = p->g;
  if (g.kh != g.kw || (g.kh != 3 && g.kh != 5) || g.sh != g.sw || (g.sh != 1 && g.sh != 2) || g.dh != 1 || g.dw != 1 ||
      setting_int("NHIP_DW_RUNS", 1) == 0)
    return false;
  return run_config(p, (int64_t)n * g.c, oh, ow).ob > 0;
}

int launch_dw_f32_runs(const nhip_conv_plan* p, const float* in, float* out, int n, int h, int w, int oh, int ow,
                       hipStream_t s) {
  DwRunArgs a{};
  a.x = in;
  a.y = out;
  a.w = p->weight;
  a.bias = p->bias;
  a.act = p->g.act;
  a.C = p->g.c;
  a.H = h;
  a.W = w;
  a.OH = oh;
  a.OW = ow;
  a.pt = p->g.pt;
  a.pl = p->g.pl;
  a.planes = n * p->g.c;
  const DwRunCfg c = run_config(p, a.planes, oh, ow);
  if (c.ob <= 0) return fail(NHIP_STATUS_UNSUPPORTED, "depthwise: input rows too wide for LDS staging");
  a.ob = c.ob;
  a.ppb = c.ppb;
  a.bands = (int)ceil_div(oh, c.ob);
  a.rgs = c.rgs;
  a.ir = c.ir;
  a.lw = c.lw;
  a.w_div = fast_div((uint32_t)w);
  a.h_div = fast_div((uint32_t)h);
  a.item_div = fast_div((uint32_t)(a.rgs * ow));
  a.ow_div = fast_div((uint32_t)ow);
  a.band_div = fast_div((uint32_t)a.bands);
  const size_t lds = (size_t)round_up((int64_t)a.ppb * a.ir * a.lw * 4, 16);
  const int64_t blocks = ceil_div(a.planes, a.ppb) * a.bands;
  if (p->g.kh == 3) return p->g.sh == 1 ? launch_ks<3, 1>(a, blocks, lds, s) : launch_ks<3, 2>(a, blocks, lds, s);
  return p->g.sh == 1 ? launch_ks<5, 1>(a, blocks, lds, s) : launch_ks<5, 2>(a, blocks, lds, s);
}

}  // namespace nhip
