// fp32 Convolution with a short reduction (reference ConvertConvolution fp32
// path, NCNNToTosa.cpp:1316-1529) as an implicit GEMM on
// v_mfma_f32_32x32x2_f32: network stems and 1x1 layers of few channels.
//
// GEMM view: D[i][j] = sum_k A[i][k] B[k][j], i an output channel, j an output
// pixel over the whole batch, k = (c, kh, kw) as the weights lie.  One workgroup
// = 4 waves (2x2) computes a 64 x 64 tile, each wave one 32x32 MFMA block; k
// advances in stages of 16 through double-buffered LDS, global loads two stages
// ahead.  MFMA k mapping: in stage-local step s (0..7) lane l supplies k = 8*(l/32)+s
// for both operands, so that a lane reads 8 consecutive k of its row.
//
// What bounds it: with one to seven stages, the chain table -> gather -> LDS ->
// MFMA -> store of a workgroup and the output's way to memory, not the matrix
// instructions.  Each input value is gathered once per 64 output channels, by
// one lane, and the weights come as rows of fp32; the split kernel
// (conv_split.hip) gathers once per 32 or 64 channels per wave, spends 5.5
// operations on a value's pieces and loads six bytes per weight, which only a
// longer reduction pays back.  1 x 3 -> 32 at 224x224, 3x3 stride 2: 7.3 us
// there, 4.8 here; 4 x 3 -> 64 at 112x112: 8.7 and 5.6; 10 x 1 -> 48 at 56x56: 9.8 and
// 5.7; 32 x 5 -> 96 at 112x112: 116 and 87.
#include "nhip_internal.h"

namespace nhip {
namespace {

constexpr int kThreads = 256;
constexpr int kBM = 64, kBN = 64, kBK = 16;
constexpr int kAS = kBK + 4;  // LDS row pitch (floats): conflict-free b128 reads
constexpr int kXcds = 8;

struct IgemmArgs {
  const float* a;        // weights [m_pad][lda]
  int lda;
  int m;                 // output channels
  const float* x;        // input NCHW
  uint32_t x_bytes;      // < 2^31
  int npix;              // output pixels of the batch
  int stages;            // of 16 k
  const int* ktab;       // c << 16 | dy << 8 | dx; c past C for the padding
  int C, H, W, OHW, OW, sh, sw, pt, pl;
  FastDiv ohw_div, ow_div;
  float* d;              // out NCHW
  const float* bias;
  const float* residual;
  int act;
};

__device__ __forceinline__ float igemm_act(float v, int act) {
  if (act == NHIP_ACT_RELU) return v < 0.0f ? 0.0f : v;
  if (act == NHIP_ACT_SIGMOID) return 1.0f / (1.0f + __expf(-v));
  return v;
}

__global__ __launch_bounds__(kThreads) void conv_igemm_kernel(IgemmArgs g) {
  // two operand buffers of each; the epilogue's 64 x 68 tile over them
  constexpr int TS = kBN + 4, OPER = 2 * (kBM + kBN) * kAS;
  __shared__ __attribute__((aligned(16))) float smem[OPER > kBM * TS ? OPER : kBM * TS];
  auto As = [&](int buf) { return smem + buf * kBM * kAS; };
  auto Bs = [&](int buf) { return smem + 2 * kBM * kAS + buf * kBN * kAS; };
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1, li = lane & 31, lh = lane >> 5;
  // consecutive tiles on one XCD (workgroups go round-robin over the XCDs):
  // the tiles of one channel block share its weights' L2
  int bx, by;
  {
    const int nbx = gridDim.x, total = nbx * gridDim.y;
    const int L = blockIdx.x + nbx * blockIdx.y, x = L % kXcds, q = L / kXcds;
    const int logical = x * (total / kXcds) + min(x, total % kXcds) + q;
    bx = logical % nbx;
    by = logical / nbx;
  }
  const int j0 = bx * kBN, i0 = by * kBM;

  // a thread's operands of a stage: four consecutive k of one weight row, and of
  // the pixel tid % 64 (k uniform over the wave)
  struct Stage {
    v4f a;
    float b[4];
  };
  const int row = tid / 4, kq = (tid % 4) * 4;
  const int jj = tid % kBN, kg = __builtin_amdgcn_readfirstlane(tid / kBN);
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(g.x, g.x_bytes);
  const int p = j0 + jj;
  const bool pix_ok = p < g.npix;
  const int pp = pix_ok ? p : 0, img = fdiv(pp, g.ohw_div), rem = pp - img * g.OHW;
  const int oh = fdiv(rem, g.ow_div), ow = rem - oh * g.OW;
  const int iy0 = oh * g.sh - g.pt, ix0 = ow * g.sw - g.pl, plane0 = img * g.C;
  auto gload = [&](Stage& st, int kt) {
    st.a = *reinterpret_cast<const v4f*>(g.a + (int64_t)(i0 + row) * g.lda + kt * kBK + kq);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = g.ktab[kt * kBK + kg * 4 + u];
      const int c = t >> 16, y = iy0 + ((t >> 8) & 255), x = ix0 + (t & 255);
      const bool in = pix_ok && c < g.C && (unsigned)y < (unsigned)g.H && (unsigned)x < (unsigned)g.W;
      st.b[u] = buf_load_f32(xr, in ? (uint32_t)(((plane0 + c) * g.H + y) * g.W + x) * 4u : kBufOOB);
    }
  };
  auto lstore = [&](const Stage& st, int buf) {
    *reinterpret_cast<v4f*>(&As(buf)[row * kAS + kq]) = st.a;
    *reinterpret_cast<v4f*>(&Bs(buf)[jj * kAS + kg * 4]) = v4f{st.b[0], st.b[1], st.b[2], st.b[3]};
  };
  v16f acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  auto compute = [&](int buf) {
    const float* pa = &As(buf)[(wm * 32 + li) * kAS + lh * 8];
    const float* pb = &Bs(buf)[(wn * 32 + li) * kAS + lh * 8];
    const v4f a0 = *reinterpret_cast<const v4f*>(pa), a1 = *reinterpret_cast<const v4f*>(pa + 4);
    const v4f b0 = *reinterpret_cast<const v4f*>(pb), b1 = *reinterpret_cast<const v4f*>(pb + 4);
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[s], b0[s], acc, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[s], b1[s], acc, 0, 0, 0);
  };
  // straight-line body: two stages per trip, odd tail peeled
  {
    const int n = g.stages;
    Stage s0, s1;
    gload(s0, 0);
    if (n > 1) gload(s1, 1);
    lstore(s0, 0);
    __syncthreads();
    int i = 0;
    for (; i + 1 < n; i += 2) {
      if (i + 2 < n) gload(s0, i + 2);
      compute(0);
      lstore(s1, 1);
      __syncthreads();
      if (i + 3 < n) gload(s1, i + 3);
      compute(1);
      if (i + 2 < n) lstore(s0, 0);
      __syncthreads();
    }
    if (i < n) compute(0);
  }
  // through LDS, so that a thread writes runs of four pixels of one channel.
  // Register r of lane l holds row (r%4) + 8*(r/4) + 4*(l/32), column l%32.
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r)
    smem[(wm * 32 + (r & 3) + 8 * (r >> 2) + 4 * lh) * TS + wn * 32 + li] = acc[r];
  __syncthreads();
  const int ohw = g.OHW;
  const bool vec = (ohw & 3) == 0;
  for (int q = tid; q < kBM * (kBN / 4); q += kThreads) {
    const int lr = q / (kBN / 4), lc = (q % (kBN / 4)) * 4, i = i0 + lr, j = j0 + lc;
    if (i >= g.m || j >= g.npix) continue;
    const float bi = g.bias[i];
    const v4f t = *reinterpret_cast<const v4f*>(&smem[lr * TS + lc]);
    if (vec) {  // (npix is then a multiple of four, and a run is in one image)
      const int ii = fdiv(j, g.ohw_div), o = (ii * g.m + i) * ohw + (j - ii * ohw);
      v4f v = t + bi;
      if (g.residual) v += *reinterpret_cast<const v4f*>(g.residual + o);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = igemm_act(v[e], g.act);
      *reinterpret_cast<v4f*>(g.d + o) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int je = j + e, ie = fdiv(je, g.ohw_div), oe = (ie * g.m + i) * ohw + (je - ie * ohw);
        if (je >= g.npix) break;
        float v = t[e] + bi;
        if (g.residual) v += g.residual[oe];
        g.d[oe] = igemm_act(v, g.act);
      }
    }
  }
}

}  // namespace

// Launches that are faster here than on the split kernel, both measured (1800
// layers of 1 to 32 images, 169 to 401408 pixels, 16 to 496 output channels; here
// / split, us).  tiles: workgroups here.
//   - Reductions that the split kernel runs by its table of taps (few channels),
//     up to 50 long: all, 0.5 to 1.0 of its time (27 long, 12544 pixels, 32
//     channels: 4.8 / 7.3).  Longer ones with more than 32 output channels from
//     three tiles per five CUs on (75 long, 6498 pixels, 100 channels 0.75, 1568
//     and 100 1.14; 99 long, 12544 pixels, 40 channels 0.84, 6498 1.10; 16 or 24
//     channels 0.99 to 1.2).
//   - Whole octets of channels per tap (1x1 mostly): up to 16 long, 0.5 to 0.95
//     with up to 48 channels, else from two tiles per five CUs (12 long, 64
//     channels: 12544 pixels 0.75, 2523 1.18).  Longer with more than 32 channels:
//     up to 50 long from three tiles per five CUs (24 long, 6498 pixels, 128
//     channels 0.84, 2523 and 100 1.13), longer from three per two CUs (72 long,
//     12544 pixels, 128 channels 0.93, 2523 and 240 1.07).
// NHIP_CONV_SMALLK=0 turns the short-reduction kernels off, this one too.
bool igemm_selected(const nhip_conv_plan* p, int n, int oh, int ow) {
  if (p->kred > kIgemmMaxKred || setting_int("NHIP_CONV_SMALLK", 1) == 0) return false;
  const int64_t tiles = ceil_div((int64_t)n * oh * ow, kBN) * ceil_div(p->g.k, kBM), cus = cu_count();
  if (!p->split_taps) return p->kred <= 50 || (p->g.k > 32 && 5 * tiles >= 3 * cus);
  if (p->kred <= 16) return p->g.k <= 48 || 5 * tiles >= 2 * cus;
  return p->g.k > 32 && (p->kred <= 50 ? 5 * tiles >= 3 * cus : 2 * tiles >= 3 * cus);
}

int launch_conv_igemm(const nhip_conv_plan* p, const float* in, const float* residual, float* out, int n, int h, int w,
                      int oh, int ow, hipStream_t s) {
  IgemmArgs g{};
  g.a = p->weight;
  g.lda = p->kred_pad;
  g.m = p->g.k;
  g.x = in;
  g.x_bytes = (uint32_t)((size_t)n * p->g.c * h * w * sizeof(float));
  g.npix = n * oh * ow;
  g.stages = p->kred_pad / kBK;
  g.ktab = p->ktab;
  g.C = p->g.c;
  g.H = h;
  g.W = w;
  g.OHW = oh * ow;
  g.OW = ow;
  g.sh = p->g.sh;
  g.sw = p->g.sw;
  g.pt = p->g.pt;
  g.pl = p->g.pl;
  g.ohw_div = fast_div((uint32_t)g.OHW);
  g.ow_div = fast_div((uint32_t)ow);
  g.d = out;
  g.bias = p->bias;
  g.residual = residual;
  g.act = p->g.act;
  const dim3 grid((unsigned)ceil_div(g.npix, kBN), (unsigned)ceil_div(g.m, kBM));
  NHIP_LAUNCH("conv_igemm_f32", conv_igemm_kernel, grid, dim3(kThreads), 0, s, g);
  return check_launch("conv_igemm_f32");
}

}  // namespace nhip
