// fp32 InnerProduct (NCNNToTosa.cpp:5254-5392: zero-init matmul, then bias) on
// v_mfma_f32_32x32x2_f32, for inputs that the other InnerProduct kernels do not
// take (not 16-byte aligned); the global-average-pooling + InnerProduct pair;
// and the choice among the fp32 convolution kernels.
//
// GEMM view: D[i][j] = sum_k A[i][k] * B[k][j], i an input row, j an output.
// One workgroup = 4 waves (2x2) computes a 64 x 64 tile; each wave one 32x32
// MFMA block.  K advances in chunks of 16 through double-buffered LDS.
//
// MFMA k mapping: in chunk-local step s (0..7) lane l supplies k = 8*(l/32)+s
// for both operands, so each lane reads 8 consecutive k of its A row (two
// ds_read_b128) instead of 16 scattered words.  Any permutation of k is valid
// for a dot product as long as A and B use the same one.
#include <algorithm>

#include "nhip_internal.h"

namespace nhip {
namespace {

constexpr int kThreads = 256;
constexpr int kBK = 16;     // K chunk of the MFMA k mapping
constexpr int kRowPad = 4;  // LDS row padding (floats): conflict-free b128 reads
constexpr int kXcds = 8;    // accelerator complex dies on MI355X

struct GemmArgs {
  const float* a;        // input [M][lda]
  int lda;
  int m;                 // input rows
  const float* b;        // W [n_pad][ldb]
  int ldb;
  int n;                 // outputs
  int kdim;              // reduction length (multiple of 16 after padding)
  int k_valid;           // valid input length (loads past it read 0)
  float* d;              // out [M][ldd], or raw partials [split][M][ldd]
  int ldd;
  const float* bias;
  int act;
  int splits;            // split-K factor
  int a_vec4;            // lda % 4 == 0 (float4 A loads allowed)
};

__device__ __forceinline__ float apply_act(float v, int act) {
  if (act == NHIP_ACT_RELU) return v < 0.0f ? 0.0f : v;
  if (act == NHIP_ACT_SIGMOID) return 1.0f / (1.0f + __expf(-v));
  return v;
}

__global__ __launch_bounds__(kThreads) void gemm_ip_kernel(GemmArgs g) {
  constexpr int BM = 64, BN = 64, AS = kBK + kRowPad;  // As[BM][AS], Bs[BN][AS]
  __shared__ __attribute__((aligned(16))) float smem[2 * (BM + BN) * AS];
  auto As = [&](int buf) { return smem + buf * BM * AS; };
  auto Bs = [&](int buf) { return smem + 2 * BM * AS + buf * BN * AS; };
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1, li = lane & 31, lh = lane >> 5;

  // Workgroups are dispatched round-robin over the XCDs (8 on MI355X, each
  // with its own L2): hardware id L runs on XCD L % 8.  Renumber so that each
  // XCD gets a contiguous range of logical tiles; tiles that share an A row
  // block (same i) then run on the same XCD and share its L2.
  int bx, by, bz;
  {
    const int nbx = gridDim.x, nby = gridDim.y;
    const int total = nbx * nby * gridDim.z;
    const int L = blockIdx.x + nbx * (blockIdx.y + nby * blockIdx.z);
    const int x = L % kXcds, q = L / kXcds;
    const int logical = x * (total / kXcds) + min(x, total % kXcds) + q;
    bx = logical % nbx;
    by = (logical / nbx) % nby;
    bz = logical / (nbx * nby);
  }
  const int j0 = bx * BN, i0 = by * BM;
  const int nk_total = g.kdim / kBK;
  const int per = (nk_total + g.splits - 1) / g.splits;
  const int kt_begin = min(nk_total, bz * per), kt_end = min(nk_total, kt_begin + per);

  // a thread's operand of a stage: 4 consecutive k of one row of each
  struct Stage {
    v4f a, b;
  };
  const int row = tid / 4, kq = (tid % 4) * 4;
  auto gload = [&](Stage& st, int kt) {
    const int k = kt * kBK + kq, r = i0 + row;
    v4f v = {0.f, 0.f, 0.f, 0.f};
    if (r < g.m) {
      const float* src = g.a + (int64_t)r * g.lda;
      if (g.a_vec4) {
        if (k < g.k_valid) v = *reinterpret_cast<const v4f*>(src + k);
      } else {
        v.x = (k + 0 < g.k_valid) ? src[k + 0] : 0.f;
        v.y = (k + 1 < g.k_valid) ? src[k + 1] : 0.f;
        v.z = (k + 2 < g.k_valid) ? src[k + 2] : 0.f;
        v.w = (k + 3 < g.k_valid) ? src[k + 3] : 0.f;
      }
    }
    st.a = v;
    st.b = *reinterpret_cast<const v4f*>(g.b + (int64_t)(j0 + row) * g.ldb + k);
  };
  auto lstore = [&](const Stage& st, int buf) {
    *reinterpret_cast<v4f*>(&As(buf)[row * AS + kq]) = st.a;
    *reinterpret_cast<v4f*>(&Bs(buf)[row * AS + kq]) = st.b;
  };

  v16f acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  auto compute = [&](int buf) {
    const float* pa = &As(buf)[(wm * 32 + li) * AS + lh * 8];
    const float* pb = &Bs(buf)[(wn * 32 + li) * AS + lh * 8];
    const v4f a0 = *reinterpret_cast<const v4f*>(pa), a1 = *reinterpret_cast<const v4f*>(pa + 4);
    const v4f b0 = *reinterpret_cast<const v4f*>(pb), b1 = *reinterpret_cast<const v4f*>(pb + 4);
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[s], b0[s], acc, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[s], b1[s], acc, 0, 0, 0);
  };

  // Two LDS buffers, global loads two stages ahead; the loop body is
  // straight-line (two stages per trip, odd tail peeled).
  const int n = kt_end - kt_begin;
  if (n > 0) {
    Stage s0, s1;
    gload(s0, kt_begin);
    if (n > 1) gload(s1, kt_begin + 1);
    lstore(s0, 0);
    __syncthreads();
    int i = 0;
    for (; i + 1 < n; i += 2) {
      if (i + 2 < n) gload(s0, kt_begin + i + 2);
      compute(0);
      lstore(s1, 1);
      __syncthreads();
      if (i + 3 < n) gload(s1, kt_begin + i + 3);
      compute(1);
      if (i + 2 < n) lstore(s0, 0);
      __syncthreads();
    }
    if (i < n) compute(0);
  }

  // 32x32 accumulator layout: register r of lane l holds row (r%4) + 8*(r/4) +
  // 4*(l/32), column l%32.
  const int j = j0 + wn * 32 + li;
  if (j >= g.n) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int i = i0 + wm * 32 + (r & 3) + 8 * (r >> 2) + 4 * lh;
    if (i >= g.m) continue;
    if (g.splits > 1)
      g.d[((int64_t)bz * g.m + i) * g.ldd + j] = acc[r];
    else
      g.d[(int64_t)i * g.ldd + j] = apply_act(acc[r] + g.bias[j], g.act);
  }
}

// Split-K reduction for InnerProduct: out = act((sum_s part[s]) + bias).
__global__ void ip_splitk_reduce(const float* part, const float* bias,
                                 float* out, int m, int n, int ldp,
                                 int splits, int act) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)m * n) return;
  const int i = (int)(idx / n), j = (int)(idx - (int64_t)i * n);
  // splits are added in order; the loads of 8 splits are issued together
  const float* src = part + (int64_t)i * ldp + j;
  const int64_t stride = (int64_t)m * ldp;
  float s = 0.f;
  int z = 0;
  for (; z + 8 <= splits; z += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = src[(z + u) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) s += v[u];
  }
  for (; z < splits; ++z) s += src[z * stride];
  out[idx] = apply_act(s + bias[j], act);
}

}  // namespace

// ------------------------------- Convolution ------------------------------
// A 1x1 stride-1 layer that runs faster on the split kernel than on the
// streaming 1x1 kernel, both measured: from 176 input channels on (288 -> 80,
// 15488 pixels: 17.9 -> 15.8 us; 448 -> 368, 6498: 37.3 -> 26.9; 168 -> 48,
// 4356: 6.0 against 6.6), and from 49 where the planes are no multiple of four
// pixels, which the streaming kernel reads one element at a time (80 -> 240,
// 57x57 x 2: 15.1 -> 11.0; 56 -> 168, 29x29 x 9: 11.3 -> 9.7), with 48 only up to one
// 64 x 64 tile per four CUs (48 -> 64, 29x29 x 3: 5.0 -> 4.6; but 48 -> 168, 29x29 x
// 9: 7.5 against 9.0; 24 -> 264, 22x22: no difference).  Up to 32768 pixels:
// launches beyond stream more than the caches hold, and there the streaming
// kernel's 16-byte loads win (192 -> 96, 50176 pixels: 25.3 against 29.6; 200
// -> 40, 100352: 28.0 against 33.9; 256 -> 128, 25088: 25.4 -> 22.0).  A forced
// 1x1 kernel (any NHIP_* switch of those kernels) is left alone.
static bool split_1x1_preferred(const nhip_conv_plan* p, int n, int oh, int ow) {
  for (const char* name : {"NHIP_POINTWISE", "NHIP_PW_CFG", "NHIP_PW_WGS", "NHIP_GEMM_DMA", "NHIP_CONV_KQ"})
    if (setting(name)) return false;
  const int64_t plane = (int64_t)oh * ow;
  if (n * plane >= 32768 || p->g.c < 48) return false;
  if (p->g.c >= 176) return true;
  return plane % 4 != 0 && (p->g.c > 48 || 4 * ceil_div(n * plane, 64) * ceil_div(p->g.k, 64) <= cu_count());
}

uint64_t conv_igemm_f32_workspace(const nhip_conv_plan* p, int n, int oh, int ow) {
  if (!split_1x1_preferred(p, n, oh, ow)) {
    if (pointwise_selected(p, n, oh, ow)) return 0;
    if (pw_dma_supported(p, n, oh, ow)) return conv_pw_dma_workspace(p, n, oh, ow);
  }
  if (igemm_selected(p, n, oh, ow)) return 0;
  return conv_split_workspace(p, n, oh, ow);
}

int launch_conv_igemm_f32(const nhip_conv_plan* p, const float* in,
                          const float* residual, float* out, int n, int h,
                          int w, int oh, int ow, void* ws, uint64_t ws_bytes,
                          hipStream_t s) {
  // (the short-reduction kernel needs no workspace; the size query above
  // keeps the split kernel's, which is then unused)
  if (smallk_supported(p, n, h, w, oh, ow)) return launch_conv_smallk(p, in, residual, out, n, h, w, oh, ow, s);
  if (kq_supported(p, n, h, w, oh, ow)) return launch_conv_kq(p, in, residual, out, n, h, w, oh, ow, s);
  if (!split_1x1_preferred(p, n, oh, ow)) {
    if (pointwise_selected(p, n, h, w)) return launch_conv_pointwise_f32(p, in, residual, out, n, h, w, s);
    if (pw_dma_supported(p, n, h, w)) return launch_conv_pw_dma(p, in, residual, out, n, h, w, ws, ws_bytes, s);
  }
  if (igemm_selected(p, n, oh, ow)) return launch_conv_igemm(p, in, residual, out, n, h, w, oh, ow, s);
  return launch_conv_split(p, in, residual, out, n, h, w, oh, ow, ws, ws_bytes, s);
}

// ------------------------------- InnerProduct -----------------------------
static int ip_splits(const nhip_ip_plan* p, int m) {
  const int64_t tiles = ceil_div(m, 64) * ceil_div(p->n_out, 64);
  const int nk = p->k_pad / kBK;
  int splits = 1;
  while (tiles * splits < 2LL * cu_count() && nk / (splits * 2) >= 8) splits *= 2;
  return splits;
}

uint64_t innerproduct_workspace(const nhip_ip_plan* p, int m) {
  const int splits = ip_splits(p, m);
  const uint64_t own = splits == 1 ? 0 : (uint64_t)splits * m * p->n_pad * sizeof(float);
  // the direct-to-LDS kernel runs when the input is 16-byte aligned; this
  // kernel otherwise: room for either
  return ip_dma_supported(p, nullptr, m) ? std::max(own, innerproduct_dma_workspace(p, m)) : own;
}

// ------------------- global average pooling + InnerProduct -----------------
// The MobileNet / ResNet head: ConvertPooling's global average
// (NCNNToTosa.cpp:1880-1990, the mean of every [H,W] plane) feeding
// ConvertInnerProduct (:5254-5392), in one pass over the input.  A
// workgroup of 16 waves owns 16 images x 256 outputs x one slice of ks <= 64
// channels.  The slice of one image is one contiguous run of ks planes: ipp
// images at a time come into LDS through 16-byte loads, one lane per plane
// sums it in element order (the CPU loop's order, so the means equal
// nhip_global_avgpool_f32's bit for bit), then the LDS holds the weight
// slice, v_mfma_f32_16x16x4_f32 multiplies, and the workgroup writes a
// split-K partial [split][n][n_out]; ip_splitk_reduce adds the splits in
// order, the bias and the activation.  The ceil(n_out / 256) workgroups of
// a slice (4 for 1000 outputs) read its planes, mostly from L2; the head is
// two launches instead of three.
namespace {
constexpr int kGapRows = 16, kGapCols = 256, kGapMaxK = 64, kGapThreads = 1024;
constexpr int kGapStage = 25600;  // floats of LDS: staged planes, then the weight slice
static_assert(kGapCols * (kGapMaxK + 4) <= kGapStage, "the weight slice fits the staging area");
static_assert(kGapThreads / 64 * 16 == kGapCols, "one 16-output MFMA block per wave");

struct GapIpArgs {
  const float* x;   // [n][C][hw]
  const float* w;   // [n_pad][k_pad], zero padded
  float* part;      // [splits][n][n_out]
  int n, C, hw, n_out, n_pad, k_pad, ks, ipp;
};

__global__ __launch_bounds__(kGapThreads) void gap_ip_kernel(GapIpArgs a) {
  __shared__ __attribute__((aligned(16))) float S[kGapStage];
  __shared__ float P[kGapRows][kGapMaxK + 4];  // pooled [image][channel of the slice]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c0 = blockIdx.x * kGapCols, z = blockIdx.y, img0 = blockIdx.z * kGapRows;
  const int k0 = z * a.ks;
  const int kv = min(a.ks, a.C - k0);  // channels of the slice inside the tensor
  const int L = kv * a.hw, L4 = L >> 2, Ls = (L + 3) & ~3;  // floats of one image's run, its LDS stride
  for (int e = tid; e < kGapRows * (kGapMaxK + 4); e += kGapThreads) (&P[0][0])[e] = 0.f;
  for (int i0 = 0; i0 < kGapRows && img0 + i0 < a.n; i0 += a.ipp) {
    const int ni = min(a.ipp, a.n - img0 - i0);
    const float* src = a.x + ((int64_t)(img0 + i0) * a.C + k0) * a.hw;
    const int64_t img_stride = (int64_t)a.C * a.hw;
    // runs of ni images: 16-byte loads (4-byte aligned sources), four in flight per lane
    for (int v0 = tid; v0 < ni * L4; v0 += 4 * kGapThreads) {
      v4f t[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int v = v0 + u * kGapThreads, i = v / max(L4, 1), q = v - i * L4;
        if (v < ni * L4) __builtin_memcpy(&t[u], src + i * img_stride + 4 * q, 16);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int v = v0 + u * kGapThreads, i = v / max(L4, 1), q = v - i * L4;
        if (v < ni * L4) *reinterpret_cast<v4f*>(&S[i * Ls + 4 * q]) = t[u];
      }
    }
    const int rem = L - 4 * L4;
    for (int e = tid; e < ni * rem; e += kGapThreads) {
      const int i = e / rem, j = e - i * rem;
      S[i * Ls + 4 * L4 + j] = src[i * img_stride + 4 * L4 + j];
    }
    __syncthreads();
    if (tid < ni * a.ks) {
      const int i = tid / a.ks, j = tid - i * a.ks;
      if (j < kv) {
        const float* pl = S + i * Ls + j * a.hw;
        float sum = 0.f;
        for (int e = 0; e < a.hw; ++e) sum = sum + pl[e];
        P[i0 + i][j] = sum / (float)a.hw;
      }
    }
    __syncthreads();
  }
  // weight slice [256 outputs][ks channels], 16-byte loads (k_pad and ks are multiples of 4)
  float (*Ws)[kGapMaxK + 4] = reinterpret_cast<float (*)[kGapMaxK + 4]>(S);
  const int kq = a.ks / 4;
  for (int e = tid; e < kGapCols * kq; e += kGapThreads) {
    const int col = e / kq, q4 = e - col * kq, k = k0 + 4 * q4;
    v4f v = v4f{0.f, 0.f, 0.f, 0.f};
    if (c0 + col < a.n_pad && k < a.k_pad) v = *reinterpret_cast<const v4f*>(a.w + (int64_t)(c0 + col) * a.k_pad + k);
    *reinterpret_cast<v4f*>(&Ws[col][4 * q4]) = v;
  }
  __syncthreads();
  // one C[16 images][16 outputs] block per wave: lane (li, q) supplies
  // A = P[li][4s + q] and B = Ws[16 wave + li][4s + q]; register r holds
  // C[image 4q + r][output li]
  const int li = lane & 15, q = lane >> 4;
  v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < kq; ++s)
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(P[li][4 * s + q], Ws[wave * 16 + li][4 * s + q], acc, 0, 0, 0);
  float* dst = a.part + (int64_t)z * a.n * a.n_out;
  const int col = c0 + wave * 16 + li;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int img = img0 + 4 * q + r;
    if (img < a.n && col < a.n_out) dst[(int64_t)img * a.n_out + col] = acc[r];
  }
}

// Channels per split: about one workgroup per CU, 16 to 64 channels per
// slice, at most 16 splits (each split's partial is n x n_out floats), and
// at least one image's slice in the staging area (4 <= ks).
int gap_ip_ks(const nhip_ip_plan* p, int n, int hw) {
  const int64_t others = ceil_div(p->n_out, kGapCols) * ceil_div(n, kGapRows);
  const int64_t splits = std::min<int64_t>(16, std::max<int64_t>(1, cu_count() / others));
  int ks = (int)round_up(ceil_div(p->k_in, splits), 4);
  ks = std::min(std::max(ks, 16), kGapMaxK);
  const int fit = (kGapStage / hw) / 4 * 4;  // run stride rounds up to 4 floats
  return std::min(ks, fit);
}

// Images per staging pass: the largest power of two up to 16 whose runs fit.
int gap_ip_ipp(int ks, int hw) {
  const int run = (int)round_up((int64_t)ks * hw, 4);
  int ipp = kGapRows;
  while (ipp > 1 && ipp * run > kGapStage) ipp /= 2;
  return ipp;
}
}  // namespace

bool gap_innerproduct_supported(int hw) { return hw >= 1 && hw <= kGapStage / 4; }

uint64_t gap_innerproduct_workspace(const nhip_ip_plan* p, int n, int hw) {
  if (!gap_innerproduct_supported(hw)) return 0;
  const int splits = (int)ceil_div(p->k_in, gap_ip_ks(p, n, hw));
  return (uint64_t)splits * n * p->n_out * sizeof(float);
}

int launch_gap_innerproduct_f32(const nhip_ip_plan* p, const float* in, float* out, int n, int hw, void* ws,
                                uint64_t ws_bytes, hipStream_t s) {
  if (!gap_innerproduct_supported(hw))
    return fail(NHIP_STATUS_CONSTRAINT_VIOLATION,
                "global_avgpool_innerproduct: planes of at most " + std::to_string(kGapStage / 4) + " pixels");
  const int ks = gap_ip_ks(p, n, hw);
  const int splits = (int)ceil_div(p->k_in, ks);
  const uint64_t need = (uint64_t)splits * n * p->n_out * sizeof(float);
  if (ws == nullptr || ws_bytes < need)
    return fail(NHIP_STATUS_OUTPUT_CAPACITY_INSUFFICIENT,
                "global_avgpool_innerproduct: workspace of " + std::to_string(need) + " bytes required");
  GapIpArgs a{in, p->weight, static_cast<float*>(ws), n, p->k_in, hw, p->n_out, p->n_pad, p->k_pad, ks,
              gap_ip_ipp(ks, hw)};
  const dim3 grid((unsigned)ceil_div(p->n_out, kGapCols), (unsigned)splits, (unsigned)ceil_div(n, kGapRows));
  NHIP_LAUNCH("gap_innerproduct_f32", gap_ip_kernel, grid, dim3(kGapThreads), 0, s, a);
  NHIP_TRY(check_launch("gap_innerproduct_f32"));
  const int64_t total = (int64_t)n * p->n_out;
  NHIP_LAUNCH("ip_splitk_reduce", ip_splitk_reduce, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, s,
              static_cast<const float*>(ws), p->bias, out, n, p->n_out, p->n_out, splits, p->act);
  return check_launch("ip_splitk_reduce");
}

int launch_innerproduct_f32(const nhip_ip_plan* p, const float* in,
                            float* out, int m, void* ws, uint64_t ws_bytes,
                            hipStream_t s) {
  if (ip_kq_supported(p, in, m)) return launch_ip_kq(p, in, out, m, s);
  if (ip_dma_supported(p, in, m)) return launch_innerproduct_dma(p, in, out, m, ws, ws_bytes, s);
  GemmArgs g{};
  g.a = in;
  g.lda = p->k_in;
  g.m = m;
  g.k_valid = p->k_in;
  g.a_vec4 = (p->k_in % 4 == 0 && (reinterpret_cast<uintptr_t>(in) & 15) == 0) ? 1 : 0;
  g.b = p->weight;
  g.ldb = p->k_pad;
  g.n = p->n_out;
  g.kdim = p->k_pad;
  g.bias = p->bias;
  g.act = p->act;
  const int splits = ip_splits(p, m);
  g.splits = splits;
  if (splits > 1) {
    const uint64_t need = innerproduct_workspace(p, m);
    if (ws == nullptr || ws_bytes < need)
      return fail(NHIP_STATUS_OUTPUT_CAPACITY_INSUFFICIENT,
                  "innerproduct: workspace of " + std::to_string(need) +
                      " bytes required");
    g.d = static_cast<float*>(ws);
    g.ldd = p->n_pad;
  } else {
    g.d = out;
    g.ldd = p->n_out;
  }
  // B rows (weights) are padded to n_pad (multiple of 64); j bounds are
  // checked in the epilogue only.
  NHIP_LAUNCH("innerproduct_f32<64,64>", gemm_ip_kernel, dim3(p->n_pad / 64, (int)ceil_div(m, 64), splits),
              dim3(kThreads), 0, s, g);
  NHIP_TRY(check_launch("innerproduct_f32<64,64>"));
  if (splits > 1) {
    const int64_t total = (int64_t)m * p->n_out;
    NHIP_LAUNCH("ip_splitk_reduce", ip_splitk_reduce, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, s,
                       static_cast<const float*>(ws), p->bias, out, m, p->n_out, p->n_pad,
                       splits, p->act);
    return check_launch("ip_splitk_reduce");
  }
  return ok();
}

}  // namespace nhip
