// rz_mlp.hip -- learned dispatch: list features and a small FP32 MLP with
// hand-written inference and training kernels.
//
// The MLP maps RZ_MLP_FEATURES features of a (list, removal list) pair to the
// predicted log2 time (us) of each of RZ_MLP_OUTPUTS methods; the dispatcher
// runs the method with the smallest prediction.  Layers: F -> 32 -> 32 -> 32
// -> C, ReLU between them, parameters row-major W[out][in] followed by b[out]
// for each layer, in order.  Training minimises the masked mean squared error
// on measured log times with Adam.  Partial gradients are written out and
// summed in a fixed order, so a gradient is the same bits on every run.
#include <cstring>
#include <mutex>
#include <vector>

#include "rz_ctx.hpp"
#include "rz_device.hpp"

namespace rz {

constexpr int F = RZ_MLP_FEATURES, H = RZ_MLP_HIDDEN, C = RZ_MLP_OUTPUTS;
constexpr int OW1 = 0, OB1 = OW1 + H * F, OW2 = OB1 + H, OB2 = OW2 + H * H, OW3 = OB2 + H, OB3 = OW3 + H * H,
              OW4 = OB3 + H, OB4 = OW4 + C * H, NP = OB4 + C;
static_assert(NP == RZ_MLP_PARAMS, "parameter count");

// ---------------------------------------------------------------------------
// features: one wave per list, a 256-entry strided sample of the removal list
// ---------------------------------------------------------------------------
// The features of list d, by one 64-lane workgroup (s_x: 256 floats of LDS);
// lanes 0 to F - 1 write them to o[0..F).  All loads of the sample are in
// flight together: one after another, with a 64-bit division each, they were
// most of the 5.6 us a list took.
__device__ __forceinline__ void list_features(const rz_list_desc& d, float* s_x, float* o) {
  const int lane = threadIdx.x;
  const double n = (double)(d.n > 0 ? d.n : 1);
  const int64_t k = d.k;
  const int64_t sz = d.n - d.k;
  const int m = k < 256 ? (int)k : 256;  // sample size
  // adjacent pairs (R[i], R[i+1]) at 128 strided positions: runs of the removal list
  const int mp = k < 2 ? 0 : (k - 1 < 128 ? (int)(k - 1) : 128);
  int32_t r[4], pa[2], pb[2];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = lane + 64 * q;  // sample j is at j k / m: m is k or 256
    r[q] = j < m ? d.removals[m < 256 ? (int64_t)j : ((int64_t)j * k) >> 8] : 0;
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int j = lane + 64 * q;  // pair j is at j (k - 1) / mp
    const int64_t i = mp < 128 ? (int64_t)j : ((int64_t)j * (k - 1)) >> 7;
    pa[q] = j < mp ? d.removals[i] : 0;
    pb[q] = j < mp ? d.removals[i + 1] : 0;
  }
  float sum = 0.f, sum2 = 0.f, tail = 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (lane + 64 * q < m) {
      const float x = (float)((double)r[q] / n);
      s_x[lane + 64 * q] = x;
      sum += x;
      sum2 += x * x;
      tail += (r[q] >= sz) ? 1.f : 0.f;
    }
  }
  float consec = 0.f, near = 0.f;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    if (lane + 64 * q < mp) {
      const int64_t a = pa[q], b = pb[q];
      consec += (b == a + 1) ? 1.f : 0.f;
      near += (b - a < 64 && a - b < 64) ? 1.f : 0.f;
    }
  }
  __syncthreads();
  float up = 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int j = lane + 64 * q;
    if (j + 1 < m) up += s_x[j + 1] > s_x[j] ? 1.f : 0.f;
  }
  sum = wave_sum(sum);
  sum2 = wave_sum(sum2);
  tail = wave_sum(tail);
  consec = wave_sum(consec);
  near = wave_sum(near);
  up = wave_sum(up);
  if (lane < F) {
    const float fm = m > 0 ? (float)m : 1.f;
    const float mean = sum / fm;
    const float var = fmaxf(sum2 / fm - mean * mean, 0.f);
    const double frac = (double)k / n;
    // one logarithm, of another argument per lane
    const double lg = log2(lane == 0 ? n : k <= 0 ? 1.0 : lane == 1 ? (double)k : frac);
    float f = 1.f;
    if (lane == 0) f = (float)(lg / 32.0);
    if (lane == 1) f = k > 0 ? (float)(lg / 32.0) : 0.f;
    if (lane == 2) f = (float)frac;
    if (lane == 3) f = k > 0 ? (float)fmax(lg / 20.0, -1.0) : -1.f;
    if (lane == 4) f = (float)d.elem_bytes / 16.f;
    if (lane == 5) f = m > 0 ? tail / fm : 0.f;
    if (lane == 6) f = mean;
    if (lane == 7) f = sqrtf(var);
    if (lane == 8) f = mp > 0 ? consec / (float)mp : 0.f;
    if (lane == 9) f = mp > 0 ? near / (float)mp : 0.f;
    if (lane == 10) f = m > 1 ? up / (float)(m - 1) : 0.f;
    o[lane] = f;
  }
}

__global__ __launch_bounds__(64) void rz_features_kernel(const rz_list_desc* __restrict__ lists, int32_t nlists,
                                                          float* __restrict__ out) {
  const int li = blockIdx.x;
  if (li >= nlists) return;
  __shared__ float s_x[256];
  list_features(lists[li], s_x, out + (size_t)li * F);
}

// ---------------------------------------------------------------------------
// MLP
// ---------------------------------------------------------------------------
// The parameters in LDS, each row of W in a stride of its own odd length (32
// lanes reading a column hit 32 banks).
constexpr int S1 = F + 1, S2 = H + 1;
struct NetShared {
  float w1[H * S1], w2[H * S2], w3[H * S2], w4[C * S2], b[3 * H + C];
};
constexpr int kNetLoads = (NP + 63) / 64;
// Parameter i of the library's layout has its place in the shared copy.
__device__ __forceinline__ void net_store(NetShared& s, int i, float v) {
  if (i < OB1) s.w1[i / F * S1 + i % F] = v;
  else if (i < OW2) s.b[i - OB1] = v;
  else if (i < OB2) s.w2[(i - OW2) / H * S2 + (i - OW2) % H] = v;
  else if (i < OW3) s.b[H + i - OB2] = v;
  else if (i < OB3) s.w3[(i - OW3) / H * S2 + (i - OW3) % H] = v;
  else if (i < OW4) s.b[2 * H + i - OB3] = v;
  else if (i < OB4) s.w4[(i - OW4) / H * S2 + (i - OW4) % H] = v;
  else s.b[3 * H + i - OB4] = v;
}

// One layer by one wave: lane o's pre-activation b[o] + sum_i W[o][i] in_i,
// in_i broadcast from lane i, summed in ascending i.
template <int NIN>
__device__ __forceinline__ float layer_wave(const float* w, float bias, float in) {
  float acc = bias;
#pragma unroll
  for (int i = 0; i < NIN; ++i)
    acc = fmaf(w[i], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(in), i)), acc);
  return acc;
}

static_assert((H & (H - 1)) == 0 && (C & (C - 1)) == 0 && H <= 64 && F <= 64, "one unit per lane");

// The network on one row by one 64-lane workgroup: lane f < F holds feature f
// on entry, p the parameters as loaded (parameter q * 64 + lane in p[q]);
// y_out (may be null) gets the C outputs.  Returns the argmin (every lane),
// ties to the lower index.
__device__ __forceinline__ int forward_wave(const float (&p)[kNetLoads], NetShared& s, float x,
                                            float* __restrict__ y_out) {
  const int lane = threadIdx.x & 63, o = lane & (H - 1), c = lane & (C - 1);
#pragma unroll
  for (int q = 0; q < kNetLoads; ++q)
    if (q * 64 + lane < NP) net_store(s, q * 64 + lane, p[q]);
  __syncthreads();
  float a = layer_wave<F>(&s.w1[o * S1], s.b[o], x);
  float h = a > 0.f ? a : 0.f;
  a = layer_wave<H>(&s.w2[o * S2], s.b[H + o], h);
  h = a > 0.f ? a : 0.f;
  a = layer_wave<H>(&s.w3[o * S2], s.b[2 * H + o], h);
  h = a > 0.f ? a : 0.f;
  const float y = layer_wave<H>(&s.w4[c * S2], s.b[3 * H + c], h);
  if (y_out && lane < C) y_out[lane] = y;
  int best = 0;
  float yb = __shfl(y, 0);
  for (int cc = 1; cc < C; ++cc) {
    const float v = __shfl(y, cc);
    if (v < yb) {
      yb = v;
      best = cc;
    }
  }
  return best;
}
__device__ __forceinline__ void net_load(const float* __restrict__ params, float (&p)[kNetLoads]) {
#pragma unroll
  for (int q = 0; q < kNetLoads; ++q) p[q] = params[min(q * 64 + (int)(threadIdx.x & 63), NP - 1)];
}

// One 64-lane workgroup per row.
__global__ __launch_bounds__(64) void rz_mlp_forward_kernel(const float* __restrict__ params,
                                                             const float* __restrict__ X, int32_t B,
                                                             float* __restrict__ Y, int32_t* __restrict__ choice) {
  __shared__ NetShared sh;
  const int b = blockIdx.x;
  if (b >= B) return;
  const int lane = threadIdx.x;
  float p[kNetLoads];
  net_load(params, p);
  const float x = lane < F ? X[(size_t)b * F + lane] : 0.f;
  const int best = forward_wave(p, sh, x, Y ? Y + (size_t)b * C : nullptr);
  if (choice && lane == 0) choice[b] = best;
}

// rz_dispatch_choose for up to kChooseArgMax lists, and rz_remove_auto: the
// descriptors come as a kernel argument (no upload), one 64-lane workgroup per
// list computes its features and the forward pass, the parameters' loads
// going out first, and lane 0 stores the choice straight into the
// caller-visible pinned staging with a system-scope store.
constexpr int kChooseArgMax = 48;
struct ChooseArgs {
  rz_list_desc d[kChooseArgMax];
};

__device__ __forceinline__ void choose_one(const rz_list_desc& d, const float* __restrict__ params,
                                           int32_t* __restrict__ h_choice) {
  __shared__ float s_x[256];
  __shared__ float s_f[F];
  __shared__ NetShared sh;
  float p[kNetLoads];
  net_load(params, p);
  list_features(d, s_x, s_f);
  __syncthreads();
  const float x = threadIdx.x < F ? s_f[threadIdx.x] : 0.f;
  const int best = forward_wave(p, sh, x, nullptr);
  if (threadIdx.x == 0) __hip_atomic_store(h_choice, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ __launch_bounds__(64) void rz_choose_kernel(ChooseArgs a, int32_t nlists, const float* __restrict__ params,
                                                        int32_t* __restrict__ h_choice) {
  const int li = blockIdx.x;
  if (li >= nlists) return;
  choose_one(a.d[li], params, h_choice + li);
}

__global__ __launch_bounds__(64) void rz_choose_one_kernel(rz_list_desc d, const float* __restrict__ params,
                                                            int32_t* __restrict__ h_choice) {
  choose_one(d, params, h_choice);
}

// ---------------------------------------------------------------------------
// Gradient of the masked MSE loss sum_b sum_c m_bc (y_bc - t_bc)^2 / sum(m).
//
// Every layer is a 32-wide product, so one wave runs a tile of 32 samples on
// v_mfma_f32_32x32x2_f32 (FP32 inputs, FP32 accumulation): three forward
// products and the output layer, the two error products and the output
// layer's, and the four weight gradients d^T h, whose sum over the tile's
// samples is the product's K dimension.  A weight gradient stays in its 16
// accumulators over all tiles of the workgroup, so a workgroup writes one
// partial gradient (NP floats and its loss) whatever the batch, and
// rz_mlp_reduce_kernel adds the partials in a fixed order.
// Bound: latency (one wave's chain of about 140 products and 9 LDS
// transposes; 20 us while the parameters were loaded a few at a time).
// B = 4,000 on MI355X: 19 us (15 and 4) where one thread per sample writing a
// gradient of its own, summed by one thread per parameter over the B samples,
// took 1,156 us (71 and 1,085).  The sums are shorter, so the gradient is
// also closer to float64 (7e-8 of its norm, 9e-7 before).
// ---------------------------------------------------------------------------
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kGradTile = 32;         // samples of a tile: the product's 32 rows
constexpr int kGradMaxGroups = 256;   // partial gradients: one wave per CU, then every wave takes more tiles
constexpr int kGradPart = NP + 1;     // floats of a partial: the gradient, then the loss
static_assert(H == 32 && F <= 32 && F % 2 == 0 && C % 2 == 0 && C <= 32, "one 32x32 product per layer");

// C[m][n] += sum_k A[m][k] B[k][n], k < K, for one wave.  a(m, k) and b(k, n)
// read the operands; register r of lane l holds row 8 (r / 4) + 4 (l / 32) +
// r % 4, column l % 32.
template <int K, typename FA, typename FB>
__device__ __forceinline__ v16f mma32(v16f acc, FA a, FB b) {
  const int l = threadIdx.x & 31, half = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int s = 0; s < K; s += 2) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a(l, s + half), b(s + half, l), acc, 0, 0, 0);
  return acc;
}
__device__ __forceinline__ int acc_row(int r) { return 8 * (r >> 2) + 4 * ((threadIdx.x >> 5) & 1) + (r & 3); }
__device__ __forceinline__ v16f splat(float v) {
  v16f x;
#pragma unroll
  for (int r = 0; r < 16; ++r) x[r] = v;
  return x;
}

// rows of 33 words: a column read by 32 lanes hits 32 banks
struct GradShared {
  float P[NP];
  float x[kGradTile][33], h1[kGradTile][33], h2[kGradTile][33], h3[kGradTile][33];
  float dy[kGradTile][33], d[kGradTile][33];  // output errors (columns C and up zero), one layer's errors
};

__global__ __launch_bounds__(64) void rz_mlp_grad_kernel(const float* __restrict__ params, const float* __restrict__ X,
                                                          const float* __restrict__ T, const float* __restrict__ M,
                                                          int32_t B, float inv_msum, float* __restrict__ part) {
  __shared__ GradShared sh;
  const int tid = threadIdx.x, n = tid & 31;
  {
    constexpr int N = (NP + 63) / 64;
    float w[N];  // all loads in flight at once: one wave has no other to hide them
#pragma unroll
    for (int j = 0; j < N; ++j) w[j] = j * 64 + tid < NP ? params[j * 64 + tid] : 0.f;
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (j * 64 + tid < NP) sh.P[j * 64 + tid] = w[j];
  }
  for (int i = tid; i < kGradTile * 33; i += 64) (&sh.dy[0][0])[i] = (&sh.x[0][0])[i] = 0.f;
  __syncthreads();
  const float b1 = sh.P[OB1 + n], b2 = sh.P[OB2 + n], b3 = sh.P[OB3 + n], b4 = n < C ? sh.P[OB4 + n] : 0.f;
  v16f g1 = splat(0.f), g2 = g1, g3 = g1, g4 = g1;  // weight gradients [out][in]
  float s1 = 0.f, s2 = 0.f, s3 = 0.f, s4 = 0.f, loss = 0.f;  // bias gradients of unit n and the loss, over this lane's rows
  const int tiles = (B - 1) / kGradTile + 1;
  for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
    const int base = t * kGradTile, rows = B - base < kGradTile ? B - base : kGradTile;
    float xx[kGradTile * F / 64];
#pragma unroll
    for (int j = 0; j < kGradTile * F / 64; ++j) {
      const int i = j * 64 + tid;
      xx[j] = i < rows * F ? X[(size_t)base * F + i] : 0.f;
    }
    float tt[16], mm[16];  // targets and masks of column n, issued before the forward products
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = acc_row(r);
      tt[r] = mm[r] = 0.f;
      if (n < C && m < rows) {
        tt[r] = T[(size_t)(base + m) * C + n];
        mm[r] = M[(size_t)(base + m) * C + n];
      }
    }
#pragma unroll
    for (int j = 0; j < kGradTile * F / 64; ++j) sh.x[(j * 64 + tid) / F][(j * 64 + tid) % F] = xx[j];
    __syncthreads();
    // relu(a) into LDS; a row past the batch stays zero, so nothing of it reaches a sum over samples
    auto store_relu = [&](float(*h)[33], const v16f& a) {
#pragma unroll
      for (int r = 0; r < 16; ++r) h[acc_row(r)][n] = acc_row(r) < rows && a[r] > 0.f ? a[r] : 0.f;
      __syncthreads();
    };
    auto rows_of = [](const float(*h)[33]) { return [h](int m, int k) { return h[m][k]; }; };
    auto cols_of = [](const float(*h)[33]) { return [h](int m, int k) { return h[k][m]; }; };
    const float* P = sh.P;
    const v16f a1 = mma32<F>(splat(b1), rows_of(sh.x), [P](int k, int o) { return P[OW1 + o * F + k]; });
    store_relu(sh.h1, a1);
    const v16f a2 = mma32<H>(splat(b2), rows_of(sh.h1), [P](int k, int o) { return P[OW2 + o * H + k]; });
    store_relu(sh.h2, a2);
    const v16f a3 = mma32<H>(splat(b3), rows_of(sh.h2), [P](int k, int o) { return P[OW3 + o * H + k]; });
    store_relu(sh.h3, a3);
    const v16f y = mma32<H>(splat(b4), rows_of(sh.h3), [P](int k, int c) { return c < C ? P[OW4 + c * H + k] : 0.f; });
    if (n < C) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float e = y[r] - tt[r];
        const float dy = acc_row(r) < rows ? 2.f * mm[r] * e * inv_msum : 0.f;
        if (acc_row(r) < rows) loss += mm[r] * e * e;
        s4 += dy;
        sh.dy[acc_row(r)][n] = dy;
      }
    }
    __syncthreads();
    // errors of one layer: the product masked by its relu, into sh.d, and summed into the layer's bias gradient
    auto store_error = [&](const v16f& e, const v16f& a, float& s) {
      __syncthreads();  // the last readers of sh.d are done
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float v = acc_row(r) < rows && a[r] > 0.f ? e[r] : 0.f;
        s += v;
        sh.d[acc_row(r)][n] = v;
      }
      __syncthreads();
    };
    auto layer_in = [](const float(*h)[33]) { return [h](int k, int i) { return h[k][i]; }; };
    g4 = mma32<kGradTile>(g4, cols_of(sh.dy), layer_in(sh.h3));
    store_error(mma32<C>(splat(0.f), rows_of(sh.dy), [P](int c, int i) { return P[OW4 + c * H + i]; }), a3, s3);
    g3 = mma32<kGradTile>(g3, cols_of(sh.d), layer_in(sh.h2));
    store_error(mma32<H>(splat(0.f), rows_of(sh.d), [P](int o, int i) { return P[OW3 + o * H + i]; }), a2, s2);
    g2 = mma32<kGradTile>(g2, cols_of(sh.d), layer_in(sh.h1));
    store_error(mma32<H>(splat(0.f), rows_of(sh.d), [P](int o, int i) { return P[OW2 + o * H + i]; }), a1, s1);
    g1 = mma32<kGradTile>(g1, cols_of(sh.d), layer_in(sh.x));
    __syncthreads();  // sh.x and sh.dy may be written again
  }
  float* g = part + (size_t)blockIdx.x * kGradPart;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int o = acc_row(r);
    if (n < F) g[OW1 + o * F + n] = g1[r];
    g[OW2 + o * H + n] = g2[r];
    g[OW3 + o * H + n] = g3[r];
    if (o < C) g[OW4 + o * H + n] = g4[r];
  }
  // the two halves of the wave hold the other rows
  s1 += __shfl_xor(s1, 32);
  s2 += __shfl_xor(s2, 32);
  s3 += __shfl_xor(s3, 32);
  s4 += __shfl_xor(s4, 32);
  loss = wave_sum(loss);
  if (tid < 32) {
    g[OB1 + n] = s1;
    g[OB2 + n] = s2;
    g[OB3 + n] = s3;
    if (n < C) g[OB4 + n] = s4;
    if (n == 0) g[NP] = loss * inv_msum;
  }
}

// grad[p] = sum of the partials, loss likewise.  64 parameters per workgroup,
// wave w adds partials w, w + 16, ... (its loads in flight together), then
// one wave adds the 16 sums: a fixed order.
__global__ __launch_bounds__(1024) void rz_mlp_reduce_kernel(const float* __restrict__ part, int32_t groups,
                                                             float* __restrict__ grad, float* __restrict__ loss) {
  __shared__ float s_sum[16][64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, p = blockIdx.x * 64 + lane;
  float acc = 0.f;
  if (p < kGradPart) {
#pragma unroll 8
    for (int g = w; g < groups; g += 16) acc += part[(size_t)g * kGradPart + p];
  }
  s_sum[w][lane] = acc;
  __syncthreads();
  if (w == 0 && p < kGradPart) {
    acc = 0.f;
#pragma unroll
    for (int q = 0; q < 16; ++q) acc += s_sum[q][lane];
    if (p < NP) grad[p] = acc;
    else if (loss) *loss = acc;
  }
}

__global__ __launch_bounds__(256) void rz_mlp_adam_kernel(float* __restrict__ P, const float* __restrict__ g,
                                                           float* __restrict__ m, float* __restrict__ v, float lr,
                                                           float b1, float b2, float eps, float c1, float c2) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= NP) return;
  const float gi = g[p];
  const float mi = b1 * m[p] + (1.f - b1) * gi;
  const float vi = b2 * v[p] + (1.f - b2) * gi * gi;
  m[p] = mi;
  v[p] = vi;
  P[p] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

}  // namespace rz

using namespace rz;

extern "C" {

rz_status rz_features(rz_ctx* ctx, const rz_list_desc* d_lists, int32_t nlists, float* d_features, void* stream) {
  if (!ctx || nlists < 0 || (nlists > 0 && (!d_lists || !d_features))) return RZ_EINVAL;
  if (nlists == 0) return RZ_OK;
  hipLaunchKernelGGL(rz_features_kernel, dim3((uint32_t)nlists), dim3(64), 0, (hipStream_t)stream, d_lists, nlists,
                     d_features);
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

rz_status rz_mlp_forward(rz_ctx* ctx, const float* d_params, const float* d_x, int32_t batch, float* d_y,
                         int32_t* d_choice, void* stream) {
  if (!ctx || !d_params || !d_x || batch < 0) return RZ_EINVAL;
  if (batch == 0) return RZ_OK;
  hipLaunchKernelGGL(rz_mlp_forward_kernel, dim3((uint32_t)batch), dim3(64), 0, (hipStream_t)stream, d_params, d_x,
                     batch, d_y, d_choice);
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

rz_status rz_mlp_grad(rz_ctx* ctx, const float* d_params, const float* d_x, const float* d_target,
                      const float* d_mask, int32_t batch, float mask_sum, float* d_grad, float* d_loss,
                      float* d_work, void* stream) {
  if (!ctx || !d_params || !d_x || !d_target || !d_mask || !d_grad || !d_work || batch < 1 || !(mask_sum > 0.f))
    return RZ_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  // one partial gradient per workgroup; d_work holds one per sample, so it always fits
  const int32_t tiles = (batch - 1) / kGradTile + 1, groups = tiles < kGradMaxGroups ? tiles : kGradMaxGroups;
  hipLaunchKernelGGL(rz_mlp_grad_kernel, dim3((uint32_t)groups), dim3(64), 0, s, d_params, d_x, d_target, d_mask, batch,
                     1.f / mask_sum, d_work);
  hipLaunchKernelGGL(rz_mlp_reduce_kernel, dim3((kGradPart + 63) / 64), dim3(1024), 0, s, (const float*)d_work, groups,
                     d_grad, d_loss);
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

rz_status rz_mlp_adam(rz_ctx* ctx, float* d_params, const float* d_grad, float* d_m, float* d_v, int32_t step,
                      float lr, void* stream) {
  if (!ctx || !d_params || !d_grad || !d_m || !d_v || step < 1) return RZ_EINVAL;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(rz_mlp_adam_kernel, dim3((NP + 255) / 256), dim3(256), 0, (hipStream_t)stream, d_params, d_grad,
                     d_m, d_v, lr, b1, b2, eps, c1, c2);
  RZ_HIP(hipGetLastError());
  return RZ_OK;
}

rz_status rz_dispatch_method_config(int32_t method, uint32_t elem_bytes, rz_tile_config* out) {
  if (!out || esz_index(elem_bytes) < 0) return RZ_EINVAL;
  if (method == RZ_METHOD_ORDERED) {
    *out = rz_tile_config{256, 4, 4096, 3, 0, 1};
    return RZ_OK;
  }
  if (method == RZ_METHOD_DENSE) {
    // 16-byte items stage half as many entries per step (LDS)
    *out = rz_tile_config{1024, elem_bytes == 16 ? 4 : 8, 1024, 5, 11, 2};
    return RZ_OK;
  }
  return RZ_EINVAL;
}

rz_status rz_dispatch_set_params(rz_ctx* ctx, const float* h_params) {
  if (!ctx) return RZ_EINVAL;
  std::lock_guard<std::mutex> lock(ctx->mu);
  int prev = -1;
  (void)hipGetDevice(&prev);
  if (prev != ctx->device) (void)hipSetDevice(ctx->device);
  rz_status st = RZ_OK;
  if (!h_params) {
    ctx->dispatch_ready = false;
  } else if ((st = ensure(ctx, ctx->dispatch, (size_t)NP * 4, nullptr)) == RZ_OK) {
    if (hipMemcpy(ctx->dispatch.ptr, h_params, (size_t)NP * 4, hipMemcpyHostToDevice) != hipSuccess) st = RZ_EHIP;
    ctx->dispatch_ready = st == RZ_OK;
  }
  if (prev >= 0 && prev != ctx->device) (void)hipSetDevice(prev);
  return st;
}

// The network's choice for one list (stream-ordered, then read back).
static rz_status auto_choose(rz_ctx* ctx, void* d_data, int64_t n, uint32_t esz, int32_t* d_removals, int64_t k,
                             hipStream_t s, int32_t* method) {
  std::lock_guard<std::mutex> lock(ctx->mu);
  if (!ctx->dispatch_ready) {
    *method = 2 * k < n ? RZ_METHOD_REDZONE : RZ_METHOD_PARTITION;
    return RZ_OK;
  }
  int prev = -1;
  (void)hipGetDevice(&prev);
  if (prev != ctx->device) (void)hipSetDevice(ctx->device);
  rz_status st = RZ_OK;
  // mapped and coherent: the choice kernel stores into it directly
  if (!ctx->auto_host &&
      (hipHostMalloc((void**)&ctx->auto_host, 256, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess ||
       hipHostGetDevicePointer((void**)&ctx->auto_host_dev, ctx->auto_host, 0) != hipSuccess)) {
    if (ctx->auto_host) (void)hipHostFree(ctx->auto_host);
    ctx->auto_host = nullptr;
    st = RZ_ENOMEM;
  }
  if (st == RZ_OK) {
    // One launch (5.8 us): a descriptor upload, the two kernels and a copy back
    // took a call of 42 us 7 us more.
    volatile int32_t* hc = (volatile int32_t*)ctx->auto_host;
    *hc = -1;
    hipLaunchKernelGGL(rz_choose_one_kernel, dim3(1), dim3(64), 0, s, rz_list_desc{d_data, d_removals, n, k, esz, 0u},
                       (const float*)ctx->dispatch.ptr, (int32_t*)ctx->auto_host_dev);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) st = RZ_EHIP;
    const int32_t c = *hc;
    if (st == RZ_OK) *method = (c >= 0 && c < RZ_MLP_OUTPUTS) ? c : (2 * k < n ? 0 : 3);
  }
  if (prev >= 0 && prev != ctx->device) (void)hipSetDevice(prev);
  return st;
}

static int32_t rule_method(const rz_list_desc& d) {
  return 2 * d.k < d.n ? RZ_METHOD_REDZONE : RZ_METHOD_PARTITION;
}

static size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

rz_status rz_dispatch_choose(rz_ctx* ctx, const float* d_params, const rz_list_desc* h_lists, int32_t nlists,
                             void* stream) {
  if (!ctx || nlists < 0 || (nlists > 0 && !h_lists)) return RZ_EINVAL;
  for (int32_t i = 0; i < nlists; ++i) {
    const rz_list_desc& d = h_lists[i];
    if (d.n < 0 || d.k < 0 || d.k > d.n || esz_index(d.elem_bytes) < 0 || (d.k > 0 && !d.removals))
      return RZ_EINVAL;
  }
  std::lock_guard<std::mutex> lock(ctx->mu);
  DeviceGuard g(ctx->device);
  hipStream_t s = (hipStream_t)stream;
  // an uncollected choice still copying back must leave the staging area first
  if (ctx->choose_n >= 0 && ctx->choose_dev) RZ_HIP(hipEventSynchronize(ctx->choose_ev));
  ctx->choose_n = -1;
  const size_t dbytes = round256((size_t)nlists * sizeof(rz_list_desc));
  const size_t fbytes = round256((size_t)nlists * RZ_MLP_FEATURES * 4);
  const size_t cbytes = round256((size_t)nlists * 4 + 4);
  if (dbytes + cbytes > ctx->choose_host_bytes) {
    if (ctx->choose_host) RZ_HIP(hipHostFree(ctx->choose_host));
    ctx->choose_host = ctx->choose_host_dev = nullptr;
    ctx->choose_host_bytes = 0;
    size_t cap = 4096;
    while (cap < dbytes + cbytes) cap *= 2;
    // mapped and coherent: the choice kernel stores into it directly
    if (hipHostMalloc((void**)&ctx->choose_host, cap, hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess) {
      ctx->choose_host = nullptr;
      return RZ_ENOMEM;
    }
    if (hipHostGetDevicePointer((void**)&ctx->choose_host_dev, ctx->choose_host, 0) != hipSuccess) {
      (void)hipHostFree(ctx->choose_host);
      ctx->choose_host = ctx->choose_host_dev = nullptr;
      return RZ_EHIP;
    }
    ctx->choose_host_bytes = cap;
  }
  if (nlists) memcpy(ctx->choose_host, h_lists, (size_t)nlists * sizeof(rz_list_desc));
  const float* params = d_params ? d_params : (ctx->dispatch_ready ? (const float*)ctx->dispatch.ptr : nullptr);
  if (!params || nlists == 0) {  // no network: the rule, on the host, at collection
    ctx->choose_dev = false;
    ctx->choose_n = nlists;
    return RZ_OK;
  }
  if (!ctx->choose_ev) RZ_HIP(hipEventCreateWithFlags(&ctx->choose_ev, hipEventDisableTiming));
  if (nlists <= kChooseArgMax) {  // one launch, no copies
    ChooseArgs a;
    memcpy(a.d, h_lists, (size_t)nlists * sizeof(rz_list_desc));
    hipLaunchKernelGGL(rz_choose_kernel, dim3((uint32_t)nlists), dim3(64), 0, s, a, nlists, params,
                       (int32_t*)(ctx->choose_host_dev + dbytes));
    RZ_HIP(hipGetLastError());
    RZ_HIP(hipEventRecord(ctx->choose_ev, s));
    ctx->choose_dev = true;
    ctx->choose_n = nlists;
    return RZ_OK;
  }
  rz_status st;
  if ((st = ensure(ctx, ctx->choose, dbytes + fbytes + cbytes, s)) != RZ_OK) return st;
  char* base = (char*)ctx->choose.ptr;
  RZ_HIP(hipMemcpyAsync(base, ctx->choose_host, (size_t)nlists * sizeof(rz_list_desc), hipMemcpyHostToDevice, s));
  if ((st = rz_features(ctx, (const rz_list_desc*)base, nlists, (float*)(base + dbytes), s)) != RZ_OK) return st;
  if ((st = rz_mlp_forward(ctx, params, (const float*)(base + dbytes), nlists, nullptr,
                           (int32_t*)(base + dbytes + fbytes), s)) != RZ_OK)
    return st;
  RZ_HIP(hipMemcpyAsync(ctx->choose_host + dbytes, base + dbytes + fbytes, (size_t)nlists * 4, hipMemcpyDeviceToHost,
                        s));
  RZ_HIP(hipEventRecord(ctx->choose_ev, s));
  ctx->choose_dev = true;
  ctx->choose_n = nlists;
  return RZ_OK;
}

rz_status rz_dispatch_collect(rz_ctx* ctx, int32_t* h_choice, int32_t nlists) {
  if (!ctx || nlists < 0 || (nlists > 0 && !h_choice)) return RZ_EINVAL;
  std::lock_guard<std::mutex> lock(ctx->mu);
  if (ctx->choose_n < 0 || ctx->choose_n != nlists) return RZ_EINVAL;
  DeviceGuard g(ctx->device);
  if (ctx->choose_dev) RZ_HIP(hipEventSynchronize(ctx->choose_ev));
  const rz_list_desc* hd = (const rz_list_desc*)ctx->choose_host;
  const int32_t* hc = (const int32_t*)(ctx->choose_host + round256((size_t)nlists * sizeof(rz_list_desc)));
  for (int32_t i = 0; i < nlists; ++i) {
    const rz_list_desc& d = hd[i];
    int32_t m = ctx->choose_dev ? hc[i] : rule_method(d);
    if (m < 0 || m >= RZ_MLP_OUTPUTS) m = rule_method(d);
    if (d.k == 0 || d.k == d.n) m = RZ_METHOD_REDZONE;  // nothing to choose: no items move
    h_choice[i] = m;
  }
  ctx->choose_n = -1;
  return RZ_OK;
}

rz_status rz_remove_auto_batched(rz_ctx* ctx, const float* d_params, const rz_list_desc* lists, int32_t nlists,
                                 int64_t batch_max_k, uint32_t flags, int32_t* methods, void* stream) {
  if (!ctx || nlists < 0 || (nlists > 0 && !lists) || nlists >= (1 << 28) || batch_max_k < 0) return RZ_EINVAL;
  std::vector<rz_list_desc> small, large;
  std::vector<int32_t> large_idx;
  small.reserve((size_t)nlists);
  for (int32_t i = 0; i < nlists; ++i) {
    rz_list_desc d = lists[i];
    d.method = 0;
    if (d.k < batch_max_k) {
      small.push_back(d);
    } else {
      large.push_back(d);
      large_idx.push_back(i);
    }
    if (methods) methods[i] = RZ_METHOD_REDZONE;
  }
  rz_status st;
  const int32_t nl = (int32_t)large.size();
  // the choice first: the device computes it while the batch below is planned
  if (nl && (st = rz_dispatch_choose(ctx, d_params, large.data(), nl, stream)) != RZ_OK) return st;
  if (!small.empty() && (st = rz_remove_batched(ctx, small.data(), (int32_t)small.size(), flags, stream)) != RZ_OK)
    return st;
  if (!nl) return RZ_OK;
  std::vector<int32_t> m((size_t)nl);
  if ((st = rz_dispatch_collect(ctx, m.data(), nl)) != RZ_OK) return st;
  for (int32_t j = 0; j < nl; ++j) {  // queued behind the batch on the stream
    const rz_list_desc& d = large[(size_t)j];
    if (m[j] == RZ_METHOD_PARTITION) {
      st = rz_partition_on(ctx, d.data, d.n, d.elem_bytes, d.removals, d.k, flags, stream);
    } else if (m[j] == RZ_METHOD_REDZONE) {
      st = rz_remove(ctx, d.data, d.n, d.elem_bytes, d.removals, d.k, flags, stream);
    } else {
      rz_tile_config cfg;
      if ((st = rz_dispatch_method_config(m[j], d.elem_bytes, &cfg)) == RZ_OK)
        st = rz_remove_config(ctx, d.data, d.n, d.elem_bytes, d.removals, d.k, flags, &cfg, stream);
    }
    if (st != RZ_OK) return st;
    if (methods) methods[large_idx[(size_t)j]] = m[j];
  }
  return RZ_OK;
}

rz_status rz_remove_auto(rz_ctx* ctx, void* d_data, int64_t n, uint32_t elem_bytes, int32_t* d_removals, int64_t k,
                         uint32_t flags, int32_t* method, void* stream) {
  if (!ctx || n < 0 || k < 0 || k > n || esz_index(elem_bytes) < 0) return RZ_EINVAL;
  if (k > 0 && (!d_data || !d_removals)) return RZ_EINVAL;
  int32_t m = RZ_METHOD_REDZONE;
  rz_status st = RZ_OK;
  if (k > 0 && k < n) st = auto_choose(ctx, d_data, n, elem_bytes, d_removals, k, (hipStream_t)stream, &m);
  if (st != RZ_OK) return st;
  if (method) *method = m;
  if (m == RZ_METHOD_PARTITION) return rz_partition_on(ctx, d_data, n, elem_bytes, d_removals, k, flags, stream);
  if (m == RZ_METHOD_REDZONE) return rz_remove(ctx, d_data, n, elem_bytes, d_removals, k, flags, stream);
  rz_tile_config cfg;
  if ((st = rz_dispatch_method_config(m, elem_bytes, &cfg)) != RZ_OK) return st;
  return rz_remove_config(ctx, d_data, n, elem_bytes, d_removals, k, flags, &cfg, stream);
}

}  // extern "C"
