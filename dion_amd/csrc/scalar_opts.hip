// Multi-tensor AdamW and Lion steps for the non-matrix parameter groups (embeddings, heads, norms,
// biases) of a model whose matrices are updated by Muon / NorMuon / Dion2 / NorDion2.
//
// One launch updates up to kMtaTensors tensors of different sizes: their pointers and element
// counts travel by value in the kernel-argument segment, each workgroup owns one run of consecutive elements of one
// tensor: kMtaChunk of them (the tensor found by bisection in a table of first workgroups, a thread with the loads
// of sixteen elements in flight at once), or in small launches a short run (mta_run; BRIEF).  All traffic is HBM streaming: AdamW reads X, G, M, V
// and writes X, M, V (28 B/element with fp32 state and gradients, 26 with bf16 gradients), Lion 20 / 18
// B/element.  The state tensors X, M, V of one launch share a dtype, fp32 or bf16 (half the bytes);
// arithmetic is fp32 either way.
// Bound by HBM.  2 x (50304 x 768) + norms, fp32 state, bf16 gradients: AdamW 580 us (3.5 TB/s) with a grid row per
// tensor and one group of four elements in flight -> 394 us (5.1 TB/s) -> 356 us (5.65 TB/s) with non-temporal accesses;
// Lion 295 -> 234 us (5.9 TB/s).  Device copy on the same card: 5.2-6.1 TB/s.
//
// Arithmetic follows dion/scalar_opts.py:7-65 (adamw_update) and :68-118 (lion_update); the step
// counters are device scalars advanced on the device, like the capturable form of
// adamw_update_foreach (dion/scalar_opts.py:196-213), and lr / weight decay are read from device
// scalars, so a captured step sees live values.
#include "elementwise.h"

namespace dion {

struct MtaTensors {
  uint64_t x[kMtaTensors], g[kMtaTensors], m[kMtaTensors], v[kMtaTensors], step[kMtaTensors];
  int64_t numel[kMtaTensors];
  unsigned wg0[kMtaTensors + 1];  // first workgroup of each tensor; wg0[n] = workgroups of the launch
  int run;                        // elements per workgroup (mta_run)
};

// Elements one workgroup updates: two rounds of 256 threads x kMtaGroups groups of four.
constexpr int kMtaGroups = 4;
constexpr int kMtaRound = 256 * 4 * kMtaGroups;
constexpr int kMtaChunk = 2 * kMtaRound;

// The tensor workgroup `wg` belongs to (wg0 ascending, wg0[n] > wg).
static __device__ __forceinline__ int mta_tensor(const MtaTensors& a, int n, unsigned wg) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (a.wg0[mid] <= wg) lo = mid;
    else hi = mid;
  }
  return lo;
}

// step[t] += 1 for every tensor of the launch (before the update kernel reads them).
__global__ void mta_advance_steps_kernel(MtaTensors a, int n) {
  const int t = threadIdx.x;
  const uint64_t mine = t < n ? a.step[t] : 0;
  // the same counter may serve several tensors: advance each distinct one once
  bool first = t < n;
  for (int u = 0; u + 1 < n; ++u) first = first && (u >= t || a.step[u] != mine);
  if (first) *(float*)mine = *(float*)mine + 1.0f;
}

struct AdamwScalars {
  float beta1, beta2, eps, wd_host;
  int cautious;
};

template <typename GT>
static __device__ __forceinline__ void adamw_one(float& x, float g, float& m, float& v, float w1,
                                                 float beta2, float w2, float inv_bc2_sqrt, float eps,
                                                 float adj_lr, float a, float coeff, int cautious) {
  m = m + w1 * (g - m);                 // lerp(M, G, 1 - beta1)
  v = v * beta2 + w2 * (g * g);         // V * beta2 + (1 - beta2) * G * G
  const float denom = sqrtf(v) * inv_bc2_sqrt + eps;
  const float upd = m / denom;
  if (cautious) {
    if (upd * x >= 0.0f) x = x - x * coeff;
  } else {
    x = x * a;
  }
  x = x - adj_lr * upd;
}

template <typename GT, typename ST, bool NT, bool BRIEF = false>
__global__ __launch_bounds__(256) void adamw_mt_kernel(MtaTensors a, int n, const float* __restrict__ lr_dev,
                                                       const float* __restrict__ wd_dev,
                                                       AdamwScalars sc) {
  const int t = BRIEF ? blockIdx.y : mta_tensor(a, n, blockIdx.x);
  const int64_t first = (int64_t)(blockIdx.x - (BRIEF ? 0 : a.wg0[t])) * a.run;
  if (BRIEF && first >= a.numel[t]) return;
  const int64_t end = a.numel[t] < first + a.run ? a.numel[t] : first + a.run;
  ST* __restrict__ x = (ST*)a.x[t];
  const GT* __restrict__ g = (const GT*)a.g[t];
  ST* __restrict__ m = (ST*)a.m[t];
  ST* __restrict__ v = (ST*)a.v[t];
  // groups of 4 elements: 16-byte accesses to fp32 tensors, 8-byte accesses to bf16 ones
  const bool vec = (((a.x[t] | a.m[t] | a.v[t]) & (sizeof(ST) == 2 ? 7 : 15)) == 0) &&
                   ((a.g[t] & (sizeof(GT) == 2 ? 7 : 15)) == 0);
  float w1, w2, inv_bc2_sqrt, adj_lr, coeff, aa;
  auto scalars = [&]() {
    const float step = *(const float*)a.step[t];
    const float lr = *lr_dev;
    const float wd = wd_dev ? *wd_dev : sc.wd_host;
    const float bc1 = 1.0f - powf(sc.beta1, step);
    const float bc2 = 1.0f - powf(sc.beta2, step);
    inv_bc2_sqrt = 1.0f / sqrtf(bc2);
    adj_lr = lr / bc1;
    coeff = lr * wd;
    aa = 1.0f - coeff;
    w1 = 1.0f - sc.beta1;
    w2 = 1.0f - sc.beta2;
  };
  if (!BRIEF && vec && end - first == kMtaChunk) {
    float xv[kMtaGroups][4], mv[kMtaGroups][4], vv[kMtaGroups][4], gv[kMtaGroups][4];
#pragma unroll 1
    for (int r = 0; r < 2; ++r) {
      const int64_t q0 = (first + r * kMtaRound) / 4 + threadIdx.x;
#pragma unroll
      for (int u = 0; u < kMtaGroups; ++u) {
        st_load4<ST, NT>(x, q0 + u * 256, xv[u]);
        st_load4<ST, NT>(m, q0 + u * 256, mv[u]);
        st_load4<ST, NT>(v, q0 + u * 256, vv[u]);
        st_load4<GT, NT>(g, q0 + u * 256, gv[u]);
      }
      if (r == 0) scalars();  // two powers: under the first loads
#pragma unroll
      for (int u = 0; u < kMtaGroups; ++u) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          adamw_one<GT>(xv[u][e], gv[u][e], mv[u][e], vv[u][e], w1, sc.beta2, w2, inv_bc2_sqrt, sc.eps, adj_lr, aa,
                        coeff, sc.cautious);
        st_store4<ST, NT>(x, q0 + u * 256, xv[u]);
        st_store4<ST, NT>(m, q0 + u * 256, mv[u]);
        st_store4<ST, NT>(v, q0 + u * 256, vv[u]);
      }
    }
    return;
  }
  // short runs, the last run of a tensor, and tensors that are not aligned
  const int64_t vend = vec ? end & ~(int64_t)3 : first;
  int64_t q = first / 4 + threadIdx.x;
  float xv[4], mv[4], vv[4], gv[4];
  auto load = [&]() {
    if (q >= vend / 4) return;
    st_load4<ST>(x, q, xv);
    st_load4<ST>(m, q, mv);
    st_load4<ST>(v, q, vv);
    st_load4<GT>(g, q, gv);
  };
  load();
  scalars();
  for (; q < vend / 4; q += 256, load()) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      adamw_one<GT>(xv[e], gv[e], mv[e], vv[e], w1, sc.beta2, w2, inv_bc2_sqrt, sc.eps, adj_lr, aa, coeff,
                    sc.cautious);
    st_store4<ST>(x, q, xv);
    st_store4<ST>(m, q, mv);
    st_store4<ST>(v, q, vv);
  }
  for (int64_t i = vend + threadIdx.x; i < end; i += 256) {
    float xs = st_load<ST>(x, i), ms = st_load<ST>(m, i), vs = st_load<ST>(v, i);
    adamw_one<GT>(xs, st_load<GT>(g, i), ms, vs, w1, sc.beta2, w2, inv_bc2_sqrt, sc.eps, adj_lr, aa, coeff,
                  sc.cautious);
    st_store<ST>(x, i, xs);
    st_store<ST>(m, i, ms);
    st_store<ST>(v, i, vs);
  }
}

static __device__ __forceinline__ void lion_one(float& x, float g, float& m, float w1, float w2, float lr,
                                                float a, float coeff, int cautious) {
  const float c = m + w1 * (g - m);  // lerp(M, G, 1 - beta1)
  const float u = c > 0.0f ? 1.0f : (c < 0.0f ? -1.0f : 0.0f);
  m = m + w2 * (g - m);              // lerp(M, G, 1 - beta2)
  if (cautious) {
    if (u * x >= 0.0f) x = x - x * coeff;
  } else {
    x = x * a;
  }
  x = x - lr * u;
}

template <typename GT, typename ST, bool NT, bool BRIEF = false>
__global__ __launch_bounds__(256) void lion_mt_kernel(MtaTensors a, int n, const float* __restrict__ lr_dev,
                                                      const float* __restrict__ wd_dev, float beta1,
                                                      float beta2, float wd_host, int cautious) {
  const int t = BRIEF ? blockIdx.y : mta_tensor(a, n, blockIdx.x);
  const int64_t first = (int64_t)(blockIdx.x - (BRIEF ? 0 : a.wg0[t])) * a.run;
  if (BRIEF && first >= a.numel[t]) return;
  const int64_t end = a.numel[t] < first + a.run ? a.numel[t] : first + a.run;
  ST* __restrict__ x = (ST*)a.x[t];
  const GT* __restrict__ g = (const GT*)a.g[t];
  ST* __restrict__ m = (ST*)a.m[t];
  const float lr = *lr_dev;
  const float wd = wd_dev ? *wd_dev : wd_host;
  const float coeff = lr * wd;
  const float aa = 1.0f - coeff;
  const float w1 = 1.0f - beta1, w2 = 1.0f - beta2;
  const bool vec = (((a.x[t] | a.m[t]) & (sizeof(ST) == 2 ? 7 : 15)) == 0) &&
                   ((a.g[t] & (sizeof(GT) == 2 ? 7 : 15)) == 0);
  if (!BRIEF && vec && end - first == kMtaChunk) {
    float xv[kMtaGroups][4], mv[kMtaGroups][4], gv[kMtaGroups][4];
#pragma unroll 1
    for (int r = 0; r < 2; ++r) {
      const int64_t q0 = (first + r * kMtaRound) / 4 + threadIdx.x;
#pragma unroll
      for (int u = 0; u < kMtaGroups; ++u) {
        st_load4<ST, NT>(x, q0 + u * 256, xv[u]);
        st_load4<ST, NT>(m, q0 + u * 256, mv[u]);
        st_load4<GT, NT>(g, q0 + u * 256, gv[u]);
      }
#pragma unroll
      for (int u = 0; u < kMtaGroups; ++u) {
#pragma unroll
        for (int e = 0; e < 4; ++e) lion_one(xv[u][e], gv[u][e], mv[u][e], w1, w2, lr, aa, coeff, cautious);
        st_store4<ST, NT>(x, q0 + u * 256, xv[u]);
        st_store4<ST, NT>(m, q0 + u * 256, mv[u]);
      }
    }
    return;
  }
  const int64_t vend = vec ? end & ~(int64_t)3 : first;
  for (int64_t q = first / 4 + threadIdx.x; q < vend / 4; q += 256) {
    float xv[4], mv[4], gv[4];
    st_load4<ST>(x, q, xv);
    st_load4<ST>(m, q, mv);
    st_load4<GT>(g, q, gv);
#pragma unroll
    for (int e = 0; e < 4; ++e) lion_one(xv[e], gv[e], mv[e], w1, w2, lr, aa, coeff, cautious);
    st_store4<ST>(x, q, xv);
    st_store4<ST>(m, q, mv);
  }
  for (int64_t i = vend + threadIdx.x; i < end; i += 256) {
    float xs = st_load<ST>(x, i), ms = st_load<ST>(m, i);
    lion_one(xs, st_load<GT>(g, i), ms, w1, w2, lr, aa, coeff, cautious);
    st_store<ST>(x, i, xs);
    st_store<ST>(m, i, ms);
  }
}

static bool past_caches(const int64_t* numel, int n, int bytes_per_element) {
  int64_t total = 0;
  for (int i = 0; i < n; ++i) total += numel[i];
  return exceeds_caches(total * bytes_per_element);
}

// Elements per workgroup.  A launch of up to 5 M elements does not fill the chip with runs of kMtaChunk: it takes short ones, a
// grid row per tensor, from a kernel of half the registers.  fp32 state, bf16 gradients, runs of 1024 / 2048 / 8192
// elements, us, AdamW: 49 x 2048 14.3 / 15.9 / 15.7, 60 x 5000 15.9 / 17.6 / 22.0, 1 M in one tensor 8.4 / 8.2 / 10.9, 4 M 22.5 /
// 20.8 / 21.9, 6 M 29.9 / 29.2 / 27.8, 38.6 M 191 / 196 / 174; Lion: 60 x 5000 4.5 / 5.4 / 8.3, 4 M 13.0 / 12.5 / 12.6,
// 38.6 M 121 / 126 / 128.
static int mta_run(int64_t total) { return total < (1 << 20) ? 1024 : total < (5 << 20) ? 2048 : kMtaChunk; }

// false: more workgroups than one launch can have
static bool fill(MtaTensors& a, const uint64_t* X, const uint64_t* G, const uint64_t* M, const uint64_t* V,
                 const uint64_t* S, const int64_t* numel, int n) {
  for (int i = 0; i < kMtaTensors; ++i) {
    const int j = i < n ? i : 0;
    a.x[i] = X[j];
    a.g[i] = G[j];
    a.m[i] = M[j];
    a.v[i] = V ? V[j] : 0;
    a.step[i] = S ? S[j] : 0;
    a.numel[i] = i < n ? numel[j] : 0;
  }
  int64_t wg = 0, total = 0;
  for (int i = 0; i < n; ++i) total += numel[i];
  a.run = mta_run(total);
  for (int i = 0; i <= kMtaTensors; ++i) {
    a.wg0[i] = (unsigned)wg;
    if (i < n) wg += (numel[i] + a.run - 1) / a.run;
    if (wg > 0x7fffffff) return false;
  }
  return true;
}

// a grid row per tensor where the runs are short
static dim3 mta_grid(const MtaTensors& a, const int64_t* numel, int n) {
  if (a.run == kMtaChunk) return dim3(a.wg0[n]);
  int64_t longest = 0;
  for (int i = 0; i < n; ++i) longest = numel[i] > longest ? numel[i] : longest;
  return dim3((unsigned)((longest + a.run - 1) / a.run), n);
}

hipError_t launch_adamw_mt(const uint64_t* X, const uint64_t* G, int g_dtype, const uint64_t* M,
                           const uint64_t* V, int s_dtype, const uint64_t* steps, const int64_t* numel, int n,
                           const float* lr_dev, float beta1, float beta2, float eps, const float* wd_dev,
                           float wd_host, int cautious, hipStream_t st) {
  MtaTensors a;
  if (!fill(a, X, G, M, V, steps, numel, n)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(mta_advance_steps_kernel, dim3(1), dim3(64), 0, st, a, n);
  if (a.wg0[n] == 0) return hipGetLastError();
  const bool nt = past_caches(numel, n, 3 * (s_dtype == 0 ? 2 : 4) + (g_dtype == 0 ? 2 : 4));
  AdamwScalars sc{beta1, beta2, eps, wd_host, cautious};
  const dim3 grid = mta_grid(a, numel, n);
#define ADAMW_LAUNCH(GT, ST)                                                                                       \
  do {                                                                                                             \
    if (a.run != kMtaChunk)                                                                                        \
      hipLaunchKernelGGL((adamw_mt_kernel<GT, ST, false, true>), grid, dim3(256), 0, st, a, n, lr_dev, wd_dev, sc); \
    else if (nt) hipLaunchKernelGGL((adamw_mt_kernel<GT, ST, true>), grid, dim3(256), 0, st, a, n, lr_dev, wd_dev, sc); \
    else hipLaunchKernelGGL((adamw_mt_kernel<GT, ST, false>), grid, dim3(256), 0, st, a, n, lr_dev, wd_dev, sc);   \
  } while (0)
  if (g_dtype == 0) {
    if (s_dtype == 0) ADAMW_LAUNCH(bf16_t, bf16_t); else ADAMW_LAUNCH(bf16_t, float);
  } else {
    if (s_dtype == 0) ADAMW_LAUNCH(float, bf16_t); else ADAMW_LAUNCH(float, float);
  }
#undef ADAMW_LAUNCH
  return hipGetLastError();
}

hipError_t launch_lion_mt(const uint64_t* X, const uint64_t* G, int g_dtype, const uint64_t* M, int s_dtype,
                          const int64_t* numel, int n, const float* lr_dev, float beta1, float beta2,
                          const float* wd_dev, float wd_host, int cautious, hipStream_t st) {
  MtaTensors a;
  if (!fill(a, X, G, M, nullptr, nullptr, numel, n)) return hipErrorInvalidValue;
  if (a.wg0[n] == 0) return hipSuccess;
  const dim3 grid = mta_grid(a, numel, n);
  const bool nt = past_caches(numel, n, 2 * (s_dtype == 0 ? 2 : 4) + (g_dtype == 0 ? 2 : 4));
#define LION_LAUNCH(GT, ST)                                                                                \
  do {                                                                                                     \
    if (a.run != kMtaChunk)                                                                                \
      hipLaunchKernelGGL((lion_mt_kernel<GT, ST, false, true>), grid, dim3(256), 0, st, a, n, lr_dev, wd_dev, \
                         beta1, beta2, wd_host, cautious);                                                 \
    else if (nt) hipLaunchKernelGGL((lion_mt_kernel<GT, ST, true>), grid, dim3(256), 0, st, a, n, lr_dev, wd_dev, \
                               beta1, beta2, wd_host, cautious);                                           \
    else hipLaunchKernelGGL((lion_mt_kernel<GT, ST, false>), grid, dim3(256), 0, st, a, n, lr_dev, wd_dev, \
                            beta1, beta2, wd_host, cautious);                                              \
  } while (0)
  if (g_dtype == 0) {
    if (s_dtype == 0) LION_LAUNCH(bf16_t, bf16_t); else LION_LAUNCH(bf16_t, float);
  } else {
    if (s_dtype == 0) LION_LAUNCH(float, bf16_t); else LION_LAUNCH(float, float);
  }
#undef LION_LAUNCH
  return hipGetLastError();
}

}  // namespace dion
