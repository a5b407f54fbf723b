// Memory-bound kernels of the Muon / NorMuon / Dion2 step for gfx950: everything around the
// Newton-Schulz GEMMs.  All of them are single-pass over their big operands, use 16-byte
// per-lane accesses where alignment allows, and reduce in a fixed order (no float atomics) so a
// step is bit-reproducible run to run.
#include "elementwise.h"

namespace dion {

static __device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Block-wide sum in a fixed order; result valid in every thread.  red: >= 16 floats of LDS.
static __device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  float s = 0.f;
  for (int i = 0; i < nw; ++i) s += red[i];
  return s;
}

template <typename T>
static __device__ __forceinline__ float load_as_bf16_f32(const T* p, int64_t i);
template <>
__device__ __forceinline__ float load_as_bf16_f32<bf16_t>(const bf16_t* p, int64_t i) {
  return bf16_to_f32(p[i]);
}
template <>
__device__ __forceinline__ float load_as_bf16_f32<float>(const float* p, int64_t i) {
  return bf16_to_f32(f32_to_bf16(p[i]));
}

// ------------------------------------------------------------------------------------------
// Frobenius pre-normalisation:  partial sums of squares of bf16(in), then 1/(||.||*s + eps).
// ------------------------------------------------------------------------------------------
// 8 consecutive elements of `p` (16-byte aligned chunk index i) as bf16-rounded floats.
template <typename T>
static __device__ __forceinline__ void load8_as_bf16(const T* p, int64_t i, float v[8]) {
  if (sizeof(T) == 2) {
    const uint4 raw = ((const uint4*)p)[i];
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[2 * e] = __uint_as_float(w[e] << 16);
      v[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
    }
  } else {
    const float4 a = ((const float4*)p)[2 * i], c = ((const float4*)p)[2 * i + 1];
    const float f[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = bf16_to_f32(f32_to_bf16(f[e]));
  }
}

template <typename T, bool VEC>
__global__ __launch_bounds__(256) void sumsq_partial_kernel(const T* __restrict__ in, int64_t numel,
                                                            int nblk, float* __restrict__ partial) {
  __shared__ float red[16];
  const int b = blockIdx.y;
  const T* src = in + (int64_t)b * numel;
  float s = 0.f;
  if (VEC) {
    const int64_t nv = numel >> 3;
    const int64_t per = (nv + nblk - 1) / nblk;
    const int64_t lo = (int64_t)blockIdx.x * per;
    int64_t hi = lo + per;
    if (hi > nv) hi = nv;
    for (int64_t i = lo + threadIdx.x; i < hi; i += 256) {
      float v[8];
      load8_as_bf16<T>(src, i, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) s += v[e] * v[e];
    }
  } else {
    const int64_t per = (numel + nblk - 1) / nblk;
    const int64_t lo = (int64_t)blockIdx.x * per;
    int64_t hi = lo + per;
    if (hi > numel) hi = numel;
    for (int64_t i = lo + threadIdx.x; i < hi; i += 256) {
      const float v = load_as_bf16_f32<T>(src, i);
      s += v * v;
    }
  }
  s = block_sum(s, red);
  if (threadIdx.x == 0) partial[(int64_t)b * nblk + blockIdx.x] = s;
}

__global__ __launch_bounds__(256) void norm_finalize_kernel(const float* __restrict__ partial, int nblk,
                                                            float norm_scale, float eps,
                                                            float* __restrict__ inv_norm, bf16_t* __restrict__ X,
                                                            int64_t elems) {
  // Fixed summation order: thread t adds partials t, t + 256, ... (four independent running sums,
  // so four loads are in flight), then the block sum.
  __shared__ float red[16];
  const int b = blockIdx.x;
  const float* src = partial + (int64_t)b * nblk;
  float s4[4] = {0.f, 0.f, 0.f, 0.f};
  int i = threadIdx.x;
  for (; i + 3 * 256 < nblk; i += 4 * 256) {
#pragma unroll
    for (int j = 0; j < 4; ++j) s4[j] += src[i + j * 256];
  }
  for (int j = 0; i < nblk; i += 256, ++j) s4[j] += src[i];
  const float s = block_sum((s4[0] + s4[1]) + (s4[2] + s4[3]), red);
  float inv = 1.0f / (sqrtf(s) * norm_scale + eps);
  // X (may be null): the matrices as they came, whose products the factor is applied to.  Where sums of such products, or
  // the factor's square, would leave the normal range of fp32, the matrix is scaled here instead (an overflown norm, a factor
  // of 0, leaves zeros; one value that is not finite, NaN).
  if (X && s != 0.f && !(s > 0x1p-80f && s < 0x1p80f)) {
    bf16_t* x = X + (int64_t)b * elems;
    for (int64_t i8 = threadIdx.x; i8 < elems / 8; i8 += 256) {
      float v[8];
      st_load8<bf16_t>(x, i8, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= inv;
      st_store8<bf16_t>(x, i8, v);
    }
    inv = 1.0f;
  }
  if (threadIdx.x == 0) inv_norm[b] = inv;
}

// in [B,R,C] -> same [B,Rp,Cp] (scaled, zero padded) and trans [B,Cp,Rp] = same^T, both bf16.
// 64x64 tiles through LDS so both stores are row-contiguous.
template <typename T>
__global__ __launch_bounds__(256) void ns_prepare_kernel(const T* __restrict__ in, int R, int C,
                                                         const float* __restrict__ inv_norm,
                                                         bf16_t* __restrict__ same, int Rp, int Cp,
                                                         int ld_same, int64_t stride_same,
                                                         bf16_t* __restrict__ trans, int ld_trans,
                                                         int64_t stride_trans) {
  __shared__ bf16_t tile[64][66];
  const int b = blockIdx.z;
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const float sc = inv_norm ? inv_norm[b] : 1.0f;  // (no factor: the values are copied as they are)
  const T* src = in + (int64_t)b * R * C;
  bf16_t* ds = same + (int64_t)b * stride_same;
  bf16_t* dt = trans + (int64_t)b * stride_trans;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll 4
  for (int i = ty; i < 64; i += 4) {
    const int r = r0 + i, c = c0 + tx;
    bf16_t v = 0;
    if (r < R && c < C) v = f32_to_bf16(load_as_bf16_f32<T>(src, (int64_t)r * C + c) * sc);
    tile[i][tx] = v;
    if (same) ds[(int64_t)r * ld_same + c] = v;
  }
  __syncthreads();
  if (!trans) return;
#pragma unroll 4
  for (int i = ty; i < 64; i += 4) {
    // trans row (c0 + i), column (r0 + tx)
    dt[(int64_t)(c0 + i) * ld_trans + r0 + tx] = tile[tx][i];
  }
}

// Same operation (either output may be null), 16-byte accesses: needs C % 8 == 0, 16-byte aligned input and row pitches.
template <typename T>
__global__ __launch_bounds__(256) void ns_prepare_vec_kernel(const T* __restrict__ in, int R, int C,
                                                             const float* __restrict__ inv_norm,
                                                             bf16_t* __restrict__ same, int ld_same,
                                                             int64_t stride_same,
                                                             bf16_t* __restrict__ trans, int ld_trans,
                                                             int64_t stride_trans) {
  __shared__ __attribute__((aligned(16))) bf16_t tile[64][72];
  const int b = blockIdx.z;
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const float sc = inv_norm ? inv_norm[b] : 1.0f;  // (no factor: the values are copied as they are)
  const T* src = in + (int64_t)b * R * C;
  bf16_t* ds = same + (int64_t)b * stride_same;
  bf16_t* dt = trans + (int64_t)b * stride_trans;
  const int chunk = threadIdx.x & 7, rr = threadIdx.x >> 3;  // 8 chunks x 32 rows per pass
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int i = rr + pass * 32;
    const int r = r0 + i, c = c0 + chunk * 8;
    uint4 o = make_uint4(0, 0, 0, 0);
    if (r < R && c < C) {
      float v[8];
      load8_as_bf16<T>(src, ((int64_t)r * C + c) >> 3, v);
      o.x = pack_bf16x2(v[0] * sc, v[1] * sc);
      o.y = pack_bf16x2(v[2] * sc, v[3] * sc);
      o.z = pack_bf16x2(v[4] * sc, v[5] * sc);
      o.w = pack_bf16x2(v[6] * sc, v[7] * sc);
    }
    *(uint4*)&tile[i][chunk * 8] = o;
    if (same) *(uint4*)(ds + (int64_t)r * ld_same + c) = o;
  }
  __syncthreads();
  if (!trans) return;
  // transposed: thread -> (trans row = column rr + 32*pass of the tile, 8 consecutive source rows)
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int col = rr + pass * 32;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = (uint32_t)tile[chunk * 8 + 2 * e][col] | ((uint32_t)tile[chunk * 8 + 2 * e + 1][col] << 16);
    *(uint4*)(dt + (int64_t)(c0 + col) * ld_trans + r0 + chunk * 8) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// Dense [B,R,C] <- padded [B,*,ld] (drops padding).
__global__ __launch_bounds__(256) void unpad_kernel(const bf16_t* __restrict__ src, int64_t src_stride,
                                                    int ld, bf16_t* __restrict__ dst, int R, int C) {
  const int b = blockIdx.z;
  for (int r = blockIdx.y; r < R; r += gridDim.y) {
    const bf16_t* s = src + (int64_t)b * src_stride + (int64_t)r * ld;
    bf16_t* d = dst + ((int64_t)b * R + r) * C;
    for (int c = blockIdx.x * 256 + threadIdx.x; c < C; c += gridDim.x * 256) d[c] = s[c];
  }
}

hipError_t launch_frobenius_inv(const void* in, int in_dtype, int batch, int64_t numel,
                                float norm_scale, float eps, float* partial, int nblk,
                                float* inv_norm, hipStream_t st) {
  const bool vec = (numel % 8 == 0) && (((uintptr_t)in) & 15) == 0;
#define SUMSQ_LAUNCH(T, V)                                                                      \
  hipLaunchKernelGGL((sumsq_partial_kernel<T, V>), dim3(nblk, batch), dim3(256), 0, st, (const T*)in, \
                     numel, nblk, partial)
  if (in_dtype == 0) {
    if (vec) SUMSQ_LAUNCH(bf16_t, true); else SUMSQ_LAUNCH(bf16_t, false);
  } else {
    if (vec) SUMSQ_LAUNCH(float, true); else SUMSQ_LAUNCH(float, false);
  }
#undef SUMSQ_LAUNCH
  return launch_norm_finalize(partial, nblk, batch, norm_scale, eps, inv_norm, nullptr, 0, st);
}

hipError_t launch_norm_finalize(const float* partial, int nblk, int batch, float norm_scale, float eps,
                                float* inv_norm, bf16_t* X, int64_t elems, hipStream_t st) {
  hipLaunchKernelGGL(norm_finalize_kernel, dim3(batch), dim3(256), 0, st, partial, nblk, norm_scale, eps,
                     inv_norm, X, elems);
  return hipGetLastError();
}

hipError_t launch_ns_prepare(const void* in, int in_dtype, int batch, int R, int C,
                             const float* inv_norm, bf16_t* same, int Rp, int Cp, int ld_same,
                             int64_t stride_same, bf16_t* trans, int ld_trans, int64_t stride_trans,
                             hipStream_t st) {
  dim3 grid(Cp / 64, Rp / 64, batch);
  const bool vec = (C % 8 == 0) && (((uintptr_t)in) & 15) == 0 && (ld_same % 8 == 0) &&
                   (ld_trans % 8 == 0) && (stride_same % 8 == 0) && (stride_trans % 8 == 0) &&
                   (((uintptr_t)same) & 15) == 0 && (((uintptr_t)trans) & 15) == 0;
  if (vec) {
    if (in_dtype == 0)
      hipLaunchKernelGGL(ns_prepare_vec_kernel<bf16_t>, grid, dim3(256), 0, st, (const bf16_t*)in, R, C,
                         inv_norm, same, ld_same, stride_same, trans, ld_trans, stride_trans);
    else
      hipLaunchKernelGGL(ns_prepare_vec_kernel<float>, grid, dim3(256), 0, st, (const float*)in, R, C,
                         inv_norm, same, ld_same, stride_same, trans, ld_trans, stride_trans);
    return hipGetLastError();
  }
  if (in_dtype == 0)
    hipLaunchKernelGGL(ns_prepare_kernel<bf16_t>, grid, dim3(256), 0, st, (const bf16_t*)in, R, C,
                       inv_norm, same, Rp, Cp, ld_same, stride_same, trans, ld_trans, stride_trans);
  else
    hipLaunchKernelGGL(ns_prepare_kernel<float>, grid, dim3(256), 0, st, (const float*)in, R, C,
                       inv_norm, same, Rp, Cp, ld_same, stride_same, trans, ld_trans, stride_trans);
  return hipGetLastError();
}

hipError_t launch_unpad(const bf16_t* src, int64_t src_stride, int ld, bf16_t* dst, int batch, int R,
                        int C, hipStream_t st) {
  int gx = (C + 255) / 256;
  if (gx > 64) gx = 64;
  hipLaunchKernelGGL(unpad_kernel, dim3(gx, R < 65535 ? R : 65535, batch), dim3(256), 0, st, src,
                     src_stride, ld, dst, R, C);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Muon pre: momentum + Nesterov + bf16 cast, list-of-parameters in, one arena out.
// ------------------------------------------------------------------------------------------
// SUMSQ (VEC only, one tile per workgroup): the workgroup also writes the sum of squares of the 4096
// bf16 values it stored, sumsq[p * gridDim.x + blockIdx.x] -- partial sums of ||U||_F^2 per matrix when
// a matrix is a whole number of tiles.
template <typename GT, typename MT, bool VEC, bool SUMSQ = false>
__global__ __launch_bounds__(256) void muon_pre_kernel(PtrTab G, PtrTab M, bf16_t* __restrict__ U,
                                                       int64_t numel, float mu, int nesterov,
                                                       float* __restrict__ sumsq = nullptr) {
  __shared__ float red[16];
  float ss = 0.f;
  const int p = blockIdx.y;
  const GT* __restrict__ g = (const GT*)G.p[p];
  MT* __restrict__ m = (MT*)M.p[p];
  bf16_t* __restrict__ u = U + (int64_t)p * numel;
  const int64_t stride = (int64_t)gridDim.x * 256;
  if (VEC) {
    // Two 8-element chunks per thread per trip, all loads issued before the arithmetic: up to 96
    // bytes of reads in flight per lane.
    // A workgroup owns contiguous tiles of 512 chunks (4096 elements), one tile per trip and normally
    // one trip: the workgroups in flight sweep one window of memory front to back.
    const int64_t nv = numel >> 3;
    for (int64_t i0 = (int64_t)blockIdx.x * 512 + threadIdx.x; i0 < nv; i0 += 2 * stride) {
      const int64_t i1 = i0 + 256;
      const bool has1 = i1 < nv;
      float gv[2][8], mv[2][8];
      st_load8<GT>(g, i0, gv[0]);
      if (has1) st_load8<GT>(g, i1, gv[1]);
      st_load8<MT>(m, i0, mv[0]);
      if (has1) st_load8<MT>(m, i1, mv[1]);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if (c == 1 && !has1) break;
        const int64_t i = c == 0 ? i0 : i1;
        float uv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          mv[c][e] = __fadd_rn(__fmul_rn(mv[c][e], mu), gv[c][e]);
          uv[e] = nesterov ? __fadd_rn(__fmul_rn(mv[c][e], mu), gv[c][e]) : mv[c][e];
        }
        st_store8<MT>(m, i, mv[c]);
        st_store8<bf16_t>(u, i, uv);
        if (SUMSQ) {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float r = st_round<bf16_t>(uv[e]);
            ss += r * r;
          }
        }
      }
    }
    if (SUMSQ) {
      ss = block_sum(ss, red);
      if (threadIdx.x == 0) sumsq[(int64_t)p * gridDim.x + blockIdx.x] = ss;
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < numel; i += stride) {
      const float gv = st_load<GT>(g, i);
      const float mv = __fadd_rn(__fmul_rn(st_load<MT>(m, i), mu), gv);
      st_store<MT>(m, i, mv);
      u[i] = f32_to_bf16(nesterov ? __fadd_rn(__fmul_rn(mv, mu), gv) : mv);
    }
  }
}

// The same update for tall matrices (rows > cols) whose orthogonalization input is wanted with the short
// side along rows: U[p][mat] is written transposed, [cols][rows].  One 64 x 64 tile per workgroup, staged
// through LDS so that G / M rows are read and U^T rows written as whole 128-byte (bf16) runs; every thread
// handles two 8-element chunks, like the flat kernel.  sumsq[(p * mats + mat) * tiles + tile]: sum of
// squares of the tile's bf16 values, tile = (row tile) * (cols / 64) + column tile.
// Needs rows % 64 == 0, cols % 64 == 0, 16-byte aligned pointers.
template <typename GT, typename MT>
__global__ __launch_bounds__(256) void muon_pre_transposed_kernel(PtrTab G, PtrTab M, bf16_t* __restrict__ U,
                                                                  int mats, int rows, int cols, float mu,
                                                                  int nesterov, float* __restrict__ sumsq) {
  __shared__ __attribute__((aligned(16))) bf16_t tile[64][72];
  __shared__ float red[16];
  const int p = blockIdx.z / mats, mat = blockIdx.z - p * mats;
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const int64_t mat_off = (int64_t)mat * rows * cols;
  const GT* __restrict__ g = (const GT*)G.p[p] + mat_off;
  MT* __restrict__ m = (MT*)M.p[p] + mat_off;
  bf16_t* __restrict__ ut = U + ((int64_t)p * mats + mat) * rows * cols;
  const int chunk = threadIdx.x & 7, rr = threadIdx.x >> 3;  // 8 chunks x 32 rows per pass
  float gv[2][8], mv[2][8];
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int64_t i8 = ((int64_t)(r0 + rr + pass * 32) * cols + c0 + chunk * 8) >> 3;
    st_load8<GT>(g, i8, gv[pass]);
    st_load8<MT>(m, i8, mv[pass]);
  }
  float ss = 0.f;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int64_t i8 = ((int64_t)(r0 + rr + pass * 32) * cols + c0 + chunk * 8) >> 3;
    float uv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      mv[pass][e] = __fadd_rn(__fmul_rn(mv[pass][e], mu), gv[pass][e]);
      uv[e] = nesterov ? __fadd_rn(__fmul_rn(mv[pass][e], mu), gv[pass][e]) : mv[pass][e];
    }
    st_store8<MT>(m, i8, mv[pass]);
    uint4 o;
    o.x = pack_bf16x2(uv[0], uv[1]);
    o.y = pack_bf16x2(uv[2], uv[3]);
    o.z = pack_bf16x2(uv[4], uv[5]);
    o.w = pack_bf16x2(uv[6], uv[7]);
    *(uint4*)&tile[rr + pass * 32][chunk * 8] = o;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float r = st_round<bf16_t>(uv[e]);
      ss += r * r;
    }
  }
  ss = block_sum(ss, red);  // (its barriers also order the tile writes before the reads below)
  if (threadIdx.x == 0)
    sumsq[((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = ss;
  // transposed: thread -> (U^T row = column rr + 32 * pass of the tile, 8 consecutive source rows)
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int col = rr + pass * 32;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = (uint32_t)tile[chunk * 8 + 2 * e][col] | ((uint32_t)tile[chunk * 8 + 2 * e + 1][col] << 16);
    *(uint4*)(ut + (int64_t)(c0 + col) * rows + r0 + chunk * 8) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// ------------------------------------------------------------------------------------------
// Matrices that do not fill whole GEMM tiles, into the zero-padded form the iteration carries: X [mat][Mp][Np] bf16,
// short side along rows, plus the sum of squares of every 64 x 64 tile of it.  One such tile per workgroup; a thread
// brings sixteen elements, V side by side (V divides the row length, so a group never straddles a row's end; with
// V = 8 a lane moves 16 or 32 bytes), all of them requested before the first is used, and the tile goes through LDS so
// that X is written 16 bytes a lane whatever V and the orientation are.  The sums are taken there, in X order: a matrix
// and its transpose give the same bits.
// Bound: HBM.  12 x (2730 x 1000) fp32, momentum update included: 95 us beside another stream's GEMMs, where the update
// (76), the norm's pass over its result (14) and the scaled copy (30) took 120; 4 x (2730 x 1000) fp32 copied: 15.0 us
// where copy and norm took 23.4.  Selected rows gathered here instead of copied a second time: NorDion2 on 12 layers of 1600,
// a step, 4130 -> 3935 us (bf16 state 3594 -> 3372).
// ------------------------------------------------------------------------------------------
template <typename T, int V>
static __device__ __forceinline__ void load_group(const T* p, int64_t i, float* v) {
  if constexpr (V == 8) st_load8<T>(p, i >> 3, v);
  else if constexpr (V == 2 && sizeof(T) == 2) {
    const uint32_t w = *(const uint32_t*)(p + i);
    v[0] = __uint_as_float(w << 16);
    v[1] = __uint_as_float(w & 0xffff0000u);
  } else if constexpr (V == 2) {
    const float2 w = *(const float2*)(p + i);
    v[0] = w.x;
    v[1] = w.y;
  } else v[0] = st_load<T>(p, i);
}
template <typename T, int V>
static __device__ __forceinline__ void store_group(T* p, int64_t i, const float* v) {
  if constexpr (V == 8) st_store8<T>(p, i >> 3, v);
  else if constexpr (V == 2 && sizeof(T) == 2) *(uint32_t*)(p + i) = pack_bf16x2(v[0], v[1]);
  else if constexpr (V == 2) *(float2*)(p + i) = make_float2(v[0], v[1]);
  else st_store<T>(p, i, v[0]);
}

// Where the elements come from.  A plain tensor:
template <typename T>
struct PadCopyOp {
  const T* in;
  struct At { const T* p; };
  __device__ __forceinline__ At at(int mat, int mats, int64_t mat_elems) const { return {in + (int64_t)mat * mat_elems}; }
  struct Raw { float v[8]; };
  template <int V>
  static __device__ __forceinline__ void load(const At& a, int row, int c, int C, Raw& r) {
    load_group<T, V>(a.p, (int64_t)row * C + c, r.v);
  }
  template <int V>
  __device__ __forceinline__ void finish(const At&, int, int, int, Raw& r, float* u) const {
#pragma unroll
    for (int e = 0; e < V; ++e) u[e] = r.v[e];
  }
};
// the momentum update of muon_pre_kernel:
template <typename GT, typename MT>
struct PadPreOp {
  PtrTab G, M;
  float mu;
  int nesterov;
  struct At { const GT* g; MT* m; };
  __device__ __forceinline__ At at(int mat, int mats, int64_t mat_elems) const {
    const int p = mat / mats;
    const int64_t off = (int64_t)(mat - p * mats) * mat_elems;
    return {(const GT*)G.p[p] + off, (MT*)M.p[p] + off};
  }
  struct Raw { float g[8], m[8]; };
  template <int V>
  static __device__ __forceinline__ void load(const At& a, int row, int c, int C, Raw& r) {
    load_group<GT, V>(a.g, (int64_t)row * C + c, r.g);
    load_group<MT, V>(a.m, (int64_t)row * C + c, r.m);
  }
  template <int V>
  __device__ __forceinline__ void finish(const At& a, int row, int c, int C, Raw& r, float* u) const {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      r.m[e] = __fadd_rn(__fmul_rn(r.m[e], mu), r.g[e]);
      u[e] = nesterov ? __fadd_rn(__fmul_rn(r.m[e], mu), r.g[e]) : r.m[e];
    }
    store_group<MT, V>(a.m, (int64_t)row * C + c, r.m);
  }
};
// the selected rows of dion2_gather_kernel, which decay where they lie.  (Columns are not taken: a tile's ends fall inside lines
// that two workgroups then write, and a step of 12 layers of 1600 took 3250 us instead of 3220.)
template <typename MT>
struct PadGatherRowsOp {
  PtrTab M;
  const int32_t* idx;
  int rows, cols, k;
  float ef_decay;
  struct At { MT* m; const int32_t* id; };
  __device__ __forceinline__ At at(int mat, int mats, int64_t) const {
    const int p = mat / mats;
    return {(MT*)M.p[p] + (int64_t)(mat - p * mats) * rows * cols, idx + (int64_t)mat * k};
  }
  struct Raw { float v[8]; int64_t at; };
  template <int V>
  static __device__ __forceinline__ void load(const At& a, int row, int c, int C, Raw& r) {
    r.at = (int64_t)a.id[row] * C + c;
    load_group<MT, V>(a.m, r.at, r.v);
  }
  template <int V>
  __device__ __forceinline__ void finish(const At& a, int, int, int, Raw& r, float* u) const {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      u[e] = r.v[e];
      r.v[e] = __fmul_rn(r.v[e], ef_decay);
    }
    store_group<MT, V>(a.m, r.at, r.v);
  }
};

template <class Op, int V, bool TALL>
__global__ __launch_bounds__(256) void pad_tile_kernel(const Op op, int mats, int R, int C, bf16_t* __restrict__ X,
                                                       int Mp, int Np, float* __restrict__ partial) {
  constexpr int CPR = 64 / V, RPP = 256 / CPR, NP = 64 / RPP;  // groups per tile row, rows per pass, passes
  __shared__ __attribute__((aligned(16))) bf16_t tile[64][72];
  __shared__ float red[16];
  const int mat = blockIdx.z;
  const int x0 = blockIdx.y * 64, y0 = blockIdx.x * 64;  // tile of X: first row, first column
  const int r0 = TALL ? y0 : x0, c0 = TALL ? x0 : y0;    // and of the source
  const auto at = op.at(mat, mats, (int64_t)R * C);
  const int grp = threadIdx.x % CPR, rr = threadIdx.x / CPR;
  const int c = c0 + grp * V;
  typename Op::Raw raw[NP];
#pragma unroll
  for (int ps = 0; ps < NP; ++ps) {
    const int r = r0 + rr + ps * RPP;
    if (r < R && c < C) op.template load<V>(at, r, c, C, raw[ps]);
  }
#pragma unroll
  for (int ps = 0; ps < NP; ++ps) {
    const int i = rr + ps * RPP, r = r0 + i;
    float u[V];
#pragma unroll
    for (int e = 0; e < V; ++e) u[e] = 0.f;
    if (r < R && c < C) op.template finish<V>(at, r, c, C, raw[ps], u);
    store_group<bf16_t, V>(&tile[i][0], grp * V, u);
  }
  __syncthreads();
  bf16_t* x = X + ((int64_t)mat * Mp + x0) * Np + y0;
  const int chunk = threadIdx.x & 7, row = threadIdx.x >> 3;
  float ss = 0.f;
#pragma unroll
  for (int ps = 0; ps < 2; ++ps) {
    const int i = row + ps * 32;  // row of X, eight columns from 8 * chunk on
    u32x4_t w;
    if (!TALL) w = *(const u32x4_t*)&tile[i][chunk * 8];
    else
#pragma unroll
      for (int e = 0; e < 4; ++e)
        w[e] = (uint32_t)tile[chunk * 8 + 2 * e][i] | ((uint32_t)tile[chunk * 8 + 2 * e + 1][i] << 16);
    *(u32x4_t*)(x + (int64_t)i * Np + chunk * 8) = w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = __uint_as_float(w[e] << 16), hi = __uint_as_float(w[e] & 0xffff0000u);
      ss += lo * lo;
      ss += hi * hi;
    }
  }
  ss = block_sum(ss, red);
  if (threadIdx.x == 0) partial[((int64_t)mat * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = ss;
}

template <class Op>
static hipError_t launch_pad_tile(const Op& op, int n_mat, int mats, int R, int C, bool aligned, bf16_t* X, int Mp, int Np,
                                  float* partial, hipStream_t st) {
  const dim3 grid(Np / 64, Mp / 64, n_mat);
  const int v = !aligned ? 1 : C % 8 == 0 ? 8 : C % 2 == 0 ? 2 : 1;
#define PAD_LAUNCH(V, T) \
  hipLaunchKernelGGL((pad_tile_kernel<Op, V, T>), grid, dim3(256), 0, st, op, mats, R, C, X, Mp, Np, partial)
  if (R > C) {
    if (v == 8) PAD_LAUNCH(8, true); else if (v == 2) PAD_LAUNCH(2, true); else PAD_LAUNCH(1, true);
  } else {
    if (v == 8) PAD_LAUNCH(8, false); else if (v == 2) PAD_LAUNCH(2, false); else PAD_LAUNCH(1, false);
  }
#undef PAD_LAUNCH
  return hipGetLastError();
}

hipError_t launch_ns_pad_copy(const void* in, int in_dtype, int batch, int R, int C, bf16_t* X, int Mp, int Np,
                              float* partial, hipStream_t st) {
  const bool aligned = (((uintptr_t)in) & 15) == 0;
  if (in_dtype == 0)
    return launch_pad_tile(PadCopyOp<bf16_t>{(const bf16_t*)in}, batch, 1, R, C, aligned, X, Mp, Np, partial, st);
  return launch_pad_tile(PadCopyOp<float>{(const float*)in}, batch, 1, R, C, aligned, X, Mp, Np, partial, st);
}

template <typename GT, typename MT>
static hipError_t muon_pre_padded(const PtrTab& G, const PtrTab& M, bf16_t* X, float* sumsq, int n, int mats, int rows,
                                  int cols, int mp, int np, float mu, int nesterov, bool aligned, hipStream_t st) {
  PadPreOp<GT, MT> op;
  op.G = G;
  op.M = M;
  op.mu = mu;
  op.nesterov = nesterov;
  return launch_pad_tile(op, n * mats, mats, rows, cols, aligned, X, mp, np, sumsq, st);
}

hipError_t launch_muon_pre_padded(const PtrTab& G, int g_dtype, const PtrTab& M, int m_dtype, bf16_t* X, float* sumsq,
                                  int n, int mats, int rows, int cols, int mp, int np, float mu, int nesterov,
                                  bool aligned, hipStream_t st) {
  if (g_dtype == 0)
    return m_dtype == 0 ? muon_pre_padded<bf16_t, bf16_t>(G, M, X, sumsq, n, mats, rows, cols, mp, np, mu, nesterov, aligned, st)
                        : muon_pre_padded<bf16_t, float>(G, M, X, sumsq, n, mats, rows, cols, mp, np, mu, nesterov, aligned, st);
  return m_dtype == 0 ? muon_pre_padded<float, bf16_t>(G, M, X, sumsq, n, mats, rows, cols, mp, np, mu, nesterov, aligned, st)
                      : muon_pre_padded<float, float>(G, M, X, sumsq, n, mats, rows, cols, mp, np, mu, nesterov, aligned, st);
}

hipError_t launch_dion2_gather_padded(const PtrTab& M, int m_dtype, int n_mat, int mats_per_ptr, int rows, int cols,
                                      const int32_t* idx, int k, float ef_decay, bf16_t* X, int mp, int np, float* sumsq,
                                      bool aligned, hipStream_t st) {
  if (m_dtype == 0)
    return launch_pad_tile(PadGatherRowsOp<bf16_t>{M, idx, rows, cols, k, ef_decay}, n_mat, mats_per_ptr, k, cols, aligned, X,
                           mp, np, sumsq, st);
  return launch_pad_tile(PadGatherRowsOp<float>{M, idx, rows, cols, k, ef_decay}, n_mat, mats_per_ptr, k, cols, aligned, X, mp,
                         np, sumsq, st);
}

// Workgroups for the tile-per-workgroup kernels: one per 512 chunks, at most 2^20.
static int ew_tiles(int64_t chunks) {
  int64_t b = (chunks + 511) / 512;
  if (b > (1 << 20)) b = 1 << 20;
  if (b < 1) b = 1;
  return (int)b;
}

static int ew_blocks(int64_t work_items) {
  int64_t b = (work_items + 255) / 256;
  if (b > 2048) b = 2048;
  if (b < 1) b = 1;
  return (int)b;
}

hipError_t launch_muon_pre(const PtrTab& G, int g_dtype, const PtrTab& M, int m_dtype, bf16_t* U, int n,
                           int64_t numel, float mu, int nesterov, bool vec, hipStream_t st) {
  dim3 grid(vec ? ew_tiles(numel >> 3) : ew_blocks(numel), n);
#define PRE_LAUNCH(GT, MT, V) \
  hipLaunchKernelGGL((muon_pre_kernel<GT, MT, V>), grid, dim3(256), 0, st, G, M, U, numel, mu, nesterov)
#define PRE_LAUNCH_M(GT, V) \
  do { if (m_dtype == 0) PRE_LAUNCH(GT, bf16_t, V); else PRE_LAUNCH(GT, float, V); } while (0)
  if (g_dtype == 0) {
    if (vec) PRE_LAUNCH_M(bf16_t, true); else PRE_LAUNCH_M(bf16_t, false);
  } else {
    if (vec) PRE_LAUNCH_M(float, true); else PRE_LAUNCH_M(float, false);
  }
#undef PRE_LAUNCH_M
#undef PRE_LAUNCH
  return hipGetLastError();
}

hipError_t launch_muon_pre_prepared(const PtrTab& G, int g_dtype, const PtrTab& M, int m_dtype, bf16_t* U,
                                    float* sumsq, int n, int mats, int rows, int cols, float mu,
                                    int nesterov, hipStream_t st) {
  if (rows > cols) {
    dim3 grid(cols / 64, rows / 64, n * mats);
#define PRET_LAUNCH(GT, MT)                                                                            \
  hipLaunchKernelGGL((muon_pre_transposed_kernel<GT, MT>), grid, dim3(256), 0, st, G, M, U, mats, rows, cols, \
                     mu, nesterov, sumsq)
    if (g_dtype == 0) {
      if (m_dtype == 0) PRET_LAUNCH(bf16_t, bf16_t); else PRET_LAUNCH(bf16_t, float);
    } else {
      if (m_dtype == 0) PRET_LAUNCH(float, bf16_t); else PRET_LAUNCH(float, float);
    }
#undef PRET_LAUNCH
    return hipGetLastError();
  }
  // one 4096-element tile per workgroup, so that blockIdx.x is the tile number within the parameter
  const int64_t numel = (int64_t)mats * rows * cols;
  dim3 grid((unsigned)(numel / 4096), n);
#define PRES_LAUNCH(GT, MT)                                                                             \
  hipLaunchKernelGGL((muon_pre_kernel<GT, MT, true, true>), grid, dim3(256), 0, st, G, M, U, numel, mu, \
                     nesterov, sumsq)
  if (g_dtype == 0) {
    if (m_dtype == 0) PRES_LAUNCH(bf16_t, bf16_t); else PRES_LAUNCH(bf16_t, float);
  } else {
    if (m_dtype == 0) PRES_LAUNCH(float, bf16_t); else PRES_LAUNCH(float, float);
  }
#undef PRES_LAUNCH
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Muon / NorMuon post: decoupled weight decay (plain or cautious) + scaled update.
// ------------------------------------------------------------------------------------------
template <typename UT, typename XT, bool VEC>
__global__ __launch_bounds__(256) void muon_post_kernel(PtrTab X, const UT* __restrict__ U,
                                                        int64_t numel, int cols,
                                                        const float* __restrict__ row_scale,
                                                        const float* __restrict__ lr_dev,
                                                        const float* __restrict__ adj_lr_dev,
                                                        float adj_ratio,
                                                        const float* __restrict__ wd_dev,
                                                        float wd_host, int cautious) {
  const int p = blockIdx.y;
  XT* __restrict__ x = (XT*)X.p[p];
  const UT* __restrict__ u = U + (int64_t)p * numel;
  const float lr = *lr_dev;
  const float wd = wd_dev ? *wd_dev : wd_host;
  const float coeff = __fmul_rn(lr, wd);
  const float a = __fsub_rn(1.0f, coeff);
  const float b = adj_lr_dev ? *adj_lr_dev : __fmul_rn(lr, adj_ratio);
  const int64_t rows = numel / cols;
  const float* rs = row_scale ? row_scale + (int64_t)p * rows : nullptr;
  const int64_t stride = (int64_t)gridDim.x * 256;
  if (VEC) {
    // contiguous tiles of 512 chunks (4096 elements) per workgroup, two chunks per lane, all loads first
    const int64_t nv = numel >> 3;
    for (int64_t i0 = (int64_t)blockIdx.x * 512 + threadIdx.x; i0 < nv; i0 += 2 * stride) {
      const int64_t i1 = i0 + 256;
      const bool has1 = i1 < nv;
      float uv[2][8], xv[2][8];
      st_load8<UT>(u, i0, uv[0]);
      if (has1) st_load8<UT>(u, i1, uv[1]);
      st_load8<XT>(x, i0, xv[0]);
      if (has1) st_load8<XT>(x, i1, xv[1]);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if (c == 1 && !has1) break;
        const int64_t i = c == 0 ? i0 : i1;
        if (rs) {  // cols % 8 == 0 on this path, so the 8 elements share a row
          const float s = rs[(i << 3) / cols];
#pragma unroll
          for (int e = 0; e < 8; ++e) uv[c][e] = __fmul_rn(uv[c][e], s);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) xv[c][e] = muon_post_one(xv[c][e], uv[c][e], a, coeff, b, cautious);
        st_store8<XT>(x, i, xv[c]);
      }
    }
  } else {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < numel; i += stride) {
      float uv = st_load<UT>(u, i);
      if (rs) uv = __fmul_rn(uv, rs[i / cols]);
      st_store<XT>(x, i, muon_post_one(st_load<XT>(x, i), uv, a, coeff, b, cautious));
    }
  }
}

hipError_t launch_muon_post(const PtrTab& X, int x_dtype, const void* U, int u_dtype, int n, int64_t numel,
                            int cols, const float* row_scale, const float* lr_dev, const float* adj_lr_dev,
                            float adj_ratio, const float* wd_dev, float wd_host, int cautious, bool vec,
                            hipStream_t st) {
  dim3 grid(vec ? ew_tiles(numel >> 3) : ew_blocks(numel), n);
#define POST_LAUNCH(UT, XT, V)                                                                      \
  hipLaunchKernelGGL((muon_post_kernel<UT, XT, V>), grid, dim3(256), 0, st, X, (const UT*)U, numel, \
                     cols, row_scale, lr_dev, adj_lr_dev, adj_ratio, wd_dev, wd_host, cautious)
#define POST_LAUNCH_X(UT, V) \
  do { if (x_dtype == 0) POST_LAUNCH(UT, bf16_t, V); else POST_LAUNCH(UT, float, V); } while (0)
  if (u_dtype == 0) {
    if (vec) POST_LAUNCH_X(bf16_t, true); else POST_LAUNCH_X(bf16_t, false);
  } else {
    if (vec) POST_LAUNCH_X(float, true); else POST_LAUNCH_X(float, false);
  }
#undef POST_LAUNCH_X
#undef POST_LAUNCH
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// out[row][:] = U[row][:] * scale[row]: the normalised update itself, for callers that want it as a
// tensor (the optimizers fold the scale into the update kernels instead).
// ------------------------------------------------------------------------------------------
template <typename OT>
__global__ __launch_bounds__(256) void scale_rows_kernel(const bf16_t* __restrict__ U,
                                                         const float* __restrict__ scale,
                                                         OT* __restrict__ out, int cols) {
  const int64_t row = blockIdx.x;
  const float s = scale[row];
  const bf16_t* u = U + row * cols;
  OT* o = out + row * cols;
  for (int c = threadIdx.x; c < cols; c += 256) st_store<OT>(o, c, __fmul_rn(bf16_to_f32(u[c]), s));
}

hipError_t launch_scale_rows(const bf16_t* U, const float* scale, void* out, int out_dtype, int64_t n_rows,
                             int cols, hipStream_t st) {
  if (n_rows <= 0 || cols <= 0) return hipSuccess;
  if (n_rows > 0x7fffffff) return hipErrorInvalidValue;
  if (out_dtype == 0)
    hipLaunchKernelGGL((scale_rows_kernel<bf16_t>), dim3((unsigned)n_rows), dim3(256), 0, st, U, scale,
                       (bf16_t*)out, cols);
  else
    hipLaunchKernelGGL((scale_rows_kernel<float>), dim3((unsigned)n_rows), dim3(256), 0, st, U, scale,
                       (float*)out, cols);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// NorMuon: per-row second moment EMA and the Frobenius-preserving row scales.
// ------------------------------------------------------------------------------------------
// Row r of matrix mat keeps its second moment at V[mat][row_idx ? row_idx[mat][r] : r]; V holds
// v_rows entries per matrix (v_rows == rows without row_idx).  The indirection serves updates made
// of selected rows only (NorDion2, dion/nordion2.py:430-447).  A negative row_idx entry marks a row
// that is not part of the update (an all-zero row of a masked full-size tensor,
// dion/nordion2.py:485-497): its second moment is left alone and its scale is 0.
// Pass 1: one wavefront per row.  V <- lerp(V, mean(u^2), w);  tmp[row] = sum(u^2).  u_sq is the square of a factor that the
// rows count with (1: as they lie).
template <typename VT>
__global__ __launch_bounds__(256) void normuon_rows_kernel(const bf16_t* __restrict__ U, PtrTab V,
                                                           int mats_per_ptr, int rows, int cols,
                                                           const int32_t* __restrict__ row_idx,
                                                           int v_rows, float w, float u_sq,
                                                           float* __restrict__ rowsq) {
  const int mat = blockIdx.y;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const bf16_t* u = U + ((int64_t)mat * rows + row) * cols;
  float s = 0.f;
  if ((cols & 7) == 0 && (((uintptr_t)u) & 15) == 0) {
    for (int c = lane * 8; c < cols; c += 512) {
      const uint4 raw = *(const uint4*)(u + c);
      const uint32_t wv[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = __uint_as_float(wv[e] << 16), hi = __uint_as_float(wv[e] & 0xffff0000u);
        s += lo * lo;
        s += hi * hi;
      }
    }
  } else {
    for (int c = lane; c < cols; c += 64) {
      const float v = bf16_to_f32(u[c]);
      s += v * v;
    }
  }
  s = wave_sum(s) * u_sq;
  if (lane == 0) {
    const int vr = row_idx ? row_idx[(int64_t)mat * rows + row] : row;
    if (vr >= 0) {
      VT* v = (VT*)V.p[mat / mats_per_ptr] + (int64_t)(mat % mats_per_ptr) * v_rows + vr;
      const float mean = s / (float)cols;
      const float vo = st_load<VT>(v, 0);
      st_store<VT>(v, 0, vo + w * (mean - vo));  // torch.lerp for weight < 0.5
    }
    rowsq[(int64_t)mat * rows + row] = vr >= 0 ? s : 0.f;
  }
}

// Pass 2: one block per matrix.  scale[row] = (1/d) * sqrt(S1) / max(sqrt(S2), 1e-8) with
// d = sqrt(V)+1e-8, S1 = sum rowsq, S2 = sum rowsq/d^2.  In place over rowsq.
template <typename VT>
__global__ __launch_bounds__(1024) void normuon_scale_kernel(PtrTab V, int mats_per_ptr, int rows,
                                                             const int32_t* __restrict__ row_idx,
                                                             int v_rows, float* __restrict__ scale) {
  __shared__ float red[16];
  const int mat = blockIdx.x;
  const VT* v = (const VT*)V.p[mat / mats_per_ptr] + (int64_t)(mat % mats_per_ptr) * v_rows;
  const int32_t* ri = row_idx ? row_idx + (int64_t)mat * rows : nullptr;
  float* sc = scale + (int64_t)mat * rows;
  float s1 = 0.f, s2 = 0.f;
  for (int r = threadIdx.x; r < rows; r += 1024) {
    const float q = sc[r];
    const int vr = ri ? ri[r] : r;
    const float inv = vr >= 0 ? 1.0f / (sqrtf(st_load<VT>(v, vr)) + 1e-8f) : 0.f;
    s1 += q;
    s2 += q * inv * inv;
  }
  s1 = block_sum(s1, red);
  s2 = block_sum(s2, red);
  const float ratio = sqrtf(s1) / fmaxf(sqrtf(s2), 1e-8f);
  __syncthreads();
  for (int r = threadIdx.x; r < rows; r += 1024) {
    const int vr = ri ? ri[r] : r;
    sc[r] = vr >= 0 ? (1.0f / (sqrtf(st_load<VT>(v, vr)) + 1e-8f)) * ratio : 0.f;
  }
}

hipError_t launch_normuon_stats(const bf16_t* U, const PtrTab& V, int v_dtype, int n_mat, int mats_per_ptr,
                                int rows, int cols, const int32_t* row_idx, int v_rows, float w, float u_sq,
                                float* row_scale, hipStream_t st) {
  // U / row_scale / row_idx are offset to the first matrix by the caller; V is the table chunk
  // covering them.
  if (v_dtype == 0) {
    hipLaunchKernelGGL(normuon_rows_kernel<bf16_t>, dim3((rows + 3) / 4, n_mat), dim3(256), 0, st, U, V,
                       mats_per_ptr, rows, cols, row_idx, v_rows, w, u_sq, row_scale);
    hipLaunchKernelGGL(normuon_scale_kernel<bf16_t>, dim3(n_mat), dim3(1024), 0, st, V, mats_per_ptr, rows,
                       row_idx, v_rows, row_scale);
  } else {
    hipLaunchKernelGGL(normuon_rows_kernel<float>, dim3((rows + 3) / 4, n_mat), dim3(256), 0, st, U, V,
                       mats_per_ptr, rows, cols, row_idx, v_rows, w, u_sq, row_scale);
    hipLaunchKernelGGL(normuon_scale_kernel<float>, dim3(n_mat), dim3(1024), 0, st, V, mats_per_ptr, rows,
                       row_idx, v_rows, row_scale);
  }
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------------
// Dion2: accumulate + slice L1 norms, top-k, gather with error-feedback decay, fused post.
// ------------------------------------------------------------------------------------------
template <typename GT>
static __device__ __forceinline__ float g_load(const GT* g, int64_t i) {
  return sizeof(GT) == 2 ? bf16_to_f32(((const bf16_t*)g)[i]) : ((const float*)g)[i];
}

// select rows: one wavefront per row, norms[mat][row] = sum_j |M+G| (of the values as stored).  A lane adds the
// columns lane, lane + 64, ... in that order, whatever the batch it loads them in.
// Bound by HBM: sixteen columns' loads in flight per lane, non-temporal past the caches.  24 x (2048 x 8192), fp32 momentum,
// bf16 gradients: 824 us (4.9 TB/s) one column at a time -> 730 us (5.5 TB/s); bf16 momentum 600 -> 420 us;
// 12 x (768 x 3072) 52 -> 42 us.
template <int B, typename GT, typename MT, bool NT>
static __device__ __forceinline__ void acc_row_batch(const GT* __restrict__ g, MT* __restrict__ m, int c, float& s) {
  float gv[B], mv[B];
#pragma unroll
  for (int i = 0; i < B; ++i) {
    mv[i] = st_load<MT, NT>(m, c + 64 * i);
    gv[i] = st_load<GT, NT>(g, c + 64 * i);
  }
#pragma unroll
  for (int i = 0; i < B; ++i) {
    const float v = st_round<MT>(__fadd_rn(mv[i], gv[i]));
    st_store<MT, NT>(m, c + 64 * i, v);
    s += fabsf(v);
  }
}

template <typename GT, typename MT, bool NT>
__global__ __launch_bounds__(256) void dion2_acc_rows_kernel(PtrTab G, PtrTab M, int mats_per_ptr,
                                                             int rows, int cols,
                                                             float* __restrict__ norms) {
  const int mat = blockIdx.y;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int64_t base = ((int64_t)(mat % mats_per_ptr) * rows + row) * cols;
  const GT* __restrict__ g = (const GT*)G.p[mat / mats_per_ptr] + base;
  MT* __restrict__ m = (MT*)M.p[mat / mats_per_ptr] + base;
  float s = 0.f;
  int c = 0;
  for (; c + 64 * 16 <= cols; c += 64 * 16) acc_row_batch<16, GT, MT, NT>(g, m, c + lane, s);
  for (; c + 64 * 4 <= cols; c += 64 * 4) acc_row_batch<4, GT, MT, NT>(g, m, c + lane, s);
  for (c += lane; c < cols; c += 64) acc_row_batch<1, GT, MT, NT>(g, m, c, s);
  s = wave_sum(s);
  if (lane == 0) norms[(int64_t)mat * rows + row] = s;
}

// select columns: each block owns 64 columns of one matrix and walks all rows (4 rows at a time).
template <typename GT, typename MT>
__global__ __launch_bounds__(256) void dion2_acc_cols_kernel(PtrTab G, PtrTab M, int mats_per_ptr,
                                                             int rows, int cols,
                                                             float* __restrict__ norms) {
  __shared__ float red[4][64];
  const int mat = blockIdx.y;
  const int c = blockIdx.x * 64 + (threadIdx.x & 63);
  const int ry = threadIdx.x >> 6;
  const int64_t base = (int64_t)(mat % mats_per_ptr) * rows * cols;
  const GT* g = (const GT*)G.p[mat / mats_per_ptr] + base;
  MT* m = (MT*)M.p[mat / mats_per_ptr] + base;
  float s = 0.f;
  if (c < cols) {
    for (int r = ry; r < rows; r += 4) {
      const int64_t i = (int64_t)r * cols + c;
      const float v = st_round<MT>(__fadd_rn(st_load<MT>(m, i), g_load<GT>(g, i)));
      st_store<MT>(m, i, v);
      s += fabsf(v);
    }
  }
  red[ry][threadIdx.x & 63] = s;
  __syncthreads();
  if (ry == 0 && c < cols)
    norms[(int64_t)mat * cols + c] = (red[0][threadIdx.x] + red[1][threadIdx.x]) +
                                     (red[2][threadIdx.x] + red[3][threadIdx.x]);
}

template <int B, typename GT, typename MT, bool NT, bool STORE>
static __device__ __forceinline__ void acc_cols_batch(const GT* __restrict__ g, MT* __restrict__ m, int64_t i, int cols,
                                                      float4& s) {
  float gv[B][4], mv[B][4];
#pragma unroll
  for (int b = 0; b < B; ++b) {  // cols % 4 == 0 on this path
    st_load4<MT, NT>(m, (i >> 2) + (int64_t)b * cols, mv[b]);
    st_load4<GT, NT>(g, (i >> 2) + (int64_t)b * cols, gv[b]);
  }
#pragma unroll
  for (int b = 0; b < B; ++b) {
#pragma unroll
    for (int e = 0; e < 4; ++e) mv[b][e] = st_round<MT>(__fadd_rn(mv[b][e], gv[b][e]));
    if (STORE) st_store4<MT, NT>(m, (i >> 2) + (int64_t)b * cols, mv[b]);
    s.x += fabsf(mv[b][0]);
    s.y += fabsf(mv[b][1]);
    s.z += fabsf(mv[b][2]);
    s.w += fabsf(mv[b][3]);
  }
}

// 4 columns per thread (8- / 16-byte accesses): each block owns 256 columns, four row lanes.
// Bound by HBM: eight rows' loads in flight per thread, non-temporal past the caches (24 x (8192 x 2048), fp32 momentum, bf16
// gradients: 844 us (4.8 TB/s) with four -> 717 us (5.6 TB/s); 12 x (3072 x 768) 52 us either way).
// With gridDim.z row slabs the block writes its slab's partial sums to out[(slab*n_mat + mat)*cols]
// (n_mat = gridDim.y); dion2_sum_slabs_kernel adds the slabs in a fixed order.
// STORE false: the norms alone, M stays as it is (dion2_add_gather_cols_kernel updates it).
template <typename GT, typename MT, bool NT, bool STORE = true>
__global__ __launch_bounds__(256) void dion2_acc_cols_vec_kernel(PtrTab G, PtrTab M, int mats_per_ptr,
                                                                 int rows, int cols, int slab_rows,
                                                                 float* __restrict__ norms) {
  __shared__ float4 red[4][64];
  const int mat = blockIdx.y;
  const int r0 = blockIdx.z * slab_rows;
  const int r1 = (r0 + slab_rows) < rows ? (r0 + slab_rows) : rows;
  norms += (int64_t)blockIdx.z * gridDim.y * cols;
  const int c = (blockIdx.x * 64 + (threadIdx.x & 63)) * 4;
  const int ry = threadIdx.x >> 6;
  const int64_t base = (int64_t)(mat % mats_per_ptr) * rows * cols;
  const GT* __restrict__ g = (const GT*)G.p[mat / mats_per_ptr] + base;
  MT* __restrict__ m = (MT*)M.p[mat / mats_per_ptr] + base;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (c < cols) {
    int r = r0 + ry;
    // eight rows' loads in flight, added in row order
    for (; r + 28 < r1; r += 32) acc_cols_batch<8, GT, MT, NT, STORE>(g, m, (int64_t)r * cols + c, cols, s);
    for (; r < r1; r += 4) acc_cols_batch<1, GT, MT, NT, STORE>(g, m, (int64_t)r * cols + c, cols, s);
  }
  red[ry][threadIdx.x & 63] = s;
  __syncthreads();
  if (ry == 0 && c < cols) {
    const int t = threadIdx.x;
    float4 o;
    o.x = (red[0][t].x + red[1][t].x) + (red[2][t].x + red[3][t].x);
    o.y = (red[0][t].y + red[1][t].y) + (red[2][t].y + red[3][t].y);
    o.z = (red[0][t].z + red[1][t].z) + (red[2][t].z + red[3][t].z);
    o.w = (red[0][t].w + red[1][t].w) + (red[2][t].w + red[3][t].w);
    *(float4*)(norms + (int64_t)mat * cols + c) = o;
  }
}

__global__ __launch_bounds__(256) void dion2_sum_slabs_kernel(const float* __restrict__ part,
                                                             int64_t n, int slabs,
                                                             float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float s = part[i];
  for (int z = 1; z < slabs; ++z) s += part[(int64_t)z * n + i];
  out[i] = s;
}

int dion2_acc_slabs(int n_mat, int rows, int cols) {
  const int64_t blocks = (int64_t)((cols / 4 + 63) / 64) * n_mat;
  int64_t s = (2048 + blocks - 1) / blocks;
  const int64_t s_max = rows / 64 > 0 ? rows / 64 : 1;
  if (s > s_max) s = s_max;
  if (s > 32) s = 32;
  return s < 1 ? 1 : (int)s;
}

hipError_t launch_dion2_accumulate(const PtrTab& G, int g_dtype, const PtrTab& M, int m_dtype, int n_mat,
                                   int mats_per_ptr, int rows, int cols, int select_rows,
                                   float* norms, bool vec4, float* slab_scratch, int slabs, bool store,
                                   hipStream_t st) {
  if (!store && (select_rows || !vec4)) return hipErrorInvalidValue;
  const bool nt = exceeds_caches((int64_t)n_mat * rows * cols * ((m_dtype == 0 ? 4 : 8) + (g_dtype == 0 ? 2 : 4)));
  // the four (gradient, momentum) dtype pairs; NTV... is empty for kernels without a non-temporal form
#define ACC_LAUNCH_T(K, GRID, NTV, ...)                                                                 \
  do {                                                                                                  \
    if (g_dtype == 0 && m_dtype == 0)                                                                   \
      hipLaunchKernelGGL((K<bf16_t, bf16_t NTV>), GRID, dim3(256), 0, st, __VA_ARGS__);                  \
    else if (g_dtype == 0)                                                                              \
      hipLaunchKernelGGL((K<bf16_t, float NTV>), GRID, dim3(256), 0, st, __VA_ARGS__);                   \
    else if (m_dtype == 0)                                                                              \
      hipLaunchKernelGGL((K<float, bf16_t NTV>), GRID, dim3(256), 0, st, __VA_ARGS__);                   \
    else                                                                                                \
      hipLaunchKernelGGL((K<float, float NTV>), GRID, dim3(256), 0, st, __VA_ARGS__);                    \
  } while (0)
#define ACC_NT , true
#define ACC_T , false
#define ACC_NT_NORMS , true, false
#define ACC_T_NORMS , false, false
#define ACC_LAUNCH(K, GRID, ...)                             \
  do {                                                       \
    if (nt) ACC_LAUNCH_T(K, GRID, ACC_NT, __VA_ARGS__);      \
    else ACC_LAUNCH_T(K, GRID, ACC_T, __VA_ARGS__);          \
  } while (0)
  if (select_rows) {
    dim3 grid((rows + 3) / 4, n_mat);
    ACC_LAUNCH(dion2_acc_rows_kernel, grid, G, M, mats_per_ptr, rows, cols, norms);
  } else if (vec4) {
    if (!slab_scratch) slabs = 1;
    const int slab_rows = ((rows + slabs - 1) / slabs + 3) / 4 * 4;
    slabs = (rows + slab_rows - 1) / slab_rows;
    float* dst = slabs > 1 ? slab_scratch : norms;
    dim3 grid((cols / 4 + 63) / 64, n_mat, slabs);
    if (store) ACC_LAUNCH(dion2_acc_cols_vec_kernel, grid, G, M, mats_per_ptr, rows, cols, slab_rows, dst);
    else if (nt) ACC_LAUNCH_T(dion2_acc_cols_vec_kernel, grid, ACC_NT_NORMS, G, M, mats_per_ptr, rows, cols, slab_rows, dst);
    else ACC_LAUNCH_T(dion2_acc_cols_vec_kernel, grid, ACC_T_NORMS, G, M, mats_per_ptr, rows, cols, slab_rows, dst);
    if (slabs > 1) {
      const int64_t n = (int64_t)n_mat * cols;
      hipLaunchKernelGGL(dion2_sum_slabs_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                         slab_scratch, n, slabs, norms);
    }
  } else {
    dim3 grid((cols + 63) / 64, n_mat);
    ACC_LAUNCH_T(dion2_acc_cols_kernel, grid, , G, M, mats_per_ptr, rows, cols, norms);
  }
#undef ACC_NT
#undef ACC_T
#undef ACC_NT_NORMS
#undef ACC_T_NORMS
#undef ACC_LAUNCH_T
#undef ACC_LAUNCH
  return hipGetLastError();
}

// The k largest of every row, ties to the lower index, NaN as +inf: ascending positions in idx, the inverse in map
// (-1 for what is not selected).  One workgroup per matrix finds the k-th largest value two bits at a time -- each step
// counts the entries at or above three candidates with ballots, one LDS counter per candidate and step, one barrier --
// and stops as soon as a candidate has exactly k entries above it; a pass over 1024 entries at a time then places the
// selected ones in index order.  Bound by the chain of at most sixteen counting steps (about 0.2 us each), not by
// its dim * 4 bytes.  Keys stay in registers up to 1024 * 8 entries; longer rows are read again at every step.
// 24 rows of 2048 (k = 512), the launch alone: 43.4 us counting every entry's rank (2048^2 compares a row) and compacting in a
// second launch -> 8.2 us; 12 rows of 768: 20.9 -> 7.0; 300 rows of 64: 6.2 -> 7.0.  Inside a step it takes longer: a workgroup
// of 16 wavefronts waits for a CU that another stream's kernels leave (205 us a launch on average in a Dion2 step
// over matrices of 2048 x 8192).
// unsigned keys in the order of the values (NaN = +inf, -0 = +0); never 0
static __device__ __forceinline__ uint32_t topk_key(float x) {
  if (x != x) x = INFINITY;
  const uint32_t b = __float_as_uint(x + 0.0f);
  return b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
}

// R: keys per thread held in registers (dim <= 1024 * R); 0: any dim
template <int R>
__global__ __launch_bounds__(1024) void dion2_topk_kernel(const float* __restrict__ norms, int dim, int k,
                                                          int32_t* __restrict__ idx, int32_t* __restrict__ map) {
  __shared__ int count[16][4];   // [step][candidate]
  __shared__ int2 wave_tot[2][16];
  const int mat = blockIdx.x, tid = threadIdx.x;
  const int lane = tid & 63, w = tid >> 6;
  const float* v = norms + (int64_t)mat * dim;
  uint32_t key[R ? R : 1];
  auto load = [&](int base) -> uint32_t { return base + tid < dim ? topk_key(v[base + tid]) : 0u; };
#pragma unroll
  for (int r = 0; r < R; ++r) key[r] = load(r * 1024);
  if (tid < 64) ((int*)count)[tid] = 0;
  __syncthreads();
  // invariant: at least k keys are >= bar, `above` (fewer than k) are >= the next value the open bits allow
  uint32_t bar = 0;
  int above = 0, need = 0;
  bool exact = k == 0;  // k == 0: nothing is selected
  if (exact) bar = 0xffffffffu;
  for (int step = 0; step < 16 && !exact; ++step) {
    const int shift = 30 - 2 * step;
    const uint32_t c1 = bar | (1u << shift), c2 = bar | (2u << shift), c3 = bar | (3u << shift);
    int n1 = 0, n2 = 0, n3 = 0;
    if (R) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        n1 += __popcll(__ballot(key[r] >= c1));
        n2 += __popcll(__ballot(key[r] >= c2));
        n3 += __popcll(__ballot(key[r] >= c3));
      }
    } else {
      for (int base = 0; base < dim; base += 1024) {
        const uint32_t x = load(base);
        n1 += __popcll(__ballot(x >= c1));
        n2 += __popcll(__ballot(x >= c2));
        n3 += __popcll(__ballot(x >= c3));
      }
    }
    if (lane < 3) atomicAdd(&count[step][lane], lane == 0 ? n1 : (lane == 1 ? n2 : n3));
    __syncthreads();
    n1 = count[step][0];
    n2 = count[step][1];
    n3 = count[step][2];
    int here = 0;  // entries >= the bar this step chose (0: unchanged)
    if (n3 >= k) {
      bar = c3;
      here = n3;
    } else if (n2 >= k) {
      bar = c2;
      here = n2;
      above = n3;
    } else if (n1 >= k) {
      bar = c1;
      here = n1;
      above = n2;
    } else {
      above = n1;
    }
    if (here == k) {  // the entries >= bar are the selection
      exact = true;
      bar -= 1;
    }
  }
  if (!exact) need = k - above;  // how many of the entries equal to bar are selected
  int run_gt = 0, run_eq = 0;    // entries of either kind before the current 1024
  auto place = [&](int base, uint32_t x, int buf) {
    const int i = base + tid;
    const bool gt = x > bar, eq = x == bar;
    const unsigned long long bg = __ballot(gt), be = __ballot(eq), below = (1ull << lane) - 1ull;
    if (lane == 0) wave_tot[buf][w] = make_int2(__popcll(bg), __popcll(be));
    __syncthreads();
    int g = run_gt + __popcll(bg & below), e = run_eq + __popcll(be & below);
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int2 t = wave_tot[buf][q];
      if (q < w) {
        g += t.x;
        e += t.y;
      }
      run_gt += t.x;
      run_eq += t.y;
    }
    if (i < dim) {
      const bool sel = gt || (eq && e < need);
      const int pos = g + (e < need ? e : need);
      if (sel) idx[(int64_t)mat * k + pos] = i;
      map[(int64_t)mat * dim + i] = sel ? pos : -1;
    }
  };
  if (R) {
#pragma unroll
    for (int r = 0; r < R; ++r) place(r * 1024, key[r], r & 1);
  } else {
    int buf = 0;
    for (int base = 0; base < dim; base += 1024, buf ^= 1) place(base, load(base), buf);
  }
}

hipError_t launch_dion2_topk(const float* norms, int n_mat, int dim, int k, int32_t* idx,
                             int32_t* map, hipStream_t st) {
  const int r = (dim + 1023) / 1024;
  auto* kernel = r <= 1   ? dion2_topk_kernel<1>
                 : r <= 2 ? dion2_topk_kernel<2>
                 : r <= 4 ? dion2_topk_kernel<4>
                 : r <= 8 ? dion2_topk_kernel<8>
                          : dion2_topk_kernel<0>;
  hipLaunchKernelGGL(kernel, dim3(n_mat), dim3(1024), 0, st, norms, dim, k, idx, map);
  return hipGetLastError();
}

// U_sel = bf16(M[sel]); M[sel] *= ef_decay.
// rows selected: block (j, mat) copies row idx[j]; columns selected: block (row, mat) gathers the k
// selected columns (ascending, so the reads walk the row forwards).
// SUMSQ: the block also writes the sum of squares of the bf16 values of its slice of U, sumsq[mat * gridDim.x +
// blockIdx.x] -- one partial sum of ||U_mat||_F^2 per selected row (rows selected) or per row (columns).
template <typename MT, bool VEC, bool SUMSQ = false>
__global__ __launch_bounds__(256) void dion2_gather_kernel(PtrTab M, int mats_per_ptr, int rows,
                                                           int cols, int select_rows,
                                                           const int32_t* __restrict__ idx, int k,
                                                           float ef_decay, bf16_t* __restrict__ U,
                                                           float* __restrict__ sumsq = nullptr) {
  __shared__ float red[16];
  float ss = 0.f;
  const int mat = blockIdx.y;
  MT* m = (MT*)M.p[mat / mats_per_ptr] + (int64_t)(mat % mats_per_ptr) * rows * cols;
  const int32_t* id = idx + (int64_t)mat * k;
  if (select_rows) {
    const int j = blockIdx.x;
    MT* src = m + (int64_t)id[j] * cols;
    bf16_t* u = U + ((int64_t)mat * k + j) * cols;
    if (VEC) {
      for (int c4 = threadIdx.x; c4 < cols / 4; c4 += 256) {
        float v[4];
        st_load4<MT>(src, c4, v);
        st_store4<bf16_t>(u, c4, v);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (SUMSQ) {
            const float r = st_round<bf16_t>(v[e]);
            ss += r * r;
          }
          v[e] = __fmul_rn(v[e], ef_decay);
        }
        st_store4<MT>(src, c4, v);
      }
    } else {
      for (int c = threadIdx.x; c < cols; c += 256) {
        const float v = st_load<MT>(src, c);
        u[c] = f32_to_bf16(v);
        if (SUMSQ) {
          const float r = st_round<bf16_t>(v);
          ss += r * r;
        }
        st_store<MT>(src, c, __fmul_rn(v, ef_decay));
      }
    }
  } else {
    const int r = blockIdx.x;
    MT* src = m + (int64_t)r * cols;
    bf16_t* u = U + ((int64_t)mat * rows + r) * k;
    for (int j = threadIdx.x; j < k; j += 256) {
      const int c = id[j];
      const float v = st_load<MT>(src, c);
      u[j] = f32_to_bf16(v);
      if (SUMSQ) {
        const float q = st_round<bf16_t>(v);
        ss += q * q;
      }
      st_store<MT>(src, c, __fmul_rn(v, ef_decay));
    }
  }
  if (SUMSQ) {
    ss = block_sum(ss, red);
    if (threadIdx.x == 0) sumsq[(int64_t)mat * gridDim.x + blockIdx.x] = ss;
  }
}

// Columns selected from tall matrices, U written transposed ([k][rows]: the short side along rows, the
// layout the orthogonalization carries): one tile of 64 rows x 64 selected columns per workgroup, staged
// through LDS so that U^T rows leave as whole 128-byte runs.  sumsq[(mat * row_tiles + row tile) * (k / 64) +
// column tile]: sum of squares of the tile's bf16 values.  rows % 64 == 0, k % 64 == 0.
template <typename MT>
__global__ __launch_bounds__(256) void dion2_gather_cols_transposed_kernel(PtrTab M, int mats_per_ptr, int rows,
                                                                           int cols,
                                                                           const int32_t* __restrict__ idx, int k,
                                                                           float ef_decay, bf16_t* __restrict__ U,
                                                                           float* __restrict__ sumsq) {
  __shared__ __attribute__((aligned(16))) bf16_t tile[64][72];
  __shared__ float red[16];
  const int mat = blockIdx.z;
  MT* m = (MT*)M.p[mat / mats_per_ptr] + (int64_t)(mat % mats_per_ptr) * rows * cols;
  const int r0 = blockIdx.y * 64, j0 = blockIdx.x * 64;
  const int j = threadIdx.x & 63, rsub = threadIdx.x >> 6;
  const int c = idx[(int64_t)mat * k + j0 + j];
  float ss = 0.f;
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = st_load<MT>(m, (int64_t)(r0 + rsub + 4 * i) * cols + c);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const bf16_t b = f32_to_bf16(v[i]);
    tile[rsub + 4 * i][j] = b;
    const float q = bf16_to_f32(b);
    ss += q * q;
    st_store<MT>(m, (int64_t)(r0 + rsub + 4 * i) * cols + c, __fmul_rn(v[i], ef_decay));
  }
  ss = block_sum(ss, red);  // (its barriers also order the tile writes before the reads below)
  if (threadIdx.x == 0)
    sumsq[((int64_t)mat * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = ss;
  bf16_t* ut = U + (int64_t)mat * k * rows;
  const int chunk = threadIdx.x & 7, rr = threadIdx.x >> 3;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    const int col = rr + pass * 32;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      w[e] = (uint32_t)tile[chunk * 8 + 2 * e][col] | ((uint32_t)tile[chunk * 8 + 2 * e + 1][col] << 16);
    *(uint4*)(ut + (int64_t)(j0 + col) * rows + r0 + chunk * 8) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// The same U^T and decay with M += G in the same pass over whole rows: every element of M is read and written once, in
// whole lines.  A workgroup takes 64 rows and the columns from its 64 selected ones' first up to the next workgroup's
// (the outermost to the matrix's edge), both rounded down to 64 columns -- with ranges that ended inside a line the launch
// below took 1058 us.  It writes the selected columns that fall into its range (at most 127) and one partial sum of their
// squares; the partial sums of a matrix add up as those of the kernel above do.
// map [n_mat][cols]: position among the selected, or -1.  cols % 4 == 0, G and M 16-byte aligned, rows % 64 == 0, k % 64 == 0.
// Bound by HBM.  Beside norms that do not write M this moves 16 bytes an element of an fp32 momentum with bf16 gradients
// where accumulating first (715 us) and gathering a scattered quarter of every line (754) moved 18: 24 x (8192 x 2048).
template <typename GT, typename MT, bool NT>
__global__ __launch_bounds__(256) void dion2_add_gather_cols_kernel(PtrTab G, PtrTab M, int mats_per_ptr, int rows,
                                                                    int cols, const int32_t* __restrict__ idx,
                                                                    const int32_t* __restrict__ map, int k,
                                                                    float ef_decay, bf16_t* __restrict__ U,
                                                                    float* __restrict__ sumsq) {
  __shared__ __attribute__((aligned(16))) bf16_t tile[128][72];  // [selected column][row]
  __shared__ float red[16];
  const int mat = blockIdx.z, lane = threadIdx.x & 63;
  const int64_t base = (int64_t)(mat % mats_per_ptr) * rows * cols;
  const int r0 = blockIdx.y * 64, j0 = blockIdx.x * 64, j1 = j0 + 64;
  const GT* __restrict__ g = (const GT*)G.p[mat / mats_per_ptr] + base + (int64_t)r0 * cols;
  MT* __restrict__ m = (MT*)M.p[mat / mats_per_ptr] + base + (int64_t)r0 * cols;
  const int32_t* id = idx + (int64_t)mat * k;
  const int c_lo = j0 == 0 ? 0 : id[j0] & ~63, c_hi = j1 == k ? cols : id[j1] & ~63;
  // selected columns of the range: [s_lo, s_hi); at most 63 of those before a bound's own share its 64 columns
  const int s_lo = j0 - __popcll(__ballot(j0 > lane && id[j0 > lane ? j0 - 1 - lane : 0] >= c_lo));
  const int s_hi = j1 == k ? k : j1 - __popcll(__ballot(id[j1 - 1 - lane] >= c_hi));
  const int q0 = c_lo >> 2;
  const unsigned nq = (unsigned)((c_hi >> 2) - q0), total = nq * 64;  // groups of four columns a row, in the tile
  const int4* mp = (const int4*)(map + (int64_t)mat * cols) + q0;
  constexpr int B = 8;  // groups in flight a thread
  for (unsigned t0 = threadIdx.x; t0 < total; t0 += B * 256) {
    float mv[B][4], gv[B][4];
    int4 slot[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const unsigned t = t0 + b * 256;
      if (t >= total) continue;
      const unsigned row = t / nq, grp = t - row * nq;
      const int64_t i4 = (((int64_t)row * cols) >> 2) + q0 + grp;
      st_load4<MT, NT>(m, i4, mv[b]);
      st_load4<GT, NT>(g, i4, gv[b]);
      slot[b] = mp[grp];
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const unsigned t = t0 + b * 256;
      if (t >= total) continue;
      const unsigned row = t / nq, grp = t - row * nq;
      const int s[4] = {slot[b].x, slot[b].y, slot[b].z, slot[b].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        mv[b][e] = st_round<MT>(__fadd_rn(mv[b][e], gv[b][e]));
        if (s[e] >= s_lo && s[e] < s_hi) {
          tile[s[e] - s_lo][row] = f32_to_bf16(mv[b][e]);
          mv[b][e] = __fmul_rn(mv[b][e], ef_decay);
        }
      }
      st_store4<MT, NT>(m, (((int64_t)row * cols) >> 2) + q0 + grp, mv[b]);
    }
  }
  __syncthreads();
  bf16_t* ut = U + ((int64_t)mat * k + s_lo) * rows + r0;
  float ss = 0.f;
  for (int i = threadIdx.x; i < (s_hi - s_lo) * 8; i += 256) {
    const int col = i >> 3, chunk = i & 7;
    const u32x4_t w = *(const u32x4_t*)&tile[col][chunk * 8];
    *(u32x4_t*)(ut + (int64_t)col * rows + chunk * 8) = w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = __uint_as_float(w[e] << 16), hi = __uint_as_float(w[e] & 0xffff0000u);
      ss += lo * lo;
      ss += hi * hi;
    }
  }
  ss = block_sum(ss, red);
  if (threadIdx.x == 0) sumsq[((int64_t)mat * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = ss;
}

hipError_t launch_dion2_add_gather_cols(const PtrTab& G, int g_dtype, const PtrTab& M, int m_dtype, int n_mat,
                                        int mats_per_ptr, int rows, int cols, const int32_t* idx, const int32_t* map,
                                        int k, float ef_decay, bf16_t* U, float* sumsq, hipStream_t st) {
  const bool nt = exceeds_caches((int64_t)n_mat * rows * cols * ((m_dtype == 0 ? 2 : 4) + (g_dtype == 0 ? 2 : 4)));
  const dim3 grid(k / 64, rows / 64, n_mat);
#define ADDG_LAUNCH(GT, MT)                                                                                           \
  do {                                                                                                                \
    if (nt)                                                                                                           \
      hipLaunchKernelGGL((dion2_add_gather_cols_kernel<GT, MT, true>), grid, dim3(256), 0, st, G, M, mats_per_ptr, rows, \
                         cols, idx, map, k, ef_decay, U, sumsq);                                                      \
    else                                                                                                              \
      hipLaunchKernelGGL((dion2_add_gather_cols_kernel<GT, MT, false>), grid, dim3(256), 0, st, G, M, mats_per_ptr,    \
                         rows, cols, idx, map, k, ef_decay, U, sumsq);                                                \
  } while (0)
  if (g_dtype == 0) {
    if (m_dtype == 0) ADDG_LAUNCH(bf16_t, bf16_t); else ADDG_LAUNCH(bf16_t, float);
  } else {
    if (m_dtype == 0) ADDG_LAUNCH(float, bf16_t); else ADDG_LAUNCH(float, float);
  }
#undef ADDG_LAUNCH
  return hipGetLastError();
}

hipError_t launch_dion2_gather(const PtrTab& M, int m_dtype, int n_mat, int mats_per_ptr, int rows, int cols,
                               int select_rows, const int32_t* idx, int k, float ef_decay, bf16_t* U,
                               bool vec4, hipStream_t st) {
  dim3 grid(select_rows ? k : rows, n_mat);
#define GATHER_LAUNCH(MT, V)                                                                          \
  hipLaunchKernelGGL((dion2_gather_kernel<MT, V>), grid, dim3(256), 0, st, M, mats_per_ptr, rows, cols, \
                     select_rows, idx, k, ef_decay, U)
  if (m_dtype == 0) {
    if (vec4) GATHER_LAUNCH(bf16_t, true); else GATHER_LAUNCH(bf16_t, false);
  } else {
    if (vec4) GATHER_LAUNCH(float, true); else GATHER_LAUNCH(float, false);
  }
#undef GATHER_LAUNCH
  return hipGetLastError();
}

hipError_t launch_dion2_gather_prepared(const PtrTab& M, int m_dtype, int n_mat, int mats_per_ptr, int rows,
                                        int cols, int select_rows, const int32_t* idx, int k, float ef_decay,
                                        bf16_t* U, float* sumsq, bool vec4, hipStream_t st) {
  if (!select_rows && rows > k) {
    dim3 grid(k / 64, rows / 64, n_mat);
    if (m_dtype == 0)
      hipLaunchKernelGGL(dion2_gather_cols_transposed_kernel<bf16_t>, grid, dim3(256), 0, st, M, mats_per_ptr, rows,
                         cols, idx, k, ef_decay, U, sumsq);
    else
      hipLaunchKernelGGL(dion2_gather_cols_transposed_kernel<float>, grid, dim3(256), 0, st, M, mats_per_ptr, rows,
                         cols, idx, k, ef_decay, U, sumsq);
    return hipGetLastError();
  }
  dim3 grid(select_rows ? k : rows, n_mat);
#define GATHERS_LAUNCH(MT, V)                                                                               \
  hipLaunchKernelGGL((dion2_gather_kernel<MT, V, true>), grid, dim3(256), 0, st, M, mats_per_ptr, rows, cols, \
                     select_rows, idx, k, ef_decay, U, sumsq)
  if (m_dtype == 0) {
    if (vec4) GATHERS_LAUNCH(bf16_t, true); else GATHERS_LAUNCH(bf16_t, false);
  } else {
    if (vec4) GATHERS_LAUNCH(float, true); else GATHERS_LAUNCH(float, false);
  }
#undef GATHERS_LAUNCH
  return hipGetLastError();
}

// x = a*x - b*u[map] on selected slices, x = a*x elsewhere; one rounding of the sum.  u is bf16 or fp32 (UT).
template <typename UT>
static __device__ __forceinline__ float u_load(const UT* u, int64_t i) {
  return sizeof(UT) == 2 ? bf16_to_f32(((const bf16_t*)u)[i]) : ((const float*)u)[i];
}
struct Dion2PostArgs {
  const int32_t* map;
  const float *row_scale, *lr_dev, *adj_lr_dev, *wd_dev;
  float adj_ratio, wd_host;
};
// x = a*x - b*u
static __device__ __forceinline__ void dion2_post_coeffs(const Dion2PostArgs& p, float& a, float& b) {
  const float lr = *p.lr_dev;
  const float wd = p.wd_dev ? *p.wd_dev : p.wd_host;
  a = __fsub_rn(1.0f, __fmul_rn(lr, wd));
  b = __fmul_rn(p.adj_lr_dev ? *p.adj_lr_dev : lr, p.adj_ratio);
}

// Any size and alignment, one element at a time; block (row group of 8, mat).
template <typename UT, typename XT>
__global__ __launch_bounds__(256) void dion2_post_kernel(PtrTab X, int mats_per_ptr, int rows, int cols, int select_rows,
                                                         const UT* __restrict__ U, int k, Dion2PostArgs p) {
  const int mat = blockIdx.y;
  XT* x = (XT*)X.p[mat / mats_per_ptr] + (int64_t)(mat % mats_per_ptr) * rows * cols;
  float a, b0;
  dion2_post_coeffs(p, a, b0);
  const int32_t* mp = p.map + (int64_t)mat * (select_rows ? rows : cols);
  const UT* u = U + (int64_t)mat * (select_rows ? (int64_t)k * cols : (int64_t)rows * k);
  const int r_end = (blockIdx.x * 8 + 8) < rows ? (blockIdx.x * 8 + 8) : rows;
  for (int r = blockIdx.x * 8; r < r_end; ++r) {
    XT* xr = x + (int64_t)r * cols;
    const int jr = select_rows ? mp[r] : 0;
    // per-row scale of the selected slice (rows selected only): u is multiplied by it first
    const float b = p.row_scale && jr >= 0 ? __fmul_rn(b0, p.row_scale[(int64_t)mat * k + jr]) : b0;
    const UT* ur = u + (select_rows ? (int64_t)(jr < 0 ? 0 : jr) * cols : (int64_t)r * k);
    for (int c = threadIdx.x; c < cols; c += 256) {
      const int j = select_rows ? (jr < 0 ? -1 : c) : mp[c];
      const float uv = j >= 0 ? u_load<UT>(ur, j) : 0.f;
      st_store<XT>(xr, c, fmaf(a, st_load<XT>(xr, c), -(b * uv)));
    }
  }
}

// Rows selected, groups of W consecutive elements (8 of bf16 X where rows allow it: 16-byte accesses, else 4): a
// workgroup owns 8192 consecutive elements of a matrix whatever rows they lie in, a thread has sixteen elements of X (and,
// in the selected rows, of U) in flight.
// Bound by HBM (non-temporal past the caches).  24 x (2048 x 8192), k = 512, fp32 X: 682 us (5.0 TB/s) a row at a time ->
// 570 us (6.0 TB/s); bf16 X 363 -> 276 us.
constexpr int kPostRun = 8192;
template <bool NT, int W, typename UT, typename XT>
__global__ __launch_bounds__(256) void dion2_post_rows_kernel(PtrTab X, int mats_per_ptr, int rows, int cols,
                                                              const UT* __restrict__ U, int k, Dion2PostArgs p) {
  constexpr int N = 16 / W, kRound = 256 * N;  // groups per thread / per workgroup and round
  const int mat = blockIdx.y;
  const unsigned w = (unsigned)cols / W;
  const int64_t n = (int64_t)rows * w;
  XT* __restrict__ x = (XT*)X.p[mat / mats_per_ptr] + (int64_t)(mat % mats_per_ptr) * rows * cols;
  const int32_t* __restrict__ mp = p.map + (int64_t)mat * rows;
  const UT* __restrict__ u = U + (int64_t)mat * k * cols;
  for (int round = 0; round < kPostRun / (kRound * W); ++round) {
    const int64_t first = (int64_t)blockIdx.x * (kPostRun / W) + round * kRound;
    if (first >= n) return;
    const int row0 = (int)(first / w);
    const unsigned rem0 = (unsigned)(first - (int64_t)row0 * w);
    float v[N][W], uv[N][W], b[N];
    int j[N];
    unsigned c[N];
#pragma unroll
    for (int g = 0; g < N; ++g) {
      const unsigned q = threadIdx.x + g * 256;
      if (first + q < n) st_loadw<XT, W, NT>(x, first + q, v[g]);
      const unsigned dr = (rem0 + q) / w;
      c[g] = rem0 + q - dr * w;
      j[g] = first + q < n ? mp[row0 + dr] : -1;
    }
    float a, b0;
    dion2_post_coeffs(p, a, b0);
#pragma unroll
    for (int g = 0; g < N; ++g) {
#pragma unroll
      for (int e = 0; e < W; ++e) uv[g][e] = 0.f;
      b[g] = b0;
      if (j[g] >= 0) {
        st_loadw<UT, W>(u, (int64_t)j[g] * w + c[g], uv[g]);
        // per-row scale of the selected slice: u is multiplied by it first
        if (p.row_scale) b[g] = __fmul_rn(b0, p.row_scale[(int64_t)mat * k + j[g]]);
      }
    }
#pragma unroll
    for (int g = 0; g < N; ++g) {
#pragma unroll
      for (int e = 0; e < W; ++e) v[g][e] = fmaf(a, v[g][e], -(b[g] * uv[g][e]));
      if (first + threadIdx.x + g * 256 < n) st_storew<XT, W, NT>(x, first + threadIdx.x + g * 256, v[g]);
    }
  }
}

// Columns selected, groups of four: a workgroup owns `rpb` rows; their selected values, rpb * k consecutive elements of U,
// go through LDS (gathered from memory two bytes a lane they cost as much as X itself), a thread keeps its columns'
// positions in registers and has four rows of X in flight.
// Bound by HBM.  24 x (8192 x 2048), k = 512, fp32 X: 785 us (4.35 TB/s) with the gathers from memory -> 557 us (6.1 TB/s);
// bf16 X 605 -> 271 us.
template <bool NT, typename UT, typename XT>
__global__ __launch_bounds__(256) void dion2_post_cols_kernel(PtrTab X, int mats_per_ptr, int rows, int cols, int rpb,
                                                              const UT* __restrict__ U, int k, Dion2PostArgs p) {
  extern __shared__ float4 post_lds[];
  UT* lu = (UT*)post_lds;
  const int mat = blockIdx.y;
  const int r0 = blockIdx.x * rpb;
  const int nr = rows - r0 < rpb ? rows - r0 : rpb;
  XT* __restrict__ x = (XT*)X.p[mat / mats_per_ptr] + (int64_t)(mat % mats_per_ptr) * rows * cols + (int64_t)r0 * cols;
  const int32_t* __restrict__ mp = p.map + (int64_t)mat * cols;
  const UT* __restrict__ u = U + ((int64_t)mat * rows + r0) * k;
  const int nu = nr * k;
  const int nv = (((uintptr_t)u) & 15) == 0 ? nu * (int)sizeof(UT) / 16 : 0;  // whole 16-byte pieces
  for (int i = threadIdx.x; i < nv; i += 256) post_lds[i] = ((const float4*)u)[i];
  for (int i = nv * (16 / (int)sizeof(UT)) + threadIdx.x; i < nu; i += 256) lu[i] = u[i];
  float a, b;
  dion2_post_coeffs(p, a, b);
  __syncthreads();
  for (int c4 = threadIdx.x; c4 < cols / 4; c4 += 256) {
    const int4 j4 = *(const int4*)(mp + c4 * 4);
    const int j[4] = {j4.x, j4.y, j4.z, j4.w};
    int jl[4];  // (an unselected column reads the row's first value and drops it)
#pragma unroll
    for (int e = 0; e < 4; ++e) jl[e] = j[e] < 0 ? 0 : j[e];
    auto rows_of = [&](int r, int n) {
      float v[4][4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q < n) st_load4<XT, NT>(x, (((int64_t)(r + q) * cols) >> 2) + c4, v[q]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q >= n) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float uv = u_load<UT>(lu, (r + q) * k + jl[e]);
          v[q][e] = fmaf(a, v[q][e], -(b * (j[e] >= 0 ? uv : 0.f)));
        }
        st_store4<XT, NT>(x, (((int64_t)(r + q) * cols) >> 2) + c4, v[q]);
      }
    };
    int r = 0;
    for (; r + 4 <= nr; r += 4) rows_of(r, 4);
    for (; r < nr; ++r) rows_of(r, 1);
  }
}

constexpr int kPostLds = 32 * 1024;  // selected values of one workgroup's rows; five workgroups per CU

template <typename UT, typename XT>
static void dion2_post_dispatch(const PtrTab& X, int n_mat, int mats_per_ptr, int rows, int cols, int select_rows,
                                const UT* U, int k, const Dion2PostArgs& p, bool vec4, hipStream_t st) {
  const bool nt = exceeds_caches((int64_t)n_mat * rows * cols * 2 * (int)sizeof(XT));
  const int64_t wg = ((int64_t)rows * cols + kPostRun - 1) / kPostRun;
  if (vec4 && select_rows && wg <= (1 << 23)) {
    const dim3 grid((unsigned)wg, n_mat);
    const bool w8 = sizeof(XT) == 2 && cols % 8 == 0;
    auto* kernel = w8 ? (nt ? dion2_post_rows_kernel<true, 8, UT, XT> : dion2_post_rows_kernel<false, 8, UT, XT>)
                      : (nt ? dion2_post_rows_kernel<true, 4, UT, XT> : dion2_post_rows_kernel<false, 4, UT, XT>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, X, mats_per_ptr, rows, cols, U, k, p);
    return;
  }
  const int64_t row_bytes = (int64_t)k * sizeof(UT);
  if (vec4 && !select_rows && k > 0 && row_bytes <= kPostLds) {
    const int rpb = row_bytes * 8 <= kPostLds ? 8 : (row_bytes * 4 <= kPostLds ? 4 : 1);
    const dim3 grid((rows + rpb - 1) / rpb, n_mat);
    const size_t lds = (size_t)(rpb * row_bytes + 15) / 16 * 16;
    auto* kernel = nt ? dion2_post_cols_kernel<true, UT, XT> : dion2_post_cols_kernel<false, UT, XT>;
    hipLaunchKernelGGL(kernel, grid, dim3(256), lds, st, X, mats_per_ptr, rows, cols, rpb, U, k, p);
    return;
  }
  hipLaunchKernelGGL((dion2_post_kernel<UT, XT>), dim3((rows + 7) / 8, n_mat), dim3(256), 0, st, X, mats_per_ptr, rows, cols,
                     select_rows, U, k, p);
}

hipError_t launch_dion2_post(const PtrTab& X, int x_dtype, int n_mat, int mats_per_ptr, int rows, int cols,
                             int select_rows, const void* U, int u_dtype, int k, const int32_t* map,
                             const float* row_scale, const float* lr_dev, const float* adj_lr_dev,
                             float adj_ratio, const float* wd_dev, float wd_host, bool vec4,
                             hipStream_t st) {
  const Dion2PostArgs p{map, row_scale, lr_dev, adj_lr_dev, wd_dev, adj_ratio, wd_host};
#define D2POST(UT, XT) \
  dion2_post_dispatch<UT, XT>(X, n_mat, mats_per_ptr, rows, cols, select_rows, (const UT*)U, k, p, vec4, st)
  if (u_dtype == 0) {
    if (x_dtype == 0) D2POST(bf16_t, bf16_t); else D2POST(bf16_t, float);
  } else {
    if (x_dtype == 0) D2POST(float, bf16_t); else D2POST(float, float);
  }
#undef D2POST
  return hipGetLastError();
}

// map[m][idx[m][j]] = j for the k (distinct, unordered) int64 indices of every matrix, -1 elsewhere.
// One block per matrix: the fill and the scatter are separated by a block barrier.
__global__ __launch_bounds__(256) void dion2_index_map_kernel(const int64_t* __restrict__ idx, int k,
                                                              int dim, int32_t* __restrict__ map) {
  const int mat = blockIdx.x;
  int32_t* mp = map + (int64_t)mat * dim;
  for (int i = threadIdx.x; i < dim; i += 256) mp[i] = -1;
  __syncthreads();
  const int64_t* id = idx + (int64_t)mat * k;
  for (int j = threadIdx.x; j < k; j += 256) {
    const int64_t i = id[j];
    if (i >= 0 && i < dim) mp[i] = j;
  }
}

hipError_t launch_dion2_index_map(const int64_t* idx, int n_mat, int k, int dim, int32_t* map,
                                  hipStream_t st) {
  hipLaunchKernelGGL(dion2_index_map_kernel, dim3(n_mat), dim3(256), 0, st, idx, k, dim, map);
  return hipGetLastError();
}

}  // namespace dion
