// Whole Newton-Schulz / Polar-Express orthogonalization of one small matrix per workgroup, in registers
// from the Frobenius normalisation to the last iteration: the per-head regime (e.g. 64 x 768 attention
// heads), where the general path is 15 launches of GEMMs too small to fill a CU.
//
// Follows the same arithmetic as the batched driver (dion/newton_schulz_triton.py:508-522,
// dion/polar_express.py:30-50): X = bf16(G) / (||.||_F * s + eps); A = X X^T; B = c A A + b A + a I;
// X = B X, with A, B and X rounded to bf16 once per iteration and fp32 MFMA accumulation.
#include "elementwise.h"

namespace dion {

constexpr int kMaxLds = 160 * 1024 - 1024;  // dynamic LDS of one workgroup; the static part takes the rest

// ------------------------------------------------------------------------------------------
// A wavefront owns groups of 32 columns of X and keeps them as MFMA fragments: lane l of fragment x[g][t] holds row
// l % 16 of row tile t and eight columns of group g.  That is an operand of A = X X^T as it is (the reduction runs over
// columns, in any order both operands share), so the Gram product reads nothing.  X' = B X reduces over rows, which lie
// across lanes: a product with the identity (exact: one term of each sum is not zero) turns a fragment so that lanes
// run along columns, and X'^T = X^T B, with B symmetric, comes out in the layout x started in.  What crosses
// wavefronts is only A's partial sums, A and B (16 MT square), through LDS; X crosses memory once in and once out.
// Rows and columns are numbered so that the four consecutive indices a lane receives of each of two neighbouring 16-wide
// tiles are eight consecutive ones: 16 bytes a lane from and to memory, and 16-byte reads of B.
//
// MT row tiles (rows padded to 16 MT), at most KC column groups per wavefront (of which the first KF exist in every
// wavefront), NW wavefronts.  NW = 4 leaves room for two workgroups per CU: one's reduction and load phases run under the
// other's MFMAs.
//
// What bounds it, 432 x (64 x 768), 38.8 us: 16.8 us are the 84 MB in and out (5 TB/s, no iteration), 4.4 us an iteration of
// two matrices on one CU (20.6, 25.2, 29.6, 34.4, 38.8 us with one to five), of which 2.8 are MFMA time (the turning products
// are a quarter of it); the rest is the latency of three barriers and A's partial sums through LDS.  The form with X in
// LDS and one workgroup per CU took 55.0.
// 256 x (64 x 2048) 55 us, 300 x (128 x 768) 135, 200 x (80 x 1000) 54, 400 x (128 x 1024) 163, where the GEMM chain on
// matrices padded to 128 rows took many times that (1074, 724, 296 for the first three); 16 x (128 x 256) 42 against 90.
// ------------------------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(4))) unsigned rx4;
static __device__ __forceinline__ f32x4 mfma_rx(rx4 a, rx4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <typename T>
static __device__ __forceinline__ rx4 load8_bf16(const T* p) {
  if constexpr (sizeof(T) == 2) return *(const rx4*)p;
  else {
    const float4 a = ((const float4*)p)[0], b = ((const float4*)p)[1];
    return rx4{pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w), pack_bf16x2(b.x, b.y), pack_bf16x2(b.z, b.w)};
  }
}

template <int MT, int NW>
struct RegCfg {
  static constexpr int MR = MT * 16, AP = MR * 2 + 16;
  static constexpr int NTILE = MT * (MT + 1) / 2;   // tiles of the symmetric A
  static constexpr int PASSES = NTILE <= 10 ? 1 : NTILE <= 21 ? 3 : 4;
  static constexpr int GT = (NTILE + PASSES - 1) / PASSES;  // tiles of A summed across wavefronts at a time
  static constexpr int LDS = 2 * MR * AP + NW * GT * 1024;
};

template <int MT, int KC, int NW, int KF, typename T>
__global__ __launch_bounds__(NW * 64, 2) void ns_reg_kernel(const T* __restrict__ in, bf16_t* __restrict__ out, int rows,
                                                            int cols, NsCoeffs co, float norm_scale, float eps) {
  typedef RegCfg<MT, NW> C;
  constexpr int MR = C::MR, AP = C::AP, GT = C::GT, ST = MT / 2;
  // x takes 4 MT KC registers: past 96 a second turned group gains nothing (256 x (64 x 2048) 54.8 us, 54.7 with it; 400 x (128 x
  // 1024) 162 and 167)
  constexpr bool PIPE = MT * KC <= 24;
  // Matrices the GEMMs would take otherwise are not rounded after the scaling there, and so not here; the multiplications cost
  // 5 % of an iteration, which the shapes that never ran anywhere else (up to 64 x 1024) are spared.
  constexpr bool LATE = MT > 4 || KC * NW > 32;
  constexpr bool BREG = MT <= 4;  // B's fragments stay in registers over the column groups
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  __shared__ float red[NW];
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  char* const As = lds;
  char* const Bs = As + MR * AP;
  f32x4* const Ps = (f32x4*)(Bs + MR * AP);  // [wavefront][tile][lane]
  const bool tall = rows > cols;
  const int m = tall ? cols : rows, n = tall ? rows : cols;
  const int64_t first = (int64_t)blockIdx.x * rows * cols;
  const T* const src = in + first;
  bf16_t* const dst = out + first;
  const bool vec = cols % 8 == 0 && (((uintptr_t)in) & 15) == 0;
  const bool ovec = cols % 8 == 0 && (((uintptr_t)out) & 15) == 0;
  auto col0 = [&](int g) { return (wave + g * NW) * 32; };       // first column of the wavefront's group g
  auto absent = [&](int g) { return g >= KF && col0(g) >= n; };
  const int sub = 8 * (l16 >> 2) + (l16 & 3);                     // index l16 of tile 2 s + h is 32 s + sub + 4 h
  const uint32_t one = 0x3f80u;
  const uint32_t i0 = (4 * q == l16 ? one : 0u) | (4 * q + 1 == l16 ? one << 16 : 0u);
  const uint32_t i1 = (4 * q + 2 == l16 ? one : 0u) | (4 * q + 3 == l16 ? one << 16 : 0u);
  const rx4 eye[2] = {rx4{i0, i1, 0u, 0u}, rx4{0u, 0u, i0, i1}};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  // eight consecutive elements from `at` on, those at or past `left` zero
  auto fetch = [&](const T* at, bool ok, int left) -> rx4 {
    rx4 w = {0u, 0u, 0u, 0u};
    if (!ok) return w;
    if (vec) return load8_bf16<T>(at);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t lo = 0, hi = 0;
      if (2 * e < left) lo = sizeof(T) == 2 ? (uint32_t)(uint16_t)((const bf16_t*)at)[2 * e] : (uint32_t)(uint16_t)f32_to_bf16(((const float*)at)[2 * e]);
      if (2 * e + 1 < left) hi = sizeof(T) == 2 ? (uint32_t)(uint16_t)((const bf16_t*)at)[2 * e + 1] : (uint32_t)(uint16_t)f32_to_bf16(((const float*)at)[2 * e + 1]);
      w[e] = lo | (hi << 16);
    }
    return w;
  };
  auto store = [&](bf16_t* at, bool ok, int left, rx4 w) {
    if (!ok) return;
    if (ovec) {
      *(rx4*)at = w;
      return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (2 * e < left) at[2 * e] = (bf16_t)(w[e] & 0xffffu);
      if (2 * e + 1 < left) at[2 * e + 1] = (bf16_t)(w[e] >> 16);
    }
  };

  rx4 x[KC][MT];
  // ---- load.  A tall matrix lies with its columns contiguous: fetched with lanes along columns and turned.
#pragma unroll
  for (int g = 0; g < KC; ++g) {
    const int c0 = col0(g);
    if (!tall) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int r = 32 * (t >> 1) + sub + 4 * (t & 1), c = c0 + 8 * q;
        x[g][t] = fetch(src + (int64_t)r * cols + c, r < m && c < n, n - c);
      }
    } else {
      rx4 p[2][ST];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int s = 0; s < ST; ++s) {
          const int c = c0 + sub + 4 * h, r = 32 * s + 8 * q;
          p[h][s] = fetch(src + (int64_t)c * cols + r, r < m && c < n, m - r);
        }
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 d = mfma_rx(p[h][t >> 1], eye[t & 1], zero);
          x[g][t][2 * h] = pack_bf16x2(d[0], d[1]);
          x[g][t][2 * h + 1] = pack_bf16x2(d[2], d[3]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // Between two passes over x: without this the compiler keeps the values it unpacked for one as floats for the next, twice
  // the registers of x, and the forms of 96 and 128 registers of x went through scratch memory (up to 444 bytes a lane:
  // 256 x (64 x 2048) 72 us, 55 without; 256 x (32 x 4096) 73 and 52; 400 x (128 x 1024) 211 and 163).
  auto settle = [&]() {
    if constexpr (!LATE && MT * KC < 24) return;
#pragma unroll
    for (int g = 0; g < KC; ++g)
#pragma unroll
      for (int t = 0; t < MT; ++t) asm volatile("" : "+v"(x[g][t]));
  };
  // ---- Frobenius norm, scale
  float ss = 0.f;
#pragma unroll
  for (int g = 0; g < KC; ++g)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = __uint_as_float(x[g][t][e] << 16), hi = __uint_as_float(x[g][t][e] & 0xffff0000u);
        ss += lo * lo;
        ss += hi * hi;
      }
  settle();
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) total += red[w];
  const float sc = 1.0f / (sqrtf(total) * norm_scale + eps);
  // LATE: the factor rides on the fp32 sums of the first iteration, squared on A's and once on those of X'.  Scaled here, x is
  // rounded a second time, which the steep first polynomials carry far (16 x (128 x 256), singular values over 2.5 decades,
  // Polar-Express, distance to float64: 5.8e-2, and 4.1e-2 without; folded into B before B is rounded, it shifts all of B's
  // diagonal by one rounding, 64 x (32 x 4096) of Gaussian values 1.23e-2 -> 1.65e-2).  It is scaled here all the same where no
  // iteration follows and where sums of products of the values as they came would leave the normal range of fp32.
  const bool late = LATE && co.n > 0 && total > 0x1p-80f && total < 0x1p80f;
  if (!late) {
#pragma unroll
    for (int g = 0; g < KC; ++g)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          x[g][t][e] = pack_bf16x2(__uint_as_float(x[g][t][e] << 16) * sc, __uint_as_float(x[g][t][e] & 0xffff0000u) * sc);
    if (LATE) settle();
  }
  // (the same for every lane: say so, the factors live in scalar registers)
  auto uniform = [](float v) { return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v))); };
  float sa = uniform(late ? sc * sc : 1.0f), sx = uniform(late ? sc : 1.0f);

  // group g with lanes along columns: p[h][s] holds, of column tile h, the rows of tiles 2 s and 2 s + 1
  auto turn = [&](int g, rx4 (&p)[2][ST]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const f32x4 d = mfma_rx(x[g][t], eye[h], zero);
        p[h][t >> 1][2 * (t & 1)] = pack_bf16x2(d[0], d[1]);
        p[h][t >> 1][2 * (t & 1) + 1] = pack_bf16x2(d[2], d[3]);
      }
  };

  for (int it = 0; it < co.n; ++it) {
    const float a = co.c[it][0], b = co.c[it][1], c = co.c[it][2];
    // ---- A = X X^T, GT tiles at a time: every wavefront's share, then one wavefront per tile adds them in order
#pragma unroll
    for (int ps = 0; ps < C::PASSES; ++ps) {
      f32x4 acc[GT];
#pragma unroll
      for (int k = 0; k < GT; ++k) acc[k] = zero;
#pragma unroll
      for (int g = 0; g < KC; ++g) {
        if (absent(g)) continue;
#pragma unroll
        for (int t1 = 0; t1 < MT; ++t1)
#pragma unroll
          for (int t2 = t1; t2 < MT; ++t2) {
            const int k = t1 * MT - t1 * (t1 - 1) / 2 + (t2 - t1) - ps * GT;
            if (k >= 0 && k < GT) acc[k] = mfma_rx(x[g][t1], x[g][t2], acc[k]);
          }
      }
      if (ps > 0) __syncthreads();  // the sums of the tiles before have been read
#pragma unroll
      for (int k = 0; k < GT; ++k) Ps[(wave * GT + k) * 64 + lane] = acc[k];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < (GT + NW - 1) / NW; ++i) {
        const int k = wave + i * NW;
        if (k >= GT || ps * GT + k >= C::NTILE) continue;
        int t1 = 0, t2 = ps * GT + k;
        while (t2 >= MT - t1) {
          t2 -= MT - t1;
          ++t1;
        }
        t2 += t1;
        f32x4 s = Ps[k * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) s += Ps[(w * GT + k) * 64 + lane];
        if (LATE) s *= sa;
        const uint32_t w0 = pack_bf16x2(s[0], s[1]), w1 = pack_bf16x2(s[2], s[3]);
        const int row = 16 * t1 + 4 * q, col = 16 * t2 + l16;
        *(uint2*)(As + col * AP + row * 2) = make_uint2(w0, w1);
        if (t1 != t2) {
          *(uint16_t*)(As + row * AP + col * 2) = (uint16_t)w0;
          *(uint16_t*)(As + (row + 1) * AP + col * 2) = (uint16_t)(w0 >> 16);
          *(uint16_t*)(As + (row + 2) * AP + col * 2) = (uint16_t)w1;
          *(uint16_t*)(As + (row + 3) * AP + col * 2) = (uint16_t)(w1 >> 16);
        }
      }
    }
    __syncthreads();
    // ---- B = c A A + b A + a I.  A is symmetric, and so, bit for bit, is B: element (row, col) is stored as (col, row).
#pragma unroll 4
    for (int i = 0; i < (MT * MT + NW - 1) / NW; ++i) {
      const int u = wave + i * NW;
      if (MT * MT % NW != 0 && u >= MT * MT) continue;
      const int t1 = u / MT, t2 = u - t1 * MT;
      f32x4 acc = zero;
#pragma unroll
      for (int s = 0; s < ST; ++s)
        acc = mfma_rx(*(const rx4*)(As + (16 * t1 + l16) * AP + s * 64 + q * 16),
                      *(const rx4*)(As + (16 * t2 + l16) * AP + s * 64 + q * 16), acc);
      const int row = 16 * t1 + 4 * q, col = 16 * t2 + l16;
      const uint2 av = *(const uint2*)(As + col * AP + row * 2);
      float v[4];
      v[0] = c * acc[0] + b * __uint_as_float(av.x << 16);
      v[1] = c * acc[1] + b * __uint_as_float(av.x & 0xffff0000u);
      v[2] = c * acc[2] + b * __uint_as_float(av.y << 16);
      v[3] = c * acc[3] + b * __uint_as_float(av.y & 0xffff0000u);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (row + r == col) v[r] += a;
      // (columns of B in the order a turned fragment holds its rows)
      *(uint2*)(Bs + col * AP + (32 * (t1 >> 1) + 8 * q + 4 * (t1 & 1)) * 2) =
          make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    }
    __syncthreads();
    // ---- X = B X
    auto bfrag = [&](int t, int s) { return *(const rx4*)(Bs + (16 * t + l16) * AP + s * 64 + q * 16); };
    rx4 bf[BREG ? MT : 1][ST];
    if constexpr (BREG)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int s = 0; s < ST; ++s) bf[t][s] = bfrag(t, s);
    // (where the registers reach for it, the next group is turned beside the products of this one)
    rx4 p[2][2][ST];
    if (PIPE && !absent(0)) turn(0, p[0]);
#pragma unroll
    for (int g = 0; g < KC; ++g) {
      if (absent(g)) continue;
      if constexpr (!PIPE) turn(g, p[g & 1]);
      else if (g + 1 < KC && !absent(g + 1)) turn(g + 1, p[(g + 1) & 1]);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        rx4 b1[ST];
#pragma unroll
        for (int k = 0; k < ST; ++k) b1[k] = BREG ? bf[BREG ? t : 0][k] : bfrag(t, k);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          f32x4 acc = zero;
#pragma unroll
          for (int k = 0; k < ST; ++k) acc = mfma_rx(p[g & 1][h][k], b1[k], acc);
          if (LATE) acc *= sx;
          x[g][t][2 * h] = pack_bf16x2(acc[0], acc[1]);
          x[g][t][2 * h + 1] = pack_bf16x2(acc[2], acc[3]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // no more than two groups' temporaries at a time
    }
    sa = sx = 1.0f;
  }
  // ---- out
#pragma unroll
  for (int g = 0; g < KC; ++g) {
    if (absent(g)) continue;
    if (!tall) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int r = 32 * (t >> 1) + sub + 4 * (t & 1), c = col0(g) + 8 * q;
        store(dst + (int64_t)r * cols + c, r < m && c < n, n - c, x[g][t]);
      }
    } else {
      rx4 p[2][ST];
      turn(g, p);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int s = 0; s < ST; ++s) {
          const int c = col0(g) + sub + 4 * h, r = 32 * s + 8 * q;
          store(dst + (int64_t)c * cols + r, r < m && c < n, m - r, p[h][s]);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

template <int MT, int KC, int NW, int KF>
static hipError_t launch_reg(const void* in, int in_dtype, bf16_t* out, int batch, int rows, int cols, const NsCoeffs& co,
                             float norm_scale, float eps, hipStream_t st) {
  static std::atomic<uint64_t> done[2];
  constexpr int bytes = RegCfg<MT, NW>::LDS;
  static_assert(bytes <= kMaxLds, "");
  if (in_dtype == 0) {
    if (hipError_t e = set_max_dynamic_lds_once((const void*)ns_reg_kernel<MT, KC, NW, KF, bf16_t>, bytes, done[0])) return e;
    hipLaunchKernelGGL((ns_reg_kernel<MT, KC, NW, KF, bf16_t>), dim3(batch), dim3(NW * 64), bytes, st, (const bf16_t*)in, out,
                       rows, cols, co, norm_scale, eps);
  } else {
    if (hipError_t e = set_max_dynamic_lds_once((const void*)ns_reg_kernel<MT, KC, NW, KF, float>, bytes, done[1])) return e;
    hipLaunchKernelGGL((ns_reg_kernel<MT, KC, NW, KF, float>), dim3(batch), dim3(NW * 64), bytes, st, (const float*)in, out,
                       rows, cols, co, norm_scale, eps);
  }
  return hipGetLastError();
}

// Longest long side the kernel takes at a short side of m: 128 registers of X per lane; 0: none.
static int ns_reg_max_cols(int m) { return m <= 32 ? 4096 : m <= 64 ? 2048 : m <= 96 ? 1280 : m <= 128 ? 1024 : 0; }

hipError_t launch_ns_small(const void* in, int in_dtype, bf16_t* out, int batch, int rows, int cols, const NsCoeffs& co,
                           float norm_scale, float eps, hipStream_t st) {
  const int m = rows < cols ? rows : cols, n = rows < cols ? cols : rows;
  const int groups = (n + 31) / 32;
  // Up to a workgroup per CU eight wavefronts share a matrix (24 x (64 x 768): 26.8 -> 22.0 us), past that four, two
  // workgroups per CU.  The forms of 128 registers of X check every group for being there: the straight-line code of
  // the others makes the compiler keep more of them in flight than fit (256 x (64 x 2048) 55 -> 82 us).
  const bool wide = batch <= 256;
#define REG(MT, KC, NW, KF)                                                                               \
  if (groups <= KC * NW && groups >= KF * NW)                                                             \
  return launch_reg<MT, KC, NW, KF>(in, in_dtype, out, batch, rows, cols, co, norm_scale, eps, st)
  if (m <= 32) {
    if (!wide) {
      REG(2, 2, 4, 0); REG(2, 4, 4, 2); REG(2, 8, 4, 4);
    }
    REG(2, 4, 8, 0); REG(2, 8, 8, 4); REG(2, 16, 8, 0);
  } else if (m <= 64) {
    if (!wide) {
      REG(4, 2, 4, 0); REG(4, 4, 4, 2); REG(4, 6, 4, 4);
    }
    REG(4, 1, 8, 0); REG(4, 2, 8, 1); REG(4, 3, 8, 2); REG(4, 4, 8, 3); REG(4, 6, 8, 4); REG(4, 8, 8, 0);
  } else if (m <= 96) {
    REG(6, 2, 8, 0); REG(6, 3, 8, 2); REG(6, 4, 8, 3); REG(6, 5, 8, 0);
  } else if (m <= 128) {
    REG(8, 2, 8, 0); REG(8, 3, 8, 2); REG(8, 4, 8, 0);
  }
#undef REG
  return hipErrorInvalidValue;
}

// Short sides up to 64 and long sides up to 1024 whatever the batch.  Past that only batches of 16 and more, from 256 columns
// on (a group for every wavefront).  The line is where the widest matrices break even, a whole call in us, GEMM chain / this
// kernel: 128 x 1024, one of them 78 / 77, 15 85 / 79, 128 of them 196 (the chain before 64-wide tiles) / 82.  It is
// on the safe side for the others, which would gain below it too: 15 x (128 x 256) 71 / 43, 15 x (96 x 768) 83 / 43,
// 15 x (64 x 2048) 107 / 49, one of 32 x 4096 125 / 40, 16 x (128 x 128) 67 / 38, 128 x (96 x 192) 101 / 28.  Rows that are no
// multiple of 16 bytes are fetched element by element and lose at short batches: 16 x (100 x 500) 75 / 81.
bool ns_small_fits(int batch, int rows, int cols) {
  const int m = rows < cols ? rows : cols, n = rows < cols ? cols : rows;
  if (m <= 64 && n <= 1024) return true;
  return batch >= 16 && n >= 256 && n <= ns_reg_max_cols(m);
}

}  // namespace dion
