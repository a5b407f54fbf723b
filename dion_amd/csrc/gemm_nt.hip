// Batched bf16 GEMM for gfx950 (CDNA4):  C = alpha * P * Q^T + beta * D (+ diag * I), fp32 accumulate.
//
// Every GEMM of the Newton-Schulz / Polar-Express iteration is an instance of this one kernel:
//   A  = X X^T                     P = Q = X            (tri: upper tiles + mirrored store)
//   B  = c A A + b A + a I         P = Q = A (A = A^T)  (tri, D = A, a on the diagonal)
//   X' = B X  (= a X + (B - aI) X)  P = B, Q = X
// P is always read with the reduction index contiguous ("K-contiguous" rows).  Q comes in two forms:
// K-contiguous rows [N][K] like P (Q^T is then what multiplies P: the Gram products above, or
// X' = B X given X^T, which also stores (X')^T for the next round), or -- QK -- stored with the
// reduction index along rows, [K][N]: X' = B X then reads X as it lies, its MFMA fragments come from
// ds_read_b64_tr_b16 (transposing LDS read), and no X^T has to be kept or written.  QK is the form
// the orthogonalization driver uses.
// This replaces the reference's ns_line_1 / ns_line_2 / ns_line_3
// (dion/newton_schulz_triton.py:88-157, :206-287, :384-447) and the baddbmm of
// dion/newton_schulz_triton.py:557-563.
//
// Kernel structure: one workgroup per BM x BN output tile, WM x WN wavefronts (64 lanes) each
// owning a (BM/WM) x (BN/WN) sub-tile as 16x16 MFMA accumulators (v_mfma_f32_16x16x32_bf16: per
// FLOP half the accumulator register traffic of the 32x32x16 form, which on this power-limited part is
// worth 5 % of clock).  Operand tiles reach an LDS ring through direct-to-LDS loads, no VGPR staging: two slots
// filled by global_load_lds_dwordx4 with 256-wide tiles, two or four filled by buffer loads with 128-wide ones, and
// a two-slot ring of its own per wavefront with 64-wide ones (gemm_k64_kernel).  XOR swizzles keep the LDS writes and
// the fragment reads bank-conflict free.
#include <type_traits>

#include "common.h"

namespace dion {

#define LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
#define GLB_PTR(p) ((const __attribute__((address_space(1))) void*)(p))

template <int BM_, int BN_, int BK_, int WM_, int WN_, int NSTAGE_, bool AHEAD_ = false>
struct TileCfg {
  static constexpr bool AHEAD = AHEAD_;  // fragments of a whole slab requested one slab ahead (see the kernel)
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_, NSTAGE = NSTAGE_;
  static_assert(NSTAGE_ == 2 || (AHEAD_ && NSTAGE_ == 4), "two-slot ring, or a four-slot one for launches that leave a CU one workgroup");
  static constexpr int NT = WM * WN * 64;
  static constexpr int CPR = BK / 8;            // 16-byte chunks per tile row
  static constexpr int ROWS_PER_LOAD = NT / CPR; // tile rows covered by one load instruction
  static constexpr int P_BYTES = BM * BK * 2;
  static constexpr int Q_BYTES = BN * BK * 2;
  static constexpr int STAGE_BYTES = P_BYTES + Q_BYTES;
  // Epilogue staging of the transposed tile: per wavefront WTN rows of WTM bf16 (+16 B pad).
  static constexpr int STG_PITCH = (BM / WM_) * 2 + 16;
  static constexpr int STG_BYTES = (BN / WN_) * STG_PITCH;
  static constexpr int RING_BYTES = STAGE_BYTES * NSTAGE;
  static constexpr int LDS_BYTES =
      RING_BYTES > STG_BYTES * WM_ * WN_ ? RING_BYTES : STG_BYTES * WM_ * WN_;
  static constexpr int P_LOADS = BM / ROWS_PER_LOAD;
  static constexpr int Q_LOADS = BN / ROWS_PER_LOAD;
  static constexpr int LOADS_PER_STAGE = P_LOADS + Q_LOADS;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int TM = WTM / 16, TN = WTN / 16;  // 16 x 16 accumulator tiles of a wavefront tile
  static constexpr int ST = BK / 32;                  // 32-deep MFMA steps per slab
  // The MFMAs of a step run in halves of sixteen: four A fragments against the four B fragments.
  static constexpr int HALVES = TM / 4;
  static_assert(TN == 4 && (TM == 4 || TM == 8) && ST == 2, "wavefront tiles of 64 or 128 rows by 64 columns, 64-deep slabs");
  // gfx950 LDS: 64 banks x 4 B = 256-byte bank rows, and a ds_read_b128 is served 16 lanes at a
  // time.  16 consecutive tile rows must therefore land in 16 distinct 16-byte slots of a bank
  // row: the 256/(2*BK) tile rows that share a bank row take one swizzle value.
  static constexpr int SWZ_DIV = 256 / (BK * 2);
  static_assert(BM % ROWS_PER_LOAD == 0 && BN % ROWS_PER_LOAD == 0, "tile/threads mismatch");
  static_assert(CPR == 8 || CPR == 4, "BK must be 64 or 32");
};

// s_waitcnt with only vmcnt constrained (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8]
// | vmcnt_hi[15:14]).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | 0x0F70);
}

// Compile-time loop: f(std::integral_constant<int, I>()) for I in [I0, N).
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    static_for<I + 1, N>(f);
  }
}

// Issue order of the fragment reads.  A 32-deep step of a wavefront tile is HALVES halves of sixteen MFMAs
// (A fragment i = q / 4 against B fragment j = q % 4); a slab is ST steps, i.e. P = HALVES * ST halves.  While
// the MFMAs of one half issue, the fragments of the next half are requested behind them:
//   next half starts a step:   A0 B0 B1 B2 B3 A1 A2 A3 of that step, read r behind MFMA r, the order in
//                              which the MFMAs first need them;
//   next half is a second half: its A fragments 4..7, read r behind MFMA 4 r + 1 (B stays).
// Every fragment is requested fifteen or more MFMAs before its first use.  Every read is an assembly
// statement and so is every wait: the LDS returns in order, so "all but the newest N LDS instructions have
// returned" is exactly "the fragments MFMA q needs are in their registers", with N counted here from the
// issue order -- the LDS instructions issued after the later of the two fragments q needs.  Every MFMA
// carries its wait, also where an earlier one already covers its fragments: dropping those nine of sixteen
// measured 0.5-1.5 % slower on the polynomial and K-major launches.  (Left to the
// compiler, every group of MFMAs starts with a wait for all outstanding reads, the last of which was
// issued two MFMAs earlier.)  A K-major B fragment is two transposing reads.
template <int HALVES, int ST, bool QK>
struct FragSched {
  static constexpr int P = HALVES * ST, NM = 16;
  static constexpr bool issues_full(int hp) { return (hp + 1) % HALVES == 0; }
  static constexpr int read_behind(int hp, int q) {
    if (issues_full(hp)) return q < 8 ? q : -1;
    return (q % 4 == 1) ? q / 4 : -1;
  }
  static constexpr int instrs_full(int r) { return (QK && r >= 1 && r <= 4) ? 2 : 1; }
  static constexpr int lds_behind(int hp, int q) {
    const int r = read_behind(hp, q);
    if (r < 0) return 0;
    return issues_full(hp) ? instrs_full(r) : 1;
  }
  // LDS instructions that may still be outstanding when MFMA q of half hp issues
  static constexpr int allowed(int hp, int q) {
    const int i = q / 4, j = q % 4;
    const int prev = (hp + P - 1) % P;
    int need_q = 0;  // MFMA of the half before behind which the later of q's two fragments was requested
    if (hp % HALVES == 0) {
      const int ra = i == 0 ? 0 : 4 + i, rb = 1 + j;
      need_q = ra > rb ? ra : rb;
    } else {
      need_q = 4 * i + 1;  // A fragment 4 + i; the B fragments arrived a half earlier
    }
    int n = 0;
    for (int qq = need_q + 1; qq < NM; ++qq) n += lds_behind(prev, qq);
    for (int qq = 0; qq < q; ++qq) n += lds_behind(hp, qq);
    return n < 15 ? n : 15;  // lgkmcnt is a four-bit field; waiting for more than needed is harmless
  }
};

// Fragment wait: an asm statement that takes the fragments it guards as read-write operands, so that to
// the compiler they are (re)defined here and no use of them can be scheduled ahead of the wait.
template <int N>
__device__ __forceinline__ void frag_wait(bf16x8& a, bf16x8& b) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a), "+v"(b) : "n"(N));
}
// 16-byte LDS read at addr + OFF, issued from assembly (the compiler does not know it is in flight: the
// matching frag_wait is what its consumers wait on).
template <int OFF>
__device__ __forceinline__ void lds_read16(bf16x8& dst, uint32_t addr) {
  static_assert(OFF >= 0 && OFF < 65536, "ds offset field");
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
// K-major fragment: two transposing reads, rows k..k+3 and k+4..k+7 of the tile (HI bytes apart)
template <int OFF, int HI>
__device__ __forceinline__ void lds_read_tr(bf16x8& dst, uint32_t addr) {
  static_assert(OFF >= 0 && OFF + HI < 65536, "ds offset field");
  typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
  typedef __attribute__((ext_vector_type(4))) unsigned u32x4f;
  u32x2 lo, hi;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(addr), "n"(OFF));
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "n"(OFF + HI));
  const u32x4f v = {lo[0], lo[1], hi[0], hi[1]};
  dst = __builtin_bit_cast(bf16x8, v);
}

// Eight transposing reads and the wait for them in one statement (through the builtin, the compiler waits for every
// outstanding store before each of them).
typedef __attribute__((ext_vector_type(2))) unsigned tr_u32x2;
__device__ __forceinline__ void lds_read_tr8(tr_u32x2 (&d)[8], const uint32_t (&a)[8]) {
  asm volatile("ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %9\n\tds_read_b64_tr_b16 %2, %10\n\t"
               "ds_read_b64_tr_b16 %3, %11\n\tds_read_b64_tr_b16 %4, %12\n\tds_read_b64_tr_b16 %5, %13\n\t"
               "ds_read_b64_tr_b16 %6, %14\n\tds_read_b64_tr_b16 %7, %15\n\ts_waitcnt lgkmcnt(0)"
               : "=&v"(d[0]), "=&v"(d[1]), "=&v"(d[2]), "=&v"(d[3]), "=&v"(d[4]), "=&v"(d[5]), "=&v"(d[6]), "=&v"(d[7])
               : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7])
               : "memory");
}

// Enumeration of the upper triangle (ti <= tj) of a T x T tile grid in super-blocks of SB x SB
// tiles, so that the ~32 workgroups an XCD runs side by side touch as few distinct operand row
// blocks as possible (their L2 is what feeds the LDS): a diagonal super-block has SB(SB+1)/2
// tiles over only SB row blocks; an off-diagonal one is walked in SB x 4 column groups.
__device__ __forceinline__ void tri_tile(int t, int T, int& ti, int& tj) {
  constexpr int SB = 8;
  const int nb = (T + SB - 1) / SB;
  for (int I = 0; I < nb; ++I) {
    const int r = (T - I * SB) < SB ? (T - I * SB) : SB;  // tile rows in super-row I
    const int diag = r * (r + 1) / 2;
    if (t < diag) {
      // row-major triangle of side r
      int i = 0, rem = t;
      while (rem >= r - i) {
        rem -= r - i;
        ++i;
      }
      ti = I * SB + i;
      tj = I * SB + i + rem;
      return;
    }
    t -= diag;
    for (int J = I + 1; J < nb; ++J) {
      const int c = (T - J * SB) < SB ? (T - J * SB) : SB;
      const int cnt = r * c;
      if (t < cnt) {
        const int per_group = r * 4;
        const int g = t / per_group;
        const int gw = (c - g * 4) < 4 ? (c - g * 4) : 4;  // columns in this group
        const int tg = t - g * per_group;
        ti = I * SB + tg / gw;
        tj = J * SB + g * 4 + tg % gw;
        return;
      }
      t -= cnt;
    }
  }
  ti = tj = 0;  // unreachable for t < T(T+1)/2
}

// Quotient and remainder by a divisor the host knows: inv = (2^32 - 1) / d gives the quotient or one less for x < 2^31.
__device__ __forceinline__ int div_known(int x, int d, uint32_t inv, int& rem) {
  int q = (int)__umulhi((uint32_t)x, inv);
  rem = x - q * d;
  if (rem >= d) {
    rem -= d;
    ++q;
  }
  return q;
}

// Tile number `pid` of a launch of `total` tiles -> (batch, tile row, tile column).  Hardware deals workgroups
// round-robin over the 8 XCDs; each XCD (own L2) gets one contiguous run of the tile list, so that neighbours share
// operands, or -- xcd_interleave -- 32 consecutive tiles of every 256: the 8 XCDs then work on neighbouring tile
// groups (same matrix, same operand row panels) at the same time, and what one of them fetches from memory the
// others find in the memory-side cache.  The latter pays when a matrix's operands are much larger than an XCD's L2.
// Every workgroup starts with this, alone on its CU: no division by a number the host can divide by (four of them and
// the triangle's loop were 0.5 us of the 9 us a launch of 10 x (640 x 640) takes).
template <int BM, int BN, bool TRI>
__device__ __forceinline__ void tile_of(const GemmParams& p, int pid, int total, int& b, int& ti, int& tj) {
  const int tilesM = p.M / BM, tilesN = p.N / BN;
  int base = 0, lt;
  if constexpr (BM == 256) base = p.xcd_interleave ? total & ~255 : 0;  // (the only tiles that are interleaved)
  if (BM == 256 && pid < base) {
    const int j = pid & 255;
    lt = (pid & ~255) + (j & 7) * 32 + (j >> 3);
  } else {
    const int xcd = pid & 7, loc = (pid - base) >> 3;
    const int q = (total - base) >> 3, r = total & 7;
    lt = base + xcd * q + (xcd < r ? xcd : r) + loc;
  }
  int t;
  if constexpr (TRI) {
    b = div_known(lt, (tilesM * (tilesM + 1)) / 2, p.inv_mat, t);
    if (tilesM <= 8) {
      // row-major triangle: tile row i starts at i * tilesM - i (i - 1) / 2.  The root is off by less than one.  (Wider ones
      // stay in super-blocks: X X^T of one 768 x 3072 on 64-wide tiles 10.2 us so, 12.9 row by row.)
      const float e = (float)(2 * tilesM + 1);
      int i = (int)(0.5f * (e - __builtin_amdgcn_sqrtf(e * e - 8.0f * (float)t)));
      i = __builtin_amdgcn_readfirstlane(i);
      int start = i * tilesM - i * (i - 1) / 2;
      if (t < start) {
        --i;
        start -= tilesM - i;
      } else if (t >= start + tilesM - i) {
        start += tilesM - i;
        ++i;
      }
      ti = i;
      tj = i + t - start;
    } else {
      tri_tile(t, tilesM, ti, tj);
    }
  } else {
    constexpr int GM = 8;
    const int per_group = GM * tilesN;
    b = div_known(lt, tilesM * tilesN, p.inv_mat, t);
    int tg;
    const int first = div_known(t, per_group, p.inv_group, tg) * GM;
    if (tilesM - first >= GM) {
      ti = first + (tg & (GM - 1));
      tj = tg / GM;
    } else {
      int row;
      tj = div_known(tg, tilesM - first, p.inv_tail, row);
      ti = first + row;
    }
  }
  // (the same for every lane: say so, tile bases live in scalar registers)
  b = __builtin_amdgcn_readfirstlane(b);
  ti = __builtin_amdgcn_readfirstlane(ti);
  tj = __builtin_amdgcn_readfirstlane(tj);
}

// What tile_of needs of the host: the reciprocals of its divisors (tiles of a matrix, of a group of eight tile rows, rows
// of the last group), and the order of the list.
static void set_tile_order(GemmParams& p, int bm, int bn) {
  const int64_t tm = p.M / bm, tn = p.N / bn;
  const int64_t per_mat = p.tri ? tm * (tm + 1) / 2 : tm * tn;
  p.inv_mat = (uint32_t)(0xffffffffu / per_mat);
  p.inv_group = (uint32_t)(0xffffffffu / (8 * tn));
  p.inv_tail = tm % 8 ? (uint32_t)(0xffffffffu / (tm % 8)) : 0;
  // Interleaved 32-tile chunks for 256-wide tiles of large matrices.  us a launch, one contiguous run per XCD / interleaved:
  //  * symmetric products from 16 MB of X and reductions of 3584 on: X X^T of 32 x (4096 x 14336) 6364 / 5688, of 4 x 967 / 877, of
  //    12 x (2560 x 6912) 491 / 444, of 10 x (2304 x 9216) 461 / 415, of 20 x (1536 x 6144) 283 / 262, of 24 x (2048 x 8192)
  //    699 / 682, of 32 x (1024 x 8192) 328 / 323, A A of 5 x (5120 x 5120) 622 / 574; shorter ones 4 x (6144 x 2048) 252 / 271,
  //    8 x (3072 x 3072) 198 / 201.  (4 x (3584 x 3584), five iterations, 3310 / 3223 less 31 for the rest below.)
  //  * full products from 16 MB of B on: B X of 32 x (4096 x 14336) 11310 / 11064, of 5 x (5120 x 5120) 1055 / 976, between 386 /
  //    386 (8 x (3072 x 3072)) and 467 / 473 (4 x (3072 x 8192)).  (From 8 MB on, the walking kernel's 24 x (2048 x 8192) takes
  //    1306 / 1279 alone, but a whole step of such groups on two streams no less.)
  // 128-wide tiles are two to a CU, 64 of them side by side on an XCD: X X^T of 8 x (1024 x 14336) 132 / 164, of 2 x (2048 x 5504)
  // 62 / 68, of 40 x (1408 x 5632) 482 / 511.
  // The tiles past the last whole 256 are one contiguous run per XCD in either order: dealt out singly, no two workgroups
  // of an XCD shared an operand there (repeated on one operand, X X^T of 6 x (1024 x 8192), 216 tiles, 101 us instead of 53, of
  // 12 x (1536 x 6144) 180 instead of 141; B X of 32 x (4096 x 14336) 11208 instead of 11064).
  const int64_t p_mb = ((int64_t)p.M * p.K * 2) >> 20;
  if (bm != 256) p.xcd_interleave = 0;
  else p.xcd_interleave = p_mb >= 16 && (p.q_kmajor || p.K >= 3584) ? 1 : 0;
}

// Workgroup barrier preceded by the counter waits the software pipeline needs: every LDS read
// this wave issued has returned (the ring slot they read is about to be refilled) and all but the
// newest VM_LEFT direct-to-LDS loads of this wave have landed.  The "memory" clobber keeps the
// compiler from moving LDS accesses across it.
template <int VM_LEFT>
__device__ __forceinline__ void pipeline_barrier() {
  static_assert(VM_LEFT >= 0 && VM_LEFT < 64, "vmcnt range");
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  // vmcnt = VM_LEFT, lgkmcnt = 0, expcnt unconstrained (gfx9 s_waitcnt encoding).
  __builtin_amdgcn_s_waitcnt((VM_LEFT & 0xF) | ((VM_LEFT >> 4) << 14) | 0x0070);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

typedef __attribute__((ext_vector_type(4))) short s16x4;

// A pointer every lane holds the same value of, moved to scalar registers (where the compiler cannot
// prove uniformity it wraps each buffer access in a loop over the distinct values).
template <typename T>
__device__ __forceinline__ T* uniform_ptr(T* p) {
  const uint64_t v = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return (T*)(((uint64_t)hi << 32) | lo);
}

// Parameter accesses of the fused update go through buffer instructions: a descriptor based at the
// wavefront's tile of X (wave-uniform, scalar registers), a wave-uniform byte offset per instruction
// (scalar) and one per-lane byte offset shared by all accesses -- no 64-bit address per row in vector
// registers.  Offsets are 32-bit: the launcher checks that a wavefront tile spans less than 2 GiB.
typedef __attribute__((ext_vector_type(4))) unsigned bx_u32x4;
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t bx_resource(T* base) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)0xffffffffu, 0x00020000);
}
template <typename T>
__device__ __forceinline__ float bx_load(__amdgpu_buffer_rsrc_t rs, int lane_bytes, int uni_bytes) {
  if constexpr (sizeof(T) == 2)
    return bf16_to_f32((bf16_t)__builtin_amdgcn_raw_buffer_load_b16(rs, lane_bytes, uni_bytes, 0));
  else return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, lane_bytes, uni_bytes, 0));
}
template <typename T>
__device__ __forceinline__ void bx_store(__amdgpu_buffer_rsrc_t rs, int lane_bytes, int uni_bytes, float v) {
  if constexpr (sizeof(T) == 2)
    __builtin_amdgcn_raw_buffer_store_b16((unsigned short)f32_to_bf16(v), rs, lane_bytes, uni_bytes, 0);
  else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rs, lane_bytes, uni_bytes, 0);
}
// 16 bytes per lane.  A store of more than 8 bytes reads its data after it has issued: a VALU instruction that writes one of
// those registers within the next two wait states can get ahead of it, and the lanes read last store the new value.  The
// compiler keeps that distance where the store has no scalar offset and relies on the hardware where it has one; here it does not
// hold (32 wrong elements in 40 % of the tiles of a B X that had `v_mul v98` right behind a store of v[98:101]).  The
// statement behind the store keeps the data's registers until the distance is there.
__device__ __forceinline__ void bx_store_b128(__amdgpu_buffer_rsrc_t rs, int lane_bytes, int uni_bytes, bx_u32x4 o) {
  __builtin_amdgcn_raw_buffer_store_b128(o, rs, lane_bytes, uni_bytes, 0);
  asm volatile("s_nop 1" ::"v"(o));
}
// eight bf16 or four fp32 elements
template <typename T>
__device__ __forceinline__ void bx_load16(__amdgpu_buffer_rsrc_t rs, int lane_bytes, int uni_bytes, float* v) {
  const bx_u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(rs, lane_bytes, uni_bytes, 0);
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[2 * e] = __uint_as_float(w[e] << 16);
      v[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = __uint_as_float(w[e]);
  }
}
template <typename T>
__device__ __forceinline__ void bx_store16(__amdgpu_buffer_rsrc_t rs, int lane_bytes, int uni_bytes,
                                           const float* v) {
  bx_u32x4 o;
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = pack_bf16x2(v[2 * e], v[2 * e + 1]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = __float_as_uint(v[e]);
  }
  bx_store_b128(rs, lane_bytes, uni_bytes, o);
}

// POST: 0 stores the product; 1 / 2 feed it to the fused Muon update of fp32 / bf16 parameters
// (HAS_C then means "update X[row][col]", HAS_CT "update X[col][row]"; nothing else is stored).
template <int POST>
struct PostSel {
  typedef NoPost arg;
  typedef float xt;
};
template <>
struct PostSel<1> {
  typedef FusedPost arg;
  typedef float xt;
};
template <>
struct PostSel<2> {
  typedef FusedPost arg;
  typedef bf16_t xt;
};

// Lines of a staged transposed tile to a bounded destination (GemmParams::out_rows): EPL consecutive elements per lane
// (2 where every line starts on a pair), `stg` + line * pitch is line `line` of the tile, line < n_lines and element <
// n_elems are stored.  POST 0 stores bf16 values to dst + line * ld, else the Muon update of X is applied there: sixteen
// lines' parameters are requested before the first is updated (one at a time, every line cost a round trip to memory:
// 12 x (2730 x 1000) fp32 222 us a launch).
template <int EPL, int WIDTH, int LINES, int POST, typename XT>
__device__ __forceinline__ void store_lines_bounded(const char* stg, int pitch, int lane, XT* dst, int ld, int n_lines,
                                                    int n_elems, float pa, float pcoeff, float pb, int cautious) {
  constexpr int PL = WIDTH / EPL < 64 ? WIDTH / EPL : 64;  // lanes per line
  constexpr int LPP = 64 / PL;                             // lines per pass
  constexpr int EP = WIDTH / EPL / PL;                     // passes per line
  constexpr int NP = LINES / LPP, BI = NP < 16 ? NP : 16;  // passes, passes in flight
  static_assert(NP % BI == 0, "");
  const int l0 = lane / PL, e0 = (lane % PL) * EPL;
  typedef std::conditional_t<EPL == 1, XT, std::conditional_t<sizeof(XT) == 4, uint2, uint32_t>> raw_t;
#pragma unroll
  for (int ep = 0; ep < EP; ++ep) {
    const int el = e0 + ep * PL * EPL;
    if (el >= n_elems) continue;
    XT* const x = dst + (int64_t)l0 * ld + el;
    const char* const q = stg + l0 * pitch + el * 2;
#pragma unroll
    for (int c0 = 0; c0 < NP; c0 += BI) {
      raw_t xv[BI];
      if constexpr (POST != 0) {
#pragma unroll
        for (int k = 0; k < BI; ++k) {
          const int c = (c0 + k) * LPP;
          if (l0 + c < n_lines) xv[k] = *(const raw_t*)(x + (int64_t)c * ld);
        }
      }
#pragma unroll
      for (int k = 0; k < BI; ++k) {
        const int c = (c0 + k) * LPP;
        if (l0 + c >= n_lines) continue;
        raw_t* const o = (raw_t*)(x + (int64_t)c * ld);
        if constexpr (POST == 0) {
          *o = *(const raw_t*)(q + c * pitch);
        } else if constexpr (EPL == 2) {
          const uint32_t w = *(const uint32_t*)(q + c * pitch);
          float v[2];
          st_unpack2<XT>(xv[k], v);
          v[0] = muon_post_one(v[0], __uint_as_float(w << 16), pa, pcoeff, pb, cautious);
          v[1] = muon_post_one(v[1], __uint_as_float(w & 0xffff0000u), pa, pcoeff, pb, cautious);
          *o = st_pack2<XT>(v);
        } else {
          const float u = bf16_to_f32(*(const bf16_t*)(q + c * pitch));
          st_store<XT>((XT*)o, 0, muon_post_one(st_load<XT>(&xv[k], 0), u, pa, pcoeff, pb, cautious));
        }
      }
      if constexpr (POST != 0) asm volatile("" ::: "memory");  // the next batch of loads stays behind these stores
    }
  }
}

// BND: the destination is dense, p.out_rows x p.out_cols, and smaller than the padded product (GemmParams): the last
// product of a call then needs no pass that drops the padding (4 x (2730 x 1000): 22 us; 12 x: 100), and no separate
// update pass (65 us more).  256-wide tiles take this kernel for it, not the tile-walking one.
template <class Cfg, bool HAS_D, bool HAS_C, bool HAS_CT, bool QK = false, int POST = 0, bool BND = false>
__global__ __launch_bounds__(Cfg::NT, 2) void gemm_nt_kernel(const GemmParams p, const typename PostSel<POST>::arg post) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK;
  constexpr int TM = Cfg::TM, TN = Cfg::TN, ST = Cfg::ST, HALVES = Cfg::HALVES, NSTAGE = Cfg::NSTAGE;
  constexpr int HP = HALVES * ST;  // halves (sixteen MFMAs each) per slab
  constexpr int NM = 16;
  constexpr int LPS = Cfg::LOADS_PER_STAGE;
  static_assert(LPS <= NM / 2, "one refill load behind every second MFMA of a slab's last half");
  static_assert(!BND || (QK && !HAS_D && HAS_C != HAS_CT), "bounded destinations: the last product of a call");
  // Refill of the slot a slab occupied: all of it during the slab's last half, or -- the plain product of two
  // K-contiguous operands on 256-wide tiles, i.e. X X^T -- half then and half during the next slab's first half.
  // Measured: X X^T 2-3 % faster that way; the polynomial GEMM (its last refills bring the addend) 1 % slower, the
  // K-major form (two-instruction fragment reads in the same half) 3 % slower, 128-wide tiles 10 % slower.
  constexpr bool SPREAD = !QK && !HAS_D && BM == 256;
  extern __shared__ __attribute__((aligned(1024))) char lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;

  int b, ti, tj;
  constexpr bool TRI = HAS_C && HAS_CT && !QK;  // (the launcher's combinations)
  tile_of<BM, BN, TRI>(p, blockIdx.x, gridDim.x, b, ti, tj);
  const float factor = p.scale_vec ? p.scale_vec[b] : 1.0f;  // (requested here, used behind the main loop)

  // ---- global -> LDS addressing.  Chunk q = j*NT + tid of a tile lands at LDS byte q*16; it holds
  // logical 16-byte chunk (q % CPR) ^ swz(row) of tile row q / CPR.
  const int ld_row = tid / Cfg::CPR;
  const int ld_phys = tid % Cfg::CPR;
  const int ld_chunk = ld_phys ^ ((ld_row / Cfg::SWZ_DIV) % Cfg::CPR);
  const char* gP = (const char*)(p.P + (int64_t)b * p.strideP + (int64_t)(ti * BM) * p.ldp);
  // QK: the Q tile is BK rows (reduction index) of BN bf16; chunk q lands at LDS byte q*16 and holds
  // logical chunk ((c >> 2) ^ (row & 3)) << 2 | ((c & 3) ^ 2 * ((row >> 3) & 1)), c = q % QCPR, of tile row
  // q / QCPR: the four rows one transposing read gathers land in four distinct 64-byte bank groups, and
  // the rows 8 apart that neighbouring 16-lane groups read in the two 32-byte halves of a group.
  constexpr int QCPR = BN / 8;               // 16-byte chunks per K-major tile row
  constexpr int QROWS_PER_LOAD = Cfg::NT / QCPR;
  static_assert(!QK || (BK % QROWS_PER_LOAD == 0 && QROWS_PER_LOAD % 16 == 0), "K-major tile/threads");
  const int qk_row = tid / QCPR;
  const int qk_chunk = ((((tid % QCPR) >> 2) ^ (qk_row & 3)) << 2) | ((tid & 3) ^ (((qk_row >> 3) & 1) << 1));
  const char* gQ = QK ? (const char*)(p.Q + (int64_t)b * p.strideQ + tj * BN)
                      : (const char*)(p.Q + (int64_t)b * p.strideQ + (int64_t)(tj * BN) * p.ldq);
  uint32_t offP = (uint32_t)(ld_row * p.ldp + ld_chunk * 8) * 2u;
  uint32_t offQ = QK ? (uint32_t)(qk_row * p.ldq + qk_chunk * 8) * 2u
                           : (uint32_t)(ld_row * p.ldq + ld_chunk * 8) * 2u;
  const uint32_t stepP = (uint32_t)(Cfg::ROWS_PER_LOAD * p.ldp) * 2u;
  const uint32_t stepQ = (uint32_t)((QK ? QROWS_PER_LOAD : Cfg::ROWS_PER_LOAD) * p.ldq) * 2u;
  const int64_t slabQ = QK ? (int64_t)BK * p.ldq * 2 : (int64_t)BK * 2;  // bytes between k-slabs of Q
  const int KT = p.K / BK;

  // One direct-to-LDS load (index j of the LPS that make up a stage) of k-slab kt into ring
  // slot buf.  kt past the end re-fetches the last slab (never read): the refill count per stage
  // stays fixed, which is what the vmcnt bookkeeping in pipeline_barrier relies on.
  // A diagonal tile of a symmetric product of one matrix with itself (A = X X^T, A A) needs one operand
  // tile, not two: Q's loads are skipped and its fragments are read from P's half of the slot.  (With a
  // two-slot ring the barrier waits for every outstanding load, so the load count per slab is free to vary.)
  const bool one_operand = !QK && TRI && ti == tj && p.P == p.Q && p.ldp == p.ldq && p.strideP == p.strideQ;
  // LDS layout of the ring: [P slot 0][P slot 1][Q slot 0][Q slot 1].  With the two slots of an operand
  // side by side, slot, wavefront-tile row block and k step all fit the offset field of the LDS read
  // instructions: the per-lane address registers below are all the address arithmetic the loop needs.
  static_assert(Cfg::P_BYTES == Cfg::Q_BYTES, "square tiles: a one-operand tile reads Q's fragments from P's slots");
  auto issue_load = [&](int kt, int buf, int j) {
    if (one_operand && j >= Cfg::P_LOADS) return;
    const int k = kt < KT ? kt : KT - 1;
    char* l = lds + buf * Cfg::P_BYTES + wave * (64 * 16);
    // Address = wave-uniform 64-bit base (scalar registers; slab and load index folded in) + one 32-bit
    // per-lane offset per operand.  The empty asm (re)defines both right at the load, so that the
    // instruction is selected in its scalar-base form: left to the compiler, base and offset are
    // folded and hoisted out of the loop as a 64-bit address in vector registers per load.
    if (j < Cfg::P_LOADS) {
      const char* src = gP + (int64_t)k * (BK * 2) + (uint64_t)j * stepP;
      asm volatile("" : "+s"(src), "+v"(offP));
      __builtin_amdgcn_global_load_lds(GLB_PTR(src + offP), LDS_PTR(l + j * (Cfg::NT * 16)), 16, 0, 0);
    } else {
      const int jq = j - Cfg::P_LOADS;
      const char* src = gQ + k * slabQ + (uint64_t)jq * stepQ;
      asm volatile("" : "+s"(src), "+v"(offQ));
      __builtin_amdgcn_global_load_lds(GLB_PTR(src + offQ), LDS_PTR(l + NSTAGE * Cfg::P_BYTES + jq * (Cfg::NT * 16)),
                                       16, 0, 0);
    }
  };

  // ---- addend.  A wavefront fetches its part of D with direct-to-LDS loads into its own eighths of a ring slot that is
  // no longer needed: 64 rows of 128 bytes, load n brings rows 8 n .. 8 n + 7, the 16-byte chunk c of row r lies at
  // c ^ 2 * ((r >> 1) & 3), so that the transposing reads of the epilogue cover all banks.
  constexpr int D_LOADS = 8;
  static_assert(!HAS_D || LPS == D_LOADS, "a wavefront's share of a slot is 64 rows of 64 columns");
  const char* gD = HAS_D ? (const char*)(p.D + (int64_t)b * p.strideD + (int64_t)(ti * BM + wm * Cfg::WTM) * p.ldd +
                                         tj * BN + wn * Cfg::WTN)
                         : nullptr;
  uint32_t offD = HAS_D ? (uint32_t)((lane >> 3) * p.ldd + ((lane & 7) ^ ((lane >> 4) << 1)) * 8) * 2u : 0;
  auto issue_addend = [&](int buf, int h, int n) {  // rows 64 h + 8 n .. of the wavefront tile, into slot buf
    const char* src = gD + (int64_t)(h * 64 + n * 8) * p.ldd * 2;
    char* l = lds + buf * Cfg::P_BYTES + wave * (64 * 16) + (n & 3) * (Cfg::NT * 16) + (n >> 2) * (NSTAGE * Cfg::P_BYTES);
    asm volatile("" : "+s"(src), "+v"(offD));
    __builtin_amdgcn_global_load_lds(GLB_PTR(src + offD), LDS_PTR(l), 16, 0, 0);
  };

  // ---- LDS -> register fragment addressing.  A fragment of v_mfma_f32_16x16x32_bf16: lane l holds row (or
  // column) l % 16 and the eight reduction indices 8 * (l / 16) .. + 7 of a 32-deep step -- one 16-byte chunk.
  const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;
  const int l16 = lane & 15, quad = lane >> 4;
  const int fswz = (l16 / Cfg::SWZ_DIV) % Cfg::CPR;  // (every fragment's first row is a multiple of 16)
  uint32_t aoff[ST], boff[ST];
#pragma unroll
  for (int st = 0; st < ST; ++st) {
    const int chunk = ((st * 4 + quad) ^ fswz) * 16;
    aoff[st] = lds_base + (uint32_t)((wm * Cfg::WTM + l16) * (BK * 2) + chunk);
    boff[st] = lds_base + (uint32_t)((one_operand ? 0 : NSTAGE * Cfg::P_BYTES) + (wn * Cfg::WTN + l16) * (BK * 2) + chunk);
  }

  // QK fragments: a transposing read hands each 16-lane group a 4 (reduction index) x 16 (column) block, lane i
  // its column i; within the group, lane 4r+q addresses row r / 4-element piece q of the block.  Group g takes
  // reduction indices 8 g .. 8 g + 7 of the step (two reads of 4 rows); the 16 columns of fragment j are half
  // of a 64-byte group of the tile row; the swizzle keys the group on the row's index modulo 4 and the half
  // on bit 3 of the row (= g & 1), so the 32 lanes served together cover all 64 banks once.
  uint32_t qoff[TN];
  if (QK) {
    const int t16 = lane & 15;
#pragma unroll
    for (int j = 0; j < TN; ++j)
      qoff[j] = lds_base + (uint32_t)(NSTAGE * Cfg::P_BYTES + (8 * quad + (t16 >> 2)) * (BN * 2) +
                                      ((((wn * Cfg::WTN + j * 16) >> 5) ^ (t16 >> 2)) << 6) + ((j ^ quad) & 1) * 32 +
                                      (t16 & 3) * 8);
  }

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  typedef std::integral_constant<int, 0> ic0;

  if constexpr (Cfg::AHEAD) {
    // ---- main loop of 64 x 64 wavefront tiles (128-wide tiles).  A wavefront holds the fragments of a whole slab and
    // requests those of the next one behind this one's MFMAs: one wait and one barrier per slab, and the slot of a
    // slab is free for its refill a slab earlier than with fragments read half a slab ahead.  Four wavefronts share a
    // CU's four SIMDs here, or eight with two workgroups, so nothing hides what a wavefront issues besides its MFMAs:
    // an instruction costs four cycles, an MFMA sixteen, hence slots as constants of the unrolled loop and
    // refills without address arithmetic.  The LDS allows 0.3 us a slab: 64 KB of fragments and 32 KB of refills are
    // 750 cycles at 128 bytes per cycle, 512 are MFMA time.  Measured, X X^T of b x (1024 x K) on the four-slot ring, K from
    // 1024 to 4096: 0.28-0.31 us with up to 144 workgroups whatever the operands hold, 0.39 with 252.  Of those 0.39,
    // operands of zeros give back 0.07 (the clock, on this power-limited part) and one matrix for all workgroups 0.02-0.04 (the
    // way from memory to L2); both, 0.30.  (Half-slab fragments and accumulators in AGPRs, which the compiler copied
    // around every MFMA, took 0.42 where this takes 0.31: __launch_bounds__' second figure
    // keeps them out).  Short reductions pay for what is outside: first loads 1.3 us behind the tile's coordinates, the
    // epilogue 1.4.  X X^T of 12 x (768 x 3072) 27.1 -> 24.4 us, of 4 x (1024 x 2816) 23.1 -> 19.8, of 24 x (512 x 8192)
    // 62.6 -> 51.7, of 8 x (1024 x 4096), two workgroups per CU, 49.6 -> 41.2, of 10 x (640 x 640) 9.5 -> 8.3, A A of
    // those 10.6 -> 9.1, of 24 x (512 x 512) 10.4 -> 9.1; B X of 10 x (640 x 640) 9.5 -> 8.7.  256 x 128 tiles
    // on the same loop (eight wavefronts, three slots) take 0.57 us a slab for twice the work, in a launch longer than either
    // neighbour (12 x (768 x 768): 14.7 against 13.8 us).
    static_assert(TM == 4 && ST == 2 && LPS <= 8, "64 x 64 wavefront tiles");
    bf16x8 fa[2][ST][4], fb[2][ST][TN];  // by parity of the slab
    // read r (0..15) of the fragments of the slab in ring slot `slotc` (0, 1) of the pair the offsets point to
    auto read_frag = [&](auto slotc, auto rc) {
      constexpr int slot = decltype(slotc)::value, par = slot;
      constexpr int r = decltype(rc)::value, st = r / 8, f = r % 8;
      if constexpr (f < 4) lds_read16<slot * Cfg::P_BYTES + f * (16 * BK * 2)>(fa[par][st][f], aoff[st]);
      else if constexpr (QK) lds_read_tr<slot * Cfg::Q_BYTES + st * (32 * BN * 2), 4 * BN * 2>(fb[par][st][f - 4], qoff[f - 4]);
      else lds_read16<slot * Cfg::Q_BYTES + (f - 4) * (16 * BK * 2)>(fb[par][st][f - 4], boff[st]);
    };
    // every fragment of that parity has arrived
    auto landed = [&](auto parc) {
      auto& a = fa[decltype(parc)::value];
      auto& b = fb[decltype(parc)::value];
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(a[0][0]), "+v"(a[0][1]), "+v"(a[0][2]), "+v"(a[0][3]), "+v"(a[1][0]), "+v"(a[1][1]), "+v"(a[1][2]),
                     "+v"(a[1][3]));
      asm volatile("" : "+v"(b[0][0]), "+v"(b[0][1]), "+v"(b[0][2]), "+v"(b[0][3]), "+v"(b[1][0]), "+v"(b[1][1]),
                        "+v"(b[1][2]), "+v"(b[1][3]));
    };
    // Refills go through buffer descriptors, always LPS of them per slab.  Those past the last slab -- and all of Q's on a
    // tile that has one operand -- have a descriptor of no records, so they touch no memory; the loop is the same
    // code for every slab, and the waits are constants.  (With branches around the loads of the last slabs those slabs
    // ran in a second copy of the loop, cold, with a branch per load: X X^T of 10 x (640 x 640) had six of its ten slabs
    // there.)  The place behind the last slab is the addend's.
    const char *nextP = gP, *nextQ = gQ;  // what to load next
    uint32_t voff[LPS];
#pragma unroll
    for (int j = 0; j < LPS; ++j)
      voff[j] = j < Cfg::P_LOADS ? offP + j * stepP : QK ? offQ : offQ + (j - Cfg::P_LOADS) * stepQ;
    uint64_t rowsQ = QK ? stepQ : 0;  // between two loads of a K-major Q, 64 of whose rows may span more than a 32-bit offset
    const int keepQ = __builtin_amdgcn_readfirstlane(one_operand ? 0 : -1);
    int recsP = -1, recsQ = keepQ, nxt = 0;
    auto load = [&](int slot_at, auto jc) {  // slot_at: offset of the slot in either operand's half of the ring
      constexpr int j = decltype(jc)::value, jq = j < Cfg::P_LOADS ? 0 : j - Cfg::P_LOADS;
      const char* src = j < Cfg::P_LOADS ? nextP : QK ? nextQ + jq * rowsQ : nextQ;
      char* l = lds + slot_at + (j < Cfg::P_LOADS ? j * (Cfg::NT * 16) : NSTAGE * Cfg::P_BYTES + jq * (Cfg::NT * 16));
      const __amdgpu_buffer_rsrc_t rs =
          __builtin_amdgcn_make_buffer_rsrc((void*)src, 0, j < Cfg::P_LOADS ? recsP : recsQ, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS_PTR(l + wave * (64 * 16)), 16, (int)voff[j], 0, 0, 0);
    };
    auto loaded = [&]() {
      ++nxt;
      int left = nxt - KT;
      asm volatile("" : "+s"(left));  // (recognised as a comparison, its result would come through vector registers)
      recsP = left >> 31;  // all ones while there are slabs
      recsQ = recsP & keepQ;
      nextP += recsP & (BK * 2);
      nextQ += (int64_t)recsP & slabQ;
      if constexpr (HAS_D) {
        if (nxt == KT) {
          // loads 0-3 bring rows 0-31 of the wavefront's part of D, loads 4-7 rows 32-63
          nextP = gD;
          nextQ = gD + (int64_t)32 * p.ldd * 2;
          rowsQ = 0;
          recsP = recsQ = -1;
#pragma unroll
          for (int j = 0; j < LPS; ++j) voff[j] = offD + (uint32_t)((j & 3) * 8 * p.ldd) * 2u;
        }
      }
    };
    static_for<0, NSTAGE>([&](auto sc) {
      static_for<0, LPS>([&](auto jc) { load(decltype(sc)::value * Cfg::P_BYTES, jc); });
      loaded();
    });
    pipeline_barrier<(NSTAGE - 1) * LPS>();
    static_for<0, 16>([&](auto rc) { read_frag(ic0(), rc); });
    // Slab kt, in slot kt % NSTAGE: its fragments are on their way or there, slab kt + 1 has to be in the ring, and slab
    // kt + NSTAGE goes where this one was.  The loop is two slabs long; in a four-slot ring the addresses alternate
    // between the two pairs of slots.
    uint32_t to_pair = NSTAGE == 4 ? 2 * Cfg::P_BYTES : 0;  // from this pair to the other, then back
    int pair_at = 0;
    auto slab = [&](auto slotc) {
      constexpr int slot = decltype(slotc)::value;
      typedef std::integral_constant<int, slot ^ 1> nextc;
      pipeline_barrier<(NSTAGE - 2) * LPS>();
      landed(slotc);
      if constexpr (NSTAGE == 4 && slot == 1) {
#pragma unroll
        for (int st = 0; st < ST; ++st) {
          aoff[st] += to_pair;
          if (!QK) boff[st] += to_pair;
        }
        if (QK)
#pragma unroll
          for (int j = 0; j < TN; ++j) qoff[j] += to_pair;
      }
      __builtin_amdgcn_sched_barrier(0);
      static_for<0, 32>([&](auto qc) {
        constexpr int q = decltype(qc)::value, st = q / 16, i = (q % 16) / 4, j = q % 4;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[slot][st][i], fb[slot][st][j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        // a refill behind every E-th MFMA: spread over the slab, or early in it where it is needed a slab later
        constexpr int E = NSTAGE == 2 ? 2 : 4;
        constexpr bool refill = q % E == E - 1 && q / E < LPS;
        constexpr int before = q / E < LPS ? q / E : LPS;  // refills behind the MFMAs before this one
        constexpr int r = q - before;
        if constexpr (refill) load(pair_at + slot * Cfg::P_BYTES, std::integral_constant<int, q / E>());
        else if constexpr (r < 16) read_frag(nextc(), std::integral_constant<int, r>());
        __builtin_amdgcn_sched_barrier(0);
      });
      loaded();
      if constexpr (NSTAGE == 4 && slot == 1) {
        pair_at += (int)to_pair;
        to_pair = 0u - to_pair;
      }
    };
    for (int kt = 0; kt < KT; kt += 2) {  // (KT is even)
      slab(ic0());
      slab(std::integral_constant<int, 1>());
    }
    wait_vmcnt<0>();
    landed(ic0());  // the reads behind the last slab's MFMAs, which nobody uses, before their registers are let go
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        asm volatile("" ::"v"(fa[0][st][i]));
        asm volatile("" ::"v"(fb[0][st][i]));
      }
  } else {
    typedef FragSched<HALVES, ST, QK> FS;
    // A fragments: two sets of four, alternating by half; B fragments: two sets of TN, alternating by step
    bf16x8 fa[2][4], fb[2][TN];
    // Read r of the fragments half hn (0..HP-1) of ring slot buf needs: the first half of a step takes
    // A0 B0 B1 B2 B3 A1 A2 A3 (r = 0..7), a second half its A fragments 4..7 (r = 0..3).  All compile-time
    // constants, which end up in the instruction's offset field.
    auto read_frag = [&](auto bufc, auto hnc, auto rc) {
      constexpr int buf = decltype(bufc)::value, hn = decltype(hnc)::value, r = decltype(rc)::value;
      constexpr int st = hn / HALVES, part = hn % HALVES, fs = hn & 1, bs = st & 1;
      if constexpr (part != 0) {
        lds_read16<buf * Cfg::P_BYTES + (4 + r) * (16 * BK * 2)>(fa[fs][r], aoff[st]);
      } else if constexpr (r == 0 || r > 4) {
        constexpr int i = r == 0 ? 0 : r - 4;
        lds_read16<buf * Cfg::P_BYTES + i * (16 * BK * 2)>(fa[fs][i], aoff[st]);
      } else if constexpr (QK) {
        constexpr int j = r - 1;
        lds_read_tr<buf * Cfg::Q_BYTES + st * (32 * BN * 2), 4 * BN * 2>(fb[bs][j], qoff[j]);
      } else {
        constexpr int j = r - 1;
        lds_read16<buf * Cfg::Q_BYTES + j * (16 * BK * 2)>(fb[bs][j], boff[st]);
      }
    };

    // ---- prologue: fill one ring slot, wait for slab 0, read its first fragments, start the other slot.
    static_assert(NSTAGE == 2, "");
#pragma unroll
    for (int j = 0; j < LPS; ++j) issue_load(0, 0, j);
    pipeline_barrier<0>();
    static_for<0, 8>([&](auto rc) { read_frag(ic0(), ic0(), rc); });
#pragma unroll
    for (int j = 0; j < (SPREAD ? LPS / 2 : LPS); ++j) issue_load(1, 1, j);
    __builtin_amdgcn_sched_barrier(0);

    // ---- main loop.  Halves run back to back across slab boundaries: while the MFMAs of one half issue, the
    // fragment reads of the next half (and, from the last half of a slab on, the refill of the slot that slab
    // occupied) are slotted behind them.  sched_barrier pins that order.  KT is a multiple of NSTAGE
    // (launcher checks) so ring slots are compile-time constants.  The refills of the last round have no slab to
    // fetch: they bring the addend, whose 64-row blocks are as large as a wavefront's share of a slot.
    auto round = [&](int kt0, auto finalc) {
      static_for<0, NSTAGE * HP>([&](auto shc) {
        constexpr int s = decltype(shc)::value / HP, hp = decltype(shc)::value % HP;
        constexpr int st = hp / HALVES, part = hp % HALVES, fs = hp & 1, bs = st & 1;
        constexpr bool last = (hp == HP - 1);
        // slab kt+1 landed, slab kt fully read
        if constexpr (last) pipeline_barrier<(NSTAGE - 2) * LPS>();
        static_for<0, NM>([&](auto qc) {
          constexpr int q = decltype(qc)::value, i = q / 4, j = q % 4;
          frag_wait<FS::allowed(hp, q)>(fa[fs][i], fb[bs][j]);
          acc[part * 4 + i][j] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[fs][i], fb[bs][j], acc[part * 4 + i][j], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (FS::read_behind(hp, q) >= 0) {
            typedef std::integral_constant<int, FS::read_behind(hp, q)> rc;
            if constexpr (last) read_frag(std::integral_constant<int, (s + 1) % NSTAGE>(), ic0(), rc());
            else read_frag(std::integral_constant<int, s>(), std::integral_constant<int, hp + 1>(), rc());
          }
          if constexpr (SPREAD) {
            if constexpr (last && q % 4 == 3 && q / 4 < LPS / 2) issue_load(kt0 + s + NSTAGE, s, q / 4);
            if constexpr (hp == 0 && q % 4 == 3 && LPS / 2 + q / 4 < LPS)
              issue_load(kt0 + s - 1 + NSTAGE, (s + NSTAGE - 1) % NSTAGE, LPS / 2 + q / 4);
          } else if constexpr (last && (q & 1) && q / 2 < LPS) {
            if constexpr (HAS_D && decltype(finalc)::value) issue_addend(s, s, q / 2);
            else issue_load(kt0 + s + NSTAGE, s, q / 2);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      });
    };
    int kt0 = 0;
    for (; kt0 + (HAS_D ? NSTAGE : 0) < KT; kt0 += NSTAGE) round(kt0, std::false_type());
    if constexpr (HAS_D) round(kt0, std::true_type());
    wait_vmcnt<0>();  // drain the redundant tail refills before LDS is reused / the wave exits
    // The read-ahead of the last half issued reads whose results nobody uses.  The compiler does not know
    // they are in flight; were their destination registers dead here, it would hand them to whatever comes
    // next (the lane index, store addresses) and a read landing late would overwrite that.  So: wait for the
    // LDS queue to drain, and only then let go of the fragment registers -- the empty asm statements below
    // are their last use and sit behind the wait.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int f = 0; f < 2; ++f) {
#pragma unroll
      for (int i = 0; i < 4; ++i) asm volatile("" ::"v"(fa[f][i]));
#pragma unroll
      for (int j = 0; j < TN; ++j) asm volatile("" ::"v"(fb[f][j]));
    }
  }

  // ---- epilogue.  Accumulator element e of lane l holds row 4 * (l / 16) + e, column l % 16 of its 16 x 16
  // tile.  Whole tiles are stored: destinations are padded to the tile.
  const float alpha = gemm_alpha(p, factor), beta = p.beta;
  const int row_base = ti * BM + wm * Cfg::WTM;
  const int col_base = tj * BN + wn * Cfg::WTN;
  const bool mirror = HAS_CT && !(TRI && ti == tj);  // a diagonal tile is its own mirror
  const bool on_diag = TRI && ti == tj && p.diag != 0.0f;
  const int ldc = p.ldc, ldct = p.ldct;

  // Whole tiles.  C goes out straight from registers (16 lanes x 2 B = one 32-byte run per row and instruction, neighbouring
  // tiles completing the lines; staged through LDS and stored as 16 bytes per lane it took 0.3-0.5 us longer, two LDS
  // round trips with nothing beside them).  The transposed copy would be 8-byte pieces scattered over 16 rows per
  // instruction, so 64 x 64 blocks of it are staged [column][row] in the wavefront's own part of a ring slot nobody
  // reads any more.  The addend lies there already (see issue_addend); loaded here, 2 bytes per lane, it made the
  // epilogue 0.8 us longer.
  if constexpr (POST == 0 && !BND) {
    constexpr int PIECE = Cfg::NT * 16, FAR = NSTAGE * Cfg::P_BYTES;  // lines 8 n .. of a block: n % 4 pieces on, n / 4 far
    const int slot0 = Cfg::AHEAD ? KT % NSTAGE : 0;
    bf16_t* Cp = HAS_C ? p.C + (int64_t)b * p.strideC + (int64_t)(row_base + 4 * quad) * ldc + col_base + l16 : nullptr;
    const int line = (l16 >> 2), half = (l16 & 1) * 8, pair = (l16 >> 1) & 1;  // transposing reads: line of four, piece
    const int sw_w = ((l16 >> 1) & 1) << 1 | ((l16 >> 3) & 1) << 2 | ((l16 >> 2) & 1);
    static_for<0, TM / 4>([&](auto hc) {
      constexpr int h = decltype(hc)::value;
      char* const blk = lds + (slot0 + h) * Cfg::P_BYTES + wave * (64 * 16);
      const uint32_t blk_a = lds_base + (uint32_t)((slot0 + h) * Cfg::P_BYTES + wave * (64 * 16));
      tr_u32x2 dv[2][8];  // [row block / 2][row block % 2, column block]
      if constexpr (HAS_D) {
        // lane: column l16 of the tile, rows 4 quad ..: a transposing read over four rows of D
        const uint32_t q = blk_a + (quad >> 1) * PIECE + ((quad & 1) * 4 + line) * 128 + half;
        const int sw = ((line >> 1) | (quad & 1) << 1) << 1;
        uint32_t at[8];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) at[i * 4 + j] = q + i * 2 * PIECE + ((2 * j + pair) ^ sw) * 16;
        lds_read_tr8(dv[0], at);
#pragma unroll
        for (int r = 0; r < 8; ++r) at[r] += FAR;
        lds_read_tr8(dv[1], at);
      }
      // line j * 16 + l16 (a column) of the staged block: chunk c (rows 8 c ..) lies at c ^ f(column), so that the writes of
      // sixteen columns cover all banks
      char* const w = blk + (l16 >> 3) * PIECE + (l16 & 7) * 128 + (quad & 1) * 8;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = alpha * acc[h * 4 + i][j][e];
          if (HAS_D) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t d = dv[i >> 1][(i & 1) * 4 + j][e >> 1];
              v[e] = fmaf(alpha, acc[h * 4 + i][j][e], beta * __uint_as_float((e & 1) ? (d & 0xffff0000u) : (d << 16)));
            }
          }
          if (i == j && on_diag && row_base + h * 64 == col_base) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = l16 - 4 * quad == e ? v[e] + p.diag : v[e];
          }
          if (HAS_C) {
#pragma unroll
            for (int e = 0; e < 4; ++e) Cp[(int64_t)(h * 64 + i * 16 + e) * ldc + j * 16] = f32_to_bf16(v[e]);
          }
          if (!HAS_CT) continue;
          uint2 pk;
          pk.x = pack_bf16x2(v[0], v[1]);
          pk.y = pack_bf16x2(v[2], v[3]);
          *(uint2*)(w + (j & 1) * 2 * PIECE + (j >> 1) * FAR + (((2 * i + (quad >> 1)) ^ sw_w) * 16)) = pk;
        }
      asm volatile("" ::: "memory");
    });
    if (HAS_CT && mirror) {
      // lines of TM / 4 * 128 bytes
      constexpr int LL = TM * 2, LPI = 64 / LL;  // lanes per line, lines per instruction
      const int sub = lane / LL, h = (lane >> 3) & (TM / 4 - 1), ch = lane & 7;
      bf16_t* o = p.Ct + (int64_t)b * p.strideCt + (int64_t)(col_base + sub) * ldct + row_base + h * 64 + ch * 8;
      const char* blk = lds + (slot0 + h) * Cfg::P_BYTES + wave * (64 * 16) + sub * 128;
#pragma unroll
      for (int n = 0; n < 64 / LPI; ++n) {
        const int c = n * LPI + sub;
        const int sw = ((c >> 1) & 1) << 1 | ((c >> 3) & 1) << 2 | ((c >> 2) & 1);
        const int piece = n * LPI / 8, in_piece = n * LPI % 8;
        const uint4 q = *(const uint4*)(blk + (piece & 3) * PIECE + (piece >> 2) * FAR + in_piece * 128 + ((ch ^ sw) * 16));
        *(uint4*)(o + (int64_t)(n * LPI) * ldct) = q;
      }
    }
    return;
  }

  // BND: rows / columns of this wavefront's tile that exist; per lane, those left from its first row / column on
  const int rows_in = BND ? p.out_rows - row_base : 0, cols_in = BND ? p.out_cols - col_base : 0;
  const int lrows = rows_in - 4 * quad, lcols = cols_in - l16;
  typedef typename PostSel<POST>::xt XT;
  float pa = 0.f, pcoeff = 0.f, pb = 0.f;
  int pcautious = 0, pvec = 0;
  XT* xmat = nullptr;
  if constexpr (POST != 0) {
    const float lr = *post.lr_dev;
    const float wd = post.wd_dev ? *post.wd_dev : post.wd_host;
    muon_post_coeffs(lr, wd, post.adj_ratio, pa, pcoeff, pb);
    pcautious = post.cautious;
    pvec = post.vec_ok;
    const int pi = b / post.mats_per_ptr;
    xmat = (XT*)post.X.p[pi] + (int64_t)(b - pi * post.mats_per_ptr) * (HAS_C ? p.strideC : p.strideCt);
  }
  char* stg = lds + wave * Cfg::STG_BYTES;
  if (HAS_CT) __syncthreads();  // every wavefront is done with the operand ring

  if constexpr (POST != 0 && HAS_C) {
    // Update X[row][col] from registers.  The products are rounded to bf16 first, two per register,
    // which frees half of the accumulator registers: the parameter values of half a wavefront tile
    // are then loaded in one go (one round trip to memory per half, not one per tile).
    // 16 lanes x one element: a 64-byte (fp32) or 32-byte (bf16) run of X per row.
    uint32_t pk[TM][TN][2];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          pk[i][j][q] = pack_bf16x2(alpha * acc[i][j][2 * q], alpha * acc[i][j][2 * q + 1]);
    const __amdgpu_buffer_rsrc_t xr = bx_resource(uniform_ptr(xmat + (int64_t)row_base * ldc + col_base));
    const int xl = (4 * quad * ldc + l16) * (int)sizeof(XT);  // per lane
    constexpr int HM = BND ? 2 : TM / 2;
    auto run = [&](auto caut) {
      constexpr int CAUT = decltype(caut)::value;
#pragma unroll
      for (int i0 = 0; i0 < TM; i0 += HM) {
        float xv[HM][TN][4];
#pragma unroll
        for (int ii = 0; ii < HM; ++ii)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if constexpr (BND) {
                xv[ii][j][e] = 0.f;
                if ((i0 + ii) * 16 + e >= lrows || j * 16 >= lcols) continue;
              }
              xv[ii][j][e] = bx_load<XT>(xr, xl, (((i0 + ii) * 16 + e) * ldc + j * 16) * (int)sizeof(XT));
            }
#pragma unroll
        for (int ii = 0; ii < HM; ++ii)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if constexpr (BND)
                if ((i0 + ii) * 16 + e >= lrows || j * 16 >= lcols) continue;
              const uint32_t w = pk[i0 + ii][j][e >> 1];
              const float u = __uint_as_float((e & 1) ? (w & 0xffff0000u) : (w << 16));
              bx_store<XT>(xr, xl, (((i0 + ii) * 16 + e) * ldc + j * 16) * (int)sizeof(XT),
                           muon_post_one(xv[ii][j][e], u, pa, pcoeff, pb, CAUT));
            }
        asm volatile("" ::: "memory");  // the next batch of loads stays behind these stores
      }
    };
    if (pcautious) run(std::integral_constant<int, 1>());
    else run(std::integral_constant<int, 0>());
    return;
  }

  // (here: the update of a transposed parameter, or a bounded destination)
  bf16_t* Cp = HAS_C ? p.C + (int64_t)b * p.strideC + (int64_t)(row_base + 4 * quad) * ldc + col_base + l16 : nullptr;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = alpha * acc[i][j][e];
      if (HAS_C) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (i * 16 + e >= lrows || j * 16 >= lcols) continue;
          Cp[(int64_t)(i * 16 + e) * ldc + j * 16] = f32_to_bf16(v[e]);
        }
      }
      if (HAS_CT) {
        // four consecutive rows of column j * 16 + l16: 8 bytes of the staged [column][row] tile
        uint2 pk;
        pk.x = pack_bf16x2(v[0], v[1]);
        pk.y = pack_bf16x2(v[2], v[3]);
        *(uint2*)(stg + (j * 16 + l16) * Cfg::STG_PITCH + (i * 16 + 4 * quad) * 2) = pk;
      }
    }
  }
  if constexpr (BND && HAS_CT) {
    typedef std::conditional_t<POST == 0, bf16_t, XT> OT;
    OT* dst;
    bool pair = (ldct & 1) == 0;
    if constexpr (POST != 0) {
      dst = xmat + (int64_t)col_base * ldct + row_base;
      pair = pair && pvec;
    } else {
      dst = p.Ct + (int64_t)b * p.strideCt + (int64_t)col_base * ldct + row_base;
    }
    if (pair) store_lines_bounded<2, Cfg::WTM, Cfg::WTN, POST>(stg, Cfg::STG_PITCH, lane, dst, ldct, cols_in, rows_in, pa, pcoeff, pb, pcautious);
    else store_lines_bounded<1, Cfg::WTM, Cfg::WTN, POST>(stg, Cfg::STG_PITCH, lane, dst, ldct, cols_in, rows_in, pa, pcoeff, pb, pcautious);
  } else if constexpr (HAS_CT && POST != 0) {
    // The staged bf16 tile is the update.  One 16-byte access of X per lane and step (4 fp32 or 8 bf16
    // elements), lanes side by side along the row: every instruction covers whole contiguous runs.
    constexpr int EPL = 16 / (int)sizeof(XT);   // elements per lane
    constexpr int PCH = Cfg::WTM / EPL;          // lanes per staged row
    constexpr int PRPI = 64 / PCH;               // staged rows per instruction
    constexpr int NIT = Cfg::WTN / PRPI;
    constexpr int BI = NIT < (EPL == 4 ? 16 : 8) ? NIT : (EPL == 4 ? 16 : 8);
    static_assert(64 % PCH == 0 && Cfg::WTN % PRPI == 0 && NIT % BI == 0, "staged rows per wavefront");
    const int prow = lane / PCH, pchunk = lane % PCH;
    const char* pp = stg + prow * Cfg::STG_PITCH + pchunk * (EPL * 2);
    const __amdgpu_buffer_rsrc_t xr = bx_resource(uniform_ptr(xmat + (int64_t)col_base * ldct + row_base));
    const int xl = (prow * ldct + pchunk * EPL) * (int)sizeof(XT);  // per lane
    auto run = [&](auto caut) {
      constexpr int CAUT = decltype(caut)::value;
#pragma unroll
      for (int it0 = 0; it0 < NIT; it0 += BI) {
        float uv[BI][EPL], xv[BI][EPL];
#pragma unroll
        for (int k = 0; k < BI; ++k) {
          const char* q = pp + (it0 + k) * PRPI * Cfg::STG_PITCH;
          if constexpr (EPL == 8) st_load8<bf16_t>((const bf16_t*)q, 0, uv[k]);
          else st_load4<bf16_t>((const bf16_t*)q, 0, uv[k]);
        }
        if (pvec) {
#pragma unroll
          for (int k = 0; k < BI; ++k)
            bx_load16<XT>(xr, xl, (it0 + k) * PRPI * ldct * (int)sizeof(XT), xv[k]);
        } else {
#pragma unroll
          for (int k = 0; k < BI; ++k)
#pragma unroll
            for (int e = 0; e < EPL; ++e)
              xv[k][e] = bx_load<XT>(xr, xl, ((it0 + k) * PRPI * ldct + e) * (int)sizeof(XT));
        }
#pragma unroll
        for (int k = 0; k < BI; ++k)
#pragma unroll
          for (int e = 0; e < EPL; ++e) xv[k][e] = muon_post_one(xv[k][e], uv[k][e], pa, pcoeff, pb, CAUT);
        if (pvec) {
#pragma unroll
          for (int k = 0; k < BI; ++k)
            bx_store16<XT>(xr, xl, (it0 + k) * PRPI * ldct * (int)sizeof(XT), xv[k]);
        } else {
#pragma unroll
          for (int k = 0; k < BI; ++k)
#pragma unroll
            for (int e = 0; e < EPL; ++e)
              bx_store<XT>(xr, xl, ((it0 + k) * PRPI * ldct + e) * (int)sizeof(XT), xv[k][e]);
        }
      }
    };
    if (pcautious) run(std::integral_constant<int, 1>());
    else run(std::integral_constant<int, 0>());
  }
}

// ---------------------------------------------------------------------------------------------
// X' = P Q with Q stored [K][N] (the dominant launch of the iteration), one workgroup per CU walking a
// list of output tiles.  What the one-tile-per-workgroup kernel above pays at every tile boundary --
// the store acknowledgements a wavefront waits for before it may end, the dispatch of the next
// workgroup, and the latency of its first operand loads, together 5-8 us per 256x256 tile with the
// MFMA pipes idle -- is overlapped here:
//   * the operand ring runs on across tiles: the refills issued during the last two slabs of a tile
//     fetch the first two slabs of the workgroup's next tile, so the next tile's first MFMAs issue right
//     after this tile's epilogue;
//   * the epilogue goes through a private 4 KB LDS slice per wavefront next to the ring (not over
//     it: the ring is already receiving the next tile) and leaves as sixteen 16-byte stores per
//     lane, each instruction writing whole 128-byte lines.  Sixteen outstanding stores also stay countable
//     next to the ring's loads (the wait counter has six bits), and their acknowledgements come back
//     under the next tile's first slab.
// OUT_T false stores C[row][col]: the MFMA operands are swapped, so that a lane's four accumulator
// elements are four consecutive columns of one output row (8 bytes of a C row).
// OUT_T true stores Ct[col][row] (the product of a tall input, kept in the wide layout): operands
// in the usual order, the four elements are four consecutive rows = 8 bytes of a Ct row.
// Either way a staged chunk is 32 lines x 128 bytes from eight 16x16 accumulator tiles.
template <class Cfg, bool OUT_T>
__global__ __launch_bounds__(Cfg::NT) void gemm_qk_walk_kernel(const GemmParams p, const int total_tiles) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK;
  constexpr int TM = Cfg::TM, TN = Cfg::TN, ST = Cfg::ST, HALVES = Cfg::HALVES, NSTAGE = Cfg::NSTAGE;
  constexpr int HP = HALVES * ST, NM = 16, LPS = Cfg::LOADS_PER_STAGE;
  static_assert(NSTAGE == 2 && TM == 8 && TN == 4 && LPS <= NM / 2, "written for 128x64 wavefront tiles, two-slot ring");
  constexpr int STG_WAVE = 32 * 128;  // staging bytes per wavefront: 32 lines of 128 bytes
  extern __shared__ __attribute__((aligned(1024))) char lds[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WN, wn = wave % Cfg::WN;
  const int KT = p.K / BK;

  // ---- global -> LDS addressing (see the kernel above): per-lane offsets are the same for every tile,
  // the tile only moves the wave-uniform base pointers.
  const int ld_row = tid / Cfg::CPR;
  const int ld_phys = tid % Cfg::CPR;
  const int ld_chunk = ld_phys ^ ((ld_row / Cfg::SWZ_DIV) % Cfg::CPR);
  constexpr int QCPR = BN / 8;
  constexpr int QROWS_PER_LOAD = Cfg::NT / QCPR;
  static_assert(BK % QROWS_PER_LOAD == 0 && QROWS_PER_LOAD % 16 == 0, "K-major tile/threads");
  const int qk_row = tid / QCPR;
  const int qk_chunk = ((((tid % QCPR) >> 2) ^ (qk_row & 3)) << 2) | ((tid & 3) ^ (((qk_row >> 3) & 1) << 1));
  uint32_t offP = (uint32_t)(ld_row * p.ldp + ld_chunk * 8) * 2u;
  uint32_t offQ = (uint32_t)(qk_row * p.ldq + qk_chunk * 8) * 2u;
  const uint32_t stepP = (uint32_t)(Cfg::ROWS_PER_LOAD * p.ldp) * 2u;
  const uint32_t stepQ = (uint32_t)(QROWS_PER_LOAD * p.ldq) * 2u;
  const int64_t slabQ = (int64_t)BK * p.ldq * 2;

  int b_c, ti_c, tj_c, b_n, ti_n, tj_n;
  int pid = blockIdx.x;
  tile_of<BM, BN, false>(p, pid, total_tiles, b_c, ti_c, tj_c);
  auto base_p = [&](int b, int ti) { return (const char*)(p.P + (int64_t)b * p.strideP + (int64_t)(ti * BM) * p.ldp); };
  auto base_q = [&](int b, int tj) { return (const char*)(p.Q + (int64_t)b * p.strideQ + tj * BN); };
  const char* gP_c = base_p(b_c, ti_c);
  const char* gQ_c = base_q(b_c, tj_c);
  const char *gP_n = gP_c, *gQ_n = gQ_c;
  auto look_ahead = [&]() {
    // the tile after the current one; past the end of the list the current tile stands in (its slabs are
    // fetched again and never read, which keeps the load count per slab fixed)
    const int np = pid + (int)gridDim.x;
    if (np < total_tiles) {
      tile_of<BM, BN, false>(p, np, total_tiles, b_n, ti_n, tj_n);
      gP_n = base_p(b_n, ti_n);
      gQ_n = base_q(b_n, tj_n);
    } else {
      b_n = b_c; ti_n = ti_c; tj_n = tj_c;
      gP_n = gP_c; gQ_n = gQ_c;
    }
  };
  look_ahead();

  // slab kt of the current tile, or slab kt - KT of the next one, into ring slot buf (load j of LPS);
  // ring layout [P slot 0][P slot 1][Q slot 0][Q slot 1] as in the kernel above
  auto issue_load = [&](int kt, int buf, int j) {
    const bool nx = kt >= KT;
    const int k = nx ? kt - KT : kt;
    char* l = lds + buf * Cfg::P_BYTES + wave * (64 * 16);
    // wave-uniform base in scalar registers + one per-lane offset per operand (see the kernel above)
    if (j < Cfg::P_LOADS) {
      const char* src = (nx ? gP_n : gP_c) + (int64_t)k * (BK * 2) + (uint64_t)j * stepP;
      asm volatile("" : "+s"(src), "+v"(offP));
      __builtin_amdgcn_global_load_lds(GLB_PTR(src + offP), LDS_PTR(l + j * (Cfg::NT * 16)), 16, 0, 0);
    } else {
      const int jq = j - Cfg::P_LOADS;
      const char* src = (nx ? gQ_n : gQ_c) + k * slabQ + (uint64_t)jq * stepQ;
      asm volatile("" : "+s"(src), "+v"(offQ));
      __builtin_amdgcn_global_load_lds(GLB_PTR(src + offQ), LDS_PTR(l + NSTAGE * Cfg::P_BYTES + jq * (Cfg::NT * 16)), 16, 0, 0);
    }
  };

  // ---- LDS -> register fragments (see the kernel above)
  const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds;
  const int l16 = lane & 15, quad = lane >> 4;
  const int fswz = (l16 / Cfg::SWZ_DIV) % Cfg::CPR;
  uint32_t aoff[ST];
#pragma unroll
  for (int st = 0; st < ST; ++st)
    aoff[st] = lds_base + (uint32_t)((wm * Cfg::WTM + l16) * (BK * 2) + ((st * 4 + quad) ^ fswz) * 16);
  uint32_t qoff[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j)
    qoff[j] = lds_base + (uint32_t)(NSTAGE * Cfg::P_BYTES + (8 * quad + (l16 >> 2)) * (BN * 2) +
                                    ((((wn * Cfg::WTN + j * 16) >> 5) ^ (l16 >> 2)) << 6) + ((j ^ quad) & 1) * 32 +
                                    (l16 & 3) * 8);
  typedef FragSched<HALVES, ST, true> FS;
  bf16x8 fa[2][4], fb[2][TN];
  auto read_frag = [&](auto bufc, auto hnc, auto rc) {
    constexpr int buf = decltype(bufc)::value, hn = decltype(hnc)::value, r = decltype(rc)::value;
    constexpr int st = hn / HALVES, part = hn % HALVES, fs = hn & 1, bs = st & 1;
    if constexpr (part != 0) {
      lds_read16<buf * Cfg::P_BYTES + (4 + r) * (16 * BK * 2)>(fa[fs][r], aoff[st]);
    } else if constexpr (r == 0 || r > 4) {
      constexpr int i = r == 0 ? 0 : r - 4;
      lds_read16<buf * Cfg::P_BYTES + i * (16 * BK * 2)>(fa[fs][i], aoff[st]);
    } else {
      constexpr int j = r - 1;
      lds_read_tr<buf * Cfg::Q_BYTES + st * (32 * BN * 2), 4 * BN * 2>(fb[bs][j], qoff[j]);
    }
  };
  typedef std::integral_constant<int, 0> ic0;

  f32x4 acc[TM][TN];
  auto clear_acc = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  clear_acc();

  // ---- epilogue addressing: lane = (line l16 of a tile, 8-byte piece quad) when staging, (line rl, 16-byte
  // piece rq) when storing
  char* stg = lds + Cfg::RING_BYTES + wave * STG_WAVE;
  const int rl = lane >> 3, rq = lane & 7;
  const int ld_out = OUT_T ? p.ldct : p.ldc;

  auto store_tile = [&](int b, int ti, int tj) {
    const int row_base = ti * BM + wm * Cfg::WTM;
    const int col_base = tj * BN + wn * Cfg::WTN;
    bf16_t* out = OUT_T ? p.Ct + (int64_t)b * p.strideCt + (int64_t)col_base * ld_out + row_base
                        : p.C + (int64_t)b * p.strideC + (int64_t)row_base * ld_out + col_base;
    const __amdgpu_buffer_rsrc_t rs = bx_resource(uniform_ptr(out));
    const int lane_bytes = (rl * ld_out + rq * 8) * 2;
    const float alpha = gemm_alpha(p, p.scale_vec ? p.scale_vec[b] : 1.0f);  // 1 unless a per-matrix factor rides on this launch
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      // chunk c: 32 output lines of 128 bytes.  OUT_T false: C rows 32 c .. 32 c + 31 of the wavefront tile
      // (accumulator tiles i = 2 c, 2 c + 1, all j); OUT_T true: Ct lines = C columns 32 (c / 2) .. + 31
      // (j = 2 (c / 2), + 1) by C rows 64 (c % 2) .. + 63 (i = 4 (c % 2) .. + 3).
      const int line0 = OUT_T ? (c >> 1) * 32 : c * 32;   // first output line of the chunk (relative)
      const int run0 = OUT_T ? (c & 1) * 64 : 0;          // first element of the chunk within a line
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const f32x4& a = OUT_T ? acc[4 * (c & 1) + (t & 3)][2 * (c >> 1) + (t >> 2)] : acc[2 * c + (t >> 2)][t & 3];
        uint2 pk;
        pk.x = pack_bf16x2(alpha * a[0], alpha * a[1]);
        pk.y = pack_bf16x2(alpha * a[2], alpha * a[3]);
        // 8-byte piece 4 (t % 4) + quad of line 16 (t / 4) + l16; XOR with twice the line pair number spreads
        // the 16 lines of half a wavefront over all 64 banks and keeps 16-byte pairs together
        const int line = 16 * (t >> 2) + l16;
        *(uint2*)(stg + line * 128 + (((4 * (t & 3) + quad) ^ (((line >> 1) & 7) << 1)) << 3)) = pk;
      }
      asm volatile("" ::: "memory");
      uint4 v[4];
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int line = rl + 8 * it;
        v[it] = *(const uint4*)(stg + line * 128 + (((2 * rq) ^ (((line >> 1) & 7) << 1)) << 3));
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const bx_u32x4 o = {v[it].x, v[it].y, v[it].z, v[it].w};
        bx_store_b128(rs, lane_bytes, ((line0 + 8 * it) * ld_out + run0) * 2, o);
      }
    }
  };

  // ---- prologue: slab 0 of the first tile, its first fragments, slab 1
#pragma unroll
  for (int j = 0; j < LPS; ++j) issue_load(0, 0, j);
  pipeline_barrier<0>();
  static_for<0, 8>([&](auto rc) { read_frag(ic0(), ic0(), rc); });
#pragma unroll
  for (int j = 0; j < LPS; ++j) issue_load(1, 1, j);
  __builtin_amdgcn_sched_barrier(0);

  for (;;) {
    // ---- one tile: the main loop of the kernel above; refills past the tile's last slab fetch the next tile
    for (int kt0 = 0; kt0 < KT; kt0 += NSTAGE) {
      static_for<0, NSTAGE * HP>([&](auto shc) {
        constexpr int s = decltype(shc)::value / HP, hp = decltype(shc)::value % HP;
        constexpr int st = hp / HALVES, part = hp % HALVES, fs = hp & 1, bs = st & 1;
        constexpr bool last = (hp == HP - 1);
        if constexpr (last) pipeline_barrier<0>();
        static_for<0, NM>([&](auto qc) {
          constexpr int q = decltype(qc)::value, i = q / 4, j = q % 4;
          frag_wait<FS::allowed(hp, q)>(fa[fs][i], fb[bs][j]);
          if constexpr (OUT_T)
            acc[part * 4 + i][j] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[fs][i], fb[bs][j], acc[part * 4 + i][j], 0, 0, 0);
          else
            acc[part * 4 + i][j] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[bs][j], fa[fs][i], acc[part * 4 + i][j], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (FS::read_behind(hp, q) >= 0) {
            typedef std::integral_constant<int, FS::read_behind(hp, q)> rc;
            if constexpr (last) read_frag(std::integral_constant<int, (s + 1) % NSTAGE>(), ic0(), rc());
            else read_frag(std::integral_constant<int, s>(), std::integral_constant<int, hp + 1>(), rc());
          }
          if constexpr (last && (q & 1) && q / 2 < LPS) issue_load(kt0 + s + NSTAGE, s, q / 2);
          __builtin_amdgcn_sched_barrier(0);
        });
      });
    }
    // The first fragments of the next tile are on their way into set 0.  Let them land before the epilogue:
    // its register traffic must not meet a transposing read still in flight.
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(fa[0][0]), "+v"(fa[0][1]), "+v"(fa[0][2]), "+v"(fa[0][3]), "+v"(fb[0][0]), "+v"(fb[0][1]),
                   "+v"(fb[0][2]), "+v"(fb[0][3]));
    store_tile(b_c, ti_c, tj_c);
    pid += (int)gridDim.x;
    if (pid >= total_tiles) break;
    clear_acc();
    b_c = b_n; ti_c = ti_n; tj_c = tj_n;
    gP_c = gP_n; gQ_c = gQ_n;
    look_ahead();
    __builtin_amdgcn_sched_barrier(0);
  }
  wait_vmcnt<0>();  // the stand-in refills of the last tile must land before the LDS is given back
}

// ---------------------------------------------------------------------------------------------
// The same product for launches of few tiles: 64 x 64 tiles, the reduction of a tile split over the four
// wavefronts of its workgroup.  With a handful of 128-wide tiles most CUs idle and each busy one walks the whole
// reduction at the pace of its own operand stream (0.3-0.4 us per 64-deep slab, 64 slabs for 1024 x 4096); four times
// as many tiles, each pulling a quarter of the bytes at once through four private rings, use the CUs that are
// there.  A wavefront takes every fourth slab (64 x 64 of each operand) into a two-slot ring of its own and never
// meets a barrier until its partial sums are added; the 64 x 64 wavefront tile keeps the fragment schedule of the
// 128-wide kernel.  Per CU 64 KB of loads stay in flight.
struct CfgK64 {
  static constexpr int BM = 64, BN = 64, BK = 64, NT = 256, KW = 4;  // KW wavefronts share a reduction
  static constexpr int OP_BYTES = 64 * 64 * 2;                       // one operand of one slab
  static constexpr int WAVE_BYTES = 4 * OP_BYTES;                    // [P slot 0][P slot 1][Q slot 0][Q slot 1]
  static constexpr int STG_PITCH = 64 * 2 + 16;
  static constexpr int LDS_BYTES = KW * WAVE_BYTES;
  // after the loop: partial sums [wavefront][row block][column block][lane] f32x4, then the staged transposed tile
  static constexpr int PART_BYTES = KW * 16 * 64 * 16;
  static_assert(PART_BYTES + 64 * STG_PITCH <= LDS_BYTES, "reduction and staging areas");
};

template <bool HAS_D, bool HAS_C, bool HAS_CT, bool QK, int POST = 0, bool BND = false>
__global__ __launch_bounds__(CfgK64::NT, 2) void gemm_k64_kernel(const GemmParams p, const typename PostSel<POST>::arg post) {
  typedef CfgK64 Cfg;
  typedef typename PostSel<POST>::xt XT;
  constexpr int OPB = Cfg::OP_BYTES, KW = Cfg::KW, BK = Cfg::BK;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int b, ti, tj;
  constexpr bool TRI = HAS_C && HAS_CT && !QK;
  tile_of<64, 64, TRI>(p, blockIdx.x, gridDim.x, b, ti, tj);
  const float factor = p.scale_vec ? p.scale_vec[b] : 1.0f;
  const bool one_operand = !QK && TRI && ti == tj && p.P == p.Q && p.ldp == p.ldq && p.strideP == p.strideQ;

  // ---- global -> LDS: a load moves 8 tile rows of 128 bytes; lane l brings 16-byte chunk l % 8 of row l / 8.  The
  // swizzles are those of the kernel above; a load's first row is a multiple of 8, and they differ between
  // even and odd multiples, hence two offsets per operand.
  const int lrow = lane >> 3, lchunk = lane & 7;
  uint32_t offP[2], offQ[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    const int pc = lchunk ^ ((o * 4 + (lrow >> 1)) & 7);
    offP[o] = (uint32_t)(lrow * p.ldp + pc * 8) * 2u;
    // K-major rows are 128 bytes: the four rows of a transposing read fall into the two halves of a 256-byte bank
    // row twice; rows 2 and 3 swap their 64-byte groups, rows 8 apart their 32-byte halves
    const int qc = QK ? ((((lchunk >> 2) ^ ((lrow >> 1) & 1)) << 2) | ((lchunk & 3) ^ (o << 1))) : pc;
    offQ[o] = (uint32_t)(lrow * p.ldq + qc * 8) * 2u;
  }
  const char* gP = (const char*)(p.P + (int64_t)b * p.strideP + (int64_t)(ti * 64) * p.ldp);
  const char* gQ = QK ? (const char*)(p.Q + (int64_t)b * p.strideQ + tj * 64)
                      : (const char*)(p.Q + (int64_t)b * p.strideQ + (int64_t)(tj * 64) * p.ldq);
  const uint32_t stepP = (uint32_t)(8 * p.ldp) * 2u, stepQ = (uint32_t)(8 * p.ldq) * 2u;
  const int64_t slabQ = QK ? (int64_t)BK * p.ldq * 2 : (int64_t)BK * 2;
  const int KT = p.K / BK;
  const int nw = KT > wave ? (KT - wave + KW - 1) / KW : 0;  // slabs of this wavefront: wave, wave + KW, ...
  char* const ring = lds + wave * Cfg::WAVE_BYTES;
  constexpr int LPS = 16;
  auto issue_load = [&](int t, int slot, int j) {
    if (one_operand && j >= 8) return;
    const int kt = wave + t * KW;
    if (j < 8) {
      const char* src = gP + (int64_t)kt * (BK * 2) + (uint64_t)j * stepP;
      asm volatile("" : "+s"(src), "+v"(offP[j & 1]));
      __builtin_amdgcn_global_load_lds(GLB_PTR(src + offP[j & 1]), LDS_PTR(ring + slot * OPB + j * 1024), 16, 0, 0);
    } else {
      const int jq = j - 8;
      const char* src = gQ + kt * slabQ + (uint64_t)jq * stepQ;
      asm volatile("" : "+s"(src), "+v"(offQ[jq & 1]));
      __builtin_amdgcn_global_load_lds(GLB_PTR(src + offQ[jq & 1]), LDS_PTR(ring + (2 + slot) * OPB + jq * 1024), 16, 0, 0);
    }
  };

  // ---- LDS -> register fragments (see the kernel above)
  const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)ring;
  const int l16 = lane & 15, quad = lane >> 4;
  uint32_t aoff[2], boff[2], qoff[4];
#pragma unroll
  for (int st = 0; st < 2; ++st) {
    const int chunk = ((st * 4 + quad) ^ (l16 >> 1)) * 16;
    aoff[st] = lds_base + (uint32_t)(l16 * 128 + chunk);
    boff[st] = aoff[st] + (one_operand ? 0 : 2 * OPB);
  }
  if (QK) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      qoff[j] = lds_base + (uint32_t)(2 * OPB + (8 * quad + (l16 >> 2)) * 128 + (((j >> 1) ^ (l16 >> 3)) << 6) +
                                      ((j ^ quad) & 1) * 32 + (l16 & 3) * 8);
  }
  typedef FragSched<1, 2, QK> FS;
  bf16x8 fa[2][4], fb[2][4];
  auto read_frag = [&](auto hnc, auto rc) {
    constexpr int st = decltype(hnc)::value, r = decltype(rc)::value;
    if constexpr (r == 0 || r > 4) {
      constexpr int i = r == 0 ? 0 : r - 4;
      lds_read16<i * 2048>(fa[st][i], aoff[st]);
    } else if constexpr (QK) {
      lds_read_tr<st * 4096, 512>(fb[st][r - 1], qoff[r - 1]);
    } else {
      lds_read16<(r - 1) * 2048>(fb[st][r - 1], boff[st]);
    }
  };
  typedef std::integral_constant<int, 0> ic0;
  typedef std::integral_constant<int, 1> ic1;

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- main loop over this wavefront's slabs: no other wavefront touches its ring, so its own load counter is all
  // the synchronisation there is
  if (nw > 0) {
#pragma unroll
    for (int j = 0; j < LPS; ++j) issue_load(0, 0, j);
    if (nw > 1)
#pragma unroll
      for (int j = 0; j < LPS; ++j) issue_load(1, 1, j);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    if (nw > 1) {
      if (one_operand) wait_vmcnt<LPS / 2>();
      else wait_vmcnt<LPS>();
    } else wait_vmcnt<0>();
    __builtin_amdgcn_sched_barrier(0);
    static_for<0, 8>([&](auto rc) { read_frag(ic0(), rc); });
    __builtin_amdgcn_sched_barrier(0);
    uint32_t step = OPB;  // to the other slot: + OPB, then - OPB, ...
    auto slab = [&](int t, auto refill) {
      static_for<0, 2>([&](auto hc) {
        constexpr int hp = decltype(hc)::value;
        if constexpr (hp == 1) {
          // the other slab has landed, and every read of this one has returned: its slot may be refilled
          asm volatile("" ::: "memory");
          __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt 0, lgkmcnt 0
          asm volatile("" ::: "memory");
#pragma unroll
          for (int st = 0; st < 2; ++st) {
            aoff[st] += step;
            if (!QK) boff[st] += step;
          }
          if (QK)
#pragma unroll
            for (int j = 0; j < 4; ++j) qoff[j] += step;
          step = 0u - step;
          __builtin_amdgcn_sched_barrier(0);
        }
        static_for<0, 16>([&](auto qc) {
          constexpr int q = decltype(qc)::value, i = q / 4, j = q % 4;
          frag_wait<FS::allowed(hp, q)>(fa[hp][i], fb[hp][j]);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[hp][i], fb[hp][j], acc[i][j], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (FS::read_behind(hp, q) >= 0) {
            typedef std::integral_constant<int, FS::read_behind(hp, q)> rc;
            if constexpr (hp == 1) read_frag(ic0(), rc());
            else read_frag(ic1(), rc());
          }
          if constexpr (decltype(refill)::value && hp == 1) issue_load(t + 2, t & 1, q);
          __builtin_amdgcn_sched_barrier(0);
        });
      });
    };
    int t = 0;
    for (; t + 2 < nw; ++t) slab(t, std::true_type());
    for (; t < nw; ++t) slab(t, std::false_type());
  }
  wait_vmcnt<0>();
  // (see the kernel above: the read-ahead of the last half must land before its registers are let go)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      asm volatile("" ::"v"(fa[f][i]));
      asm volatile("" ::"v"(fb[f][i]));
    }

  // ---- partial sums -> tile.  Wavefront w finishes row block w (16 rows): every other wavefront hands it its share
  // through LDS, added in wavefront order.
  const int row_base = ti * 64 + wave * 16, col_base = tj * 64;
  const int lrows = BND ? p.out_rows - row_base - 4 * quad : 0, lcols = BND ? p.out_cols - col_base - l16 : 0;
  float pa = 0.f, pcoeff = 0.f, pb = 0.f;
  XT* xmat = nullptr;
  if constexpr (POST != 0) {
    const float wd = post.wd_dev ? *post.wd_dev : post.wd_host;
    muon_post_coeffs(*post.lr_dev, wd, post.adj_ratio, pa, pcoeff, pb);
    const int pi = b / post.mats_per_ptr;
    xmat = (XT*)post.X.p[pi] + (int64_t)(b - pi * post.mats_per_ptr) * (HAS_C ? p.strideC : p.strideCt);
  }
  bf16_t dreg[4][4];
  if (HAS_D) {
    const bf16_t* Dp = p.D + (int64_t)b * p.strideD + (int64_t)(row_base + 4 * quad) * p.ldd + col_base + l16;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) dreg[j][e] = Dp[(int64_t)e * p.ldd + j * 16];
  }
  __syncthreads();  // every wavefront is done with its ring
  f32x4* part = (f32x4*)lds;  // [wavefront][row block][column block][lane]
  static_for<0, 4>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int j = 0; j < 4; ++j) part[((wave * 4 + i) * 4 + j) * 64 + lane] = acc[i][j];
  });
  __syncthreads();
  const float alpha = gemm_alpha(p, factor), beta = p.beta;
  const bool on_diag = TRI && ti == tj && p.diag != 0.0f;
  char* stg = lds + Cfg::PART_BYTES;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f32x4 s = part[(wave * 4 + j) * 64 + lane];
#pragma unroll
    for (int w = 1; w < KW; ++w) s += part[((w * 4 + wave) * 4 + j) * 64 + lane];
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = alpha * s[e];
    if (HAS_D) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += beta * bf16_to_f32(dreg[j][e]);
    }
    if (on_diag) {
      const int dcol = col_base + j * 16 + l16 - (row_base + 4 * quad);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (dcol == e) v[e] += p.diag;
    }
    if (HAS_C) {
      const int64_t at = (int64_t)(row_base + 4 * quad) * p.ldc + col_base + l16 + j * 16;
      if constexpr (POST != 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (BND && (e >= lrows || j * 16 >= lcols)) continue;
          st_store<XT>(xmat, at + (int64_t)e * p.ldc,
                       muon_post_one(st_load<XT>(xmat, at + (int64_t)e * p.ldc), bf16_to_f32(f32_to_bf16(v[e])), pa,
                                     pcoeff, pb, post.cautious));
        }
      } else {
        bf16_t* Cp = p.C + (int64_t)b * p.strideC + at;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (BND && (e >= lrows || j * 16 >= lcols)) continue;
          Cp[(int64_t)e * p.ldc] = f32_to_bf16(v[e]);
        }
      }
    }
    if (HAS_CT) {
      uint2 pk;
      pk.x = pack_bf16x2(v[0], v[1]);
      pk.y = pack_bf16x2(v[2], v[3]);
      *(uint2*)(stg + (j * 16 + l16) * Cfg::STG_PITCH + (wave * 16 + 4 * quad) * 2) = pk;
    }
  }
  if (HAS_CT) {
    __syncthreads();
    if constexpr (BND) {
      // (a wavefront takes 16 of the 64 lines)
      typedef std::conditional_t<POST == 0, bf16_t, XT> OT;
      OT* dst;
      int cautious = 0;
      bool pair = (p.ldct & 1) == 0;
      if constexpr (POST != 0) {
        dst = xmat + (int64_t)(col_base + wave * 16) * p.ldct + ti * 64;
        pair = pair && post.vec_ok;
        cautious = post.cautious;
      } else {
        dst = p.Ct + (int64_t)b * p.strideCt + (int64_t)(col_base + wave * 16) * p.ldct + ti * 64;
      }
      const char* sp = stg + wave * 16 * Cfg::STG_PITCH;
      const int nl = p.out_cols - (col_base + wave * 16), ne = p.out_rows - ti * 64;
      if (pair) store_lines_bounded<2, 64, 16, POST>(sp, Cfg::STG_PITCH, lane, dst, p.ldct, nl, ne, pa, pcoeff, pb, cautious);
      else store_lines_bounded<1, 64, 16, POST>(sp, Cfg::STG_PITCH, lane, dst, p.ldct, nl, ne, pa, pcoeff, pb, cautious);
    } else if constexpr (POST != 0) {
      // the staged bf16 tile is the update of X[col][row]: a wavefront takes 16 of the 64 rows of X, lanes along a row
      XT* xt = xmat + (int64_t)(col_base + wave * 16) * p.ldct + ti * 64 + lane;
#pragma unroll 8
      for (int c = 0; c < 16; ++c) {
        const float u = bf16_to_f32(*(const bf16_t*)(stg + (wave * 16 + c) * Cfg::STG_PITCH + lane * 2));
        const int64_t at = (int64_t)c * p.ldct;
        st_store<XT>(xt, at, muon_post_one(st_load<XT>(xt, at), u, pa, pcoeff, pb, post.cautious));
      }
    } else if (!(TRI && ti == tj)) {  // a diagonal tile is its own mirror
      bf16_t* Ctp = p.Ct + (int64_t)b * p.strideCt + (int64_t)col_base * p.ldct + ti * 64;
#pragma unroll
      for (int it = 0; it < 2; ++it) {
        const int c = (tid >> 3) + it * 32, ch = tid & 7;
        *(uint4*)(Ctp + (int64_t)c * p.ldct + ch * 8) = *(const uint4*)(stg + c * Cfg::STG_PITCH + ch * 16);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
typedef TileCfg<128, 128, 64, 2, 2, 2, true> Cfg128;   // 4 wavefronts, 64x64 each; two workgroups per CU
typedef TileCfg<128, 128, 64, 2, 2, 4, true> Cfg128d;  // the same on a four-slot ring: one workgroup per CU
typedef TileCfg<256, 256, 64, 2, 4, 2> Cfg256w8;       // 8 wavefronts, 128x64 each: two per SIMD, one workgroup per CU
constexpr int kWalkMaxK = 2048;                    // longest reduction the tile-walking kernel is used for

template <class Cfg, bool HAS_D, bool HAS_C, bool HAS_CT, bool QK = false, int POST = 0, bool BND = false>
static hipError_t launch_epi(const GemmParams& p, hipStream_t stream,
                             const typename PostSel<POST>::arg& post = typename PostSel<POST>::arg()) {
  static std::atomic<uint64_t> attr_done{0};
  auto kern = gemm_nt_kernel<Cfg, HAS_D, HAS_C, HAS_CT, QK, POST, BND>;
  if (hipError_t e = set_max_dynamic_lds_once((const void*)kern, Cfg::LDS_BYTES, attr_done)) return e;
  const int tilesM = p.M / Cfg::BM, tilesN = p.N / Cfg::BN;
  const int64_t per_mat = p.tri ? (int64_t)tilesM * (tilesM + 1) / 2 : (int64_t)tilesM * tilesN;
  const int64_t total = per_mat * p.batch;
  if (total <= 0) return hipSuccess;
  if (total > 0x7fffffff) return hipErrorInvalidValue;
  GemmParams pp = p;
  set_tile_order(pp, Cfg::BM, Cfg::BN);
  hipLaunchKernelGGL(kern, dim3((unsigned)total), dim3(Cfg::NT), Cfg::LDS_BYTES, stream, pp, post);
  return hipGetLastError();
}

enum TileKind { kTile64, kTile128Deep, kTile128, kTile256 };

// The kernels keep the byte offset of a lane's row from its tile's first one in 32 bits (and some of the products it is
// made of in an int): 128 rows of a K-contiguous operand, 64 with 256-wide tiles; 16 rows of a K-major one; 32 of the addend,
// 8 with 256-wide tiles.  The 64-wide kernel spans 8 rows of an operand, and the addend's rows have 64-bit addresses there.
static bool rows_addressable(const GemmParams& p, TileKind k) {
  auto fits = [](int64_t rows, int ld) { return rows * ld < (int64_t(1) << 31); };
  if (k == kTile64) return fits(8, p.ldp) && fits(8, p.ldq);
  const int rows = k == kTile256 ? 64 : 128;
  return fits(rows, p.ldp) && fits(p.q_kmajor ? 16 : rows, p.ldq) && (!p.D || fits(k == kTile256 ? 8 : 32, p.ldd));
}

template <bool HAS_D, bool HAS_C, bool HAS_CT, bool QK, int POST = 0, bool BND = false>
static hipError_t launch_k64_epi(const GemmParams& p, hipStream_t stream,
                                 const typename PostSel<POST>::arg& post = typename PostSel<POST>::arg()) {
  static std::atomic<uint64_t> attr_done{0};
  auto kern = gemm_k64_kernel<HAS_D, HAS_C, HAS_CT, QK, POST, BND>;
  if (hipError_t e = set_max_dynamic_lds_once((const void*)kern, CfgK64::LDS_BYTES, attr_done)) return e;
  if (p.M % 64 || p.N % 64 || p.K % 64 || !rows_addressable(p, kTile64)) return hipErrorInvalidValue;
  const int64_t T = p.M / 64;
  const int64_t total = (p.tri ? T * (T + 1) / 2 : T * (p.N / 64)) * p.batch;
  if (total <= 0) return hipSuccess;
  if (total > 0x7fffffff) return hipErrorInvalidValue;
  GemmParams pp = p;
  set_tile_order(pp, 64, 64);
  hipLaunchKernelGGL(kern, dim3((unsigned)total), dim3(CfgK64::NT), CfgK64::LDS_BYTES, stream, pp, post);
  return hipGetLastError();
}

// One workgroup per CU, each walking its share of the tile list.
template <class Cfg, bool OUT_T>
static hipError_t launch_walk(const GemmParams& p, hipStream_t stream) {
  static std::atomic<uint64_t> attr_done{0};
  constexpr int kLds = Cfg::RING_BYTES + Cfg::WM * Cfg::WN * 32 * 128;
  auto kern = gemm_qk_walk_kernel<Cfg, OUT_T>;
  if (hipError_t e = set_max_dynamic_lds_once((const void*)kern, kLds, attr_done)) return e;
  const int64_t total = (int64_t)(p.M / Cfg::BM) * (p.N / Cfg::BN) * p.batch;
  if (total <= 0) return hipSuccess;
  if (total > 0x7fffffff) return hipErrorInvalidValue;
  // a wavefront's output tile is addressed with 32-bit byte offsets from its first element
  if ((int64_t)(OUT_T ? p.ldct : p.ldc) * 129 * 2 > 0x7fffffffLL) return hipErrorInvalidValue;
  static std::atomic<int> cu_count[64];
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev)) return e;
  int cus = cu_count[dev & 63].load(std::memory_order_relaxed);
  if (cus == 0) {
    if (hipError_t e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) return e;
    if (cus <= 0) return hipErrorInvalidValue;
    cu_count[dev & 63].store(cus, std::memory_order_relaxed);
  }
  GemmParams pp = p;
  set_tile_order(pp, Cfg::BM, Cfg::BN);
  const unsigned grid = (unsigned)(total < cus ? total : cus);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(Cfg::NT), kLds, stream, pp, (int)total);
  return hipGetLastError();
}

static bool bounded(const GemmParams& p) { return p.out_rows > 0; }
static bool bounds_ok(const GemmParams& p) {
  return p.out_rows > 0 && p.out_rows <= p.M && p.out_cols > 0 && p.out_cols <= p.N && p.q_kmajor && !p.tri && !p.D;
}

// The operand / result combinations the Newton-Schulz drivers use.
template <class Cfg>
static hipError_t launch_cfg(const GemmParams& p, hipStream_t stream) {
  if (p.M % Cfg::BM || p.N % Cfg::BN || p.K % 128) return hipErrorInvalidValue;
  const bool d = p.D != nullptr, c = p.C != nullptr, ct = p.Ct != nullptr;
  if (bounded(p)) {
    if (!bounds_ok(p) || c == ct) return hipErrorInvalidValue;
    return c ? launch_epi<Cfg, false, true, false, true, 0, true>(p, stream)
             : launch_epi<Cfg, false, false, true, true, 0, true>(p, stream);
  }
  if (p.q_kmajor) {
    if (p.tri) return hipErrorInvalidValue;
    if constexpr (Cfg::BM == 256) {
      // Short reductions go to the tile-walking kernel: what it saves is a fixed cost per tile, 13 % of the
      // launch at 32 slabs and nothing at 64 (where its static tile order costs as much as it saves).
      if (p.K <= kWalkMaxK && p.alpha == 1.0f) {  // (the drivers' X' products are unscaled)
        if (!d && c && !ct) return launch_walk<Cfg, false>(p, stream);  // X' = B X
        if (!d && !c && ct) return launch_walk<Cfg, true>(p, stream);   // (B X)^T only
      }
    }
    if (!d && c && !ct) return launch_epi<Cfg, false, true, false, true>(p, stream);  // X' = B X
    if (!d && !c && ct) return launch_epi<Cfg, false, false, true, true>(p, stream);  // (B X)^T only
    if (d && c && !ct) return launch_epi<Cfg, true, true, false, true>(p, stream);    // a X + B X
    return hipErrorInvalidValue;
  }
  if (p.tri && !d && c && ct) return launch_epi<Cfg, false, true, true>(p, stream);   // A = X X^T, R = T Z
  if (p.tri && d && c && ct) return launch_epi<Cfg, true, true, true>(p, stream);     // B = c A A + b A (+ a I)
  if (!p.tri && !d && c && !ct) return launch_epi<Cfg, false, true, false>(p, stream); // full product of two symmetric matrices
  return hipErrorInvalidValue;
}

static hipError_t launch_k64(const GemmParams& p, hipStream_t stream) {
  const bool d = p.D != nullptr, c = p.C != nullptr, ct = p.Ct != nullptr;
  if (bounded(p)) {
    if (!bounds_ok(p) || c == ct) return hipErrorInvalidValue;
    return c ? launch_k64_epi<false, true, false, true, 0, true>(p, stream)
             : launch_k64_epi<false, false, true, true, 0, true>(p, stream);
  }
  if (p.q_kmajor && !p.tri) {
    if (!d && c && !ct) return launch_k64_epi<false, true, false, true>(p, stream);
    if (!d && !c && ct) return launch_k64_epi<false, false, true, true>(p, stream);
    if (d && c && !ct) return launch_k64_epi<true, true, false, true>(p, stream);  // (rows too long for the other kernels)
    return hipErrorInvalidValue;
  }
  if (p.tri && !d && c && ct) return launch_k64_epi<false, true, true, false>(p, stream);
  if (p.tri && d && c && ct) return launch_k64_epi<true, true, true, false>(p, stream);
  if (!p.tri && !d && c && !ct) return launch_k64_epi<false, true, false, false>(p, stream);
  return hipErrorInvalidValue;
}

bool gemm_pad_is_chosen(int m, int batch) {
  const int64_t m256 = ((int64_t)m + 255) / 256;
  return m256 * (m256 + 1) / 2 * batch >= 256;
}

int gemm_pad_granule(int m, int n, int batch) {
  // To 256 once whole 256-wide tiles make more than one round of the CUs for the symmetric products, so that every product may
  // use them -- unless the padding to 128 leaves 18 % of the operations out: 256-wide tiles take up to 13 % less time for the same
  // operations, no more.  NS5, us a call padded to 256 / 128, and the operations to 256 over those to 128: 64 x (640 x 640) 862 / 553
  // (1.73), 100 x (384 x 1536) 1017 / 742 (1.82), 48 x (640 x 2560) 1483 / 1290 (1.46), 18 x (1152 x 1152) 804 / 690 (1.37), 30 x
  // (896 x 3584) 2257 / 1836 (1.32), 16 x (1408 x 1408) 1323 / 1072 and 40 x 3000 / 2841 (1.30), 50 x (1152 x 4608) 6165 / 6070
  // (1.245); but 12 x (1920 x 1920) 1880 / 1936 (1.21), 40 x (1408 x 5632) 7970 / 8150 (1.20), 20 x (1664 x 6656) 6396 / 6702
  // (1.17), 24 x (1920 x 7680) 11020 / 11777 (1.14), 3 x (4224 x 4224) 4150 / 4618 (1.09).  Between 1.1 and 1.2 rounds of the CUs
  // decide some square ones the other way: 10 x (2176 x 2176) 2371 / 2195 (1.19), 8 x (2432 x 2432) 2569 / 2328 (1.17).
  // (Taken with whole 128-wide tiles read where they lie; a plain call copies them, 1-4 % more of a wide bf16 one: NsPlan::ranged.)
  // The Gram form, whose products are others, loses nowhere: padded to 256 / by this rule 100 x (384 x 1536) 819 / 552, 90 x (300 x
  // 1000) 636 / 426, 48 x (640 x 2560) 1090 / 860, 30 x (896 x 3584) 1543 / 1229, 50 x (1152 x 4608) 4716 / 4322; the same extents for
  // 40 x (1408 x 5632) 6067 / 6066.
  if (!gemm_pad_is_chosen(m, batch)) return 128;
  auto padded_ops = [&](int64_t g) {
    const int64_t mp = (m + g - 1) / g, np = (n + g - 1) / g;  // (in tiles: no overflow)
    return (double)(g * mp) * (double)(g * mp) * (double)(g * (3 * np + mp));
  };
  return padded_ops(256) >= 1.22 * padded_ops(128) ? 128 : 256;
}

int gemm_pad_long(int mp, int n, int batch, int granule) {
  // The long side of a matrix that is padded to 128: to 256 where B X then offers more than a round and a half of the CUs
  // (384 tiles) on 256-wide tiles.  128-wide ones take twice the operand bytes there: B X of 24 x (512 x 8064) 167 us where
  // 24 x (512 x 8192) takes 118.  NS5, us a call padded to 128 / 256: 24 x (512 x 8056) 1245 / 1064, 6 x (1280 x 3448) 725 / 658, 30 x
  // (512 x 1656) 415 / 380, 12 x (1024 x 3448) 857 / 799, 24 x (512 x 2168) 374 / 352, 12 x (768 x 2936) 468 / 446, 9 x (1024 x
  // 2680) 559 / 545, 48 x (512 x 2168) 706 / 700, 6 x (1536 x 4216) 1032 / 1029; at 384 tiles 24 x (500 x 1920) 325 / 328, 16 x
  // (768 x 1912) 458 / 450, fewer 24 x (512 x 1400) 286 / 291, and where B has one row of tiles 60 x (256 x 2168) 331 / 344.  A Muon
  // step of 10 layers of 1530 x 4100 7051 / 6510, NorMuon, 8 of 1280 x 3400, 3448 / 3292, 24 of 512 x 2168 1327 / 1313.
  // Gram form 24 x (512 x 8056) 674 / 600, 12 x (1024 x 3448) 660 / 628, 48 x (512 x 2168) 538 / 527, 24 x (512 x 2168) 283 / 279.
  const int np = (n + granule - 1) / granule * granule;
  const bool fits = mp % 256 == 0 && mp >= 512 && np % 256 == 128;
  return fits && (int64_t)(mp / 256) * ((np + 128) / 256) * batch > 384 ? np + 128 : np;
}

// Which kernel a product runs on, by the number of tiles it offers the 256 CUs.  Figures: us per launch on one box, a launch
// repeated on the same operands unless it says otherwise.  In a call, behind the launch that wrote an operand, a launch
// of few tiles takes up to 3 us more (X X^T of one 768 x 3072 13.0, B X 10.1).
//  * 256-wide tiles, a symmetric product: when 128-wide ones are more than two per CU (512) and 256-wide ones at most one;
//    past that from the count on where 128-wide ones need a fourth round of two per CU (1536) where the reduction is as long
//    as the matrix is wide, and soon into the third (1152, or its begin, 1024) where it is longer.  X X^T on 256- / 128-wide
//    tiles: 130 / 468 tiles of 13 x (1024 x 1024) 26.1 / 19.5, 144 / 544 of 4 x (2048 x 2048) 42.6 /
//    48.8, 200 / 720 of 20 x (1024 x 3072) 65.0 / 71.8, 260 / 936 of 26 x (1024 x 1024) 50.8 / 36.7, of 26 x (1024 x 3072) 124 /
//    81, 270 / 900 of 90 x (512 x 2048) 84.9 / 55.8, 399 / 1482 of 19 x (1536 x 1536) 74.5 / 70.4, 420 / 1560 of 20 x 76.4 / 86.9.
//    The third round's lines are those of whole calls, whose X the product before has just written (five NS5 iterations, X X^T
//    on 256- / 128-wide tiles): 1344 tiles of 64 x (768 x 1536) 1303 / 1343, 1296 of 36 x (1024 x 2048) 1574 / 1622, 1512 of
//    42 x 1781 / 1846, but 1050 of 10 x (1792 x 3584) 2127 / 2085, 1044 of 29 x (1024 x 2048) 1339 / 1315, 1152 of
//    32 x (1024 x 1280) 1032 / 1025; from reductions four times the width on 1100 of 110 x (512 x 2048) 1412 / 1467, 1134 of
//    54 x (768 x 3072) 2018 / 2053, outside these widths 1026 of 342 x (256 x 1024) 855 / 836, 1050 of 10 x (1792 x 7168) 3835 /
//    3755.  A full product: when they make one round of the CUs where 128-wide ones make more than one of
//    two workgroups each (129-256 tiles), or most of two (from 336, with reductions past 1024 or an epilogue that reads memory --
//    an addend, a fused update -- from 384); the update of transposed padded parameters, whose epilogue is the longest, not
//    on one round of reductions up to 512.  B X on 128- / 256-wide tiles: 128 tiles of 8 x (1024 x 1024) 20.5 / 25.2, 144 of 9 x
//    27.2 / 24.3, 256 of 16 x 33.7 / 31.4, 272 of 17 x 46.6 / 49.1, 135 of 15 x (768 x 768) 24.2 / 22.1, 129 of 43 x (256 x 768)
//    12.4 / 11.4, 216 of 27 x (512 x 1024) 23.0 / 19.9, 252 of 7 x (1536 x 1536) 50.0 / 44.1, 360 of 10 x 71.4 / 72.1, 192 of one
//    3072 x 4096 75.9 / 66.7, 256 of one 4096 x 4096 112 / 100, 336 of 42 x (512 x 1024) 33.9 / 31.2 (on another box 28.8 / 29.5),
//    of 21 x (1024 x 1024) 52.0 / 50.6.  With an addend 144 of 9 x (1024 x 1024) 28.3 / 25.8, 129 of 43 x (256 x 768) 13.2 / 12.8,
//    336 of 42 x (512 x 1024) 34.6 / 36.5.  Updates of fp32 parameters 144 of 9 x (1024 x 1024) 33.4 / 32.1, 192 of one
//    3072 x 4096 81.6 / 71.4, 336 of 21 x (1024 x 1024) 65.8 / 71.8, 352 of 44 x (512 x 1024) 54.4 / 51.4; padded and transposed
//    144 of 9 x (1024 x 1024) 50.7 / 49.7, 135 of 15 x (768 x 768) 46.0 / 46.3, 132 of 33 x (512 x 512) 40.1 / 42.3, 130 of
//    65 x (256 x 512) 35.3 / 38.2, 336 of 42 x (512 x 1024) 70.7 / 84.3.
//  * 64-wide tiles with the reduction split over a workgroup's wavefronts (gemm_k64_kernel) when they are at most one
//    per CU.  64- / 128-wide tiles: X X^T of one 768 x 3072 matrix 10.1 / 17.8 (78 tiles), of 1024 x 4096 16.3 / 23.7, of
//    4 x (640 x 2560) 10.6 / 15.9, A A of one 1024 x 1024 6.4 / 9.8; B X of one 1024 x 1024 (256 tiles) 5.8 / 8.6, its update 8.0 /
//    10.3, past that no more: 288 of 2 x (768 x 768) 8.6 / 7.3, 576 of one 768 x 3072 13.0 / 7.9.  Whole calls with X X^T on
//    64- / 128-wide tiles: one 768 x 3072 163 / 200, 3 x (768 x 3072) 184 / 220, 60 x (128 x 2048) 155 / 169.
//    Symmetric products of up to two per CU where the reduction is not short: 128-wide tiles take less time there (X X^T of
//    2 x (1024 x 4096) 30.6 / 24.0, of 13 x (512 x 2048) 17.8 / 14.9, of 113 x (128 x 2048) 17.4 / 14.1, of 6 x (768 x 3072) 25.3 /
//    22.1, of 8 x (512 x 2048) 14.0 / 14.0; A A of 5 x (768 x 768) 10.4 / 9.0), but add a reduction up in one chain where
//    these have four partial sums, and one chain carries twice the rounding error: sums of 2048 products of unit variance
//    that cancel, 3.7e-6 rms on 64-wide tiles, 8.1e-6 on others.  Short ones, a slab or two to a wavefront: X X^T of
//    128 x (128 x 128) 6.6 / 4.7, of 40 x (256 x 256) 7.3 / 5.8, of 150 x (128 x 512) 8.4 / 6.8.
//  * 128-wide tiles, at most one per CU: the CU is one workgroup's alone, and a ring of four slots keeps three slabs
//    of loads in flight instead of one.  Four / two slots: X X^T of 12 x (768 x 3072) 25.6 / 32.1, of 4 x (1024 x 2816) 19.8 / 28.1, of
//    12 x (768 x 768) 10.9 / 10.9; a full product gains only when its reduction is long (B X of one 2048 x 2048 17.9 / 24.7, of
//    one 1536 x 2048 13.4 / 17.7, of one 1024 x 4096 11.5 / 11.4).
//  * else 128-wide tiles on a two-slot ring, two workgroups per CU (288 tiles of 8 x (1024 x 4096): 42.0, on four slots 50.1).
static TileKind tile_by_count(const GemmParams& p, UpdateKind update) {
  auto tiles = [&](int edge) -> int64_t {
    const int64_t T = p.M / edge;
    return (p.tri ? T * (T + 1) / 2 : T * (p.N / edge)) * (p.rule_batch > 0 ? p.rule_batch : p.batch);
  };
  if (p.M % 256 == 0 && p.N % 256 == 0) {
    const int64_t t = tiles(256), t128 = tiles(128);
    const int most128 = p.K / 4 >= p.M && p.M >= 512 && p.M <= 1024 ? 1024 : p.K > p.M || p.K > 2048 ? 1152 : 1536;
    const bool sym = t128 > 512 && (t <= 256 || t128 > most128);
    const bool one_round = t > 128 && t <= 256 && !(update == kUpdateTransposed && bounded(p) && p.K <= 512);
    const bool full = t >= 384 || one_round || (t >= 336 && p.K <= 1024 && update == kNoUpdate && !p.D);
    if (p.tri ? sym : full) return kTile256;
  }
  const int short_k = p.M < 256 ? 1024 : p.M < 384 ? 512 : 384;
  const int most64 = p.tri && p.K >= short_k ? 512 : 256;
  if (tiles(64) <= most64 && !(p.D && !p.tri)) return kTile64;
  if (tiles(128) <= 256 && (p.tri || p.K > 1024)) return kTile128Deep;
  return kTile128;
}

static TileKind pick_tile(const GemmParams& p, UpdateKind update = kNoUpdate) {
  const TileKind k = tile_by_count(p, update);
  return rows_addressable(p, k) ? k : kTile64;
}

int gemm_tile_edge(const GemmParams& p) {
  const TileKind k = pick_tile(p);
  return k == kTile256 ? 256 : k == kTile64 ? 64 : 128;
}

int gemm_kernel(const GemmParams& p, UpdateKind update) {
  const TileKind k = pick_tile(p, update);
  return k == kTile256 ? 256 : k == kTile64 ? 64 : k == kTile128Deep ? 129 : 128;
}

template <class Cfg, int POST, bool BND>
static hipError_t launch_post_cfg(const GemmParams& p, const FusedPost& post, bool transposed, hipStream_t stream) {
  if (p.M % Cfg::BM || p.N % Cfg::BN || p.K % 128) return hipErrorInvalidValue;
  return transposed ? launch_epi<Cfg, false, false, true, true, POST, BND>(p, stream, post)
                    : launch_epi<Cfg, false, true, false, true, POST, BND>(p, stream, post);
}

template <int POST, bool BND>
static hipError_t launch_post(const GemmParams& p, const FusedPost& post, bool transposed, hipStream_t stream) {
  switch (pick_tile(p, transposed ? kUpdateTransposed : kUpdate)) {
    case kTile256: return launch_post_cfg<Cfg256w8, POST, BND>(p, post, transposed, stream);
    case kTile128Deep: return launch_post_cfg<Cfg128d, POST, BND>(p, post, transposed, stream);
    case kTile64:
      return transposed ? launch_k64_epi<false, false, true, true, POST, BND>(p, stream, post)
                        : launch_k64_epi<false, true, false, true, POST, BND>(p, stream, post);
    default: return launch_post_cfg<Cfg128, POST, BND>(p, post, transposed, stream);
  }
}

hipError_t launch_gemm_nt_post(const GemmParams& p, const FusedPost& post, int x_dtype, bool transposed,
                               hipStream_t stream) {
  if (p.M <= 0 || p.N <= 0 || p.K <= 0 || p.batch <= 0) return hipSuccess;
  // the epilogue addresses a wavefront tile of X (at most 128 rows) with 32-bit byte offsets
  if ((int64_t)(transposed ? p.ldct : p.ldc) * 129 * 4 > 0x7fffffffLL) return hipErrorInvalidValue;
  if (!p.q_kmajor || p.tri || p.D || post.mats_per_ptr <= 0 || !post.lr_dev ||
      p.batch > (int64_t)kMaxPtrs * post.mats_per_ptr || (x_dtype != 0 && x_dtype != 1))
    return hipErrorInvalidValue;
  if (bounded(p)) {
    if (!bounds_ok(p)) return hipErrorInvalidValue;
    return x_dtype == 1 ? launch_post<1, true>(p, post, transposed, stream)
                        : launch_post<2, true>(p, post, transposed, stream);
  }
  return x_dtype == 1 ? launch_post<1, false>(p, post, transposed, stream)
                      : launch_post<2, false>(p, post, transposed, stream);
}

hipError_t launch_gemm_nt(const GemmParams& p, hipStream_t stream) {
  if (p.M <= 0 || p.N <= 0 || p.K <= 0 || p.batch <= 0) return hipSuccess;
  if (p.tri && (p.M != p.N)) return hipErrorInvalidValue;
  switch (pick_tile(p)) {
    case kTile256: return launch_cfg<Cfg256w8>(p, stream);
    case kTile128Deep: return launch_cfg<Cfg128d>(p, stream);
    case kTile64: return launch_k64(p, stream);
    default: return launch_cfg<Cfg128>(p, stream);
  }
}

}  // namespace dion
