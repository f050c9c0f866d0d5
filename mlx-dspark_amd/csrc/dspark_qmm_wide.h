// Affine quantized matmul over many rows (prefill widths) on the gfx950 matrix cores.
//
// y[m, n] = sum_g s[n, g] * (x[m, g] . q[n, g]) + b[n, g] * sum x[m, g]    (groups g of 64 along K)
//
// x is bf16 and the integer fields q (0..255, or 16 + 0..15) are exact in bf16, so every product
// is exact in fp32; scales are applied in fp32 to each group's dot product and the weight is
// never rounded. The bias term is one more contraction over g: the group sums of x are held as
// three bf16 pieces (24 significand bits, wide_xsum_kernel) and multiplied by the bf16 biases on
// the same MFMA, 3 G / K = 5% more of them.
//
// What bounds it: the MFMA pipe, with the VALU close behind (per 16 x 16 x 64 step two MFMAs of
// 16 cycles against 4 FMAs of the scale, 16 cycles, and the field unpacking). Hence:
//   * a workgroup is 4 waves side by side along N, each with all BM = 16 MT rows and its own
//     16 NT columns: a weight is read and unpacked by one wave only, straight from global memory
//     to registers, and the unpacking is paid once for 16 MT rows (at MT = 8, NT = 4 it is 384 of
//     about 900 VALU cycles beside 1024 MFMA cycles per group);
//   * x tiles (BM x 64) are copied global -> LDS without passing registers, double buffered, one
//     barrier per group, 16-byte chunks XOR-swizzled by the row so the fragment reads are free
//     of bank conflicts; all four waves read every fragment (LDS time is half the MFMA time);
//   * the tile order keeps the row tiles of one weight strip on one XCD, next to each other, so
//     a strip comes from HBM once.
// Measured (with the group sums and the K-slice sum): 2048 x 12288 x 4096, 8-bit, 241 us (857
// TFLOP/s; a large bf16 matrix product of the library reaches 1150 to 1220 here) where an fp32
// product of dequantized weights took 1450 us; 93 x 17408 x 5120, 4-bit, 43 us against 1363 us.
// At 2048 rows the matrix pipe is busy 38% of the time and the VALU issues 47% of it: MFMAs in sequence
// with their FMAs, without the interleaving in tile_loop, took 280 us.
#pragma once

#include "dspark_qmm_core.h"

namespace dspark {
namespace wide {

constexpr int kThreads = 256;
constexpr int kPieces = 3;  // bf16 pieces of a group sum

// lane quarter q's k offset / 8 inside a group: 16q (8-bit rows: 16 bytes per quarter), or the
// packed 4-bit tiles' order 16 (2 (q & 1) + (q >> 1)), used for row-major 4-bit rows too so both
// layouts give the same bits
template <int BITS>
__device__ __forceinline__ int k_chunk(int q) {
  return BITS == 4 ? 2 * (2 * (q & 1) + (q >> 1)) : 2 * q;
}

// 8 nibbles of a word as 8 bf16 (16 + nibble) in field order: 16 + n is 0x4180 | n << 3, so even
// and odd nibbles go to bits 3..6 of bytes 0x80, the bytes are interleaved in order and each is
// paired with the byte 0x41. The offset is kept small because its term, -16 s sum x, cancels in
// the fp32 sum: with 128 + n (two instructions a word less) the error grew by 5e-6 of itself.
__device__ __forceinline__ u32x4_t unpack_u4_ordered(u32 w) {
  const u32 m = opaque_sgpr(0x78787878u), b = opaque_vgpr(0x80808080u), c = opaque_vgpr(0x41414141u);
  const u32 e = and_or(w << 3, m, b), o = and_or(w >> 1, m, b);
  const u32 lo = __builtin_amdgcn_perm(o, e, 0x05010400u), hi = __builtin_amdgcn_perm(o, e, 0x07030602u);
  return u32x4_t{__builtin_amdgcn_perm(c, lo, 0x04010400u), __builtin_amdgcn_perm(c, lo, 0x04030402u),
                 __builtin_amdgcn_perm(c, hi, 0x04010400u), __builtin_amdgcn_perm(c, hi, 0x04030402u)};
}

template <int BITS>
struct Raw;
template <>
struct Raw<8> {
  u32x4_t v;
};
template <>
struct Raw<4> {
  u32x2_t v;
};

// x copies of a wave per group: 8 rows each, 32 of the workgroup's
template <int MT>
constexpr int kCopies = (MT + 1) / 2;

// Everything of a tile that does not depend on the group.
template <int MT, int NT>
struct Tile {
  const char* xb;        // x, the base of the row offsets
  u32 xoff[kCopies<MT>];      // byte offset of this lane's 16-byte chunk of each x copy it issues
  const u16* xs;         // group-sum pieces
  u32 xsoff[MT];         // element offset of this lane's row of every row tile
  long xs_piece;         // elements between pieces
  const char* wb[2];     // weight strip bases (second: the up matrix of a SwiGLU pair)
  u32 woff[NT];          // byte offset of this lane's fields at group 0
  const u16* srow;       // this thread's scale row (kThreads rows are staged), at group 0
  const u16* brow[NT];   // this lane's bias rows
  const u16* sown[NT];   // this lane's scale rows (the 4-bit offset term)
  int G, gs, ge;
  bool vec;              // scale / bias rows are whole aligned 16-byte chunks (chunk_rows)
};

// Whether rows of G scales and biases are whole aligned 16-byte chunks
inline bool chunk_rows(int G, const void* s, const void* b) { return G % 8 == 0 && aligned(s, 16) && aligned(b, 16); }

template <int BITS, bool PW>
__device__ __forceinline__ u32 w_step(int g) {  // byte offset of group g along a row / packed tile
  if constexpr (PW) return BITS == 8 ? (u32)g * 1024u : (u32)(g >> 1) * 1024u + (u32)(g & 1) * 8u;
  else return (u32)g * (BITS == 8 ? 64u : 32u);
}

// Rows that are not whole 16-byte chunks are read as the aligned words that hold them: word i of a
// row holds its elements 2 i - odd_start and the next
__device__ __forceinline__ int odd_start(const u16* row) { return (int)(reinterpret_cast<uintptr_t>(row) >> 1) & 1; }
__device__ __forceinline__ const u32* row_words(const u16* row) {
  return reinterpret_cast<const u32*>(reinterpret_cast<uintptr_t>(row) & ~(uintptr_t)3);
}

// 8 consecutive bf16 of a row of G starting at g0 (a multiple of 8), zeros past its end
__device__ __forceinline__ u32x4_t row8(const u16* row, int g0, int G, bool vec) {
  if (vec) return g0 < G ? ldg128(row + g0) : u32x4_t{0u, 0u, 0u, 0u};
  const int odd = odd_start(row), last = (odd + G - 1) >> 1;
  const u32* p = row_words(row);
  u32 w[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) w[i] = p[min((g0 >> 1) + i, last)];
  u32x4_t o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int a = g0 + 2 * i;
    const u32 v = __builtin_amdgcn_alignbit(w[i + 1], w[i], 16 * odd);
    o[i] = a + 1 < G ? v : a < G ? v & 0xFFFFu : 0u;
  }
  return o;
}

// 8 bf16 times -16 (exact short of overflow)
__device__ __forceinline__ u32x4_t times_m16(u32x4_t v) {
  u32x4_t o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = pack_bf16x2(-16.0f * bf2f(v[i] & 0xFFFFu), -16.0f * bf2f(v[i] >> 16));
  return o;
}

// Groups held ahead of the one being multiplied. The largest tiles have the work of two waves per
// SIMD (and no registers) to cover a load. Smaller tiles hold three groups, but the scale chunk's
// conditional load makes the compiler wait, after each barrier, for every request before it issues
// the next group's: a group is requested one step's length ahead or a little more, whatever is held.
// One group ahead instead: 1024 x 4096 x 4032 4-bit 69 -> 73 us, 200 x 8192 x 2048 29.4 -> 27.9, the
// others of 17 shapes within 4%, either way.
template <int MT, int NT>
constexpr int kAhead = MT * NT >= 24 ? 1 : 3;

template <int MT, int NT>
struct __attribute__((aligned(16))) Smem {
  u16 xa[kAhead<MT, NT> + 1][32 * kCopies<MT> * 64];
  u16 sc[2][kThreads * 8];
};

// The group loop of one tile: acc[mt][nt] = this lane's 4 outputs (rows 16 mt + 4 q + r, the
// wave's column 16 nt + c16) over groups [gs, ge); gs is a multiple of 8. bias_phase / bias_step:
// of the 32-group steps of the bias term this call takes those t with t % bias_step == bias_phase
// (the K slices share them out).
template <int BITS, int MT, int NT, bool PW, bool PAIR>
__device__ __forceinline__ void tile_loop(const Tile<MT, NT>& t, Smem<MT, NT>& sm, int GP, int bias_phase,
                                          int bias_step, f32x4_t (&acc)[MT][NT]) {
  constexpr int PD = kAhead<MT, NT>, NBUF = PD + 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int c16 = lane & 15, q = lane >> 4;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  typedef __attribute__((address_space(3))) u16 lds_u16;
  typedef const __attribute__((address_space(1))) u16 glb_u16;

  auto copy_x = [&](int g, int buf) {
#pragma unroll
    for (int j = 0; j < kCopies<MT>; ++j)
      __builtin_amdgcn_global_load_lds((glb_u16*)(t.xb + (size_t)g * 128 + t.xoff[j]),
                                       (lds_u16*)&sm.xa[buf][(wave * kCopies<MT> + j) * 512], 16, 0, 0);
  };
  auto load_w = [&](int g, Raw<BITS> (&raw)[NT]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const char* p = t.wb[PAIR && nt >= NT / 2 ? 1 : 0] + w_step<BITS, PW>(g) + t.woff[nt];
      if constexpr (BITS == 8) raw[nt].v = ldg128(p);
      else raw[nt].v = ldg64(p);
    }
  };

  // groups past the end repeat the last one: their loads are never used
  Raw<BITS> raw[PD][NT];
  u32x4_t scn = tid < 64 * NT ? row8(t.srow, t.gs, t.G, t.vec) : u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
  for (int u = 0; u < PD; ++u) {
    load_w(min(t.gs + u, t.ge - 1), raw[u]);
    copy_x(min(t.gs + u, t.ge - 1), u);
  }

#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = zero;
  for (int tb = bias_phase; tb < GP / 32; tb += bias_step) {
    const int g0 = 32 * tb + 8 * q;
    u32x4_t bf[NT], sf[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      bf[nt] = row8(t.brow[nt], g0, t.G, t.vec);
      if constexpr (BITS == 4) sf[nt] = times_m16(row8(t.sown[nt], g0, t.G, t.vec));
    }
#pragma unroll 1
    for (int p = 0; p < kPieces; ++p) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const u32x4_t a = ldg128(t.xs + p * t.xs_piece + t.xsoff[mt] + g0);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          acc[mt][nt] = mfma16x16x32(a, bf[nt], acc[mt][nt]);
          if constexpr (BITS == 4) acc[mt][nt] = mfma16x16x32(a, sf[nt], acc[mt][nt]);
        }
      }
    }
  }

  // The requests above are the compiler's to order, so no count of later ones says that the first x
  // tile has landed: all of them are waited for, once. In the loop the count holds, since the memory
  // clobbers at a step's barrier keep its requests behind those of the steps before.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (tid < 64 * NT) *reinterpret_cast<u32x4_t*>(&sm.sc[(t.gs >> 3) & 1][tid * 8]) = scn;
  const int abase = c16 * 64 + ((k_chunk<BITS>(q) ^ ((c16 >> 1) & 7)) << 3);  // the second chunk: ^ 8
  const int sbase = (wave * 16 * NT + c16) * 8;
  int buf = 0;
  auto step = [&](int g, Raw<BITS> (&rw)[NT]) {
    // x tile g and the staged scales are in LDS once every wave's copies have landed; the loads
    // of the PD - 1 groups after g need not have (a __syncthreads would wait for them). Every LDS
    // read of the step before has been used by then.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((PD - 1) * (NT + kCopies<MT>)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    u32x4_t b[NT][2];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if constexpr (BITS == 8) {
        b[nt][0] = unpack_u8(rw[nt].v.x, rw[nt].v.y);
        b[nt][1] = unpack_u8(rw[nt].v.z, rw[nt].v.w);
      } else {
        b[nt][0] = unpack_u4_ordered(rw[nt].v.x);
        b[nt][1] = unpack_u4_ordered(rw[nt].v.y);
      }
    }
    float s[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) s[nt] = bf2f(sm.sc[(g >> 3) & 1][sbase + nt * 128 + (g & 7)]);
    // scales of the next 8 groups: requested at a chunk's first group, stored at its last
    if ((g & 7) == 7 && g + 1 < t.ge && tid < 64 * NT)
      *reinterpret_cast<u32x4_t*>(&sm.sc[((g >> 3) + 1) & 1][tid * 8]) = scn;
    if ((g & 7) == 0 && g + 8 < t.ge && tid < 64 * NT) scn = row8(t.srow, g + 8, t.G, t.vec);
    const int gn = min(g + PD, t.ge - 1);
    load_w(gn, rw);
    copy_x(gn, buf == 0 ? NBUF - 1 : buf - 1);  // the buffer read in the step before
    // Row tiles in turn, each step issuing the tile's MFMAs between the scale FMAs of the tile
    // before (one MFMA occupies the matrix pipe for 16 cycles, two FMAs issue in 8) and reading
    // the next tile's x fragments. Raised priority: the other workgroup's wave on this SIMD
    // unpacks its weights in the gaps.
    const u16* xa = sm.xa[buf];
    u32x4_t a[2][2];
    f32x4_t p[2][NT];
    __builtin_amdgcn_s_setprio(1);
    a[0][0] = *reinterpret_cast<const u32x4_t*>(xa + abase);
    a[0][1] = *reinterpret_cast<const u32x4_t*>(xa + (abase ^ 8));
#pragma unroll
    for (int mt = 0; mt <= MT; ++mt) {
      if (mt + 1 < MT) {
        a[(mt + 1) & 1][0] = *reinterpret_cast<const u32x4_t*>(xa + (mt + 1) * 1024 + abase);
        a[(mt + 1) & 1][1] = *reinterpret_cast<const u32x4_t*>(xa + (mt + 1) * 1024 + (abase ^ 8));
      }
      if (mt < MT) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) p[mt & 1][nt] = mfma16x16x32(a[mt & 1][0], b[nt][0], zero);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) p[mt & 1][nt] = mfma16x16x32(a[mt & 1][1], b[nt][1], p[mt & 1][nt]);
      }
      if (mt > 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[mt - 1][nt][r] = __builtin_fmaf(s[nt], p[(mt - 1) & 1][nt][r], acc[mt - 1][nt][r]);
      }
      if (mt + 1 < MT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // the LDS reads first
      if (mt > 0 && mt < MT) {
#pragma unroll
        for (int i = 0; i < 2 * NT; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
          __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two VALU
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_amdgcn_s_setprio(0);
    buf = buf + 1 == NBUF ? 0 : buf + 1;
  };
  for (int g = t.gs; g < t.ge; g += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u)
      if (g + u < t.ge) step(g + u, raw[u]);
  }
}

// This thread's chunk of the x copies: LDS chunk l of copy j lies in tile row 8 (..) + (l >> 3);
// row r holds its eight 16-byte chunks in the order chunk ^ ((r >> 1) & 7), which with the row's
// parity spreads 16 rows read at one chunk over the banks.
template <int MT>
__device__ __forceinline__ int copy_row(int j) {
  return 8 * ((int)(threadIdx.x >> 6) * kCopies<MT> + j) + ((threadIdx.x & 63) >> 3);
}
__device__ __forceinline__ int copy_chunk(int row) { return (threadIdx.x & 7) ^ ((row >> 1) & 7); }

// ---------------------------------------------------------------- the dense matrix

struct Args {
  const u16* x;
  const u16* xs;  // [kPieces][M][GP]
  const u32* w;
  const u16* s;
  const u16* b;
  const u16* bias;  // nullable [N]
  u16* y;
  float* part;  // [S][M][N] when S > 1
  long ldx, ldy;
  int M, N, K, G, GP, S, mtiles, ntiles, per_xcd;
  bool vec;
};

// exact fp32 value of one weight as an elementwise dequantization rounds it
template <int BITS>
__device__ __forceinline__ float dequant_at(const Args& a, int n, int k) {
#pragma clang fp contract(off)
  const u32 word = a.w[(long)n * (a.K / (32 / BITS)) + k / (32 / BITS)];
  const float qv = (float)((word >> (BITS * (k % (32 / BITS)))) & ((1u << BITS) - 1u));
  const float p = bf2f(a.s[(long)n * a.G + (k >> 6)]) * qv;
  return p + bf2f(a.b[(long)n * a.G + (k >> 6)]);
}

// The factored sums turn an infinite x into a NaN (inf * 0 for a zero field, inf - inf with the bias
// term) where the dequantized product is infinite, so outputs that are not finite are computed again.
// Where the row of x has values that are not finite (and the weights have none, infinite_weights), their
// terms are the output: acc becomes the sum of x[k] weight(k) over them, for the lanes of a wave (one
// output each, all of row xr) that take part. False if the row has none. An infinity in one row of 93 x
// 17408 x 5120, 4-bit: 82 us where a call without takes 74; in every row 116; with each output's whole
// product by its lane 6.9 and 134 ms.
template <class W>
__device__ __forceinline__ bool infinite_terms(const u16* xr, int K, bool take, float& acc, W weight) {
  const int lane = threadIdx.x & 63;
  acc = 0.f;
  bool found = false;
#pragma unroll 1
  for (int k0 = 0; k0 < K; k0 += 512) {
    const int k = k0 + 8 * lane;
    u32 mine = 0;  // bit j: x[k + j] is not finite
    if (k < K) {
      const u32x4_t v = ldg128(xr + k);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        mine |= ((v[j >> 1] >> (16 * (j & 1))) & 0x7F80u) == 0x7F80u ? 1u << j : 0u;
    }
#pragma unroll 1
    for (unsigned long long any = __builtin_amdgcn_ballot_w64(mine != 0); any; any &= any - 1) {
      const int src = __builtin_ctzll(any);
      found = true;
#pragma unroll 1
      for (u32 bits = __builtin_amdgcn_readlane((int)mine, src); bits; bits &= bits - 1) {
        const int kk = k0 + 8 * src + __builtin_ctz(bits);
        if (take) acc = __builtin_fmaf(bf2f(xr[kk]), weight(kk), acc);
        if (!__builtin_amdgcn_ballot_w64(take && acc == acc)) return true;  // all NaN
      }
    }
  }
  return found;
}

// Whether a scale or bias of weight rows [n, n + rows) is not finite: by a wave, the rows' values in order
__device__ __forceinline__ bool infinite_weights(const u16* s, const u16* b, long n, int rows, int G, bool vec) {
  const long count = (long)rows * G;
  s += n * G;
  b += n * G;
  bool any = false;
  if (vec) {
#pragma unroll 8
    for (long i = 8 * (threadIdx.x & 63); i < count; i += 512) {
      const u32x4_t x = ldg128(s + i), y = ldg128(b + i);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        any |= (x[j] & 0x7F80u) == 0x7F80u || (x[j] & 0x7F800000u) == 0x7F800000u ||
               (y[j] & 0x7F80u) == 0x7F80u || (y[j] & 0x7F800000u) == 0x7F800000u;
    }
  } else {
#pragma unroll 8
    for (long i = threadIdx.x & 63; i < count; i += 64)
      any |= (s[i] & 0x7F80u) == 0x7F80u || (b[i] & 0x7F80u) == 0x7F80u;
  }
  return __builtin_amdgcn_ballot_w64(any) != 0;
}

// One output as the dequantized product in fp32
template <int BITS>
__device__ float plain_dot(const Args& a, int m, int n) {
  float acc = 0.f;
  for (int k = 0; k < a.K && acc == acc; ++k)
    acc = __builtin_fmaf(bf2f(a.x[(long)m * a.ldx + k]), dequant_at<BITS>(a, n, k), acc);
  return acc;
}

__device__ __forceinline__ bool not_finite(float v) { return !(__builtin_fabsf(v) < __builtin_inff()); }

__device__ __forceinline__ u16 finish(const Args& a, float v, int n) {
  const u16 r = f2bf(v);
  return a.bias ? f2bf(bf2f(r) + bf2f(a.bias[n])) : r;  // the module's bias is added to the bf16 product
}

// Outputs y[m, n] again, by one wave: m is the wave's, n the lane's, take whether it has one, whole
// whether weights of the wave's columns are not finite.
template <int BITS>
__device__ __forceinline__ void plain_outputs(const Args& a, int m, int n, bool take, bool whole) {
  float acc;
  const bool terms = infinite_terms(a.x + (long)m * a.ldx, a.K, take, acc, [&](int k) { return dequant_at<BITS>(a, n, k); });
  if (take && (whole || !terms)) acc = plain_dot<BITS>(a, m, n);
  if (take) a.y[(long)m * a.ldy + n] = finish(a, acc, n);
}

template <int BITS, int MT, int NT>
__global__ __launch_bounds__(kThreads, 2) void wide_kernel(const Args a) {
  __shared__ Smem<MT, NT> sm;
  // one XCD's workgroups (ids equal modulo 8) take consecutive tiles
  const int id = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if (id >= a.mtiles * a.ntiles * a.S) return;
  const int mt_ = id % a.mtiles, rest = id / a.mtiles;
  const int z = rest % a.S, nt_ = rest / a.S;
  const int m0 = mt_ * 16 * MT, n0 = nt_ * 64 * NT;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int c16 = lane & 15, q = lane >> 4;
  constexpr int kRowShift = BITS == 8 ? 0 : 1;  // bytes of a row = K >> kRowShift

  Tile<MT, NT> t;
  t.G = a.G;
  t.vec = a.vec;
  const int units = (a.G + 7) >> 3;
  t.gs = 8 * (int)(((long)z * units) / a.S);
  t.ge = min(8 * (int)(((long)(z + 1) * units) / a.S), a.G);
  t.xb = reinterpret_cast<const char*>(a.x + (long)m0 * a.ldx);
  const int mlast = a.M - 1 - m0;  // rows past M repeat the last one; their outputs are dropped
#pragma unroll
  for (int j = 0; j < kCopies<MT>; ++j) {
    const int r = copy_row<MT>(j);
    t.xoff[j] = (u32)(min(r, mlast) * (int)a.ldx * 2 + copy_chunk(r) * 16);
  }
  t.xs = a.xs + (long)m0 * a.GP;
  t.xs_piece = (long)a.M * a.GP;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) t.xsoff[mt] = (u32)(min(16 * mt + c16, mlast) * a.GP);
  t.wb[0] = t.wb[1] = reinterpret_cast<const char*>(a.w) + (long)n0 * (a.K >> kRowShift);
  const int nlast = a.N - 1 - n0;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int nr = min(wave * 16 * NT + nt * 16 + c16, nlast);
    t.woff[nt] = (u32)nr * (u32)(a.K >> kRowShift) + (u32)k_chunk<BITS>(q) * (BITS == 8 ? 8u : 4u);
    t.brow[nt] = a.b + (long)(n0 + nr) * a.G;
    t.sown[nt] = a.s + (long)(n0 + nr) * a.G;
  }
  t.srow = a.s + (long)(n0 + min(tid, nlast)) * a.G;

  f32x4_t acc[MT][NT];
  tile_loop<BITS, MT, NT, false, false>(t, sm, a.GP, z, a.S, acc);

  if (a.S > 1) {
    float* part = a.part + (long)z * a.M * a.N;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + 16 * mt + 4 * q + r;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          const int n = n0 + wave * 16 * NT + nt * 16 + c16;
          if (m < a.M && n < a.N) part[(long)m * a.N + n] = acc[mt][nt][r];
        }
      }
    return;
  }
  bool bad = false;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = m0 + 16 * mt + 4 * q + r;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int n = n0 + wave * 16 * NT + nt * 16 + c16;
        bad |= not_finite(acc[mt][nt][r]);
        if (m < a.M && n < a.N) a.y[(long)m * a.ldy + n] = finish(a, acc[mt][nt][r], n);
      }
    }
  if (!__builtin_amdgcn_ballot_w64(bad)) return;
  __threadfence_block();  // the wave's outputs are read back by other lanes
  const int n = n0 + wave * 16 * NT + lane;
  const int c0 = n0 + wave * 16 * NT;
  const bool whole = infinite_weights(a.s, a.b, c0, min(16 * NT, a.N - c0), a.G, a.vec);
#pragma unroll 1
  for (int m = m0; m < min(m0 + 16 * MT, a.M); ++m) {
    const bool take = lane < 16 * NT && n < a.N && not_finite(bf2f(a.y[(long)m * a.ldy + min(n, a.N - 1)]));
    if (__builtin_amdgcn_ballot_w64(take)) plain_outputs<BITS>(a, m, n, take, whole);
  }
}

// y = the K slices' partial sums in slice order
template <int BITS>
__global__ __launch_bounds__(256) void wide_reduce_kernel(const Args a) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4, total = (long)a.M * a.N;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  const int cnt = (int)max(0L, min(4L, total - i));
  if (a.N % 4 == 0) {
    if (cnt)
      for (int z = 0; z < a.S; ++z) {
        const f32x4_t p = *reinterpret_cast<const f32x4_t*>(a.part + z * total + i);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += p[j];
      }
  } else {
    for (int z = 0; z < a.S; ++z)
      for (int j = 0; j < cnt; ++j) v[j] += a.part[z * total + i + j];
  }
  u32 bad = 0;  // bit j: output i + j is not finite
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (j >= cnt) break;
    const int m = (int)((i + j) / a.N), n = (int)((i + j) - (long)m * a.N);
    a.y[(long)m * a.ldy + n] = finish(a, v[j], n);
    bad |= not_finite(v[j]) ? 1u << j : 0u;
  }
  if (!__builtin_amdgcn_ballot_w64(bad != 0)) return;
  // the columns of the wave's 256 outputs, which may go on at the first one
  const long i0 = i - 4 * (threadIdx.x & 63);
  const int c0 = (int)(i0 % a.N), cols = min(256, a.N), to_end = min(cols, a.N - c0);
  const bool whole = infinite_weights(a.s, a.b, c0, to_end, a.G, a.vec) ||
                     infinite_weights(a.s, a.b, 0, cols - to_end, a.G, a.vec);
#pragma unroll 1
  for (int j = 0; j < 4; ++j) {
    const int m = (int)((i + j) / a.N), n = (int)((i + j) - (long)m * a.N);
    // the lanes of one row of x at a time
    for (unsigned long long left = __builtin_amdgcn_ballot_w64((bad >> j) & 1); left;) {
      const int row = __builtin_amdgcn_readlane(m, __builtin_ctzll(left));
      const bool take = ((bad >> j) & 1) && m == row;
      left &= ~__builtin_amdgcn_ballot_w64(take);
      plain_outputs<BITS>(a, row, n, take, whole);
    }
  }
}

// Group sums of x [M, K = 64 G] as bf16 pieces xs[p][m][g], rows of GP entries (g >= G zero)
int launch_group_sums(const u16* x, long ldx, long M, int G, int GP, u16* xs, hipStream_t s);

}  // namespace wide
}  // namespace dspark
