// Attention over many query rows (prefill widths) on the gfx950 matrix cores.
//
// out[h, i] = softmax(scale * q[h, i] . k^T) . v with fp32 scores, softmax and sums, causal (row i
// sees keys 0 .. L - M + i) or over all keys. q, k and v are bf16 or fp16, so every product of
// q . k^T is exact; the probabilities go to the matrix cores as kPieces pieces of the input type
// whose sum is their fp32 value. bf16 pieces (8 bits each) have fp32's exponents. The fp16 ones
// (11 bits) are of p * 2^15, the largest that fits, and the second and third, which lie below the
// unit of the first, are scaled by another kLow = 2^12 and summed apart within a tile: the pieces are
// exact from p = 2^-28 of the row's largest on, and below that less than 2^-51 of it short. (With two
// pieces in one sum p = 2^-26 was 2^-14 off, and a quarter of all p 2^-23.)
//
// What bounds it: the MFMA pipe (at D = 128, per 32 queries x 64 keys 512 cycles of q . k^T and
// 512 kPieces of p . v) and beside it the VALU (about 10 instructions a score, the exponential at
// a quarter of the rate). Hence:
//   * the rows of one KV head are (position, query head of the group), heads fastest: a workgroup
//     of 4 waves takes 128 of them, 32 a wave, so a K/V tile is shared by the group's heads and a
//     short prompt still fills the rows;
//   * S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_32x32x16: a lane holds 16 keys of one query,
//     the row maximum is in-lane but for one exchange of lane halves, and the scores are, in
//     place, the B operand of the second product. V^T is read from the row-major V tile with the
//     transposing LDS read;
//   * K and V tiles are copied global -> LDS without passing registers, double buffered, one
//     barrier a tile; 16-byte chunks XOR-swizzled by the row, so both kinds of read are free of
//     bank conflicts;
//   * a grid that would leave CUs idle for long splits the keys (fp32 partials and a combine);
//   * the row tiles of one KV head are consecutive on one XCD, whose L2 then holds its K and V;
//     long causal tiles first.
// Tiles that hold no key a row sees are not read for it, so a value that is not finite there leaves
// it alone; within the last tiles such a value times the zero probability is a NaN, as it is anywhere
// in a product over all keys. Where a row does see it, the zero and negative pieces would make a NaN of
// an infinity too, and values near the end of bf16's range overflow the unnormalised sum: outputs that
// are not finite are looked at again (plain_row).
// Measured: 2048 rows behind 2953 keys, 32/8 heads x 128, bf16: 252 us (528 TFLOP/s of the two
// products, 1060 with the pieces) where torch's fp32 scores, softmax and product took 4042 us.
#pragma once

#include "dspark_attn.h"

namespace dspark {
namespace prefill {

using attn::BF16;
using attn::F16;

constexpr int kThreads = 256;
constexpr int kRows = 128;  // query rows of a workgroup
constexpr float kLowest = -3.402823466e38f;

constexpr int kKeys = 64;   // keys of a tile

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

struct Args {
  const u16* q;
  const u16* k;
  const u16* v;
  u16* out;              // [B, Hq, M, D]
  float* opart;          // key splits: unnormalised outputs [S][B*Hk][R][D], maxima and sums [S][B*Hk][R]
  float* mpart;
  float* lpart;
  long qsb, qsh, qss;    // element strides (batch, head, position)
  long ksb, ksh, kss;
  long vsb, vsh, vss;
  int Hk, gqa, M, L, R;  // R = gqa * M rows of a KV head
  int BH, tiles, S, per_xcd;
  float scale_log2;
  int causal;
};

template <class T>
__device__ __forceinline__ f32x16_t mfma32(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (T::kF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(attn::f16x8_t, a),
                                                   __builtin_bit_cast(attn::f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                    0, 0, 0);
}

// Chunk swizzles: the 16-byte chunk c of tile row r lies at chunk c ^ swz(r) of the row. K rows are
// read 32 at a time at one chunk, V rows 4 at a time over four chunks.
template <int D>
__device__ __forceinline__ int k_swz(int r) { return D == 64 ? (r >> 1) & 7 : r & 15; }
template <int D>
__device__ __forceinline__ int v_swz(int r) { return D == 64 ? ((r >> 1) & 1) << 2 : (r & 3) << 2; }

// Four rows of 16 columns, transposed: lane i of a 16-lane group addresses 4 columns (4 (i & 3))
// of row i >> 2 and receives column i of the four rows.
__device__ __forceinline__ u32x2_t lds_tr(const u16* p) {
  typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
}

constexpr int kPieces = 3;        // of a probability
constexpr float kLow = 4096.f;    // the scale of fp16's second and third

// Eight probabilities as pieces of the input type. fp16 rounds toward zero (two values an
// instruction), which leaves 13 and then 2 of the 24 bits.
template <class T>
__device__ __forceinline__ void split(const f32x16_t& p, int r0, u32x4_t (&o)[kPieces]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = p[r0 + 2 * i], b = p[r0 + 2 * i + 1];
#pragma unroll
    for (int n = 0; n < kPieces; ++n) {
      if constexpr (T::kF16) {
        const attn::f16x2_t h = __builtin_bit_cast(attn::f16x2_t, __builtin_amdgcn_cvt_pkrtz(a, b));
        o[n][i] = __builtin_bit_cast(u32, h);
        if (n == 0) {
          a = __builtin_fmaf((float)h.x, -kLow, a * kLow);
          b = __builtin_fmaf((float)h.y, -kLow, b * kLow);
        } else if (n == 1) {
          const float m1 = __builtin_bit_cast(float, opaque_sgpr(0xBF800000u));  // keeps it one v_fma_mix
          a = __builtin_fmaf((float)h.x, m1, a);
          b = __builtin_fmaf((float)h.y, m1, b);
        }
      } else {
        o[n][i] = attn::pack2<T>(a, b);
        if (n + 1 < kPieces) {
          a -= __builtin_bit_cast(float, o[n][i] << 16);
          b -= __builtin_bit_cast(float, o[n][i] & 0xFFFF0000u);
        }
      }
    }
  }
}

__device__ __forceinline__ bool not_finite(float v) { return !(__builtin_fabsf(v) < __builtin_inff()); }

// The D / 64 adjacent columns of a lane
template <int D>
struct LaneCols {
  u16 c[D / 64];
};

// One row (of KV head bh) that has outputs which are not finite, again, by one wave; m and l are its
// maximum and denominator. Those of columns with such values among the row's keys are the sum of
// these (a NaN, an infinity, or both infinities). Columns with such values only among the keys after
// them that share its last tile (32 positions of a wave's rows, 64 keys) stay NaN. In the others the
// unnormalised sum overflowed: they become the plain sum of fp32 probability times value. An infinite
// value in the first key of 2048 rows over 5001, 32/8 heads x 128: 5.1 ms (the torch ops 4.1).
template <class T, int D>
__device__ __forceinline__ void plain_row(const Args& a, int bh, int row, float m, float l) {
  constexpr int C = D / 64;
  const int lane = threadIdx.x & 63, b = bh / a.Hk, hk = bh - b * a.Hk;
  const int pos = row / a.gqa, hq = hk * a.gqa + (row - pos * a.gqa);
  const int keys = a.causal ? a.L - a.M + pos + 1 : a.L;
  const u16* v = a.v + b * a.vsb + hk * a.vsh + lane * C;
  auto cols = [&](int key) { return *reinterpret_cast<const LaneCols<D>*>(v + key * a.vss); };
  u16* op = a.out + (((long)b * a.Hk * a.gqa + hq) * a.M + pos) * D + lane * C;
  float sum[C] = {}, after[C] = {};
  auto add = [&](int key, float (&to)[C]) {
    const LaneCols<D> x = cols(key);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const float f = attn::to_f32<T>(x.c[c]);
      to[c] += not_finite(f) ? f : 0.f;
    }
  };
#pragma unroll 8
  for (int k = 0; k < keys; ++k) add(k, sum);
#pragma unroll 1
  for (int k = keys; k < min(keys + 32 + kKeys, a.L); ++k) add(k, after);
  bool over[C], any = false;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const bool bad = not_finite(attn::to_f32<T>(op[c]));
    over[c] = bad && !not_finite(sum[c]) && !not_finite(after[c]);
    if (bad && not_finite(sum[c])) op[c] = attn::from_f32<T>(sum[c]);
    any |= over[c];
    sum[c] = 0.f;
  }
  if (!__builtin_amdgcn_ballot_w64(any)) return;
  const u16* q = a.q + b * a.qsb + hq * a.qsh + pos * a.qss;
  const u16* kr = a.k + b * a.ksb + hk * a.ksh;
  const float inv = (T::kF16 ? 32768.f : 1.f) / l;
#pragma unroll 1
  for (int k0 = 0; k0 < keys; k0 += 64) {  // a lane takes a key's score
    const int n = min(64, keys - k0);
    const u16* kp = kr + (k0 + min(lane, n - 1)) * a.kss;
    float s = 0.f;
#pragma unroll 1
    for (int c = 0; c < D; c += 8) {
      const u32x4_t x = ldg128(q + c), y = ldg128(kp + c);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s = __builtin_fmaf(attn::to_f32<T>(x[i] & 0xFFFFu), attn::to_f32<T>(y[i] & 0xFFFFu), s);
        s = __builtin_fmaf(attn::to_f32<T>(x[i] >> 16), attn::to_f32<T>(y[i] >> 16), s);
      }
    }
    const float p = __builtin_amdgcn_exp2f((s - m) * a.scale_log2) * inv;
#pragma unroll 1
    for (int j = 0; j < n; ++j) {
      const float pj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), j));
      const LaneCols<D> x = cols(k0 + j);
#pragma unroll
      for (int c = 0; c < C; ++c) sum[c] = __builtin_fmaf(pj, attn::to_f32<T>(x.c[c]), sum[c]);
    }
  }
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (over[c]) op[c] = attn::from_f32<T>(sum[c]);
}

// Head dim 256 takes one workgroup a CU: its queries and outputs alone are 192 registers, and two
// workgroups spilled 33 over 32-key tiles (bf16, 24/4 heads, 2048 rows: 218 us, so 200; 16/8 heads,
// 1500 rows over 3000 keys 196 -> 178).
template <class T, int D>
__global__ __launch_bounds__(kThreads, D == 256 ? 1 : 2) void prefill_kernel(const Args a) {
  constexpr int KT = kKeys, SUB = KT / 32, CH = D / 8, NJ = KT * CH / kThreads, ND = D / 32, NK = D / 16;
  __shared__ __attribute__((aligned(16))) u16 sm[2][2][KT * D];  // [buffer][K, V]
  typedef __attribute__((address_space(3))) u16 lds_u16;
  typedef const __attribute__((address_space(1))) u16 glb_u16;

  // one XCD's workgroups (ids equal modulo 8) take consecutive items
  const int item = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if (item >= a.BH * a.tiles * a.S) return;
  const int bh = item / (a.tiles * a.S), rest = item - bh * a.tiles * a.S;
  const int tile = a.tiles - 1 - rest / a.S, z = rest % a.S;
  const int b = bh / a.Hk, hk = bh - b * a.Hk;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int l31 = lane & 31, half = lane >> 5, l16 = lane & 15;

  const int r0 = tile * kRows, rw = r0 + 32 * wave;          // first row of the workgroup / wave
  const int row = min(rw + l31, a.R - 1);                    // rows past R repeat the last one, dropped
  const int pos = row / a.gqa, hq = hk * a.gqa + (row - pos * a.gqa);
  const int prefix = a.L - a.M;
  // last key a row sees: this lane's, the wave's smallest and largest, the workgroup's largest
  const int last = a.L - 1;
  const int lim = a.causal ? prefix + pos : last;
  const int wmin = uniform(a.causal ? prefix + min(rw, a.R - 1) / a.gqa : last);
  const int wmax = uniform(a.causal ? prefix + min(rw + 31, a.R - 1) / a.gqa : last);
  const int bmax = a.causal ? prefix + min(r0 + kRows - 1, a.R - 1) / a.gqa : last;
  const int ntile = bmax / KT + 1;
  const int t0 = (int)((long)ntile * z / a.S), t1 = (int)((long)ntile * (z + 1) / a.S);

  const char* kb = reinterpret_cast<const char*>(a.k + b * a.ksb + hk * a.ksh);
  const char* vb = reinterpret_cast<const char*>(a.v + b * a.vsb + hk * a.vsh);
  auto copy_row = [&](int j) { return ((wave * NJ + j) * 64 + lane) / CH; };
  const u32 kstep = (u32)a.kss * 2, vstep = (u32)a.vss * 2;  // < 2^24
  auto copy = [&](int t, int buf) {
    const char* kp = kb + (long)t * KT * a.kss * 2;
    const char* vp = vb + (long)t * KT * a.vss * 2;
    const int rmax = last - t * KT;  // rows past the keys repeat the last one (and are masked)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = copy_row(j);
      const u32 off = __umul24((u32)min(r, rmax), kstep) + (u32)((lane % CH ^ k_swz<D>(r)) << 4);
      __builtin_amdgcn_global_load_lds((glb_u16*)(kp + off), (lds_u16*)&sm[buf][0][(wave * NJ + j) * 512], 16, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = copy_row(j);
      const u32 off = __umul24((u32)min(r, rmax), vstep) + (u32)((lane % CH ^ v_swz<D>(r)) << 4);
      __builtin_amdgcn_global_load_lds((glb_u16*)(vp + off), (lds_u16*)&sm[buf][1][(wave * NJ + j) * 512], 16, 0, 0);
    }
  };

  if (t0 < t1) copy(t0, 0);
  u32x4_t qf[NK];
  const u16* qp = a.q + b * a.qsb + hq * a.qsh + pos * a.qss + 8 * half;
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) qf[kk] = ldg128(qp + 16 * kk);

  f32x16_t o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
  float m = kLowest, l = 0.f;  // l: this lane's half of the keys
  const int kswz = k_swz<D>(l31), kbase = l31 * D;
  const int vrow = 4 * half + (l16 >> 2), vswz = v_swz<D>(l16 >> 2);
  const int vchunk = 2 * ((lane >> 4) & 1) + ((l16 & 3) >> 1), vbase = vrow * D + 4 * (l16 & 1);

  for (int t = t0; t < t1; ++t) {
    const int buf = (t - t0) & 1;
    // tile t has landed once every wave's copies have; every read of the other buffer is done
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (t + 1 < t1) copy(t + 1, buf ^ 1);
    const int key0 = t * KT;
    if (key0 > wmax) continue;  // wave-uniform; the barrier above is reached by all
    const u16* ks = sm[buf][0];
    const u16* vs = sm[buf][1];

    f32x16_t s[SUB];
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[u][r] = 0.f;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk)
#pragma unroll
      for (int u = 0; u < SUB; ++u)
        s[u] = mfma32<T>(*reinterpret_cast<const u32x4_t*>(ks + u * 32 * D + kbase + (((2 * kk + half) ^ kswz) << 3)),
                         qf[kk], s[u]);
    if (key0 + KT - 1 > wmin) {
#pragma unroll
      for (int u = 0; u < SUB; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (key0 + 32 * u + 8 * (r >> 2) + 4 * half + (r & 3) > lim) s[u][r] = -__builtin_inff();
    }
    float mx = m;
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[u][r]);
    mx = max_xor32(mx);
    if (__builtin_amdgcn_ballot_w64(mx > m)) {
      const float alpha = __builtin_amdgcn_exp2f((m - mx) * a.scale_log2);
      m = mx;
      l *= alpha;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
    }
    float sum = 0.f;
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        // the difference first: exact where it matters, whatever the size of the scores
        float p = __builtin_amdgcn_exp2f((s[u][r] - m) * a.scale_log2);
        if constexpr (T::kF16) p *= 32768.f;
        s[u][r] = p;
        sum += p;
      }
    }
    l += sum;
    // Head dim 64, where the products are the shorter phase: ahead of the other workgroup's softmax
    // (2000 rows over 4000 keys 53 -> 46 us, 2048 over 2048 32.6 -> 29.2; at 128 a first chunk lost 9%)
    if constexpr (D == 64) __builtin_amdgcn_s_setprio(1);
    auto v_frag = [&](int uj, int d) {  // V^T of keys 16 uj .. 16 uj + 15, columns 32 d ..
      const u16* vp = vs + 16 * uj * D + vbase + (((4 * d + vchunk) ^ vswz) << 3);
      const u32x2_t lo = lds_tr(vp), hi = lds_tr(vp + 8 * D);
      return u32x4_t{lo.x, lo.y, hi.x, hi.y};
    };
    if constexpr (T::kF16) {
      // Two column blocks of scaled sums at a time: sums kept over the tiles (as many registers as the
      // outputs) spilled at head dim 128 and moved 1346 registers a tile at 256. Against two pieces in
      // one sum: 2048 rows over 5001 keys, 32/8 x 128, 226 -> 271 us; 24/4 x 256, 2048 rows, 155 -> 205.
      constexpr int DB = 2;
      u32x4_t p[2 * SUB][kPieces];
#pragma unroll
      for (int d0 = 0; d0 < ND; d0 += DB) {
        f32x16_t low[DB];
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) low[d][r] = 0.f;
#pragma unroll
        for (int uj = 0; uj < 2 * SUB; ++uj) {
          if (d0 == 0) split<T>(s[uj >> 1], 8 * (uj & 1), p[uj]);
          u32x4_t vf[DB];
#pragma unroll
          for (int d = 0; d < DB; ++d) vf[d] = v_frag(uj, d0 + d);
#pragma unroll
          for (int d = 0; d < DB; ++d) o[d0 + d] = mfma32<T>(vf[d], p[uj][0], o[d0 + d]);
#pragma unroll
          for (int n = 1; n < kPieces; ++n)
#pragma unroll
            for (int d = 0; d < DB; ++d) low[d] = mfma32<T>(vf[d], p[uj][n], low[d]);
        }
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[d0 + d][r] = __builtin_fmaf(low[d][r], 1.f / kLow, o[d0 + d][r]);
      }
    } else {
      constexpr int DB = ND < 4 ? ND : 4;  // V fragments in flight
#pragma unroll
      for (int uj = 0; uj < 2 * SUB; ++uj) {
        u32x4_t p[kPieces];
        split<T>(s[uj >> 1], 8 * (uj & 1), p);
#pragma unroll
        for (int d0 = 0; d0 < ND; d0 += DB) {
          u32x4_t vf[DB];
#pragma unroll
          for (int d = 0; d < DB; ++d) vf[d] = v_frag(uj, d0 + d);
#pragma unroll
          for (int n = 0; n < kPieces; ++n)
#pragma unroll
            for (int d = 0; d < DB; ++d) o[d0 + d] = mfma32<T>(vf[d], p[n], o[d0 + d]);
        }
      }
    }
    if constexpr (D == 64) __builtin_amdgcn_s_setprio(0);
  }

  l += shfl_xor(l, 32);
  const bool own = rw + l31 < a.R;
  if (a.S > 1) {
    if (!own) return;
    const long pr = ((long)z * a.BH + bh) * a.R + row;
    if (half == 0) {
      a.mpart[pr] = m;
      a.lpart[pr] = l;
    }
    float* op = a.opart + pr * D + 4 * half;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4_t*>(op + 32 * d + 8 * g) =
            f32x4_t{o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]};
    return;
  }
  const float inv = 1.0f / l;
  float zero = 0.f;  // NaN once an output is not finite
  if (own) {
    u16* op = a.out + (((long)b * a.Hk * a.gqa + hq) * a.M + pos) * D + 4 * half;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
#pragma unroll
        for (int r = 0; r < 4; ++r) zero = __builtin_fmaf(o[d][4 * g + r], 0.f, zero);
        *reinterpret_cast<u32x2_t*>(op + 32 * d + 8 * g) =
            u32x2_t{attn::pack2<T>(o[d][4 * g] * inv, o[d][4 * g + 1] * inv),
                    attn::pack2<T>(o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv)};
      }
  }
  // a denominator that is not a number came from the scores, and leaves NaN as it should
  unsigned long long bad = __builtin_amdgcn_ballot_w64(zero != 0.f && l > 0.f && l < __builtin_inff());
  if (!bad) return;
  __threadfence_block();  // the outputs above are read back by other lanes
  for (u32 rows = (u32)bad | (u32)(bad >> 32); rows; rows &= rows - 1) {
    const int i = __builtin_ctz(rows);
    auto of = [&](float x) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), i)); };
    plain_row<T, D>(a, bh, rw + i, of(m), of(l));
  }
}

// out = sum_z 2^(m_z - m) o_z / sum_z 2^(m_z - m) l_z over the key splits; 4 outputs a thread.
// A split that saw none of a row's keys has m = kLowest and l = 0.
template <class T, int D>
__global__ __launch_bounds__(256) void combine_kernel(const Args a) {
  constexpr int per = D / 4;  // threads of a row
  const long i = (long)blockIdx.x * 256 + threadIdx.x, rows = (long)a.BH * a.R;
  const bool own = i / per < rows;
  const long row = min(i / per, rows - 1);  // threads past the last row repeat it, and store nothing
  const int d = (int)(i % per) * 4;
  float m = kLowest;
  for (int z = 0; z < a.S; ++z) m = fmaxf(m, a.mpart[z * rows + row]);
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  float l = 0.f;
  for (int z = 0; z < a.S; ++z) {
    const long pr = z * rows + row;
    const float w = __builtin_amdgcn_exp2f((a.mpart[pr] - m) * a.scale_log2);
    const f32x4_t o = *reinterpret_cast<const f32x4_t*>(a.opart + pr * D + d);
    l += w * a.lpart[pr];
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] += w * o[j];
  }
  const int bh = (int)(row / a.R), r = (int)(row - (long)bh * a.R);
  const int pos = r / a.gqa, b = bh / a.Hk, hq = (bh - b * a.Hk) * a.gqa + (r - pos * a.gqa);
  const float inv = 1.0f / l;
  if (own)
    *reinterpret_cast<u32x2_t*>(a.out + (((long)b * a.Hk * a.gqa + hq) * a.M + pos) * D + d) =
        u32x2_t{attn::pack2<T>(acc[0] * inv, acc[1] * inv), attn::pack2<T>(acc[2] * inv, acc[3] * inv)};
  const float zero = acc[0] * 0.f + acc[1] * 0.f + acc[2] * 0.f + acc[3] * 0.f;
  unsigned long long bad = __builtin_amdgcn_ballot_w64(own && zero != 0.f && l > 0.f && l < __builtin_inff());
  if (!bad) return;
  __threadfence_block();
  while (bad) {
    const int lead = __builtin_ctzll(bad) / per * per;  // first lane of the row
    bad &= ~((~0ull >> (64 - per)) << lead);
    auto of = [&](int x) { return __builtin_amdgcn_readlane(x, lead); };
    plain_row<T, D>(a, of(bh), of(r), __builtin_bit_cast(float, of(__builtin_bit_cast(int, m))),
                    __builtin_bit_cast(float, of(__builtin_bit_cast(int, l))));
  }
}

}  // namespace prefill
}  // namespace dspark
