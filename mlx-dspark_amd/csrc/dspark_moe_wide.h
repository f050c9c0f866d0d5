// Grouped expert qmm for large buckets (gfx950): the fused MoE block's projections when an expert
// sees many rows (a prompt chunk: M tokens, top-k of E experts, M k / E rows a bucket). The group
// loop is that of the dense prefill product (dspark_qmm_wide.h: exact products of bf16 rows with
// the integer fields, fp32 scales per group, the bias term as a contraction over the rows' group
// sums); a workgroup takes 16 MT rows of one bucket, gathered by their pair order, and 64 NT
// weight rows (SwiGLU: 32 NT gate rows and the up rows of the same columns, so h = swiglu(gate,
// up) leaves the registers).
// What bounds it: at 32 rows a tile the instructions (per wave and group about 130 of 190 are the
// unpacking, the MFMAs and the scale FMAs, the rest the tile's beginning and end) with 2.3 TB/s of
// weights; a deeper prefetch that kept every load in flight cost the third workgroup per CU and was
// no faster (214 against 198 us below).
// Measured, 500 tokens, 128 experts top 8, 2048 x 768, 4 bits: gate/up 98 us, down 79, the block
// 194 us, where the small-bucket kernels (4 rows a pass) took 554 us with the routing in one
// workgroup (98 us of it, now 15).
#pragma once

#include "dspark_qmm_wide.h"

namespace dspark {
namespace wide {

// One row tile of the grouped product, written by the routing: rows [p0, p0 + rows) of the sorted
// pairs belong to expert e.
struct MoeTile {
  int e, p0, rows, pad;
};

struct MoeWideArgs {
  const u16* x;          // [.., K] rows
  const u16* xs;         // their group sums [kPieces][nrows][GP]
  const int* row_index;  // nullable: x row of sorted position p is row_index[p] / row_div (else p)
  const MoeTile* tiles;  // [max_tiles], entries past the last tile have rows = 0
  const char* w[2];      // plain / gate, up: [E, N, K] fields, row-major or dspark_moe_pack's form
  const u16* s[2];
  const u16* b[2];
  u16* y;                // [P, N]
  long ldx, ldy, nrows;
  int K, N, G, GP, row_div, max_tiles, strips, per_xcd;
  bool vec;              // scale / bias rows are whole aligned 16-byte chunks (chunk_rows)
};

// Field of weight row n (of one expert) at k, row-major or packed (16-row tiles in the MFMA lane
// order: lane 16 q + (n & 15) holds the 16 values of quarter q of a group; 4 bits: two groups)
template <int BITS, bool PW>
__device__ __forceinline__ u32 field_at(const char* w, int n, int k, int K) {
  long byte;
  if constexpr (!PW) {
    byte = ((long)n * K + k) * BITS / 8;
  } else {
    const int c = (k >> 4) & 3, g = k >> 6, G = K >> 6;
    const int q = BITS == 4 ? 2 * (c & 1) + (c >> 1) : c;
    const long lane = 16 * q + (n & 15);
    byte = BITS == 4 ? (((long)(n >> 4) * (G >> 1) + (g >> 1)) * 64 + lane) * 16 + (g & 1) * 8 + ((k & 15) >> 1)
                     : (((long)(n >> 4) * G + g) * 64 + lane) * 16 + (k & 15);
  }
  const u32 v = reinterpret_cast<const unsigned char*>(w)[byte];
  return BITS == 4 ? (v >> (4 * (k & 1))) & 15u : v;
}

// Exact fp32 value of one weight of expert e as an elementwise dequantization rounds it
template <int BITS, bool PW>
__device__ __forceinline__ float moe_dequant_at(const MoeWideArgs& a, int e, int which, int n, int k) {
#pragma clang fp contract(off)
  const char* w = a.w[which] + (long)e * a.N * a.K * BITS / 8;
  const long g = ((long)e * a.N + n) * a.G + (k >> 6);
  const float p = bf2f(a.s[which][g]) * (float)field_at<BITS, PW>(w, n, k, a.K);
  return p + bf2f(a.b[which][g]);
}

// One output as the dequantized product in fp32, by a lane or (where its row has terms that are not
// finite, and its weights are) the sum of those; for outputs whose factored sums are not finite
template <int BITS, bool PW>
__device__ __forceinline__ float moe_plain(const MoeWideArgs& a, int e, int which, const u16* xr, int n, bool take,
                                           bool whole) {
  auto weight = [&](int k) { return moe_dequant_at<BITS, PW>(a, e, which, n, k); };
  float acc;
  const bool terms = infinite_terms(xr, a.K, take, acc, weight);
  if (take && (whole || !terms)) {
    acc = 0.f;
    for (int k = 0; k < a.K && acc == acc; ++k) acc = __builtin_fmaf(bf2f(xr[k]), weight(k), acc);
  }
  return acc;
}

template <int BITS, int MT, int NT, bool PW, bool SWIGLU>
__global__ __launch_bounds__(kThreads, MT == 2 && BITS == 4 ? 3 : 2) void moe_wide_kernel(
    const MoeWideArgs a) {
  __shared__ Smem<MT, NT> sm;
  // one XCD's workgroups (ids equal modulo 8) take consecutive items: the strips of a row tile,
  // then the next one, so an expert's weights meet its row tiles in one L2
  const int item = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if (item >= a.max_tiles * a.strips) return;
  const int ti = item / a.strips, strip = item - ti * a.strips;
  const MoeTile tile = a.tiles[ti];
  if (tile.rows <= 0) return;
  constexpr int NW = SWIGLU ? NT / 2 : NT;  // 16-column tiles of a wave
  const int n0 = strip * 64 * NW;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int c16 = lane & 15, q = lane >> 4;

  Tile<MT, NT> t;
  t.G = a.G;
  t.gs = 0;
  t.ge = a.G;
  t.vec = a.vec;
  auto src = [&](int r) {
    const int p = tile.p0 + min(r, tile.rows - 1);  // rows past the bucket repeat its last one
    return a.row_index ? a.row_index[p] / a.row_div : p;
  };
  t.xb = reinterpret_cast<const char*>(a.x);
#pragma unroll
  for (int j = 0; j < kCopies<MT>; ++j) {
    const int r = copy_row<MT>(j);
    t.xoff[j] = (u32)src(r) * (u32)(a.ldx * 2) + copy_chunk(r) * 16;
  }
  t.xs = a.xs;
  t.xs_piece = a.nrows * a.GP;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) t.xsoff[mt] = (u32)src(16 * mt + c16) * (u32)a.GP;
  const long wbytes = (long)a.N * a.K * BITS / 8, sstride = (long)a.N * a.G;
  t.wb[0] = a.w[0] + tile.e * wbytes;
  t.wb[1] = a.w[SWIGLU ? 1 : 0] + tile.e * wbytes;
  const u16* sc[2] = {a.s[0] + tile.e * sstride, a.s[SWIGLU ? 1 : 0] + tile.e * sstride};
  const u16* bi[2] = {a.b[0] + tile.e * sstride, a.b[SWIGLU ? 1 : 0] + tile.e * sstride};
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int up = SWIGLU && nt >= NW ? 1 : 0;
    const int col = n0 + wave * 16 * NW + (nt - up * NW) * 16;
    const int n = min(col + c16, a.N - 1);
    if constexpr (PW) {  // N % 16 == 0: whole tiles
      const int tl = min(col, a.N - 16) >> 4;
      t.woff[nt] = (u32)tl * (u32)(BITS == 4 ? a.G >> 1 : a.G) * 1024u + (u32)lane * 16u;
    } else {
      t.woff[nt] = (u32)n * (u32)(a.K * BITS / 8) + (u32)k_chunk<BITS>(q) * (BITS == 8 ? 8u : 4u);
    }
    t.brow[nt] = bi[up] + (long)n * a.G;
    t.sown[nt] = sc[up] + (long)n * a.G;
  }
  {  // the scale row this thread stages: wave, tile and column in the order they are read
    const int w = (tid / (16 * NT)) & 3, nt = (tid >> 4) % NT, up = SWIGLU && nt >= NW ? 1 : 0;
    const int n = min(n0 + w * 16 * NW + (nt - up * NW) * 16 + (tid & 15), a.N - 1);
    t.srow = (up ? sc[1] : sc[0]) + (long)n * a.G;
  }

  f32x4_t acc[MT][NT];
  tile_loop<BITS, MT, NT, PW, SWIGLU>(t, sm, a.GP, 0, 1, acc);

  auto h = [](float v, float u) { return f2bf(SWIGLU ? swiglu_bf16(bf2f(f2bf(v)), bf2f(f2bf(u))) : v); };
  bool bad = false;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * mt + 4 * q + r;
#pragma unroll
      for (int nt = 0; nt < NW; ++nt) {
        const int n = n0 + wave * 16 * NW + nt * 16 + c16;
        const float v = acc[mt][nt][r], u = acc[mt][NT - NW + nt][r];
        bad |= not_finite(v) || not_finite(u);
        if (m < tile.rows && n < a.N) a.y[(long)(tile.p0 + m) * a.ldy + n] = h(v, u);
      }
    }
  // the factored sums of an infinite x: outputs that are not finite (a gate or up value that is not
  // finite leaves one) again from the plain products
  if (!__builtin_amdgcn_ballot_w64(bad)) return;
  __threadfence_block();  // the wave's outputs are read back by other lanes
  const int n = n0 + wave * 16 * NW + lane;
  bool whole[2];
#pragma unroll
  for (int j = 0; j < (SWIGLU ? 2 : 1); ++j)
    whole[j] = infinite_weights(a.s[j], a.b[j], (long)tile.e * a.N + n - lane, min(16 * NW, a.N - n + lane), a.G, a.vec);
#pragma unroll 1
  for (int m = 0; m < min(16 * MT, tile.rows); ++m) {
    u16* y = a.y + (long)(tile.p0 + m) * a.ldy + min(n, a.N - 1);
    const bool take = lane < 16 * NW && n < a.N && not_finite(bf2f(*y));
    if (!__builtin_amdgcn_ballot_w64(take)) continue;
    const u16* xr = a.x + (long)src(m) * a.ldx;
    float d[2];
#pragma unroll
    for (int j = 0; j < (SWIGLU ? 2 : 1); ++j) d[j] = moe_plain<BITS, PW>(a, tile.e, j, xr, n, take, whole[j]);
    if (take) *y = h(d[0], d[SWIGLU ? 1 : 0]);
  }
}

}  // namespace wide

// Whether the block runs its experts through this kernel rather than the small-bucket ones
bool moe_wide(long M, long H, long I, long E, long k, int bits);
// 16-row tiles of a workgroup for P pairs over E experts
int moe_wide_mt(long P, long E, int bits);
int launch_moe_wide(wide::MoeWideArgs a, bool swiglu, bool packed, int mt, int bits, hipStream_t s);

}  // namespace dspark
