// Host side of the wide (prefill) affine quantized matmul: launch plan and C entry points.
#include <algorithm>

#include "dspark_qmm_wide.h"

namespace dspark {
namespace wide {
namespace {

// Group sums of x as bf16 pieces: xs[p][m][g], sum = piece 0 + piece 1 + piece 2 to 24 bits (the
// fp32 sum); zeros for g in [G, GP). 8 lanes a (row, group).
__global__ __launch_bounds__(256) void wide_xsum_kernel(const u16* __restrict__ x, long ldx, int M, int G, int GP,
                                                        u16* __restrict__ xs) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const long rg = i >> 3;
  if (rg >= (long)M * GP) return;  // whole 8-lane groups leave together
  const int m = (int)(rg / GP), g = (int)(rg - (long)m * GP);
  float s = 0.f;
  if (g < G) {
    const u32x4_t v = ldg128(x + (long)m * ldx + 64 * g + 8 * (i & 7));
#pragma unroll
    for (int j = 0; j < 4; ++j) s += bf2f(v[j] & 0xFFFFu) + bf2f(v[j] >> 16);
  }
  s = sum8_lanes(s);
  if ((i & 7) == 0) {
    const u16 h = f2bf(s);
    const float r1 = s - bf2f(h);
    const u16 mid = f2bf(r1);
    const u16 lo = f2bf(r1 - bf2f(mid));
    const long piece = (long)M * GP, o = (long)m * GP + g;
    xs[o] = h;
    xs[o + piece] = mid;
    xs[o + 2 * piece] = lo;
  }
}

struct Plan {
  int mt, nt, S;            // 16-row tiles and 16-column tiles per wave, K slices
  int mtiles, ntiles;
  int GP;                   // group sums per row, padded to whole MFMA steps
  size_t xs_bytes, part_bytes, total;
};

// Group sums of a row, padded to whole MFMA steps
inline long padded_groups(long K) { return (K / 64 + 31) / 32 * 32; }

inline size_t round256(size_t b) { return (b + 255) / 256 * 256; }

Plan make_plan(long M, long K, long N) {
  Plan p{};
  const long G = K / 64;
  // The cheapest of the tile shapes and K slices under a model fitted to sweeps of them (M 20 to
  // 2048, N 512 to 17408, K 512 to 12288; cycles at the 2.07 GHz these kernels run at; the
  // picked plan is within 10% of the best one swept):
  //   * a workgroup takes 350 + 100 nt + 45 mt nt cycles per group of K when two share a CU (of
  //     either width: the cheaper loads of 4 bits go with the dearer unpacking);
  //   * two workgroups fill a CU, a CU's last one alone takes 1.4 of a share (2048 x 12288 x 4096:
  //     768 workgroups 247 us, but 777 rows of it in 432 workgroups 121 us, in 672 143 us);
  //   * K slices cost their fp32 partial sums, written and read once at 2000 bytes a cycle, and
  //     the launch that adds them (777 x 4096 x 12288: one slice 192 us, four 125 us).
  const long units = (G + 7) / 8;
  double best = 0;
  for (int mt : {8, 6, 4, 2}) {
    for (int nt : {4, 2}) {
      const long mtiles = (M + 16 * mt - 1) / (16 * mt), ntiles = (N + 64 * nt - 1) / (64 * nt);
      for (int S = 1; S <= std::min(units, 16L); ++S) {
        const long share = (mtiles * ntiles * S + 255) / 256;
        const double groups = 8.0 * ((units + S - 1) / S);
        double cost = (share + (share & 1 ? 0.4 : 0.0)) * groups * (350 + 100 * nt + 45 * mt * nt);
        if (S > 1) cost += 6000 + (double)S * M * N * 8 / 2000;
        if (p.mt == 0 || cost < best) {
          best = cost;
          p.mt = mt;
          p.nt = nt;
          p.S = S;
          p.mtiles = (int)mtiles;
          p.ntiles = (int)ntiles;
        }
      }
    }
  }
  p.GP = (int)padded_groups(K);
  p.xs_bytes = round256((size_t)kPieces * M * p.GP * 2);
  p.part_bytes = p.S > 1 ? round256((size_t)p.S * M * N * 4) : 0;
  p.total = p.xs_bytes + p.part_bytes;
  return p;
}

int check(long M, long K, long N, int bits, int group_size) {
  if (bits != 4 && bits != 8) return fail(DSPARK_ERR_UNSUPPORTED, "qmm_wide: bits=%d (4 or 8)", bits);
  if (group_size != 64) return fail(DSPARK_ERR_UNSUPPORTED, "qmm_wide: group_size=%d (64)", group_size);
  if (M < 1 || N < 1 || K < 64 || K % 64 || M > (1L << 24) || N > (1L << 24) || K > (1L << 22))
    return fail(DSPARK_ERR_SHAPE, "qmm_wide: M=%ld K=%ld N=%ld", M, K, N);
  // the group sums take 8 threads each, and a launch has fewer than 2^32
  if (M * padded_groups(K) > (1L << 28))
    return fail(DSPARK_ERR_SHAPE, "qmm_wide: M=%ld x %ld group sums (at most 2^28)", M, padded_groups(K));
  return DSPARK_OK;
}

template <int BITS, int NT>
void launch(const Args& a, int mt, unsigned blocks, hipStream_t s) {
  switch (mt) {
    case 2: hipLaunchKernelGGL((wide_kernel<BITS, 2, NT>), dim3(blocks), dim3(kThreads), 0, s, a); break;
    case 4: hipLaunchKernelGGL((wide_kernel<BITS, 4, NT>), dim3(blocks), dim3(kThreads), 0, s, a); break;
    case 6: hipLaunchKernelGGL((wide_kernel<BITS, 6, NT>), dim3(blocks), dim3(kThreads), 0, s, a); break;
    default: hipLaunchKernelGGL((wide_kernel<BITS, 8, NT>), dim3(blocks), dim3(kThreads), 0, s, a); break;
  }
}

}  // namespace

int launch_group_sums(const u16* x, long ldx, long M, int G, int GP, u16* xs, hipStream_t s) {
  const long threads = M * GP * 8;
  hipLaunchKernelGGL(wide_xsum_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, x, ldx, (int)M, G, GP,
                     xs);
  return check_launch("qmm_wide group sums");
}

}  // namespace wide
}  // namespace dspark

using namespace dspark;

extern "C" size_t dspark_qmm_wide_workspace(int64_t M, int64_t K, int64_t N, int bits, int group_size) {
  if (wide::check(M, K, N, bits, group_size)) return 0;
  return wide::make_plan(M, K, N).total;
}

extern "C" int dspark_qmm_wide(const void* x, int64_t ldx, int64_t M, int64_t K, const uint32_t* w, const void* scales,
                               const void* biases, int64_t N, int bits, int group_size, const void* bias, void* y,
                               int64_t ldy, void* workspace, size_t workspace_bytes, dspark_stream stream) {
  int st = wide::check(M, K, N, bits, group_size);
  if (st) return st;
  if (!x || !w || !scales || !biases || !y) return fail(DSPARK_ERR_ARG, "qmm_wide: null pointer");
  if (ldx < K || ldx > (1L << 22) || ldy < N) return fail(DSPARK_ERR_SHAPE, "qmm_wide: ldx < K, ldx > 2^22 or ldy < N");
  if (!aligned(x, 16) || ldx % 8 || !aligned(w, 16) || !aligned(scales, 2) || !aligned(biases, 2))
    return fail(DSPARK_ERR_ALIGN, "qmm_wide: x and w must be 16-byte aligned, ldx %% 8 == 0");
  const wide::Plan p = wide::make_plan(M, K, N);
  if (!workspace || workspace_bytes < p.total)
    return fail(DSPARK_ERR_WORKSPACE, "qmm_wide: workspace %zu < %zu bytes", workspace_bytes, p.total);
  if (!aligned(workspace, 256)) return fail(DSPARK_ERR_ALIGN, "qmm_wide: workspace must be 256-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  u16* xs = static_cast<u16*>(workspace);

  wide::Args a{};
  a.x = static_cast<const u16*>(x);
  a.xs = xs;
  a.w = w;
  a.s = static_cast<const u16*>(scales);
  a.b = static_cast<const u16*>(biases);
  a.bias = static_cast<const u16*>(bias);
  a.y = static_cast<u16*>(y);
  a.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + p.xs_bytes);
  a.ldx = ldx;
  a.ldy = ldy;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.G = (int)(K / 64);
  a.GP = p.GP;
  a.S = p.S;
  a.mtiles = p.mtiles;
  a.ntiles = p.ntiles;
  a.vec = wide::chunk_rows(a.G, scales, biases);
  const long tiles = (long)p.mtiles * p.ntiles * p.S;
  if (tiles > (1L << 23)) return fail(DSPARK_ERR_SHAPE, "qmm_wide: too many tiles");
  a.per_xcd = (int)((tiles + 7) / 8);

  if ((st = wide::launch_group_sums(a.x, ldx, M, a.G, p.GP, xs, s))) return st;
  const unsigned blocks = (unsigned)a.per_xcd * 8;
  if (bits == 8) {
    if (p.nt == 4) wide::launch<8, 4>(a, p.mt, blocks, s);
    else wide::launch<8, 2>(a, p.mt, blocks, s);
  } else {
    if (p.nt == 4) wide::launch<4, 4>(a, p.mt, blocks, s);
    else wide::launch<4, 2>(a, p.mt, blocks, s);
  }
  if ((st = check_launch("qmm_wide"))) return st;
  if (p.S > 1) {
    const unsigned rb = (unsigned)(((long)M * N + 1023) / 1024);
    if (bits == 8) hipLaunchKernelGGL((wide::wide_reduce_kernel<8>), dim3(rb), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((wide::wide_reduce_kernel<4>), dim3(rb), dim3(256), 0, s, a);
    return check_launch("qmm_wide reduce");
  }
  return DSPARK_OK;
}
