// Host side of the prefill attention: launch plan and C entry points.
#include <algorithm>
#include <cmath>

#include "dspark_attn_prefill.h"

namespace dspark {
namespace prefill {
namespace {

struct Plan {
  int tiles, S;
  size_t part_floats;
};

Plan make_plan(long B, long Hq, long Hk, long M, long L, long D) {
  Plan p{};
  const long R = Hq / Hk * M;
  p.tiles = (int)((R + kRows - 1) / kRows);
  const long blocks = B * Hk * p.tiles;
  // Key splits by a model of the call's time in us, fitted to sweeps of 1 to 16 splits (17 to 2048 rows,
  // 400 to 4096 keys, 8 to 376 blocks; within 15% of the best split everywhere): W workgroups a CU
  // take their key tiles in turn, a lone one (whose longest causal tile counts) at a slower pace;
  // splits cost the combine's launch and their partials, written and read at 4.1 TB/s. 32/8 heads x
  // 128: 777 rows and keys 30.8 us in one split, 37.8 in three; 300 rows over 3000 keys 91 and 49;
  // 100 over 4000 keys 34.8 in 8, 38.2 in 16; 64/8, 400 rows and keys 20.4 in one, 33.5 in three.
  const double lone = D == 256 ? 3.6 : D == 128 ? 1.76 : 1.43, shared = D == 256 ? 3.6 : D == 128 ? 1.27 : 0.96;
  const long longest = (L + kKeys - 1) / kKeys;
  const double mean = (L - 0.5 * std::min(M, L)) / kKeys, rows = (double)B * Hq * M;
  double best = 0;
  for (long s = 1; s <= std::min(64L, (longest + 3) / 4); ++s) {
    const long w = (blocks * s + 255) / 256;
    const double tiles = w == 1 ? (double)((longest + s - 1) / s) : std::max(1.0, mean / s);
    const double cost = w * tiles * (w == 1 ? lone : shared) + (s > 1 ? 6 + s * rows * D * 8 / 4.1e6 : 0);
    if (s == 1 || cost < best) {
      best = cost;
      p.S = (int)s;
    }
  }
  p.part_floats = p.S > 1 ? (size_t)p.S * B * Hk * R * (D + 2) : 0;
  return p;
}

int check(long B, long Hq, long Hk, long M, long L, long D) {
  if (D != 64 && D != 128 && D != 256)
    return fail(DSPARK_ERR_SHAPE, "prefill_attention: head_dim %ld (64, 128 or 256)", D);
  if (B < 1 || Hq < 1 || Hk < 1 || Hq % Hk || M < 1 || L < 1)
    return fail(DSPARK_ERR_SHAPE, "prefill_attention: B=%ld Hq=%ld Hk=%ld M=%ld L=%ld", B, Hq, Hk, M, L);
  if (B > 65535 || Hq > 65535 || M > (1L << 22) || L > (1L << 28) || B * Hq * M > (1L << 28))
    return fail(DSPARK_ERR_SHAPE, "prefill_attention: B=%ld Hq=%ld M=%ld L=%ld too large", B, Hq, M, L);
  return DSPARK_OK;
}

// (batch, head, position) strides in elements: 16-byte rows, offsets of a tile within 32 bits
int check_strides(const int64_t st[3], const char* what) {
  for (int i = 0; i < 3; ++i)
    if (st[i] < 0 || st[i] % 8 || (i == 2 && st[i] > (1L << 22)))
      return fail(DSPARK_ERR_ALIGN, "prefill_attention: %s strides must be multiples of 8 (position stride <= 2^22)", what);
  return DSPARK_OK;
}

template <class T, int D>
int launch(const Args& a, hipStream_t s) {
  hipLaunchKernelGGL((prefill_kernel<T, D>), dim3((unsigned)a.per_xcd * 8), dim3(kThreads), 0, s, a);
  const int st = check_launch("prefill attention");
  if (st || a.S == 1) return st;
  const long threads = (long)a.BH * a.R * (D / 4);
  hipLaunchKernelGGL((combine_kernel<T, D>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, a);
  return check_launch("prefill attention combine");
}

template <class T>
int launch_d(const Args& a, long D, hipStream_t s) {
  if (D == 64) return launch<T, 64>(a, s);
  if (D == 128) return launch<T, 128>(a, s);
  return launch<T, 256>(a, s);
}

}  // namespace
}  // namespace prefill
}  // namespace dspark

using namespace dspark;

extern "C" size_t dspark_prefill_attention_workspace(int64_t B, int64_t Hq, int64_t Hk, int64_t M, int64_t L,
                                                     int64_t D) {
  if (prefill::check(B, Hq, Hk, M, L, D)) return 0;
  return prefill::make_plan(B, Hq, Hk, M, L, D).part_floats * sizeof(float);
}

extern "C" int dspark_prefill_attention(int dtype, const void* q, const int64_t q_strides[3], int64_t B, int64_t Hq,
                                        int64_t M, int64_t D, const void* k, const void* v,
                                        const int64_t k_strides[3], const int64_t v_strides[3], int64_t Hk, int64_t L,
                                        float scale, int causal, void* out, void* workspace, size_t workspace_bytes,
                                        dspark_stream stream) {
  if (dtype != DSPARK_DTYPE_BF16 && dtype != DSPARK_DTYPE_F16)
    return fail(DSPARK_ERR_UNSUPPORTED, "prefill_attention: dtype %d", dtype);
  if (!q || !k || !v || !out || !q_strides || !k_strides || !v_strides)
    return fail(DSPARK_ERR_ARG, "prefill_attention: null pointer");
  int st = prefill::check(B, Hq, Hk, M, L, D);
  if (st) return st;
  if (causal && L < M) return fail(DSPARK_ERR_SHAPE, "prefill_attention: causal with L=%ld < M=%ld", (long)L, (long)M);
  if (!(scale > 0.0f) || !std::isfinite(scale))
    return fail(DSPARK_ERR_ARG, "prefill_attention: scale %g (finite and > 0)", (double)scale);
  if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(out, 8))
    return fail(DSPARK_ERR_ALIGN, "prefill_attention: q, k and v must be 16-byte aligned");
  if ((st = prefill::check_strides(q_strides, "q")) || (st = prefill::check_strides(k_strides, "k")) ||
      (st = prefill::check_strides(v_strides, "v")))
    return st;
  const prefill::Plan p = prefill::make_plan(B, Hq, Hk, M, L, D);
  if (p.S > 1) {
    if (!workspace || workspace_bytes < p.part_floats * sizeof(float))
      return fail(DSPARK_ERR_WORKSPACE, "prefill_attention: workspace %zu < %zu bytes", workspace_bytes,
                  p.part_floats * sizeof(float));
    if (!aligned(workspace, 16)) return fail(DSPARK_ERR_ALIGN, "prefill_attention: workspace must be 16-byte aligned");
  }
  prefill::Args a{};
  a.q = static_cast<const u16*>(q);
  a.k = static_cast<const u16*>(k);
  a.v = static_cast<const u16*>(v);
  a.out = static_cast<u16*>(out);
  a.qsb = q_strides[0], a.qsh = q_strides[1], a.qss = q_strides[2];
  a.ksb = k_strides[0], a.ksh = k_strides[1], a.kss = k_strides[2];
  a.vsb = v_strides[0], a.vsh = v_strides[1], a.vss = v_strides[2];
  a.Hk = (int)Hk;
  a.gqa = (int)(Hq / Hk);
  a.M = (int)M;
  a.L = (int)L;
  a.R = a.gqa * a.M;
  a.BH = (int)(B * Hk);
  a.tiles = p.tiles;
  a.S = p.S;
  const long rows = (long)a.BH * a.R;
  a.opart = static_cast<float*>(workspace);
  a.mpart = a.opart + rows * p.S * D;
  a.lpart = a.mpart + rows * p.S;
  a.per_xcd = (int)(((long)a.BH * a.tiles * a.S + 7) / 8);
  a.scale_log2 = scale * 1.44269504088896340736f;
  a.causal = causal ? 1 : 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == DSPARK_DTYPE_BF16 ? prefill::launch_d<attn::BF16>(a, D, s) : prefill::launch_d<attn::F16>(a, D, s);
}
