// The launches of one verify step, enqueued from native code: the sequence a caller of the single
// entry points makes, without its per-launch cost in an interpreter (a step of four small layers, hidden 1024,
// 37 launches of 184 us of kernel time, took 518 us enqueued one by one from Python and takes 189 us).
#include "dspark_common.h"

using namespace dspark;

namespace {

static_assert(sizeof(dspark_verify_layer) == 30 * 8 && sizeof(dspark_verify_args) == 29 * 8, "8-byte fields");

int qmm(const dspark_verify_args& a, const void* x, int64_t ldx, int64_t K, int bits, int count,
        const void* const* packed, void* const* y, const int64_t* n, dspark_stream s) {
  dspark_qmm_packed_problem p[3];
  for (int i = 0; i < count; ++i) p[i] = {x, ldx, packed[i], y[i], n[i], n[i], K};
  return dspark_qmm_packed_multi(p, count, a.M, bits, 64, a.qmm_ws, (size_t)a.qmm_ws_bytes, s);
}

// q/k norm + RoPE + cache write, then attention over the cache into a.att
int attention(const dspark_verify_args& a, const dspark_verify_layer& l, dspark_stream s) {
  const int64_t qw = a.Hq * a.D, kw = a.Hk * a.D, L = a.pos0 + a.M;
  const int64_t kw2[2] = {l.k_head, l.k_pos}, vw2[2] = {l.v_head, l.v_pos};
  const int64_t ks3[3] = {0, l.k_head, l.k_pos}, vs3[3] = {0, l.v_head, l.v_pos};
  const int64_t os[3] = {a.M * qw, a.D, qw};
  const float eps = (float)a.eps, base = (float)a.rope_base, scale = (float)a.scale;
  int st;
  if (!a.kv_bits) {
    if ((st = dspark_qk_norm_rope_kv(a.q, qw, a.k, kw, a.v, kw, a.M, a.Hq, a.Hk, a.D, l.q_norm, l.k_norm, eps, base,
                                     a.pos0, a.qatt, l.k_cache, kw2, l.v_cache, vw2, s)))
      return st;
    return dspark_verify_attention_typed(DSPARK_DTYPE_BF16, a.qatt, 1, a.Hq, a.M, a.D, l.k_cache, l.v_cache, ks3, vs3,
                                         a.Hk, L, scale, a.M > 1, nullptr, a.att, os, a.attn_ws,
                                         (size_t)a.attn_ws_bytes, s);
  }
  const int64_t kq2[2] = {l.ks_head, l.ks_pos}, vq2[2] = {l.vs_head, l.vs_pos};
  const int64_t kq3[3] = {0, l.ks_head, l.ks_pos}, vq3[3] = {0, l.vs_head, l.vs_pos};
  uint32_t *kc = static_cast<uint32_t*>(l.k_cache), *vc = static_cast<uint32_t*>(l.v_cache);
  if ((st = dspark_qk_norm_rope_kv_quantized(a.q, qw, a.k, kw, a.v, kw, a.M, a.Hq, a.Hk, a.D, l.q_norm, l.k_norm, eps,
                                             base, a.pos0, a.qatt, kc, l.k_scales, l.k_biases, kw2, kq2, vc,
                                             l.v_scales, l.v_biases, vw2, vq2, (int)a.kv_bits, 64, s)))
    return st;
  return dspark_verify_attention_quantized(DSPARK_DTYPE_BF16, a.qatt, 1, a.Hq, a.M, a.D, kc, l.k_scales, l.k_biases,
                                           ks3, kq3, vc, l.v_scales, l.v_biases, vs3, vq3, a.Hk, L, scale, a.M > 1,
                                           (int)a.kv_bits, 64, a.att, os, a.attn_ws, (size_t)a.attn_ws_bytes, s);
}

}  // namespace

extern "C" int dspark_verify_step(const dspark_verify_args* args, const dspark_verify_layer* layers, int64_t count,
                                  dspark_stream s) {
  if (!args || !layers) return fail(DSPARK_ERR_ARG, "verify_step: null pointer");
  if (count < 1) return fail(DSPARK_ERR_SHAPE, "verify_step: %lld layers", (long long)count);
  const dspark_verify_args& a = *args;
  const float eps = (float)a.eps;
  const int64_t qw = a.Hq * a.D, kw = a.Hk * a.D;
  const void* h = a.h;  // the residual stream
  int64_t ldh = a.H;
  int st;
  for (int64_t i = 0; i < count; ++i) {
    const dspark_verify_layer& l = layers[i];
    if (i == 0) {
      st = dspark_rmsnorm(h, ldh, nullptr, 0, l.input_norm, a.M, a.H, eps, nullptr, 0, a.y, a.H, s);
    } else {  // the add that completes the layer before writes its stream
      const dspark_verify_layer& p = layers[i - 1];
      st = dspark_rmsnorm(h, ldh, a.r, a.H, l.input_norm, a.M, a.H, eps, p.stream, p.ld_stream, a.y, a.H, s);
      h = p.stream;
      ldh = p.ld_stream;
    }
    if (st) return st;
    const void* qkv[3] = {l.q, l.k, l.v};
    void* out[3] = {a.q, a.k, a.v};
    const int64_t n[3] = {qw, kw, kw};
    if ((st = qmm(a, a.y, a.H, a.H, (int)l.qkv_bits, 3, qkv, out, n, s))) return st;
    if ((st = attention(a, l, s))) return st;
    if ((st = qmm(a, a.att, qw, qw, (int)l.o_bits, 1, &l.o, &a.r, &a.H, s))) return st;
    if ((st = dspark_rmsnorm(h, ldh, a.r, a.H, l.post_norm, a.M, a.H, eps, a.h, a.H, a.y, a.H, s))) return st;
    h = a.h;
    ldh = a.H;
    if ((st = dspark_qmm_swiglu_packed(a.y, a.H, l.gate_up, a.hm, a.I, a.I, a.H, a.M, (int)l.mlp_bits, 64, a.qmm_ws,
                                       (size_t)a.qmm_ws_bytes, s)))
      return st;
    if ((st = qmm(a, a.hm, a.I, a.I, (int)l.down_bits, 1, &l.down, &a.r, &a.H, s))) return st;
  }
  const dspark_verify_layer& p = layers[count - 1];
  if ((st = dspark_rmsnorm(h, ldh, a.r, a.H, a.final_norm, a.M, a.H, eps, p.stream, p.ld_stream, a.y, a.H, s)))
    return st;
  return qmm(a, a.y, a.H, a.H, (int)a.head_bits, 1, &a.head, &a.logits, &a.vocab, s);
}
