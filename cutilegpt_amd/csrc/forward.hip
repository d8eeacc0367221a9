// The model's prefill forward as one call: the launch sequence of
// CutileGPT.forward issued from native code.  Launching it from Python costs the
// host ~7.5 us a kernel (7 of them a layer), more than the kernels of a short
// prompt or a small model take; from here ~2.5 us.
#include "common.h"

extern "C" int cgpt_forward(const int64_t* a, int64_t n_a, const int64_t* layers, float scale, float eps,
                            cgpt_probe_fn probe, int* failed, void* stream) {
  if (failed != nullptr) *failed = CGPT_FWD_ARGS;
  if (a == nullptr || layers == nullptr || n_a != CGPT_FORWARD_ARGS) return CGPT_EINVAL;
  auto ptr = [](int64_t v) { return reinterpret_cast<void*>(static_cast<uintptr_t>(v)); };
  const int64_t B = a[0], T = a[1], D = a[2], H = a[3], V = a[4], n_layer = a[5], block = a[6];
  const int act = static_cast<int>(a[7]);
  const void *idx = ptr(a[8]), *wte = ptr(a[9]), *wpe = ptr(a[10]), *lnf_w = ptr(a[11]), *lnf_b = ptr(a[12]);
  float* x = static_cast<float*>(ptr(a[13]));
  void *h = ptr(a[14]), *qkv = ptr(a[15]), *att = ptr(a[16]), *f = ptr(a[17]);
  int* err = static_cast<int*>(ptr(a[18]));
  // Head: weight, row stride, rows, and the output's pointer, row stride, dtype;
  // last: only each sequence's last position (the output has B rows).
  const void* head = ptr(a[19]);
  const int64_t head_ld = a[20], head_n = a[21], ldc = a[23];
  void* logits = ptr(a[22]);
  const int logits_dtype = static_cast<int>(a[24]), head_tile = static_cast<int>(a[25]);
  const bool last = a[26] != 0;
  // KV cache of the whole model (0: none): layer i's keys and values at
  // k_cache + i * layer bytes, element strides (batch, head, time), t_max rows.
  uint8_t *kc = static_cast<uint8_t*>(ptr(a[27])), *vc = static_cast<uint8_t*>(ptr(a[28]));
  const int64_t c_layer = a[29], csb = a[30], csh = a[31], cst = a[32], t_max = a[33];
  const int t_qkv = static_cast<int>(a[34]), t_proj = static_cast<int>(a[35]);
  const int t_fc = static_cast<int>(a[36]), t_mlp = static_cast<int>(a[37]);
  // No sequences or no positions: nothing to do, as for every launch below; but
  // no position is no last position.
  if (B < 0 || T < 0 || (last && T == 0) || D <= 0 || H <= 0 || n_layer <= 0 || D % H != 0) return CGPT_EINVAL;
  if (act != CGPT_F32 && act != CGPT_BF16) return CGPT_EDTYPE;
  const int64_t M = B * T, hd = D / H, es = act == CGPT_F32 ? 4 : 2;
  const uint8_t* q = static_cast<const uint8_t*>(qkv);
  const void *k = q + D * es, *v = q + 2 * D * es;
  const int64_t sb = T * 3 * D, st = 3 * D;
  auto run = [&](int tag, auto launch) {
    if (failed != nullptr) *failed = tag;
    if (probe != nullptr && probe(tag, 1) != 0) return CGPT_EINVAL;
    const int rc = launch();
    if (rc == CGPT_OK && probe != nullptr && probe(tag, 0) != 0) return CGPT_EINVAL;
    return rc;
  };
#define CGPT_TRY(tag, call)                                  \
  {                                                          \
    const int rc = run(tag, [&] { return call; });           \
    if (rc != CGPT_OK) return rc;                            \
  }
  // x = wte[idx] + wpe[pos] and h = ln_1(x) of layer 0 in one pass.
  CGPT_TRY(CGPT_FWD_EMBEDDING,
           cgpt_embedding_layernorm(static_cast<const int64_t*>(idx), wte, wpe, nullptr, x, ptr(layers[0]),
                                    ptr(layers[1]), h, M, T, D, V, 0, block, eps, act, act, err, stream))
  for (int64_t i = 0; i < n_layer; ++i) {
    const int64_t* w = layers + i * 16;
    CGPT_TRY(CGPT_FWD_QKV,
             cgpt_gemm(h, ptr(w[2]), ptr(w[3]), qkv, M, 3 * D, D, D, w[12], 3 * D, act, act, act,
                       CGPT_EPI_BIAS, t_qkv, stream))
    if (kc != nullptr)
      CGPT_TRY(CGPT_FWD_KV_STORE,
               cgpt_kv_store(k, v, kc + i * c_layer, vc + i * c_layer, B, H, T, hd, 0, t_max, sb, hd, st, sb, hd,
                             st, csb, csh, cst, act, stream))
    CGPT_TRY(CGPT_FWD_ATTENTION,
             cgpt_attention_fwd(q, k, v, att, B, H, T, T, hd, sb, hd, st, sb, hd, st, sb, hd, st, T * D, hd,
                                D, scale, 1, act, stream))
    // x += att Wo^T + b (residual add in the GEMM epilogue, in place)
    CGPT_TRY(CGPT_FWD_PROJ,
             cgpt_gemm(att, ptr(w[4]), ptr(w[5]), x, M, D, D, D, w[13], D, act, act, CGPT_F32,
                       CGPT_EPI_BIAS_RESID, t_proj, stream))
    CGPT_TRY(CGPT_FWD_LN,
             cgpt_add_layernorm(x, nullptr, nullptr, ptr(w[6]), ptr(w[7]), h, M, D, eps, CGPT_F32, CGPT_F32,
                                act, act, stream))
    CGPT_TRY(CGPT_FWD_FC,
             cgpt_gemm(h, ptr(w[8]), ptr(w[9]), f, M, 4 * D, D, D, w[14], 4 * D, act, act, act,
                       CGPT_EPI_BIAS_GELU, t_fc, stream))
    CGPT_TRY(CGPT_FWD_MLP_PROJ,
             cgpt_gemm(f, ptr(w[10]), ptr(w[11]), x, M, D, 4 * D, 4 * D, w[15], D, act, act, CGPT_F32,
                       CGPT_EPI_BIAS_RESID, t_mlp, stream))
    const bool end = i + 1 == n_layer;
    CGPT_TRY(CGPT_FWD_LN,
             cgpt_add_layernorm(x, nullptr, nullptr, end ? lnf_w : ptr(w[16]), end ? lnf_b : ptr(w[17]), h, M,
                                D, eps, CGPT_F32, CGPT_F32, act, act, stream))
  }
  // The head: of every row, or of rows b * T + T - 1 of h (stride T * D).
  const uint8_t* hl = static_cast<const uint8_t*>(h) + (last ? (T - 1) * D * es : 0);
  CGPT_TRY(CGPT_FWD_HEAD,
           cgpt_gemm(hl, head, nullptr, logits, last ? B : M, head_n, D, last ? T * D : D, head_ld, ldc, act, act,
                     logits_dtype, CGPT_EPI_NONE, head_tile, stream))
  return CGPT_OK;
#undef CGPT_TRY
}
