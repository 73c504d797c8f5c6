// A prompt batch through every layer in one call: the launches of the
// engine's per-layer sequence, issued from native code. The interpreter's
// share of a launch (arguments, checks, the foreign call) was about 9 us,
// more than most of a short prompt's kernels run: 24 layers of 131 rows, 217
// launches, took 1981 us, the device idle a quarter of them; 1538 now, all busy.
#include "status.h"

extern "C" {

int wg_prefill_layers(const wg_prefill_layer *layers, int32_t count, const wg_prefill_batch *b,
                      void *stream) {
  WG_REQUIRE(b && (layers || count == 0) && count >= 0, "wg_prefill_layers: null argument");
  WG_REQUIRE(b->M >= 1 && b->D >= 1, "wg_prefill_layers: %d rows of %d", b->M, b->D);
  const int M = b->M, D = b->D, A = b->attn.heads * b->attn.head_dim;
  const int rows = (b->attn.heads + 2 * b->attn.kv_heads) * b->attn.head_dim;
  for (int i = 0; i < count; i++) {
    const wg_prefill_layer &l = layers[i];
    int rc = wg_norm_to_h2(b->h, M, D, D, l.op_norm, b->eps, b->x16, D, b->rs, stream);
    if (rc) return rc;
    if (l.conv_width) {
      rc = wg_q4_gemm(&l.in, b->x16, M, D, b->bcx, 3 * D, nullptr, 0, b->rs, nullptr, stream);
      if (!rc)
        rc = wg_short_conv(b->bcx, M, D, 3 * D, l.conv_width, l.conv_taps, l.conv_state,
                           l.conv_state, nullptr, b->c16, D, stream);
      if (!rc)
        rc = wg_q4_gemm(&l.out, b->c16, M, D, b->h, D, b->h, D, nullptr, nullptr, stream);
    } else {
      rc = wg_q4_gemm(&l.in, b->x16, M, D, b->qkv, rows, nullptr, 0, b->rs, l.col_of, stream);
      if (!rc)
        rc = wg_head_prep(b->qkv, M, rows, &b->attn, l.q_norm, l.k_norm, b->rope, b->rope_rows,
                          b->pos, b->q, A, l.k_cache, l.v_cache, b->ctx, stream);
      if (!rc)
        rc = wg_attn_prefill(b->q, M, A, &b->attn, l.k_cache, l.v_cache, b->pos, b->ctx,
                             b->att16, A, stream);
      if (!rc)
        rc = wg_q4_gemm(&l.out, b->att16, M, A, b->h, D, b->h, D, nullptr, nullptr, stream);
    }
    if (!rc) rc = wg_norm_to_h2(b->h, M, D, D, l.ffn_norm, b->eps, b->x16, D, b->rs, stream);
    if (!rc) rc = wg_q4_gemm_swiglu(&l.gate_up, b->x16, M, D, b->ff16, b->F, b->rs, stream);
    if (!rc)
      rc = wg_q4_gemm(&l.down, b->ff16, M, b->F, b->h, D, b->h, D, nullptr, nullptr, stream);
    if (rc) return rc;
  }
  return WG_OK;
}

}  // extern "C"
