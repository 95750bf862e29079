// The forward passes as one call each: the launches of every block in the reference's order, issued from native code.
// A block is seven or eight launches of 3-15 us at the sizes of a small population, and issuing one from Python (argument
// marshalling, a pointer per tensor) takes about 11 us: 8 members x 256 tokens were bound by it, not by the GPU (997 us
// per call against 668 us of kernels).
#include "../../include/noise_hip.h"

namespace {
constexpr int DM = 512, FM = 2048, NH = 8;

#define NOISE_TRY(call)       \
  do {                        \
    if (int rc_ = (call)) return rc_; \
  } while (0)
}  // namespace

extern "C" {

int noise_forward(const noise_forward_t* f, int first, int last, noise_stream_t s) {
  if (!f || !f->layers || f->n_layer <= 0 || first < 0 || first > last || last > 6 * f->n_layer + 1) return NOISE_EINVAL;
  const int m = f->members, T = f->T, ps = f->pair_shift;
  const noise_embed_t emb{f->wte, f->vocab, f->wte_a, f->wte_b, f->idx, f->tok_mstride};
  // Deferred residuals. `x = x + lowrank(c_proj, ...)` (train/val/eggroll.py:92-93) is split: the c_proj GEMM writes
  // only its bf16 dense product, and the next kernel that reads the residual stream adds the rank-1 term and the
  // residual with the same fp32 operations, in the same order (the MLP entry for the attention output; the next block
  // entry, or the head, for both outputs of a block).
  noise_pending_t pend[2] = {{f->y_ap, f->u_attn, NH, NH, 1, nullptr},
                             {f->y_mp, f->u_mlp, f->u_mlp_parts, 1, (long)m * T, nullptr}};
  for (int st = first; st < last && st < 6 * f->n_layer; ++st) {
    const int i = st / 6;
    const noise_forward_layer_t& L = f->layers[i];
    const bool ve = L.gate_w != nullptr;
    switch (st % 6) {
      case 0:
        // x0 = norm(lowrank_embed(wte)) (train/val/eggroll.py:74) is never stored: every block entry recomputes its
        // rows from the L2-resident table (the same arithmetic as noise_embed_norm)
        if (i) pend[0].a = f->layers[i - 1].a_proj, pend[1].a = f->layers[i - 1].a_mproj;
        NOISE_TRY(noise_block_entry(i ? f->x : nullptr, nullptr, f->x, f->h, f->u_qkv, L.b_q, L.b_k, L.b_v,
                                    f->lambda_r + i, f->lambda_0 + i, f->eps_r + i, f->eps_0 + i, f->eps_ld, L.gate_w,
                                    L.gate_a, L.gate_b, ve ? f->gate : nullptr, f->sign, m, T, ps, i ? pend : nullptr,
                                    i ? 2 : 0, &emb, s));
        break;
      case 1:
        NOISE_TRY(noise_qkv(f->h, L.w_qkv, L.a_q, L.a_k, L.a_v, f->u_qkv, f->sign, m, T, ps, f->rot_cos, f->rot_sin,
                            ve ? f->gate : nullptr, L.ve_w, f->vocab, L.ve_a, L.ve_b, f->idx, f->tok_mstride, f->qkv,
                            s));
        break;
      case 2:
        // q and k come out of noise_qkv RMS-normalised, so attention's bounded-score softmax applies
        NOISE_TRY(noise_attention(f->qkv, m, T, L.window, 1, NOISE_QK_F16_Q_LOG2, L.b_proj, ps, f->y, f->u_attn, nullptr,
                                  nullptr, 0, s));
        break;
      case 3:
        NOISE_TRY(noise_dense_bf16(f->y, NOISE_LAYOUT_ROWS, DM, DM, L.w_proj, NOISE_LAYOUT_ROWS, m, T, f->y_ap, s));
        break;
      case 4:
        pend[0].a = L.a_proj;
        NOISE_TRY(noise_norm_dot(f->x, f->h, L.b_fc, f->u_fc, f->sign, m, T, ps, pend, 1, s));
        break;
      default:
        // the hidden stays in the library's TILE16 layout between the two MLP GEMMs
        NOISE_TRY(noise_mlp_fc(f->h, L.w_fc, DM, FM, L.a_fc, f->u_fc, L.b_mproj, f->sign, m, T, ps, f->hidden,
                               NOISE_LAYOUT_TILE16, f->u_mlp, s));
        NOISE_TRY(noise_dense_bf16(f->hidden, NOISE_LAYOUT_TILE16, FM, DM, L.w_mproj, NOISE_LAYOUT_WTILE, m, T, f->y_mp,
                                   s));
    }
  }
  if (last > 6 * f->n_layer) {
    const noise_forward_layer_t& L = f->layers[f->n_layer - 1];
    pend[0].a = L.a_proj;
    pend[1].a = L.a_mproj;
    NOISE_TRY(noise_head_ce(f->x, 0, nullptr, f->head_w, f->head_vocab, f->head_format, f->head_a, f->head_b, f->sign,
                            f->targets, f->tok_mstride, m, T, ps, f->reduction, f->loss, f->logits, f->head_ws,
                            f->head_ws_bytes, pend, 2, s));
  }
  return NOISE_OK;
}

int noise_autocast_forward(const noise_autocast_t* f, noise_stream_t s) {
  if (!f || !f->layers || f->n_layer <= 0 || f->batch <= 0 || f->T <= 0 || (long)f->batch * f->T > 0x7fffffffL)
    return NOISE_EINVAL;
  const int B = f->batch, T = f->T, M = B * T;
  const float* z = f->zeros;  // sigma = 0: rank-1 vectors, input-side dots and signs
  for (int i = 0; i < f->n_layer; ++i) {
    const noise_forward_layer_t& L = f->layers[i];
    const bool ve = L.gate_w != nullptr;
    NOISE_TRY(noise_ac_stream(i ? f->x : nullptr, f->wte, f->vocab, f->idx, T, i ? f->y_ap : nullptr,
                              i ? f->y_mp : nullptr, f->lambda_r + i, f->lambda_0 + i, f->x, f->h, L.gate_w,
                              ve ? f->gate : nullptr, M, T, s));
    NOISE_TRY(noise_dense_bf16(f->h, NOISE_LAYOUT_ROWS, DM, 3 * DM, L.w_qkv, NOISE_LAYOUT_ROWS, B, T, f->qkv, s));
    NOISE_TRY(noise_ac_qkv(f->qkv, f->rot_cos, f->rot_sin, ve ? f->gate : nullptr, L.ve_w, ve ? f->vocab : 0, f->idx, T,
                           M, T, s));
    NOISE_TRY(noise_attention(f->qkv, B, T, L.window, 1, NOISE_QK_BF16_V_BF16, nullptr, 0, f->y, nullptr, nullptr,
                              nullptr, 0, s));
    NOISE_TRY(noise_dense_bf16(f->y, NOISE_LAYOUT_ROWS, DM, DM, L.w_proj, NOISE_LAYOUT_ROWS, B, T, f->y_ap, s));
    NOISE_TRY(noise_ac_stream(f->x, nullptr, 0, nullptr, 0, f->y_ap, nullptr, nullptr, nullptr, nullptr, f->h, nullptr,
                              nullptr, M, T, s));
    NOISE_TRY(noise_mlp_fc(f->h, L.w_fc, DM, FM, z, z, z, z, B, T, 0, f->hidden, NOISE_LAYOUT_TILE16, f->upart, s));
    NOISE_TRY(noise_dense_bf16(f->hidden, NOISE_LAYOUT_TILE16, FM, DM, L.w_mproj, NOISE_LAYOUT_WTILE, B, T, f->y_mp, s));
  }
  NOISE_TRY(noise_ac_stream(f->x, nullptr, 0, nullptr, 0, f->y_ap, f->y_mp, nullptr, nullptr, f->xf, nullptr, nullptr,
                            nullptr, M, T, s));
  return noise_head_ce(f->xf, 1, nullptr, f->head_w, f->head_vocab, NOISE_HEAD_BF16, z, z, z, f->targets, T, B, T, 0,
                       f->reduction, f->loss, f->logits, f->head_ws, f->head_ws_bytes, nullptr, 0, s);
}

}  // extern "C"
