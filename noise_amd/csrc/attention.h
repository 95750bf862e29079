// Internal interface of the attention kernel (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>

// Formats of the q and k columns (values of the C ABI's qk_format).
// QK_BF16_V_BF16: q, k and v bf16 and the probabilities rounded to bf16 for P V (torch's bf16 attention operands)
enum : int { QK_BF16 = 0, QK_F16 = 1, QK_F16_Q_LOG2 = 2, QK_BF16_V_BF16 = 3 };

// One of q, k, v: 16-bit rows of ld elements, head h at columns h*64 .. h*64+63 of row t of its member block. Member p
// reads block p % period: period = members for rows of its own, fewer where members share them (the credit reruns'
// fixed heads and values, one block per batch row).
struct AttnHeads {
  const __bf16* p;
  int ld, period;
};
struct AttnArgs {
  AttnHeads q, k, v;  // v fp16 (bf16 for QK_BF16_V_BF16)
  __bf16* y;          // [members * T, ldy], head h at columns h*64 .. h*64+63; null: only the scores below
  long ldy;
  int members, T, H, window;
  int qk_norm;        // q and k rows are RMS-normalised (scores bounded by 8.03): no running maximum
  int qk_format;      // QK_BF16, QK_F16, QK_F16_Q_LOG2 (fp16, q pre-multiplied by log2(e) / 8: noise_qkv's output) or
                      // QK_BF16_V_BF16 (bf16 q, k, v and probabilities)
  // c_proj input-side dot partials: upart[row * upart_ld + h] = sum_d y[row, h*64+d] bf16(b_proj[dir, h*64+d])
  const float* b_proj;
  long b_ld;
  int pair_shift;
  float* upart;       // nullable
  int upart_ld;
  // per-(member, head) moments of y over tokens: partials [members, H, T/128, 2, 64] reduced into
  // mom_out [members, H, 2, 64] (mean of y, mean of y^2); nullable
  float* mom;
  float* mom_out;
  // scores of the output's change: member p = draw j * score_blocks + block writes, per head and query t,
  // score[((block * H + h) * T + t) * draws + j] = sum_d (y - base) target over the head's 64 dims, base and target fp32
  // [score_blocks, T, H, 64]; nullable
  const float* base;
  const float* target;
  float* score;
  int score_blocks;
};

// Floats of the moment partials workspace.
long attention_moment_partials(int members, int T, int H);
int attention_launch(const AttnArgs& g, hipStream_t s);
