// What the steps (logits, lm_head, given log-probs) share around their loss kernel: the launch ahead of it that counts the
// mask or runs the rejection sampling, and the one behind it that finishes the stat dict and the scalar loss.  Defined
// in ppo_loss.hip.
#pragma once
#include "device_utils.h"

namespace aa {

constexpr int kFinishBlocks = 256;  // most workgroups of a launch that finishes a step
constexpr int kTableTensors = 32;   // most tensors of a moments table

// The work buffer of a step: its counters are zero before the first launch that uses it and left zero by every launch.
// Nothing in it outlives a launch: several threads may launch steps on one stream, and theirs come in any order.
struct StepWork {
  int32_t rows[2];  // row hand-out of the fused logits kernel
  int32_t total, hit, done;
  int32_t finished;
  int32_t logged;
  int32_t outside;
  int32_t pad[8];
  int32_t moments[kTableTensors];
  double partial[kFinishBlocks];
};
static_assert(sizeof(StepWork) <= AA_STEP_WORK_BYTES, "the work buffer of a step");

// Argument check of the parts of a step that these launches and the loss kernels use.
int step_args_status(const aa_ppo_step& p);
// counts (and their copy in host memory), and with rejection sampling mask_out and behave_w
int step_prepare(const aa_ppo_step& p, void* stream);
// approx_kl ... behave_kl (when wanted) and loss, from logp, stat_loss, flags
int step_finish(const aa_ppo_step& p, void* stream);

// the loss parameters with the behaviour weights that go with them
inline aa_ppo_params step_params(const aa_ppo_step& p) {
  aa_ppo_params q = p.params;
  if (p.rs.enabled) q.has_behave_weight = 1;
  return q;
}

// The scale as the loss kernels take it.  The weight of a micro-batch is the count of its whole loss mask; with
// sequence-level rejection sampling counts[0] is that of the tokens inside the sequences, and the launch that counts them
// forms the factor from all of them.  It waits in the step's own output, p.loss, which the last kernel overwrites when it
// has read it.
inline bool scale_ahead(const aa_ppo_step& p) {
  return p.scale.per_valid_token && p.rs.enabled && p.rs.level == AA_RS_LEVEL_SEQUENCE && p.T_active > 0;
}
inline aa_loss_scale step_scale(const aa_ppo_step& p) {
  return scale_ahead(p) ? aa_loss_scale{p.loss, nullptr, 1.f, 1.f, 0} : p.scale;
}

// the mask the loss is summed under
inline const uint8_t* step_mask(const aa_ppo_step& p) {
  return p.rs.enabled && p.rs.action == AA_RS_ACTION_MASK ? p.mask_out : p.mask;
}

}  // namespace aa
