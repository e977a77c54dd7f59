// A number for the layout of the structs that the Python layer, the host side of the steps and the kernels' library share: three
// binaries that are built, or written, one by one, and one memory.  FNV-1a over the name, size and place of every field.
#pragma once
#include <cstddef>
#include <cstdint>

#include "../../include/areal_amd.h"

namespace aa {

constexpr uint64_t kFnvStart = 0xcbf29ce484222325ull;

constexpr uint64_t mix(uint64_t h, const char* name, uint64_t size, uint64_t place) {
  constexpr uint64_t kPrime = 0x100000001b3ull;
  for (; *name; ++name) h = (h ^ (uint8_t)*name) * kPrime;
  h = (h ^ size) * kPrime;
  return (h ^ place) * kPrime;
}

#define AA_STRUCT(type) h = mix(h, #type, sizeof(type), 0)
#define AA_FIELD(type, field) h = mix(h, #field, sizeof(type::field), offsetof(type, field))

constexpr uint64_t layout() {
  uint64_t h = kFnvStart;
  AA_STRUCT(aa_ppo_params);
#define F(field) AA_FIELD(aa_ppo_params, field)
  F(clip_lo); F(clip_hi); F(c_clip); F(has_c_clip); F(has_behave_weight); F(loss_kind); F(sapo_tau_pos); F(sapo_tau_neg);
#undef F
  AA_STRUCT(aa_rs_params);
#define F(field) AA_FIELD(aa_rs_params, field)
  F(enabled); F(level); F(action); F(metric); F(agg); F(has_lower); F(upper); F(lower);
#undef F
  AA_STRUCT(aa_loss_scale);
#define F(field) AA_FIELD(aa_loss_scale, field)
  F(factor); F(total); F(value); F(total_value); F(per_valid_token);
#undef F
  AA_STRUCT(aa_ppo_step);
#define F(field) AA_FIELD(aa_ppo_step, field)
  F(T); F(T_active); F(prox_logp); F(old_logp); F(adv); F(mask); F(cu_seqlens); F(n_segments); F(params); F(rs); F(scale);
  F(logp); F(entropy); F(vmax); F(vmin); F(stat_loss); F(ratio); F(flags); F(approx_kl); F(clip_mask); F(dual_clip_mask);
  F(behave_mask); F(behave_kl); F(mask_out); F(behave_w); F(counts); F(counts_given); F(loss); F(host_counts); F(host_tag);
  F(work);
#undef F
  AA_STRUCT(aa_norm_params);
#define F(field) AA_FIELD(aa_norm_params, field)
  F(mean_level); F(mean_leave1out); F(std_level); F(std_unbiased); F(eps); F(group_size);
#undef F
  AA_STRUCT(aa_advantage_step);
#define F(field) AA_FIELD(aa_advantage_step, field)
  F(bs); F(L); F(loss_mask); F(loss_mask_bytes); F(roll_logp); F(logp); F(ref_logp); F(attention_mask); F(seqlens);
  F(reward_score); F(values); F(kl_ctl); F(discount); F(gae_lambda); F(kl_estimator); F(mask_no_eos_with_zero); F(norm);
  F(mask_out); F(logp_out); F(kl_rewards); F(rewards); F(advantages); F(returns); F(scratch); F(scratch_bytes); F(work);
#undef F
  AA_STRUCT(aa_score_step);
#define F(field) AA_FIELD(aa_score_step, field)
  F(rewards); F(bias); F(scaling); F(clip); F(norm);
#undef F
  return h;
}

#undef AA_STRUCT
#undef AA_FIELD

}  // namespace aa
