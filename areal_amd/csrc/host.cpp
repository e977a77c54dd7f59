// The host side of the steps that are bound by it, in native code: the arrays of a step, the description of it that the C ABI
// takes, the autograd node of the fused logits steps, and the launch of the advantage rows.  The Python layer checks the
// arguments and calls in here once per step; the kernels are reached through include/areal_amd.h like from anywhere else.
//
// What bounds a step of a few hundred tokens, or an advantage batch, is the host: some forty field assignments through ctypes, a
// dozen allocations and views, and an autograd function whose two halves are Python (the second one on autograd's own thread).
// us a pass, all of it in Python / so: PPO step on 200 x 151 936 bf16 127 / 72 (kernels 41), advantages of 512 x 4 096 36.3 / 31.7
// (kernels 31), sequence-level step from hidden states of 1 900 x 1 024 x 50 257 654 / 629; nothing where the kernels hide the
// host: supervised step on 8 192 x 32 768 201 / 201.
// Nothing here outlives a call but the autograd node, which holds tensors and no addresses.
#include <c10/core/DeviceGuard.h>
#include <c10/core/InferenceMode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/extension.h>

#include "areal_amd.h"
#include "layout.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;

namespace {

void* data(const OptTensor& t) { return t.has_value() && t->defined() ? t->data_ptr() : nullptr; }

// the stream that is current on the device, which is also the device that the caller has made current
void* stream_of(const at::Device& device) { return (void*)c10::hip::getCurrentHIPStream(device.index()).stream(); }

// NativeLibraryError with the text of areal_amd._native.check, on any thread
void check(int status, const char* what) {
  if (status == AA_OK) return;
  python_error error;
  {
    py::gil_scoped_acquire gil;
    const std::string text = std::string(what) + " failed: " + aa_status_string(status) + " (status " + std::to_string(status) + ")";
    py::object type = py::module_::import("areal_amd._native").attr("NativeLibraryError");
    PyErr_SetString(type.ptr(), text.c_str());
    error.persist();
  }
  throw error;
}

int dtype_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return AA_BF16;
    case at::kHalf: return AA_F16;
    default: return AA_F32;
  }
}

// ---- the arrays of a step ---------------------------------------------------------------------------------------------
// rows of the float and of the bool array; the counters are the last row of floats
enum { kLogp, kEntropy, kVmax, kVmin, kStatLoss, kRatio, kApproxKl, kBehaveKl, kBehaveW, kCounts, kFloatRows };
enum { kFlags, kMaskOut, kClip, kDual, kBehaveMask, kBoolRows };

// Allocates (floats, bools, loss) and enters them and the arrays that the caller brought in the aa_ppo_step at `address`.
std::tuple<Tensor, Tensor, Tensor> make_step(int64_t address, int64_t T, int64_t T_active, const Tensor& mask, const OptTensor& prox, const OptTensor& old,
                                             const OptTensor& adv, const OptTensor& cu, int64_t n_segments, bool derived, bool sampled,
                                             const OptTensor& behave_w, const OptTensor& counts, const Tensor& work,
                                             const at::Device& device) {
  const int64_t pitch = std::max<int64_t>(64, (T + 63) & ~(int64_t)63);
  const auto options = at::TensorOptions().device(device);
  Tensor floats = at::empty({kFloatRows, pitch}, options.dtype(at::kFloat));
  Tensor bools = at::empty({kBoolRows, pitch}, options.dtype(at::kBool));
  Tensor loss = at::empty({}, options.dtype(at::kFloat));
  auto f = [&](int row) { return (float*)floats.data_ptr() + row * pitch; };
  auto b = [&](int row) { return (uint8_t*)bools.data_ptr() + row * pitch; };
  aa_ppo_step& s = *(aa_ppo_step*)address;
  s.T = T;
  s.T_active = T_active;
  s.prox_logp = (const float*)data(prox);
  s.old_logp = (const float*)data(old);
  s.adv = (const float*)data(adv);
  s.mask = (const uint8_t*)mask.data_ptr();
  s.cu_seqlens = (const int32_t*)data(cu);
  s.n_segments = n_segments;
  s.logp = f(kLogp);
  s.entropy = f(kEntropy);
  s.vmax = f(kVmax);
  s.vmin = f(kVmin);
  s.stat_loss = f(kStatLoss);
  s.ratio = f(kRatio);
  s.flags = b(kFlags);
  if (derived) {
    s.approx_kl = f(kApproxKl);
    s.clip_mask = b(kClip);
    s.dual_clip_mask = b(kDual);
    if (sampled) {
      s.behave_mask = b(kBehaveMask);
      s.behave_kl = f(kBehaveKl);
    }
  }
  if (sampled) {
    s.mask_out = b(kMaskOut);
    s.behave_w = f(kBehaveW);
  } else if (behave_w.has_value()) {
    s.behave_w = (float*)data(behave_w);
  }
  s.counts = counts.has_value() ? (int32_t*)data(counts) : (int32_t*)f(kCounts);
  s.counts_given = counts.has_value() ? 1 : 0;
  s.loss = (float*)loss.data_ptr();
  s.work = work.data_ptr();
  return {floats, bools, loss};
}

Tensor row(const Tensor& rows, int i, int64_t n) {
  return rows.as_strided({n}, {1}, rows.storage_offset() + i * rows.stride(0));
}

// logp, entropy, vmax, vmin, stat_loss, ratio: [n] each
py::list step_rows(const Tensor& floats, int64_t n) {
  py::list out;
  for (int i = kLogp; i <= kRatio; ++i) out.append(row(floats, i, n));
  return out;
}

// The stat dict of ppo_actor_loss_fn (areal/utils/functional/functional.py:505-558); rows: with the per-row outputs as well.
py::dict step_stats(const Tensor& floats, const Tensor& bools, int64_t n, bool rows, bool sampled) {
  py::dict d;
  d["loss"] = row(floats, kStatLoss, n);
  d["importance_weight"] = row(floats, kRatio, n);
  d["approx_kl"] = row(floats, kApproxKl, n);
  d["clip_mask"] = row(bools, kClip, n);
  d["dual_clip_mask"] = row(bools, kDual, n);
  if (rows) {
    d["logprobs"] = row(floats, kLogp, n);
    d["entropy"] = row(floats, kEntropy, n);
    d["vocab_min_logits"] = row(floats, kVmin, n);
    d["vocab_max_logits"] = row(floats, kVmax, n);
  }
  if (sampled) {
    d["behave_approx_kl"] = row(floats, kBehaveKl, n);
    d["behave_imp_weight"] = row(floats, kBehaveW, n);
    d["behave_mask"] = row(bools, kBehaveMask, n);
  }
  return d;
}

// ---- the fused steps on logits ----------------------------------------------------------------------------------------
// An uninitialised [T, V] array for the gradient of `logits`: the same row stride, and the same place inside a 16-byte piece of
// memory, so that the kernels walk both arrays alike (the fused kernel's fast path for rows that do not start on 16-byte
// boundaries asks for that).
Tensor empty_rows_like(const Tensor& logits, int64_t stride) {
  const int64_t T = logits.size(0), V = logits.size(1);
  const int64_t lead = (int64_t)((uintptr_t)logits.data_ptr() % 16) / logits.element_size();
  if (stride == V && lead == 0) return at::empty({T, V}, logits.options());
  return at::empty({lead + (T - 1) * stride + V}, logits.options()).as_strided({T, V}, {stride, 1}, lead);
}

struct FusedLaunch {
  const aa_ppo_step* step;
  const Tensor& loss;
  const Tensor& labels;
  int64_t stride;
  float inv_temperature;
  bool inplace;
};

struct FusedLogits : torch::autograd::Function<FusedLogits> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& logits, const FusedLaunch* a) {
    // In place every kernel reads an element for the last time before it writes it, so the two arrays of the C entry point may
    // be one.
    Tensor dlogits = a->inplace ? logits.detach() : empty_rows_like(logits, a->stride);
    {
      const c10::DeviceGuard guard(logits.device());
      check(aa_logits_ppo_step(a->step, logits.data_ptr(), dtype_of(logits), logits.size(1), a->stride,
                               (const int64_t*)a->labels.data_ptr(), a->inv_temperature, dlogits.data_ptr(),
                               stream_of(logits.device())),
            "aa_logits_ppo_step");
    }
    // written through a raw pointer: an operation that saved the logits for its own backward must fail loudly
    if (a->inplace && !logits.is_inference()) logits.unsafeGetTensorImpl()->bump_version();
    ctx->save_for_backward({dlogits});
    return a->loss;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    // The gradient lies in the buffer that the forward pass wrote and is scaled there, so it can be handed out once: a second
    // backward through a retained graph would scale it again.
    if (ctx->saved_data.count("handed_out"))
      throw std::runtime_error(
          "the gradient of this fused step was already handed out; run the forward pass again "
          "instead of a second backward through a retained graph");
    ctx->saved_data["handed_out"] = true;
    Tensor dlogits = ctx->get_saved_variables()[0];
    const Tensor g = grads[0].to(at::kFloat).contiguous();
    const int64_t T = dlogits.size(0), V = dlogits.size(1);
    const c10::DeviceGuard guard(dlogits.device());
    // an upstream factor other than 1 is applied in place (the kernel returns at once when it is 1)
    check(aa_scale_rows_inplace(dlogits.data_ptr(), dtype_of(dlogits), T, V, T > 1 ? dlogits.stride(0) : V,
                                (const float*)g.data_ptr(), stream_of(dlogits.device())),
          "aa_scale_rows_inplace");
    return {dlogits, Tensor()};
  }
};

Tensor fused_logits(const Tensor& logits, int64_t address, const Tensor& loss, const Tensor& labels, int64_t stride,
                    double inv_temperature, bool inplace) {
  const FusedLaunch a{(const aa_ppo_step*)address, loss, labels, stride, (float)inv_temperature, inplace};
  return FusedLogits::apply(logits, &a);
}

// ---- advantages -------------------------------------------------------------------------------------------------------
// a float32 array that a kernel may take, and write, as it is
bool plain(const OptTensor& t, at::IntArrayRef shape, const at::Device& device) {
  return !t.has_value() || (t->scalar_type() == at::kFloat && t->layout() == at::kStrided && t->is_contiguous() && t->sizes() == shape &&
                            t->device() == device && !t->requires_grad() && (!t->is_inference() || c10::InferenceMode::is_enabled()));
}

// whether two contiguous arrays share memory
bool overlap(const Tensor& a, const OptTensor& b) {
  if (!b.has_value()) return false;
  const char *pa = (const char*)a.data_ptr(), *pb = (const char*)b->data_ptr();
  return pa < pb + b->numel() * b->element_size() && pb < pa + a.numel() * a.element_size();
}

// Whether the row kernel takes these arrays as they are.  What is masked in place (the reference log-probs, and the log-probs
// that are not rolled) is an array of its own: the kernel reads a neighbour's log-prob after that has been masked, one array as
// both policies is masked twice, and with the scores formed on the way (`scored`) a row reads the rewards of its group.
bool advantages_plain(const Tensor& loss_mask, const Tensor& logp, bool roll, const OptTensor& ref_logp, const Tensor& attention_mask,
                      const Tensor& score, const OptTensor& values, bool scored) {
  const auto shape = loss_mask.sizes();
  const auto device = loss_mask.device();
  if (!plain(logp, shape, device) || !plain(ref_logp, shape, device) || !plain(values, shape, device)) return false;
  if (ref_logp.has_value() && (overlap(*ref_logp, logp) || overlap(*ref_logp, values))) return false;
  if (!roll && overlap(logp, values)) return false;
  if (scored && ((ref_logp.has_value() && overlap(score, ref_logp)) || (!roll && overlap(score, logp)))) return false;
  return attention_mask.sizes() == shape && attention_mask.device() == device && plain(score, {shape[0]}, device);
}

using Norm = std::tuple<int, int, int, int, double, int64_t>;  // the fields of aa_norm_params, in order
aa_norm_params norm_params(const Norm& n) {
  return aa_norm_params{std::get<0>(n), std::get<1>(n), std::get<2>(n), std::get<3>(n), (float)std::get<4>(n), std::get<5>(n)};
}
using Scoring = std::tuple<double, double, double, std::optional<Norm>>;  // bias, scaling, clip, normalisation

// (mask, logp, kl_rewards, rewards, advantages, returns).  mask: bool or float32; attention (bool) or seqlens (int64); with
// `scoring` the scores are formed on the way and `score` holds the rewards; work: with a normalisation.
using SixTensors = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>;
SixTensors advantages(const Tensor& mask, const Tensor& logp, bool roll, const OptTensor& ref_logp, const OptTensor& attention,
                      const OptTensor& seqlens, const Tensor& score, const OptTensor& values, double kl_ctl, int kl_estimator,
                      double discount, double gae_lambda, bool mask_no_eos_with_zero, const std::optional<Norm>& norm,
                      const std::optional<Scoring>& scoring, const OptTensor& work) {
  const int64_t bs = mask.size(0), L = mask.size(1);
  const auto device = mask.device();
  const auto options = at::TensorOptions().device(device).dtype(at::kFloat);
  auto make = [&] { return at::empty({bs, L}, options); };
  const Tensor mask_out = make(), kl_rewards = make(), rewards = make(), adv = make(), returns = make();
  const Tensor logp_out = roll ? make() : logp;
  aa_advantage_step a{};
  a.bs = bs;
  a.L = L;
  a.loss_mask = mask.data_ptr();
  a.loss_mask_bytes = mask.scalar_type() == at::kBool ? 1 : 0;
  a.roll_logp = roll ? 1 : 0;
  a.logp = (const float*)logp.data_ptr();
  a.ref_logp = (float*)data(ref_logp);
  a.attention_mask = (const uint8_t*)data(attention);
  a.seqlens = (const int64_t*)data(seqlens);
  if (!scoring.has_value()) a.reward_score = (const float*)score.data_ptr();
  a.values = (const float*)data(values);
  a.kl_ctl = (float)kl_ctl;
  a.discount = (float)discount;
  a.gae_lambda = (float)gae_lambda;
  a.kl_estimator = kl_estimator;
  a.mask_no_eos_with_zero = mask_no_eos_with_zero ? 1 : 0;
  a.mask_out = (float*)mask_out.data_ptr();
  a.logp_out = (float*)logp_out.data_ptr();
  a.kl_rewards = (float*)kl_rewards.data_ptr();
  a.rewards = (float*)rewards.data_ptr();
  a.advantages = (float*)adv.data_ptr();
  a.returns = (float*)returns.data_ptr();
  aa_norm_params norm_c{}, score_norm{};
  Tensor scratch;
  if (norm.has_value()) {
    norm_c = norm_params(*norm);
    a.norm = &norm_c;
    a.scratch_bytes = aa_advantages_scratch_bytes(bs) / 8 * 8;
    scratch = at::empty({a.scratch_bytes / 8}, options.dtype(at::kDouble));
    a.scratch = scratch.data_ptr();
    a.work = data(work);
  }
  {
    const c10::DeviceGuard guard(device);
    if (!scoring.has_value()) {
      check(aa_advantages(&a, stream_of(device)), "aa_advantages");
    } else {
      aa_score_step s{};
      s.rewards = (const float*)score.data_ptr();
      s.bias = (float)std::get<0>(*scoring);
      s.scaling = (float)std::get<1>(*scoring);
      s.clip = (float)std::get<2>(*scoring);
      if (std::get<3>(*scoring).has_value()) {
        score_norm = norm_params(*std::get<3>(*scoring));
        s.norm = &score_norm;
      }
      check(aa_advantages_scored(&a, &s, stream_of(device)), "aa_advantages_scored");
    }
  }
  // written through a raw pointer: autograd is told
  if (ref_logp.has_value() && !ref_logp->is_inference()) ref_logp->unsafeGetTensorImpl()->bump_version();
  if (!roll && !logp.is_inference()) logp.unsafeGetTensorImpl()->bump_version();
  return {mask_out, logp_out, kl_rewards, rewards, adv, returns};
}

}  // namespace

// What allocates or launches does so without the GIL, as torch's own bindings and ctypes do: an allocation may wait for the device, a
// launch for room in the queue, and neither may stop the other threads of a trainer (one of them may have to queue the work that
// is waited for).
PYBIND11_MODULE(_host, m) {
  using without_gil = py::call_guard<py::gil_scoped_release>;
  m.attr("layout") = aa::layout();
  m.def("make_step", &make_step, without_gil());
  m.def("step_rows", &step_rows);
  m.def("step_stats", &step_stats);
  m.def("empty_rows_like", &empty_rows_like, without_gil());
  m.def("fused_logits", &fused_logits, without_gil());
  m.def("advantages_plain", &advantages_plain);
  m.def("advantages", &advantages, without_gil());
}
