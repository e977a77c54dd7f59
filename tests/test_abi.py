"""The C-ABI library builds, loads on a machine without a GPU, and exports every symbol the header declares."""
import ctypes
import re
from pathlib import Path

import pytest

from areal_amd import _native

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "areal_amd.h"


def declared_functions():
    text = HEADER.read_text()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(aa_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_expected_entry_points():
    names = declared_functions()
    for must in ("aa_logits_fwd", "aa_logits_bwd", "aa_logits_ppo_fused", "aa_rejection_sampling", "aa_ppo_loss",
                 "aa_masked_sum", "aa_lmhead_fwd", "aa_lmhead_bwd"):
        assert must in names


def test_library_exports_every_declared_symbol():
    assert _native.LIB_PATH.exists(), "build the library first: python -m areal_amd.build"
    lib = ctypes.CDLL(str(_native.LIB_PATH))
    for name in declared_functions():
        assert hasattr(lib, name), f"{name} is declared in areal_amd.h but not exported"


def test_binding_covers_header_and_loads():
    assert sorted(_native.SIGNATURES) == declared_functions()
    lib = _native.load()
    assert lib.aa_version() >= 100
    assert lib.aa_status_string(0) == b"ok"
    assert lib.aa_status_string(1) == b"invalid argument"


@pytest.mark.parametrize("load", [_native.load, _native.host])
@pytest.mark.parametrize("struct,field", [("PpoStep", "work"), ("PpoStep", "mask"), ("AdvantageStep", "bs"), ("ScoreStep", "norm")])
def test_binaries_of_another_header_are_refused(monkeypatch, load, struct, field):
    """The library and the native host side say which layout of the shared structs they were compiled with: one that lacks a
    field of the binding, or has it elsewhere, is not used."""
    load()
    known = getattr(_native, struct)
    fields = [f for f in known._fields_ if f[0] != field]
    other = type(struct, (ctypes.Structure,), {"__doc__": known.__doc__, "_fields_": fields})
    moved = type(struct, (ctypes.Structure,), {"__doc__": known.__doc__, "_fields_": known._fields_[1:] + known._fields_[:1]})
    for new in (other, moved):
        structs = tuple(new if s is known else s for s in _native._SHARED_STRUCTS)
        monkeypatch.setattr(_native._layout, "__defaults__", (structs,))
        monkeypatch.setattr(_native, "_lib" if load is _native.load else "_host", None)
        with pytest.raises(_native.NativeLibraryError, match="another include/areal_amd.h"):
            load()
        monkeypatch.undo()
    load()


def test_shared_structs_are_those_of_the_header(tmp_path):
    """Name, size and place of every field of the binding's structs, asked of a C compiler."""
    import shutil
    import subprocess

    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no gcc")
    lines = ["#include <stddef.h>", f'#include "{HEADER}"']
    for struct in _native._SHARED_STRUCTS:
        name = struct.__doc__.strip("`")
        lines.append(f"_Static_assert(sizeof({name}) == {ctypes.sizeof(struct)}, \"{name}\");")
        for field, *_ in struct._fields_:
            at = getattr(struct, field)
            lines.append(f"_Static_assert(offsetof({name}, {field}) == {at.offset} && "
                         f"sizeof((({name}*)0)->{field}) == {at.size}, \"{name}.{field}\");")
    src = tmp_path / "t.c"
    src.write_text("\n".join(lines) + "\n")
    subprocess.run([gcc, "-std=c11", "-Wall", "-Werror", "-fsyntax-only", str(src)], check=True)


def test_header_is_plain_c(tmp_path):
    import shutil
    import subprocess

    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no gcc")
    src = tmp_path / "t.c"
    src.write_text(f'#include "{HEADER}"\nint main(void) {{ return AA_OK; }}\n')
    subprocess.run([gcc, "-std=c99", "-Wall", "-Werror", "-fsyntax-only", str(src)], check=True)


def test_count_on_device_marker_agrees_with_the_header(tmp_path):
    """``AA_LMHEAD_COUNT_ON_DEVICE`` of the binding is the header's: a C program prints the macro."""
    import shutil
    import subprocess

    gcc = shutil.which("gcc")
    if gcc is None:
        pytest.skip("no gcc")
    src, exe = tmp_path / "m.c", tmp_path / "m"
    src.write_text(f'#include <stdio.h>\n#include "{HEADER}"\n'
                   'int main(void) { printf("%lld\\n", (long long)AA_LMHEAD_COUNT_ON_DEVICE); return 0; }\n')
    subprocess.run([gcc, "-std=c99", "-Wall", "-Werror", str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    assert int(out) == _native.AA_LMHEAD_COUNT_ON_DEVICE


def test_argument_validation_without_gpu():
    """Entry points reject bad arguments before touching the device."""
    lib = _native.load()
    null = ctypes.c_void_p(0)
    assert lib.aa_logits_fwd(null, 0, 1, 8, 8, null, 1.0, null, null, null, null, null, null, null) == 1
    assert lib.aa_copy_bytes(null, null, 16, null) == 1
    assert lib.aa_masked_sum(null, null, -1, null, null, null, null) == 1


def test_argument_validation_of_the_sibling_entry_points_without_gpu():
    """The losses, reductions and layout entry points return AA_ERR_INVALID_ARGUMENT (or AA_OK for empty input) before
    any launch: null outputs, negative sizes, enum values out of range."""
    lib = _native.load()
    z = ctypes.c_void_p(0)
    p = ctypes.c_void_p(256)        # a non-null address that is never dereferenced on the host
    bad, ok = 1, 0
    assert lib.aa_kl_estimate(p, p, -1, 0, 0, p, z) == bad
    assert lib.aa_kl_estimate(p, p, 4, 3, 0, p, z) == bad
    assert lib.aa_kl_estimate(z, z, 0, 0, 0, z, z) == ok
    assert lib.aa_dpo_seq_sums(p, p, p, p, -1, 4, p, p, p, z) == bad
    assert lib.aa_dpo_seq_sums(p, p, p, z, 2, 4, p, p, p, z) == bad
    assert lib.aa_dpo_seq_sums(z, z, z, z, 0, 0, z, z, z, z) == ok
    assert lib.aa_dpo_seq_sums_bwd(z, z, p, p, 2, 4, p, z) == bad
    assert lib.aa_dpo_preference_loss(p, 4, 0.1, 2, p, z, z) == bad
    assert lib.aa_dpo_preference_loss(p, 4, 0.1, 0, z, z, z) == bad
    assert lib.aa_dpo_preference_loss(z, 0, 0.1, 0, z, z, z) == ok
    assert lib.aa_dpo_pair_loss(p, p, p, p, 2, 0.1, 0, z, p, p, p, p, p, p, z) == bad
    assert lib.aa_dpo_pair_loss(p, p, p, p, 2, 0.1, 5, p, p, p, p, p, p, p, z) == bad
    assert lib.aa_rw_pair_loss(p, 4, z, 1, p, p, p, p, p, p, z, z) == bad
    assert lib.aa_rw_pair_loss(z, 4, p, 1, p, p, p, p, p, p, z, z) == bad
    assert lib.aa_sft_loss(p, p, 4, z, 2, p, z, p, z, z, p, p, z, z) == bad       # sequences without cu_seqlens
    assert lib.aa_sft_loss(p, p, 4, p, 2, z, z, p, z, z, p, p, z, z) == bad       # no token count
    assert lib.aa_sft_loss(z, z, 4, p, 2, p, z, p, z, z, p, p, z, z) == bad
    assert lib.aa_logging_stats(p, p, z, z, p, 4, 0, 1, 0, p, p, 1 << 20, z) == bad    # a method without versions
    assert lib.aa_logging_stats(p, p, z, p, p, 4, 0, 7, 1, p, p, 1 << 20, z) == bad    # errors without ground truth
    assert lib.aa_logging_stats(p, p, z, p, p, 4, 0, 8, 0, p, p, 1 << 20, z) == bad
    assert lib.aa_logging_stats(p, p, z, p, p, 4, 0, 1, 0, p, p, 8, z) == bad          # scratch too small
    assert lib.aa_logging_stats_scratch_bytes(-1) == -1 and lib.aa_logging_stats_scratch_bytes(100000) > 0
    assert lib.aa_masked_normalization(p, z, 2, 8, 0, 1e-5, p, p, 8, z) == bad         # scratch too small
    assert lib.aa_masked_normalization(z, z, 0, 8, 0, 1e-5, z, z, 0, z) == ok
    assert lib.aa_masked_normalization_scratch_bytes(4, -1) == -1
    assert lib.aa_overlong_penalty(p, p, 4, 8, 0, 1.0, 100, z) == bad                   # division by overlong_tokens
    assert lib.aa_kd_terms(p, z, p, p, 4, 1, p, p, z) == bad                            # pure form without old log-probs
    assert lib.aa_vocab_partials_combine(p, p, p, 0, 4, p, z, z, z, z) == bad       # no slice
    assert lib.aa_vocab_partials_combine(z, p, p, 2, 4, p, z, z, z, z) == bad
    assert lib.aa_vocab_partials_combine(z, z, z, 2, 0, p, z, z, z, z) == ok
    params = _native.PpoParams(clip_lo=0.8, clip_hi=1.2, loss_kind=7)
    assert lib.aa_logits_ppo_fused(p, 0, 4, 4096, 4096, p, 1.0, 4, p, p, p, z, ctypes.byref(params), p, z, p, z, z, z,
                                   p, p, p, p, z, z) == bad                             # unknown loss kind
    params = _native.PpoParams(loss_kind=2, sapo_tau_pos=1.0, sapo_tau_neg=0.0)
    assert lib.aa_logits_ppo_fused(p, 0, 4, 4096, 4096, p, 1.0, 4, p, p, p, z, ctypes.byref(params), p, z, p, z, z, z,
                                   p, p, p, p, z, z) == bad                             # SAPO gate temperature of zero
    params = _native.PpoParams(clip_lo=0.8, clip_hi=1.2, loss_kind=1)
    assert lib.aa_ppo_loss(p, p, p, p, z, 4, z, 0, 0, ctypes.byref(params), p, p, p, p, p, z) == 2   # unsupported


def test_scores_of_advantage_rows_are_validated_without_gpu():
    """``aa_advantages_scored`` takes no level over the batch and no group of more than AA_SCORE_GROUP rows (``aa_reward_scores``
    does), and refuses null scores, levels out of range and groups of nothing, before any launch."""
    lib, address = _native.load(), 256  # (never dereferenced on the host)
    step = _native.AdvantageStep(bs=4, L=8)
    for name in ("loss_mask", "logp", "attention_mask", "mask_out", "logp_out", "kl_rewards", "rewards", "advantages", "returns"):
        setattr(step, name, address)
    step.logp_out = 2 * address

    def status(*norm, rewards=address):
        scores = _native.ScoreStep(rewards, 0.0, 1.0, 5.0)
        if norm:
            scores.norm = ctypes.pointer(_native.NormParams(norm[0], 0, norm[1], 0, 1e-5, norm[2]))
        return lib.aa_advantages_scored(step, scores, None)

    assert lib.aa_advantages_scored(step, None, None) == 1 and status(rewards=None) == 1
    for levels in ((3, 0), (0, 3), (-1, 2)):
        assert status(*levels, 4) == 1
    assert status(2, 0, 0) == 1 and status(0, 2, -4) == 1
    for levels in ((1, 1), (1, 0), (2, 1)):
        assert status(*levels, 4) == 2
    assert status(2, 2, _native.SCORE_GROUP + 1) == 2
    step.bs = 0
    assert status(2, 2, 4) == 0


@pytest.mark.parametrize("V", [1, 8, 64, 65, 50257, 151936, (1 << 22) - 64, (1 << 22) - 63, (1 << 22) - 8, (1 << 22) - 1])
def test_panel_pitch(V):
    """Whole 128-byte lines of bf16, except next to 2^22: 256 rows of the panel stay below the byte offsets of a tile, or
    reach them where the multiple of 8 does."""
    pitch = int(_native.load().aa_lmhead_panel_pitch(V))
    eight = (V + 7) // 8 * 8
    assert pitch >= V and pitch % 8 == 0
    assert pitch == (V + 63) // 64 * 64 if V <= (1 << 22) - 64 else pitch == eight
