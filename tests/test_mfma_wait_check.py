"""The build's check over the kernels' assembly: for every MFMA opcode the
kernels use, a result read one wait state early on a path through a taken
branch is a finding, one read in time is not, and an opcode without a known
number of states is one."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_spec = importlib.util.spec_from_file_location(
    "mfma_wait_check", os.path.join(ROOT, "freetoken-intel_amd", "csrc", "mfma_wait_check.py"))
wait_check = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(wait_check)

# the states the compiler leaves in a block between the MFMA and a VALU read of its result
STATES = {"v_mfma_f32_16x16x32_bf16": 8, "v_mfma_f32_16x16x4_f32": 10, "v_mfma_scale_f32_16x16x128_f8f6f4": 12,
          "v_mfma_f32_32x32x1_2b_f32": 18}


def _asm(tmp_path, op, states, branch, operands="v[0:3], v[8:11], v[12:15], v[0:3]"):
    """An MFMA, ``states`` wait states (through a taken branch or not), a read of its result."""
    body = [f"\t{op} {operands}"]
    if branch:
        body += ["\ts_cbranch_scc1 .LBB0_2", "; %bb.1:", "\ts_endpgm", ".LBB0_2:"]
        states -= 1
    body += ["\ts_nop 0"] * states + ["\tv_add_f32_e32 v20, v1, v21", "\ts_endpgm"]
    path = tmp_path / "k.s"
    path.write_text("\n_Z1kPf:\n" + "\n".join(body) + "\n.Lfunc_end0:\n")
    return wait_check.check(str(path))


@pytest.mark.parametrize("branch", [False, True])
@pytest.mark.parametrize("op", sorted(STATES))
def test_a_result_read_one_state_early_is_found(tmp_path, op, branch):
    assert len(_asm(tmp_path, op, STATES[op] - 1, branch)) == 1
    assert _asm(tmp_path, op, STATES[op], branch) == []


def test_an_unknown_mfma_is_found(tmp_path):
    assert len(_asm(tmp_path, "v_mfma_f32_32x32x16_bf16", 64, False)) == 1


def test_a_register_outside_the_result_is_no_read(tmp_path):
    op = "v_mfma_f32_16x16x32_bf16"
    assert _asm(tmp_path, op, 1, False, "v[4:7], v[8:11], v[12:15], v[4:7]") == []
