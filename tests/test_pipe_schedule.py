"""The compiled form of the hand-scheduled matmul kernels: no spill traffic and no compiler-made wait for vector
memory between a kernel's first and last MFMA (either one silently drains the operand loads that the schedule keeps
in flight; results stay right, the kernel gets slower).  Compiles each instantiation to assembly with hipcc; nothing
runs on a GPU."""
import importlib.util
import os
import shutil

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SCRIPT = os.path.join(HERE, "check_pipe_schedule.py")
spec = importlib.util.spec_from_file_location("check_pipe_schedule", SCRIPT)
chk = importlib.util.module_from_spec(spec)
spec.loader.exec_module(chk)

pytestmark = pytest.mark.skipif(not (os.path.exists(chk.HIPCC) or shutil.which("hipcc")), reason="needs hipcc")


@pytest.mark.parametrize("kernel,own_waits", chk.KERNELS, ids=[k for k, _ in chk.KERNELS])
def test_scheduled_stream_is_free_of_spills_and_foreign_waits(kernel, own_waits, tmp_path):
    problems = chk.check(kernel, own_waits, str(tmp_path))
    assert not problems, "\n".join(problems[:10])


def test_int8_epilogue_branches_by_the_piece(tmp_path):
    """The INT8 kernel stores 32 pieces of four values: a handful of branches for each, not one for every value, on the output type."""
    chk.check("mx_gemm_pipe_kernel<8, 3, 256, 2, 2, 2>", set(), str(tmp_path))
    code = [ln.strip() for ln in open(tmp_path / "one_kernel.s")]
    stores = code[max(i for i, ln in enumerate(code) if ln.startswith("v_mfma")):]
    assert sum(ln.startswith("v_exp_f32") for ln in stores) == 128                                   # values of a thread
    assert sum(ln.startswith(("s_cbranch", "s_branch")) for ln in stores) < 6 * 32
