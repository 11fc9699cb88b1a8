"""The interpreter's handler tables are jumped into by place, so a handler that outgrows its place
must not assemble (gfx950 code is assembled here, none is run)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gpuropolis_amd", "csrc")
KERNEL = """
#include "gpr_device.h"
template <int KC> __device__ void eval(WaveProg p, float *out) {
    __shared__ float ls[(GPR_MAX_DEPTH + 2) * 64 * KC];
    float x[KC], T[KC];
    for (int k = 0; k < KC; k++) x[k] = out[64 * k + lane_id()];
    wave_eval_ls<KC, false>(p, x, T, ls, prog_code<KC, false>(p));
    for (int k = 0; k < KC; k++) out[64 * k + lane_id()] = T[k];
}
__global__ void k_test(WaveProg p, float *out) { KERNEL_BODY }
"""


def assemble(tmp_path, header, body):
    from gpuropolis_amd import build as B
    (tmp_path / "gpr_device.h").write_text(header)
    src = tmp_path / "t.hip"
    src.write_text(KERNEL.replace("KERNEL_BODY", body))
    for f in ("gpr_common.h", "gpr_internal.h", "gpr_index.h"):     # beside the changed header, with their own includes
        (tmp_path / f).write_text(open(os.path.join(CSRC, f)).read().replace("../../include/", os.path.join(ROOT, "include") + "/"))
    return subprocess.run([B.HIPCC, *B.HIP_FLAGS, "--offload-device-only", "-c", str(src), "-o", str(tmp_path / "t.o")],
                          capture_output=True, text=True, timeout=300)


@pytest.mark.parametrize("body", ["eval<1>(p, out);", "eval<4>(p, out);"])
def test_a_handler_that_outgrows_its_place_does_not_assemble(tmp_path, body):
    header = open(os.path.join(CSRC, "gpr_device.h")).read()
    jump = header[header.index("#define GT_JUMP"):].split("\n")[0]
    longer = jump.replace('#define GT_JUMP "', '#define GT_JUMP "' + "s_nop 0\\n\\t" * 16)      # 64 bytes
    r = assemble(tmp_path, header, body)
    assert r.returncode == 0, r.stderr[-2000:]
    r = assemble(tmp_path, header.replace(jump, longer), body)
    assert r.returncode != 0 and ".org" in r.stderr, r.stderr[-2000:]
