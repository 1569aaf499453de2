"""The matrix instructions that the tall blocks' products write out themselves (csrc/gemm_rows_tall.hip): the compiler does not see them as
such, so its wait states are not there.  In the listing of every variant: no ordinary vector instruction in the two places before a
product, and the sums read only behind the two long waits."""
import re
import subprocess

import pytest

from spyinfer_amd.kernels import build


@pytest.mark.parametrize("source,variants", [("gemm_rows_tall", 24)])
def test_no_vector_instruction_beside_a_product(source, variants, tmp_path):
    out = str(tmp_path / "tall.s")
    cmd = [build._hipcc()] + build.HIPCC_FLAGS + ["-I", build.CSRC, "-S", "--cuda-device-only", build.CSRC + "/" + source + ".hip", "-o", out]
    done = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    assert done.returncode == 0, done.stdout.decode(errors="replace")
    with open(out) as f:
        kernels = re.findall(r"^(_Z\d+%s_kernel\S*):(.*?)^\.Lfunc_end" % source, f.read(), re.S | re.M)
    assert len(kernels) == variants
    for name, body in kernels:
        lines = [x.split(";")[0].strip() for x in body.split("\n")]
        lines = [x for x in lines if x and not x.startswith(".")]                         # (labels begin with a dot)
        products = read = 0
        settled = True                                      # no product since the last two long waits
        for i, x in enumerate(lines):
            if x.startswith("v_mfma"):
                products, settled, waits = products + 1, False, 0
                for before in reversed(lines[max(0, i - 2):i]):
                    if before.startswith("s_nop"):
                        waits += int(before.split()[1], 0) + 1
                    assert waits >= 2 or before.startswith("v_mfma") or not before.startswith("v_"), (name, lines[i - 2:i + 1])
            elif (x == "s_nop 15" and lines[i - 1] == "s_nop 15") or x.startswith(("s_branch", "s_endpgm")):
                settled = True                              # (what follows a branch that is always taken does not follow a product)
            elif x.startswith("v_accvgpr_read") or (re.match(r"(ds_write|ds_store|global_store|buffer_store|scratch_store|v_)", x) and re.search(r"\ba(\d|\[)", x.split(",", 1)[-1])):
                read += 1
                assert settled, (name, lines[i - 2:i + 1])
        assert products > 0 and read > 0, name
