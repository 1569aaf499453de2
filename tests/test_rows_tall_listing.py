"""The matrix instructions that the blocks of many row tiles write out themselves (csrc/gemm_rows_tall.hip): the compiler does not see them as
such, so its wait states are not there.  In the listing of every variant: no ordinary vector instruction in the two places before a
product, and the sums read only behind the two long waits."""
import re
import subprocess

from spyinfer_amd.kernels import build


def test_no_vector_instruction_beside_a_product(tmp_path):
    out = str(tmp_path / "tall.s")
    cmd = [build._hipcc()] + build.HIPCC_FLAGS + ["-I", build.CSRC, "-S", "--cuda-device-only", build.CSRC + "/gemm_rows_tall.hip", "-o", out]
    done = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    assert done.returncode == 0, done.stdout.decode(errors="replace")
    with open(out) as f:
        kernels = re.findall(r"^(_Z\d+gemm_rows_tall_kernel\S*):(.*?)s_endpgm", f.read(), re.S | re.M)
    assert len(kernels) == 24
    for name, body in kernels:
        lines = [x.split(";")[0].strip() for x in body.split("\n")]
        lines = [x for x in lines if x and not x.startswith((".", ";"))]                  # (labels begin with a dot)
        products = [i for i, x in enumerate(lines) if x.startswith("v_mfma")]
        assert len(products) > 0
        for i in products:
            waits = 0
            for x in reversed(lines[max(0, i - 2):i]):
                if x.startswith("s_nop"):
                    waits += int(x.split()[1], 0) + 1
                assert waits >= 2 or x.startswith("v_mfma") or not x.startswith("v_"), (name, lines[i - 2:i + 1])
        first = [i for i, x in enumerate(lines) if x.startswith("v_accvgpr_read") or (re.match(r"(ds_write|global_store|buffer_store|scratch_store)", x) and re.search(r"\ba(\d|\[)", x))]
        assert first and min(first) > max(products), name
        assert [x for x in lines[max(products):min(first)] if x.startswith("s_nop")][:2] == ["s_nop 15", "s_nop 15"], name
