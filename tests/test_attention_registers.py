"""Registers of the fused decode attention as built: heads of 64 leave room for four waves a SIMD, and no variant spills."""
import re
import subprocess

from spyinfer_amd.kernels import build


def test_waves_that_fit_a_simd(tmp_path):
    out = str(tmp_path / "attention.s")
    cmd = [build._hipcc()] + build.HIPCC_FLAGS + ["-I", build.CSRC, "-S", "--cuda-device-only", build.CSRC + "/attention_mfma.hip", "-o", out]
    done = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    assert done.returncode == 0, done.stdout.decode(errors="replace")
    with open(out) as f:
        text = f.read()
    seen = {}
    for name, body in re.findall(r"^\s*\.amdhsa_kernel (\S+)(.*?)\.end_amdhsa_kernel", text, re.S | re.M):
        seen[name] = (int(re.search(r"\.amdhsa_next_free_vgpr (\d+)", body).group(1)), int(re.search(r"\.amdhsa_private_segment_fixed_size (\d+)", body).group(1)))
    fused = {d: [v for n, v in seen.items() if "attention_mfma_kernelILi%dELb1E" % d in n] for d in (64, 128, 256)}
    assert all(len(v) == 2 for v in fused.values()) and not any(spilled for _, spilled in seen.values())
    # a SIMD has 512 registers a lane, in eights
    assert all(n <= 128 for n, _ in fused[64]) and all(n <= 256 for n, _ in fused[128])
