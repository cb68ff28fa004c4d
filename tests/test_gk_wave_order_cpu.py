"""gk_dense_kernel passes rows between the lanes of a wavefront through LDS
without a workgroup barrier: in the code built for the GPU, a wave barrier stands
before and after the stores of every stage (two stages in its loop), so that the
compiler keeps the other lanes' reads on their side of them."""
import os
import re
import subprocess

from analisi_amd import build


def test_dense_kernel_orders_its_stages(tmp_path):
    asm = os.path.join(str(tmp_path), "gk.s")
    subprocess.run([build.HIPCC] + build.HIP_FLAGS + ["-w", "--cuda-device-only", "-S",
                                                      os.path.join(build.CSRC, "gk.hip"), "-o", asm], check=True)
    with open(asm) as f:
        text = f.read()
    kernels = re.findall(r"^(_ZN3anl15gk_dense_kernel\w+):(.*?)s_endpgm", text, flags=re.M | re.S)
    assert len(kernels) >= 4
    for name, body in kernels:
        assert body.count("; wave barrier") >= 4, name
