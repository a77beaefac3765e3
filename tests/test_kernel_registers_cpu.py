"""No kernel of the factorization or the sweeps keeps values in scratch memory: some are
written so that the compiler holds them in registers, and another compiler may not.
Cross-compiles the sources (no GPU)."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

from hykkt_amd import build as B


def usage(src):
    r = subprocess.run([B.HIPCC, *B.HIP_FLAGS, *B.HIP_SOURCES[src], "--cuda-device-only", "-c",
                        os.path.join(B.SRC, src), "-o", os.devnull,
                        "-Rpass-analysis=kernel-resource-usage"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return re.findall(r"Function Name: (\S+).*?ScratchSize \[bytes/lane\]: (\d+)", r.stderr, re.S)


def test_no_scratch():
    files = ["kernels_dense.hip", "kernels_trsv.hip", "kernels_forest.hip", "kernels_chol.hip"]
    with ThreadPoolExecutor(len(files)) as ex:
        kernels = [k for found in ex.map(usage, files) for k in found]
    assert len(kernels) >= 23
    spilled = {name: int(size) for name, size in kernels if int(size) > 0}
    assert not spilled
