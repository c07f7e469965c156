"""Orders that a kernel's correctness rests on and that no output shows, read
from the AMD assembly the compiler makes of the sources (no GPU)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "sinter-qwen36-nomtp-tu102_amd")


def kernels(src, tmp_path):
    """{mangled name: instructions} of a source file, with the build's flags."""
    import build
    if not (os.path.exists(build.hipcc()) or shutil.which(build.hipcc())):
        pytest.skip("no hipcc")
    flags = [f for f in build.FLAGS if f not in ("-fPIC", "-shared") and not f.startswith("-Rpass")]
    out = tmp_path / "k.s"
    subprocess.run([build.hipcc(), *flags, "--cuda-device-only", "-S", os.path.join(PKG, "csrc", src), "-o", str(out)],
                   check=True, capture_output=True)
    found, name = {}, None
    for line in out.read_text().splitlines():
        m = re.match(r"(_Z\S+|sinter_\w+):", line)
        if m:
            name = m.group(1)
            found[name] = []
        elif name and line.startswith("\t") and not line.startswith(("\t.", "\t;")):
            found[name].append(line.split(";")[0].strip())
            if "s_endpgm" in line:
                name = None
    return found


def test_gdn_scan_stages_over_no_read_in_flight(tmp_path):
    """The GDN scan refills an LDS buffer by DMA without a barrier: every LDS
    read issued before a DMA has returned by then."""
    scans = {n: k for n, k in kernels("prefill.hip", tmp_path).items() if "gdn_scan_ubatch_kernel" in n}
    assert len(scans) == 3
    for name, code in scans.items():
        flying = dmas = 0
        for ins in code:
            if ins.startswith("ds_read"):
                flying += 1
            elif m := re.search(r"s_waitcnt.*lgkmcnt\((\d+)\)", ins):
                flying = min(flying, int(m.group(1)))
            elif ins.startswith("global_load_lds"):
                dmas += 1
                assert flying == 0, f"{name}: {flying} LDS reads may be in flight at a DMA"
        assert dmas >= 4, name
