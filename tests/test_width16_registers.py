"""The width-16 kernels hold a token's state in registers: none is spilled, by the compiler's own figures."""
import re
import subprocess

from turbogpt_amd import build


def test_no_register_is_spilled(tmp_path):
    listing = tmp_path / "width16.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "-S", "--offload-device-only", str(build.CSRC / "width16.hip"), "-o", str(listing)],
                   check=True, capture_output=True)
    kernels = dict(zip(re.findall(r"^    \.name: +(\S+)", listing.read_text(), re.M),
                       map(int, re.findall(r"^    \.vgpr_spill_count: +(\d+)", listing.read_text(), re.M))))
    assert len(kernels) >= 10 and any("w16_forward_kernel" in name for name in kernels)
    assert {name: spilled for name, spilled in kernels.items() if spilled} == {}
