"""What the compiler made of the kernels, read from the metadata of the built library."""
import os
import re
import subprocess

import pytest

from bytetransformer_amd import build

LLVM = os.path.join(build.ROCM, "llvm", "bin")
KERNELS = os.path.join(build.LIB, "libbt_hip.so")


def _kernel_metadata(tmp_path):
    """{kernel: {key: number}} of every kernel in the library's gfx950 code objects."""
    fat = str(tmp_path / "fat")
    subprocess.run([os.path.join(LLVM, "llvm-objcopy"), "--dump-section", ".hip_fatbin=" + fat, KERNELS,
                    str(tmp_path / "rest")], check=True)
    data = open(fat, "rb").read()
    found = {}
    # one bundle per source file, each starting with this magic
    starts = [m.start() for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data)] + [len(data)]
    for i, (at, end) in enumerate(zip(starts, starts[1:])):
        bundle, code = str(tmp_path / ("bundle%d" % i)), str(tmp_path / ("code%d" % i))
        with open(bundle, "wb") as f:
            f.write(data[at:end])
        subprocess.run([os.path.join(LLVM, "clang-offload-bundler"), "--unbundle", "--type=o", "--input=" + bundle,
                        "--output=" + code, "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"], check=True)
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", code], check=True,
                               stdout=subprocess.PIPE, text=True).stdout
        for block in re.split(r"\n  - \.agpr_count", notes)[1:]:
            keys = dict(re.findall(r"\.(vgpr_spill_count|private_segment_fixed_size|vgpr_count): +(\d+)", block))
            found[re.search(r"\.name: +(\S+)", block).group(1)] = {k: int(v) for k, v in keys.items()}
    return found


@pytest.mark.skipif(not os.path.exists(KERNELS), reason="the kernels have not been built")
def test_no_kernel_spills(tmp_path):
    """A kernel that does not fit its registers pays for it in every tile (the wide attention kernel under mask
    and bias took 97 us in place of 75): none has spilled registers or scratch memory."""
    kernels = _kernel_metadata(tmp_path)
    assert sum("attention_grouped_kernel" in k for k in kernels) >= 12 and len(kernels) > 100
    bad = {k: v for k, v in kernels.items() if v["vgpr_spill_count"] or v["private_segment_fixed_size"]}
    assert not bad, bad
