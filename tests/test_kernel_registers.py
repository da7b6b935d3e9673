"""What the built kernels take of a CU, where a launch counts on it."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest
from test_product_waits import _code_objects


def _resources(tmp_path, pattern):
    """{kernel: (vector registers, bytes of scratch)} by its notes."""
    import vllm_amd
    library = Path(vllm_amd.__file__).parent / "_C.so"
    readelf = shutil.which("llvm-readelf",
                           path="/opt/rocm/llvm/bin:/opt/rocm/bin")
    if not library.exists() or readelf is None:
        pytest.skip("extension or readelf not there")
    out = {}
    for i, code in enumerate(_code_objects(library)):
        if not re.search(pattern.encode(), code):
            continue
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        notes = subprocess.run([readelf, "--notes", path], check=True,
                               capture_output=True, text=True).stdout
        for k in notes.split("- .agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(\S+)", k)[1]
            if re.search(pattern, name):
                out[name] = tuple(
                    int(re.search(rf"\.{f}:\s+(\d+)", k)[1])
                    for f in ("vgpr_count", "private_segment_fixed_size"))
    return out


def test_three_workgroups_of_short_prompts(tmp_path):
    """Prompts with heads of 64, alone and beside decode rows: three
    workgroups of four waves a CU (512 registers a lane of a SIMD, given out
    in eights), none with scratch."""
    kernels = _resources(tmp_path, r"(prefill|mixed)_attention_kernel.*Li64E")
    assert len(kernels) == 4 + 8
    for name, (registers, scratch) in kernels.items():
        assert (registers + 7) // 8 * 8 * 3 <= 512, name
        assert scratch == 0, name
