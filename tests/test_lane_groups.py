"""Sums, maxima and choices over neighbouring lanes go by turns within rows of 16: sizes that these cannot serve do not compile."""
import os
import subprocess

import pytest

from swifttransformer_amd.ops import library

try:
    HIPCC = library._hipcc()
except library.KernelLibraryError:
    HIPCC = None
USES = {"common.h": "__global__ void k(float* x) {{ x[threadIdx.x] = st::across_lanes<{0}, false>(x[threadIdx.x]); }}",
        "moe.hip": "__global__ void k(float* x, int* i) {{ st::group_best<{0}>(x[threadIdx.x], i[threadIdx.x]); }}"}


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
@pytest.mark.parametrize("file", sorted(USES))
@pytest.mark.parametrize("lanes,fits", [(8, False), (4, False), (48, False), (16, True), (32, True), (64, True)])
def test_which_groups_compile(tmp_path, file, lanes, fits):
    source = tmp_path / "use.hip"
    source.write_text(f'#include "{os.path.join(library.CSRC, file)}"\n' + USES[file].format(lanes) + "\n")
    flags = [f for f in library.HIPCC_FLAGS if f != "-O3"] + ["-O0"]
    done = subprocess.run([HIPCC, *flags, "-I", library.CSRC, "--cuda-device-only", "-fsyntax-only", str(source)],
                          capture_output=True, text=True, timeout=300)
    assert (done.returncode == 0) == fits and ("whole rows of 16 lanes" in done.stderr) == (not fits), done.stderr
