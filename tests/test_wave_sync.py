"""Data that the lanes of one wave hand each other through LDS passes a memory
fence: the kernels call wave_sync(), and only that function names the compiler's
wave barrier, which orders no memory by itself."""
import glob
import os
import re

from conftest import ROOT

SOURCES = glob.glob(os.path.join(ROOT, "rust-mlx_amd", "csrc", "*.h*"))


def test_wave_barriers_have_a_fence():
    uses = {}
    for path in SOURCES:
        with open(path) as f:
            text = f.read()
        n = len(re.findall(r"__builtin_amdgcn_wave_barrier", text))
        if n:
            uses[os.path.basename(path)] = n
    assert uses == {"common.hpp": 1}
    with open(os.path.join(ROOT, "rust-mlx_amd", "csrc", "common.hpp")) as f:
        body = re.search(r"void wave_sync\(\) \{(.*?)\n\}", f.read(), re.S).group(1)
    assert re.search(r"__builtin_amdgcn_fence\(__ATOMIC_ACQ_REL, \"wavefront\"\);\s*"
                     r"__builtin_amdgcn_wave_barrier\(\);", body)
