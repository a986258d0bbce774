"""Shared fixtures: the native library harness and the CPU oracle."""
import ctypes
import importlib.util
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")


def load_mx():
    """Import rust-mlx_amd (hyphenated directory) as module `rust_mlx_amd`."""
    if "rust_mlx_amd" in sys.modules:
        return sys.modules["rust_mlx_amd"]
    path = os.path.join(ROOT, "rust-mlx_amd", "__init__.py")
    spec = importlib.util.spec_from_file_location("rust_mlx_amd", path)
    mod = importlib.util.module_from_spec(spec)
    sys.modules["rust_mlx_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


@pytest.fixture(scope="session")
def mx():
    return load_mx()


@pytest.fixture(scope="session")
def orc():
    from oracle import oracle

    return oracle


@pytest.fixture(scope="session")
def gemm_plan(tmp_path_factory):
    """The form the GEMM beyond 16 rows takes: "T<32-row blocks>.<k slices>" or
    "D<16-row weight tiles>.<16-row activation tiles>"."""
    src = os.path.join(ROOT, "tests", "gemm_plan.cpp")
    so = str(tmp_path_factory.mktemp("plan") / "gemm_plan.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", src, "-o", so], check=True)
    fn = ctypes.CDLL(so).gemm_plan
    fn.argtypes = [ctypes.c_int] * 5 + [ctypes.c_size_t, ctypes.c_void_p]

    def plan(m, n, k, bits, streams=False, part_floats=0):
        out = (ctypes.c_int * 3)()
        fn(m, n, k, bits, streams, part_floats, out)
        return f"{'TD'[out[0]]}{out[1]}.{out[2]}"

    return plan
