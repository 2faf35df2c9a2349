"""Shared pytest setup: markers, import paths and the built libraries."""
import ctypes
import json
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "stwo-ml_amd"))
sys.path.insert(0, os.path.join(ROOT, "oracle"))
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

PRODUCT_SO = os.path.join(ROOT, "stwo-ml_amd", "lib", "libgkr_mi355x.so")
ORACLE_SO = os.path.join(ROOT, "oracle", "_build", "liboracle.so")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device)")
    # Build what is missing (where there is a compiler; other machines receive
    # the libraries prebuilt).
    if not os.path.exists(ORACLE_SO):
        subprocess.run(["make", "-C", os.path.join(ROOT, "oracle")], check=True)
    if not os.path.exists(PRODUCT_SO) and os.path.exists("/opt/rocm/bin/hipcc"):
        subprocess.run(["make", "-C", os.path.join(ROOT, "stwo-ml_amd")], check=True)


@pytest.fixture(scope="session")
def golden():
    with open(os.path.join(ROOT, "tests", "golden", "reference_vectors.json")) as f:
        return json.load(f)


@pytest.fixture(scope="session")
def gpu_ctx():
    import gkr_mi355x as G
    ctx = G.Context(0)
    yield ctx
    ctx.close()


@pytest.fixture(scope="session")
def write_words(gpu_ctx):
    """write_words(matrix, index, words): a matrix's device memory written from outside the library, as a
    program that owns the memory may (the library's own upload refuses words that are not canonical)."""
    copy = ctypes.CDLL("libamdhip64.so.7").hipMemcpy  # the runtime the library has loaded
    copy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]

    def write(matrix, index, words):
        w = np.array(words, dtype=np.uint32)
        assert index + len(w) <= matrix.rows * matrix.cols
        host_to_device = 1
        assert copy(matrix.device_ptr + 4 * index, w.ctypes.data, w.nbytes, host_to_device) == 0

    return write
