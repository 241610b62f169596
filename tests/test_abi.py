"""The C-ABI library loads and exports every symbol include/*.h declares; host-side
validation follows the reference status convention.  No GPU compute is issued."""

import ctypes
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from robolearn_amd import _native

ROOT = Path(__file__).resolve().parents[1]
HEADER = ROOT / "include" / "robolearn_mi355x.h"


def declared_symbols():
    text = re.sub(r"/\*.*?\*/", "", HEADER.read_text(), flags=re.S)
    return sorted(set(re.findall(r"\b(rl_[a-z0-9_]+)\s*\(", text)))


def test_header_compiles_as_c():
    compiler = shutil.which("gcc")
    if compiler is None:
        pytest.skip("gcc missing")
    subprocess.run([compiler, "-std=c99", "-Wall", "-Werror", "-fsyntax-only", "-x", "c", str(HEADER)], check=True)


def test_library_exports_every_declared_symbol():
    library = _native.load()
    names = declared_symbols()
    assert len(names) >= 60
    for name in names:
        assert hasattr(library, name), name
    # the ctypes declaration table covers the same set
    assert set(names) == set(_native.SIGNATURES)


def test_status_convention_reports_validation_errors():
    with pytest.raises(RuntimeError, match="positive"):
        _native.call("rl_gemm", 0, 0, 0, 1, 1, 0, 4, 4, 1, 1, 4, 0, 1, 4, 0, None, 1, 4, 0, None, 0, 0.0, 0, 1, None,
                     0, None, None, None, None)
    assert "GEMM" in _native.last_error()
    handle = _native.load().rl_plan_create(0, 4, 4, 0, 0, 4, 4, 4, 0, 0, 0)
    assert not handle and "positive" in _native.last_error()


def test_dense_plan_metadata_and_workspace_on_host():
    library = _native.load()
    # input_dtype 1 is the reference's IEEE fp16; 3 (bf16 operands) and 2 (fp32 stored, bf16 compute) are this
    # library's additions
    for input_dtype, precision in ((1, "fp16"), (2, "bf16"), (3, "bf16")):
        plan = _native.create("rl_plan_create_mixed", 1024, 8192, 160, 1, 0, 160, 160, 1024, 0, 0, input_dtype,
                              64 << 20)
        metadata = library.rl_plan_tuning_metadata(plan).decode()
        assert f'"mode":"{precision}"' in metadata
        assert library.rl_plan_workspace(plan) <= 64 << 20
        assert library.rl_plan_destroy(plan) == 0
    assert not library.rl_plan_create_mixed(64, 64, 64, 0, 0, 64, 64, 64, 0, 0, 4, 0)
    assert "input_dtype" in _native.last_error()


def test_exports_have_c_linkage():
    library = ctypes.CDLL(str(_native.library_path()))
    assert library.rl_last_error is not None


def plan_kernel(rows, cols, k, input_dtype, transa=1, transb=0, workspace=64 << 20):
    """The metadata's kernel for a row-major [rows, cols] product over k (the plan's view is its transpose)."""
    import json

    library = _native.load()
    plan = _native.create("rl_plan_create_mixed", cols, rows, k, transa, transb, k if transa else cols,
                          k if transb == 0 else rows, cols, 0, 0, input_dtype, workspace)
    metadata = json.loads(library.rl_plan_tuning_metadata(plan).decode())
    assert library.rl_plan_destroy(plan) == 0
    return metadata["kernel"]


@pytest.mark.parametrize("rows,cols,k,input_dtype,kernel", [
    (2048, 101, 512, 3, "mfma_64x64"),        # a head
    (4096, 512, 39, 3, "mfma_64x64"),         # an embedder
    (1, 1, 1, 3, "mfma_64x64"),
    (16384, 4096, 1024, 3, "mfma_256x256"),   # a block layer
    (16384, 4000, 1000, 3, "mfma_256x128"),   # the same, ragged
    (16384, 4000, 1000, 2, "mfma_256x128"),   # fp32 operands rounded on load
    (2048, 101, 512, 2, "mfma_256x128"),
    (2048, 101, 512, 1, "mfma_256x128"),      # fp16
    (64, 64, 64, 0, "mfma_64x64"),
    (16384, 4096, 1024, 0, "mfma_128x128"),
])
def test_dense_plan_metadata_names_the_kernel(rows, cols, k, input_dtype, kernel):
    assert plan_kernel(rows, cols, k, input_dtype) == kernel


# either side of the line in rows, K, rounds of large tiles and 16-byte rows of operands and output; (500, 16000, 1000) takes 64 us
# on the 256 x 128 tiles and 100 us on the 64 x 64 ones as a twin product
@pytest.mark.parametrize("rows,cols,k,transa,transb,kernel", [
    (500, 16000, 1000, 1, 0, "mfma_256x128"),
    (300, 16000, 1000, 1, 0, "mfma_64x64"),
    (500, 16000, 1001, 1, 0, "mfma_64x64"),
    (500, 16000, 16000, 1, 0, "mfma_256x128"),
    (16400, 400, 8200, 1, 0, "mfma_256x128"),
    (16400, 504, 8200, 0, 0, "mfma_256x128"),
    (16401, 400, 8200, 0, 1, "mfma_64x64"),
    (3000, 3000, 3000, 1, 0, "mfma_256x128"),
    (3000, 3000, 40, 1, 0, "mfma_64x64"),
    (16400, 16400, 264, 0, 1, "mfma_256x128"),
    (24, 16000, 1000, 1, 0, "mfma_64x64"),
    (65536, 101, 1024, 1, 0, "mfma_64x64"),
    (65536, 104, 1024, 1, 0, "mfma_256x128"),
])
def test_bf16_products_take_the_faster_tiles(rows, cols, k, transa, transb, kernel):
    assert plan_kernel(rows, cols, k, 3, transa, transb) == kernel
