"""The audit of the hand-counted waits (isa_audit.py) on the compiler's listing of a few grouped-GEMM kernels, and that it finds what it is for:
mistakes planted in the listing's text."""

import os
import shutil

import pytest

import isa_audit
from build import HIPCC

pytestmark = pytest.mark.skipif(shutil.which(HIPCC) is None, reason="needs hipcc")

# kinds of ragged_gemm_kernel: element type, layouts, epilogue, reduction varies, bias, gather, tall
KINDS = ["ElemBf16, true, true, EPI_SWIGLU, false, false, true, true", "ElemBf16, true, false, EPI_SWIGLU_BWD, false, false, false, true",
         "ElemF16, true, true, EPI_PLAIN, false, true, false, false", "ElemBf16, false, false, EPI_PLAIN, true, false, true, false"]  # fmt: skip


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    folder = tmp_path_factory.mktemp("isa")
    source, path = str(folder / "kinds.hip"), str(folder / "kinds.s")
    with open(source, "w") as f:
        f.write('#include "ragged_kernel.h"\nnamespace fmahip::gemm::ragged {\n')
        for kind in KINDS:
            f.write(f"template __global__ void ragged_gemm_kernel<{kind}>(const Args);\n")
        f.write("}\n")
    isa_audit.compile_to_assembly(source, path)
    return path


def test_lds_reads_have_returned_at_barriers(listing):
    assert isa_audit.audit_barriers(listing) == 0


def test_general_kernels_lds_reads_have_returned_at_barriers(tmp_path):
    path = str(tmp_path / "general.s")
    isa_audit.compile_to_assembly(os.path.join(isa_audit.CSRC, "grouped_gemm.hip"), path)
    assert isa_audit.audit_barriers(path) == 0
