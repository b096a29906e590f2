"""The audit of the hand-counted waits (isa_audit.py) on the compiler's listing of a few grouped-GEMM kernels, and that it finds what it is for:
mistakes planted in the listing's text."""

import os
import re
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


KERNEL = r"_ZN6fmahip4gemm6ragged18ragged_gemm_kernel"


def test_shapes(listing):
    assert len(list(isa_audit.kernels(listing, KERNEL))) == len(KINDS)
    assert isa_audit.audit(listing) == 0


def _lines(body, what):
    """indices of the lines that `what` holds for, at most a dozen, spread over the kernel"""
    found = [i for i, line in enumerate(body) if what(i, line.strip())]
    return found[:: max(1, len(found) // 12)]


@pytest.mark.parametrize("kind", range(len(KINDS)))
def test_finds_wrong_counts(listing, kind):
    """one wait in front of a barrier that allows for one load more, one operand load missing, one twice: each is found, wherever it is"""
    name, body = sorted(isa_audit.kernels(listing, KERNEL))[kind]

    def before_barrier(i, s):
        return s.startswith("s_waitcnt vmcnt") and body[i + 1].strip().startswith("s_barrier")

    waits = _lines(body, before_barrier)
    loads = _lines(body, lambda i, s: s.startswith("buffer_load_dwordx4") and " lds" in s)
    assert len(waits) >= 12 and len(loads) >= 12
    assert not isa_audit.audit_kernel(name, body)
    for i in waits:
        more = re.sub(r"vmcnt\((\d+)\)", lambda m: f"vmcnt({int(m.group(1)) + 1})", body[i])
        assert isa_audit.audit_kernel(name, body[:i] + [more] + body[i + 1 :]), f"line {i}: {more}"
    for i in loads:
        assert isa_audit.audit_kernel(name, body[:i] + body[i + 1 :]), f"line {i} missing"
        assert isa_audit.audit_kernel(name, body[:i] + [body[i]] + body[i:]), f"line {i} twice"


def test_finds_reads_in_flight(listing):
    """a wait in front of a barrier that leaves out the LDS reads is found where reads precede it"""
    found = 0
    for name, body in isa_audit.kernels(listing, KERNEL):
        body = [line.strip() for line in body]
        both = [i for i, s in enumerate(body) if "lgkmcnt(0)" in s and body[i + 1].startswith("s_barrier")]
        for i in both[:: max(1, len(both) // 12)]:
            reads = next(j for j in range(i - 1, -1, -1) if body[j].startswith(("ds_", "s_waitcnt lgkmcnt", "s_barrier", ".LBB")))
            if body[reads].startswith("ds_"):
                found += 1
                s = body[i].replace("lgkmcnt(0)", "")
                assert isa_audit.reads_out_at_barriers(body[:i] + [s] + body[i + 1 :]), f"{name}: line {i}"
    assert found >= 8
