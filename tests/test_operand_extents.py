"""How far a kernel's requests may reach: the buffer descriptors over operands whose rows lie further apart than they are long."""
from __future__ import annotations

import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm_amd", "csrc")


@pytest.mark.parametrize("source", ["fp8_scaled_mm.hip", "fp8_stream2_kernel.h", "fp8_quant_mm.hip"])
def test_descriptors_end_with_the_last_row(source):
    """Rows times pitch passes the end of a view of trailing columns (its last row ends with the storage), and the FP8 tile kernels request
    whole cache lines, the last of which may lie past K: a descriptor over such an operand ends (rows - 1) * pitch + K behind its start."""
    with open(os.path.join(CSRC, source)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    spans = re.findall(r"make_buffer_rsrc\(([^;]*)\);", text)
    assert spans or source == "fp8_quant_mm.hip"
    assert not [s for s in spans if re.search(r"p\.(lda|ldb)", s)]
    if source != "fp8_stream2_kernel.h":
        extents = re.findall(r"p\.([ab])_extent = ([^;]*);", text)
        assert extents
        for operand, value in extents:
            rows = "M" if operand == "a" else "N"
            assert f"(p.{rows} - 1) * p.ld{operand} + p.K" in value, value


@pytest.mark.parametrize("source", ["w4a16_strip_kernel.h", "w4a16_prefill_kernel.h"])
def test_descriptors_of_the_w4a16_tile_kernels_end_with_the_last_row(source):
    """The same of their activations.  Their 32-bit offsets wrap for rows past M where the activations end close to 4 GiB: what such
    a request finds then is at least the call's own."""
    with open(os.path.join(CSRC, source)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    spans = [s for s in re.findall(r"make_buffer_rsrc\(([^;]*)\);", text) if "p.a)" in s]
    assert len(spans) == 1
    extent = re.search(r"a_bytes = ([^;]*);", text).group(1) if "a_bytes" in spans[0] else spans[0]
    assert "(uint32_t)(p.M - 1) * (uint32_t)p.lda + (uint32_t)p.K) * 2u" in extent


def test_waits_of_the_fp8_kernel_for_some_dozen_rows_count_on_loads_that_cannot_be_merged():
    """What a wait counts on has to be there whatever the compiler makes of it: requests into LDS are, and of the scales the two loads for each of R results whose
    offsets the compiler cannot see behind the requests for activations."""
    with open(os.path.join(CSRC, "fp8_regs_kernel.h")) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    waits = re.findall(r's_waitcnt vmcnt\((%0|\d+)\)"\s*::\s*(?:"n"\(([^"]*)\)\s*:)?', text)
    assert len(waits) >= 4 and all(counted == "0" or what.strip() in ("J * LI", "2 * R") for counted, what in waits), waits
    loop = text[text.index("load_act(g);"):text.index("vmcnt(%0)\" ::\"n\"(2 * R)")]
    hidden = re.search(r'asm volatile\("" : ([^;]*)::"memory"\);', loop)
    assert hidden and all(f'"+v"(at[{i}])' in hidden.group(1) for i in range(3))
    loads = re.findall(r"raw_buffer_load_b\d+\((\w+), ([^,]*),", loop[hidden.end():])
    assert loads == [("rsa", "at[0]"), ("rsb", "at[1]"), ("rbias", "at[2]")]


@pytest.mark.parametrize("source,requests", [("fp8_scaled_mm.hip", 4), ("fp8_stream2_kernel.h", 1), ("fp8_regs_kernel.h", 2), ("w4a16_prefill_kernel.h", 2), ("w4a16_strip_kernel.h", 1)])
def test_scalar_offsets_of_requests_into_lds_stay_in_the_operand(source, requests):
    """A scalar offset past the extent leaves a negative rest to check against: a request's rows are clamped to those that are there where they stand in the
    scalar offset, and a request for nothing has scalar offset 0 or the extent."""
    with open(os.path.join(CSRC, source)) as f:
        text = re.sub(r"//[^\n]*", "", f.read())
    calls = [c.split("16, ", 1)[1] for c in re.findall(r"raw_ptr_buffer_load_lds\(([^;]*)\);", text)]
    assert len(calls) == requests
    by_row = [c for c in calls if re.search(r"lda|ldb|pitch", c)]
    assert all("min(" in c for c in by_row), by_row
    named = {"fp8_stream2_kernel.h": ["auto rows_of = [&](int nt) { return (uint32_t)(max(min(nt, nt1 - 1), 0) * 16)", "k_at[st] = (uint32_t)min(kw + st * 256, p.K)"],
             "fp8_regs_kernel.h": ["const int so = g < steps ? (int)((uint32_t)(min(nt0 + j, NT - 1) * 16)", "g < steps ? g * KT : 0"],
             "w4a16_strip_kernel.h": ["const uint32_t so = g < g_hi ? (uint32_t)g * 256u + (uint32_t)(h & 1) * 128u : a_bytes;"]}
    assert all(line in text for line in named.get(source, []))
