"""Rules that the device sources keep, read off their text."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nntrainer_amd", "csrc")
SOURCES = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")))


@pytest.mark.parametrize("path", [p for p in SOURCES if "__builtin_amdgcn_mfma" in open(p).read()], ids=os.path.basename)
def test_no_assembly_computes_beside_matrix_instructions(path):
    """A matrix instruction writes its results many cycles after it was issued, and the compiler keeps other vector
    instructions away from them; inline assembly it does not look into. Where a file issues matrix instructions, and in what
    it includes from here for them, assembly may wait and order, but names no vector instruction."""
    files = [path]
    text = open(path).read()
    files += [os.path.join(CSRC, x) for x in re.findall(r'#include "(q6k_device\.h|moe_tile_device\.h)"', text)]
    found = []
    for f in files:
        for template in re.findall(r'\basm\s*(?:volatile\s*)?\(\s*((?:"[^"]*"\s*)*)', open(f).read()):
            found += [(os.path.basename(f), x) for x in re.findall(r"\b(?:v|buffer|global|flat|ds)_\w+", template)]
    assert not found


def test_shared_arrival_counters_are_zero_before_the_word_that_ends_a_call():
    """host_done's counters belong to a stream's handle. A call on the same handle may come from another thread's queue, behind
    nothing but the word this call's last workgroup writes (hipStreamPerThread, hipq_stream_release in hipq.h): the counters
    go back to zero in the arrivals themselves, not by stores of which one may be late."""
    text = open(os.path.join(CSRC, "hipq_internal.h")).read()
    body = text[text.index("void host_done("):text.index("constexpr size_t HOST_DONE_BYTES")]
    assert re.findall(r"__hip_atomic_store\(([^,]+),", body) == ["hd.word"]
    assert len(re.findall(r"atomicInc\(hd\.count", body)) == 2 and "fetch_add" not in body


def test_loads_before_a_counted_wait_keep_their_order():
    """f6_sums waits for copies into LDS by the number of loads issued behind them (s_waitcnt vmcnt with a count): each chunk's
    copies are fenced off from the weight loads behind them, and those from the next chunk's copies, in the prologue as in
    the loop."""
    text = open(os.path.join(CSRC, "gemm_f6.hip")).read()
    body = text[text.index("f6_sums(const uint8_t *wbase"):text.index("f6_tile(const uint8_t *wbase")]
    assert re.findall(r"vmcnt\((\d+)\)", body) == ["10", "0", "7", "0"]
    fence = r"__builtin_amdgcn_sched_barrier\(0\);"
    calls = [m.end() for m in re.finditer(r"^ +(?:copy|load_dw)\([^;]*\);", body, re.M)]
    assert len(calls) == 4  # one of each in the prologue and in the loop
    for end in calls:
        assert re.match(r"\s*" + fence, body[end:]), body[end - 40:end + 80]


@pytest.mark.parametrize("path", [p for p in SOURCES if "buffer_store" in open(p).read()], ids=os.path.basename)
def test_buffer_stores_have_their_whole_place_in_the_lane_operand(path):
    """A buffer store that the descriptor's size is to drop is dropped by the lane's operand; the scalar offset beside it is
    documented as left out of that check, and stays zero."""
    calls = re.findall(r"__builtin_amdgcn_raw_(?:ptr_)?buffer_store_\w+\((.*)\);", open(path).read())
    assert calls
    for args in calls:
        assert re.search(r", 0, 0$", args), args
