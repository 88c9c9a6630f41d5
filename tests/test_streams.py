"""The library's streams do not wait for the null stream, so nothing in it is
queued there: what a null-stream copy or fill wrote would reach their kernels
in no given order."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "detectingscc_amd", "csrc")
NULL_STREAM = re.compile(r"\bhip(Memcpy|Memcpy2D|Memset|MemsetD\d+|MemcpyHtoD|MemcpyDtoH|MemcpyDtoD|MemcpyTo\w+|MemcpyFrom\w+)\s*\(")
LAUNCH = re.compile(r"<<<(.*?)>>>", re.S)


def _arguments(text):
    """Number of top-level arguments of a launch configuration."""
    depth, n = 0, 1
    for c in text:
        depth += c in "([{"
        depth -= c in ")]}"
        n += c == "," and depth == 0
    return n


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.hip"))), ids=os.path.basename)
def test_nothing_on_the_null_stream(path):
    code = re.sub(r"//[^\n]*|/\*.*?\*/", "", open(path).read(), flags=re.S)
    assert not NULL_STREAM.findall(code)
    assert all(_arguments(m) == 4 for m in LAUNCH.findall(code))
