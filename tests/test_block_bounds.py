"""Grids of more than 32,768 blocks are padded to whole rows of 32,768
(grid_blocks in csrc/common.h), so a kernel that addresses an array by its
block number has blocks beyond the array's end.  Read from the sources: such a
kernel returns before it touches the array."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pennsylvaniagpugraphclustering_amd",
                    "csrc")


def kernels():
    """(file, kernel, body) of every kernel in the sources, comments removed."""
    for path in sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h"))):
        with open(path) as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        for m in re.finditer(r"__global__[^;{]*?\b(k_\w+)\s*\(", text):
            start = pos = text.index("{", m.end())
            depth = 0
            while True:
                depth += {"{": 1, "}": -1}.get(text[pos], 0)
                if depth == 0:
                    break
                pos += 1
            yield os.path.basename(path), m.group(1), text[start:pos + 1]


INDEXED = [k for k in kernels() if "[block_id()]" in k[2]]


def test_kernels_found():
    assert len(list(kernels())) > 100
    assert {"k_uniq_sums", "k_uniq_write", "k_gnn_count"} <= {k[1] for k in INDEXED}


@pytest.mark.parametrize("kernel", INDEXED, ids=[k[1] for k in INDEXED])
def test_surplus_blocks_return_first(kernel):
    body = kernel[2]
    before = body[:body.index("[block_id()]")]
    base = re.search(r"const i64 (\w+) = block_id\(\)", before)
    names = ["block_id()"] + ([base.group(1)] if base else [])
    assert any(re.search(r"if \(%s[^;{]*>=[^;{]*\) return;" % re.escape(n), before) for n in names), kernel[:2]
