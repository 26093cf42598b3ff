"""Which responses a kernel may write to host memory: only columns that lie whole in one pinned allocation. A
column whose two ends are pinned but whose middle is not goes by the runtime's copies (CPU: the decision alone,
over a made-up address space)."""
from __future__ import annotations

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# pinned: [1000, 2000), [3000, 4000), [4000, 4500)
TABLES = [
    ("no column", [], True),
    ("first byte", [(1000, 1)], True),
    ("whole allocation", [(1000, 1000)], True),
    ("last byte", [(1999, 1)], True),
    ("one past the end", [(1999, 2)], False),
    ("one before the start", [(999, 2)], False),
    ("ordinary memory", [(2500, 10)], False),
    ("ordinary memory between two pinned ends", [(1500, 2000)], False),
    ("the same, ends at the edges", [(1999, 1002)], False),
    ("two allocations side by side", [(3500, 700)], False),
    ("columns of several allocations", [(1000, 8), (3000, 1000), (1992, 8), (4499, 1)], True),
    ("second column across the gap", [(1000, 8), (1008, 2500)], False),
    ("last column ordinary", [(1000, 8), (3000, 8), (2000, 1)], False),
]


@pytest.fixture(scope="module")
def answers(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("pinned") / "pinned_columns")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", os.path.join(ROOT, "spearhed_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "pinned_columns.cpp"), "-o", exe], check=True)
    args = []
    for i, (_, cols, _) in enumerate(TABLES):
        args += (["/"] if i else []) + [str(x) for c in cols for x in c]
    out = subprocess.run([exe, *args], capture_output=True, text=True, timeout=60, check=True).stdout.split()
    assert len(out) == len(TABLES)
    return [x == "1" for x in out]


@pytest.mark.parametrize("i", range(len(TABLES)), ids=[t[0] for t in TABLES])
def test_columns_pinned(answers, i):
    assert answers[i] == TABLES[i][2]
