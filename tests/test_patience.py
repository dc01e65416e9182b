"""The bounded wait of the resident CG engine (pp_patience.hpp), compiled for the host: all words of an exchange
share one budget of polls, and none are made once another workgroup has given up."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "phipict_amd" / "csrc"
SOURCE = r"""
#include "pp_patience.hpp"
#include <cstdio>
using namespace pp;
int main() {
    unsigned ended = 0;
    // 28 words that never come: as many polls as the budget, not 28 times as many
    Patience w{100000, &ended, 7u};
    long polls = 0;
    for (int word = 0; word < 28; ++word)
        while (w.more()) ++polls;
    std::printf("%ld\n", polls);
    // a workgroup gives up after 5000 polls: soon over
    Patience v{100000, &ended, 7u};
    polls = 0;
    for (int word = 0; word < 28; ++word)
        while (v.more())
            if (++polls == 5000) ended = 7u;
    std::printf("%ld\n", polls);
    // no budget, no poll
    ended = 0;
    Patience z{0, &ended, 7u};
    std::printf("%d\n", int(z.more()));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_one_budget_per_exchange(tmp_path):
    (tmp_path / "wait.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", str(tmp_path / "wait.cpp"), "-o", str(tmp_path / "wait")],
                   check=True)
    out = subprocess.run([str(tmp_path / "wait")], check=True, capture_output=True, text=True).stdout.split()
    spent, after, none = (int(v) for v in out)
    assert spent == 100000
    assert 5000 <= after <= 5000 + 1024 + 1
    assert none == 0
