"""The whole-number rules of csrc/nc_rules.h, compiled on the host (no GPU)."""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "nanocompile_amd" / "csrc"


@pytest.fixture
def run(tmp_path):
    """Compile and run a program over the rules; its output."""
    def go(body: str) -> str:
        source, binary = tmp_path / "rules.cpp", tmp_path / "rules"
        source.write_text('#include <initializer_list>\n#include <stdio.h>\n#include "nc_rules.h"\nint main() {\n' + body + "\nreturn 0;\n}\n")
        cxx = shutil.which("g++") or "c++"
        subprocess.run([cxx, "-O1", "-std=c++17", f"-I{CSRC}", "-o", str(binary), str(source)],
                       check=True)
        return subprocess.run([str(binary)], check=True, capture_output=True, text=True).stdout
    return go


def test_a_head_prefetch_stays_in_its_block(run):
    """Every piece the multi-row head asks for (its first ring, each refill of a stage of 16, the pieces
    past the last stage), at every width it takes: the piece itself inside the block, one of the block past it."""
    assert run("""
    long bad = 0;
    for (int pieces = 1; pieces <= 4096; ++pieces)
        for (int ring : {8, 16}) {
            auto ask = [&](int at) {
                const int got = nc::head_piece(at, pieces);
                bad += got < 0 || got >= pieces || (at < pieces && got != at);
            };
            for (int i = 0; i < ring; ++i) ask(i);
            int k4 = 0;
            for (; k4 + 16 <= pieces; k4 += 16)
                for (int j = 0; j < 16; ++j) ask(k4 + j + ring);
            for (; k4 < pieces; ++k4) ask(k4);
        }
    printf("%ld", bad);
    """) == "0"
