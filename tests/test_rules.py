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
        source.write_text('#include <initializer_list>\n#include <stdio.h>\n#include "nc_rules.h"\n'
                          "int main() {\n" + body + "\nreturn 0;\n}\n")
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


def test_head_tiles_fit_one_dimension_of_the_grid(run):
    """Rows a wave of the multi-row head, and 0 (the one-row kernels) where its workgroups of 256 threads
    would be 2^32 threads or more along the grid's first dimension."""
    shapes = [(1, 151936, 896, 0), (2, 151936, 896, 4), (4, 151936, 896, 4), (128, 151936, 896, 16),
              (65535, (1 << 20) - 256, 4, 16), (65535, 1 << 20, 4, 0), (65535, (1 << 28) + 256, 4, 0),
              (65535, (1 << 31) - 1, 4, 0), (4, (1 << 31) - 1, 4, 4)]
    said = run("".join(f'printf("%d ", nc::head_tile({m}, {v}ll, {h}));' for m, v, h, _ in shapes)).split()
    assert [int(t) for t in said] == [t for *_, t in shapes]


def test_head_rows_where_they_are_quicker(run):
    """The one-row kernels where they measured quicker than four rows a wave, four rows where those did."""
    one_row = [(64, 1024, 1024), (500, 128, 1024), (100, 896, 896), (56, 1152, 896), (2, 32768, 128), (500, 128, 128),
               (1000, 64, 64), (4000, 64, 896), (175, 512, 256), (32, 2048, 512), (8, 8192, 896), (10, 6400, 896),
               (42, 3072, 896), (125, 1024, 2048), (125, 512, 4096), (71, 1536, 1536)]
    four = [(2, 32000, 896), (3, 24000, 4096), (8, 8192, 1024), (128, 512, 8192), (400, 896, 896), (17, 8192, 896),
            (72, 896, 4864), (350, 512, 512), (88, 2048, 896), (16, 4864, 896), (32, 8192, 64), (10, 6400, 512),
            (22, 3000, 1536), (175, 512, 4096), (1000, 512, 64), (2000, 64, 4096)]
    said = run("".join(f'printf("%d ", nc::head_tile({m}, {v}, {h}));' for m, v, h in one_row + four)).split()
    wrong = [(s, t) for s, t in zip(one_row + four, said) if int(t) != (0 if s in one_row else 4)]
    assert not wrong


def test_vnni_tiles_fit_one_dimension_of_the_grid(run):
    """Weight rows a lane of matmul_i8_vnni's register tiles, 0 (a chain a lane) where they do not fit."""
    shapes = [(4, 896, 4864, 0), (17, 896, 896, 0), (18, 896, 896, 2), (128, 4864, 896, 4), (65535, 65504, 32, 4),
              (65535, 65536, 32, 0), (65535, 65537, 32, 0), (65535, (1 << 24) - 1, 32, 0),
              (256, (1 << 24) - 32, 32, 4), (257, (1 << 24) - 1, 32, 0)]
    said = run("".join(f'printf("%d ", nc::dp4_columns({m}, {n}ll, {k}));' for m, n, k, _ in shapes)).split()
    assert [int(c) for c in said] == [c for *_, c in shapes]


def test_vnni_tiles_where_they_are_quicker(run):
    """A chain a lane where that measured quicker than the register tiles, the tiles where they did."""
    chains = [(1, 16000, 896), (1, 32000, 896), (1, 151936, 64), (1, 65536, 2048), (1, 151936, 4864), (1, 24000, 4096),
              (1, 16000, 4864), (1, 32768, 8192), (1, 151936, 8192), (2, 65536, 256), (2, 16000, 128)]
    tiles = [(1, 16384, 4096), (1, 16000, 8192), (1, 32768, 16384), (2, 16000, 512), (2, 8192, 8192), (2, 151936, 896),
             (3, 16000, 256), (3, 65536, 896), (4, 4864, 896), (500, 64, 128)]
    said = run("".join(f'printf("%d ", nc::dp4_columns({m}, {n}, {k}));' for m, n, k in chains + tiles)).split()
    assert [s for s, c in zip(chains + tiles, said) if (int(c) > 0) != (s in tiles)] == []


def test_int8_tiles_fit_one_dimension_of_the_grid(run):
    """Tiles a workgroup of matmul_i8 on the matrix cores, 0 (the kernels of a grid row a row) where they do not fit."""
    shapes = [(16, 896, 4864, 0), (24, 896, 4864, 1), (128, 4864, 896, 2), (128, 896, 4864, 1), (20, 70, 24, 0),
              (20, 70, 100, 0), (65535, 131040, 32, 2), (65535, 131072, 32, 0), (65535, (1 << 24) - 1, 32, 0),
              (512, (1 << 24) - 33, 40, 2), (512, (1 << 24) - 1, 40, 0)]
    said = run("".join(f'printf("%d ", nc::chain_tiles({m}, {n}ll, {k}));' for m, n, k, _ in shapes)).split()
    assert [int(t) for t in said] == [t for *_, t in shapes]


def test_int8_on_the_matrix_cores_where_it_is_quicker(run):
    """The kernels of a grid row a row of x where they measured quicker, the matrix cores where those did."""
    rows = [(1, 20000, 896), (1, 151936, 896), (2, 10000, 896), (3, 6667, 896), (4, 5000, 896), (1, 65536, 4864),
            (2, 13000, 4864), (1, 65536, 64), (2, 151936, 128), (64, 64, 256), (16, 1024, 128), (1, 16384, 512),
            (2, 8192, 1000), (1, 32768, 1024), (1, 48000, 1536), (1, 65536, 2048)]
    cores = [(3, 20000, 896), (4, 7500, 896), (22, 1000, 896), (3, 7000, 4864), (2, 65536, 4864), (8, 65536, 896),
             (512, 64, 128), (4, 16384, 512), (256, 256, 96), (8, 4096, 256), (1, 4096, 1024), (3, 10923, 1000),
             (2, 65536, 1024), (1, 8192, 2048), (1, 16384, 4096), (1, 65536, 8192), (2, 16384, 1536)]
    said = run("".join(f'printf("%d ", nc::chain_tiles({m}, {n}, {k}));' for m, n, k in rows + cores)).split()
    assert [s for s, t in zip(rows + cores, said) if (int(t) > 0) != (s in cores)] == []


def test_pair_tiles_where_they_are_quicker(run):
    """The SwiGLU pair's tile at shapes of long k loops where each of 32 x 32, 64 x 64 and 128 x 64 measured quickest."""
    quickest = {2: [(32, 16500, 2048), (16, 20000, 2048), (64, 16500, 2048), (60, 20000, 2048), (64, 20000, 4096),
                    (200, 3300, 2048), (128, 4864, 896)],
                5: [(64, 13000, 2048), (100, 8000, 2048), (64, 26000, 2048), (257, 6400, 2048), (700, 3000, 3072),
                    (400, 4864, 2560), (300, 8192, 4096), (130, 16384, 2048), (1000, 4864, 2048), (512, 4864, 896)],
                8: [(190, 8000, 4096), (130, 8192, 4096), (100, 12800, 2048), (512, 3000, 2048), (260, 4096, 4096),
                    (384, 4096, 4096), (500, 8192, 2048), (2000, 2000, 4096)]}
    shapes = [(t, s) for t in quickest for s in quickest[t]]
    said = run("".join(f'printf("%d ", nc::pair_tile({m}, {n}, {k}));' for _, (m, n, k) in shapes)).split()
    assert [(s, int(got)) for (t, s), got in zip(shapes, said) if int(got) != t] == []


def test_prompt_attention_where_the_matrix_cores_are_quicker(run):
    """Rows a workgroup of a prompt's attention: 4 (the vector ALU) where that measured quicker, else 0."""
    vector = [(2, 8, 8, 2), (64, 8, 8, 64), (64, 8, 8, 464), (128, 4, 4, 528), (64, 16, 8, 164),
              (128, 12, 4, 128), (64, 8, 2, 464), (128, 3, 3, 528), (8, 8, 8, 4008), (2, 66, 1, 2), (5000, 130, 2, 9000)]
    matrix = [(64, 8, 8, 1264), (64, 4, 4, 1264), (128, 16, 8, 228), (256, 12, 4, 256), (128, 8, 2, 528),
              (512, 3, 3, 512), (2, 14, 2, 2), (64, 24, 4, 64), (3, 64, 1, 133), (2048, 8, 8, 2048)]
    said = run("".join(f'printf("%d ", nc::prefill_rows({m}, {h}, {kv}, {keys}));'
                       for m, h, kv, keys in vector + matrix)).split()
    assert [s for s, r in zip(vector + matrix, said) if int(r) != (4 if s in vector else 0)] == []
