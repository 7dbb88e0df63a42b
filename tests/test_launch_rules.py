"""The host rules that choose kernel forms, tiles and launch pieces (furiosa-opt_amd/csrc/launch_rules.hpp),
built with g++ and asked through tests/host_rules/rules.cpp. No GPU."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def ask(tmp_path_factory):
    exe = tmp_path_factory.mktemp("rules") / "rules"
    res = subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{ROOT / 'furiosa-opt_amd' / 'csrc'}",
                          str(ROOT / "tests" / "host_rules" / "rules.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]

    def run(questions):
        out = subprocess.run([str(exe)], input="\n".join(questions) + "\n", capture_output=True, text=True, timeout=60)
        assert out.returncode == 0
        return [line.strip() for line in out.stdout.splitlines()]
    return run


# rows, threads a row: around the first piece's end, and the shapes that one launch could not take (512
# columns from 2^26 rows, 2048 from 2^24, 4096 x 64 threads)
@pytest.mark.parametrize("rows, threads", [(1, 64), (2 ** 25 - 1, 64), (2 ** 25, 64), (2 ** 25 + 1, 64), (2 ** 26, 64),
                                           (2 ** 26 + 5, 64), (2 ** 31 + 3, 64), (2 ** 24 + 1, 256), (2 ** 23, 512),
                                           (2 ** 22 + 7, 1024), (155648, 16), (2 ** 31 - 1, 16)])
def test_row_pieces_cover_the_rows_and_fit_a_launch(ask, rows, threads):
    pieces = [tuple(map(int, p.split("+"))) for p in ask([f"pieces {rows} {threads}"])[0].split()]
    at = 0
    for first, count in pieces:
        assert first == at and count > 0
        assert -(-count // 16) * 16 * threads < 2 ** 32  # whole blocks of up to 16 rows
        assert first % 64 == 0  # no block straddles two pieces
        at += count
    assert at == rows


# heads, keys, causal -> form: both sides of each line, with the shapes whose second round of workgroups was
# slower than the 256-query form (100 x 300, 20 x 2000 and 32 x 1200 without a mask)
@pytest.mark.parametrize("heads, seq, causal, form", [
    (1, 65, 1, "2x4"), (16, 1024, 1, "2x4"), (16, 1024, 0, "2x4"), (256, 64, 1, "4x2"), (16, 1025, 1, "4x2"),
    (32, 1024, 0, "4x2"), (33, 1024, 0, "256"), (33, 1000, 1, "4x2"), (64, 600, 0, "256"), (64, 600, 1, "4x2"),
    (65, 600, 1, "256"), (100, 300, 0, "256"), (100, 300, 1, "256"), (100, 385, 1, "256"), (80, 385, 1, "4x2"),
    (86, 384, 1, "256"), (32, 1200, 0, "256"), (32, 1200, 1, "4x2"), (32, 2048, 1, "4x2"), (32, 2048, 0, "256"),
    (33, 2048, 1, "256"), (20, 2000, 0, "256"), (320, 128, 0, "4x2"), (321, 128, 0, "256"), (300, 129, 1, "256"),
    (128, 2048, 1, "256")])
def test_attention_form(ask, heads, seq, causal, form):
    assert ask([f"attention {heads} {seq} {causal}"]) == [form]


# type, batch, m, n, k -> tile (edge; 32: 32x64; 1284: 128x128 with four stages). The shapes of 129 to 143 tiles of 256x256
# whose K is long went to 128x128 once, two rounds of them and a tail; K of few stages to four-stage tiles.
@pytest.mark.parametrize("shape, tile", [
    ("bf16 1 32 4096 4096", 32), ("bf16 1 33 4096 4096", 64), ("bf16 1 500 3072 1024", 64), ("bf16 1 512 4096 4096", 64),
    ("bf16 1 1024 4096 4096", 1284), ("bf16 1 1024 4096 896", 128), ("bf16 1 1024 4096 897", 1284), ("i8 1 900 3500 1536", 128),
    ("i8 1 900 3500 1537", 1284), ("f8 1 900 3500 1152", 128), ("f8 1 900 3500 1153", 1284), ("f8 1 343 5584 384", 128),
    ("bf16 1 583 5384 512", 128), ("bf16 1 583 5384 513", 1284), ("i8 1 640 3300 896", 128), ("i8 1 640 3300 897", 1284),
    ("f8 1 583 5384 896", 128), ("f8 1 583 5384 897", 1284), ("bf16 1 1100 4096 4096", 128), ("bf16 1 2048 4096 4096", 128), ("f8 1 2048 4096 4096", 128),
    ("i8 1 2048 4096 8192", 128), ("bf16 1 1500 5500 1024", 128), ("bf16 1 1500 5500 1025", 256), ("bf16 1 2304 3840 2048", 256),
    ("i8 1 1500 5500 1024", 128), ("i8 1 1500 5500 4096", 256), ("f8 1 1500 5500 512", 128), ("f8 1 1500 5500 2048", 256),
    ("bf16 16 600 600 128", 128), ("bf16 1 2200 3900 1024", 256), ("bf16 1 4096 4096 4096", 256), ("i8 1 2048 8192 8192", 256),
    # a small side keeps its tile past 512 tiles, while a launch can hold them
    ("bf16 1 16 155648 1024", 32), ("bf16 520 16 64 256", 32), ("bf16 1 64 40000 1024", 64), ("i8 1 40000 64 1024", 64),
    ("f8 600 64 64 512", 64), ("bf16 1 65 40000 1024", 128), ("bf16 300 100 100 256", 128), ("i8 1 128 155648 8192", 128),
    ("bf16 1 129 155648 1024", 256), ("bf16 1 8 2147483647 16", 256), ("bf16 1 40 2147483647 16", 256),
    ("bf16 1 40 1073741760 16", 64), ("bf16 1 32 2147483520 16", 32), ("bf16 1 40 2147483520 16", 128), ("bf16 1 129 2147483647 16", 256)])
def test_gemm_tile(ask, shape, tile):
    assert ask([f"gemm {shape}"]) == [str(tile)]


# type, batch, m, n, k -> tile of the contraction off 16-byte rows (0: the vector-unit fold). Batches of small products
# went to 128x128 once, and a K too short for the tiles to them: i8 8 x 8 x 31 4.8 us against 3.7.
@pytest.mark.parametrize("shape, tile", [
    ("bf16 1 333 1000 777", 64), ("bf16 1 1500 2000 71", 128), ("i8 2000 32 32 63", 64), ("bf16 600 64 200 63", 64),
    ("bf16 600 65 70 63", 128), ("bf16 1 16 155648 129", 64), ("i8 1 8 1073741760 63", 64), ("i8 1 8 1073741888 63", 128),
    ("i8 1 8 2147483647 63", 0),
    ("i8 1 8 8 47", 0), ("i8 1 8 8 49", 64), ("bf16 1 8 8 19", 0), ("bf16 1 8 8 21", 64), ("i8 5000 8 8 47", 0),
    ("i8 1 500 500 31", 0), ("i8 1 500 500 33", 64), ("i8 1 700 700 15", 0), ("i8 1 700 700 17", 64), ("i8 1 1000 1000 2", 64),
    ("i8 1 9 3000 31", 0), ("i8 1 8 30000 2", 64), ("i8 1000 16 16 17", 0), ("bf16 1 100 100 7", 0), ("bf16 1 100 100 9", 64),
    ("bf16 1 500 500 2", 64), ("bf16 1 333 1000 7", 64)])
def test_gemm_any_tile(ask, shape, tile):
    assert ask([f"gemm_any {shape}"]) == [str(tile)]


# batch, inputs, hidden, outputs, whether k_mlp_split takes the shape -> form. The lines stood at in_f + hidden <= 128 up to
# 256 rows (100 x 50 and 70 x 200 were slower on k_mlp_rows, all of k_mlp's past 256 rows) and, from 65 units, at
# 256 rows of k_mlp_split (400 x 72, 1024 x 136).
@pytest.mark.parametrize("shape, form", [
    ("64 784 128 10 1", "split"), ("256 784 128 10 1", "split"), ("257 784 128 10 1", "rows"), ("257 248 128 10 1", "split"),
    ("512 400 72 10 1", "split"), ("512 1024 104 10 1", "split"), ("257 256 105 10 1", "rows"), ("512 1024 136 10 1", "split"), ("257 64 88 10 1", "rows"), ("512 64 56 10 1", "split"),
    ("513 64 16 10 1", "rows"), ("513 1024 136 10 1", "rows"),
    ("1 73 23 10 0", "thread"), ("256 100 50 10 0", "thread"), ("1 70 200 10 0", "thread"), ("64 72 201 10 0", "rows"), ("64 30 257 10 0", "rows"),
    ("257 73 23 10 0", "thread"), ("512 95 50 10 0", "thread"), ("512 96 50 10 0", "rows"), ("320 30 90 10 0", "rows"), ("513 105 105 10 0", "thread"),
    ("1024 30 129 10 0", "rows"), ("1025 100 60 10 0", "thread"), ("1025 75 75 10 0", "rows"), ("2048 73 23 10 0", "thread"),
    ("2049 73 23 10 0", "rows"), ("64 784 128 10 0", "rows"),
    ("362 123 17 50 0", "thread"), ("362 123 17 32 0", "rows"), ("257 150 131 50 0", "rows")])
def test_mlp_form(ask, shape, form):
    assert ask([f"mlp {shape}"]) == [form]


# rows, K -> cells a block. Every N past 4096 took 32 once: 16384 x 4096, 32768 and 65536 rows were slower than on 64.
@pytest.mark.parametrize("shape, cells", [
    ("4096 1024", 16), ("4097 1024", 32), ("8192 4096", 32), ("8193 1024", 64), ("16384 4096", 64), ("16385 1024", 32),
    ("24576 3584", 32), ("24576 3592", 64), ("24577 1024", 64), ("32768 200", 64), ("32769 1024", 32), ("45056 2048", 32),
    ("45057 1024", 64), ("65536 200", 64), ("90112 1024", 64), ("155648 1024", 32), ("155648 760", 64)])
def test_gemv_cells(ask, shape, cells):
    assert ask([f"gemv {shape}"]) == [str(cells)]


# rows, columns -> form. The row kernel took every number of rows of 2048 columns, and 4096 rows of 4096, once.
@pytest.mark.parametrize("shape, form", [
    ("8192 4096", "dma"), ("6144 4096", "dma"), ("6143 4096", "row"), ("4097 4096", "row"), ("4096 4096", "dma"),
    ("3840 4096", "row"), ("8192 2048", "dma"), ("8193 2048", "row"), ("7496 2048", "row"), ("7497 2048", "dma"),
    ("4096 2048", "row"), ("20000 2048", "dma"), ("32768 2048", "dma"), ("36864 2048", "row"), ("8192 1024", "row"),
    ("8192 2047", "row")])
def test_norm_form(ask, shape, form):
    assert ask([f"norm {shape}"]) == [form]
