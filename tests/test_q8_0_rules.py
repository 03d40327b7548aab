"""The rules that choose a tile of the int8 GEMM by sizes (csrc/dsx_q8_0_rules.hpp) against what was measured: token
counts on either side of each line.  The tiles have the same bits, so outputs do not tell them apart; the program is
built by __graft_entry__.build() (make -C tests/cpp)."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_build", "q8_rules")
CUS = 256


def ask(lines):
    if not os.path.exists(BIN):
        pytest.fail(f"{BIN} is not built: run `python __graft_entry__.py`")
    text = "\n".join(" ".join(map(str, line)) for line in lines)
    res = subprocess.run([BIN], input=text, stdout=subprocess.PIPE, text=True, timeout=20, check=True)
    return [int(v) for v in res.stdout.split()]


@pytest.mark.parametrize("shape,columns", [
    # (hidden, inter, experts, top): {tokens: columns per work item}
    ((7168, 2048, 256, 8), {64: 32, 256: 32, 384: 64, 512: 64, 768: 64, 1000: 64, 1700: 64, 2100: 128}),
    ((5120, 1536, 160, 6), {192: 32, 512: 64, 768: 64}),
    ((3072, 2048, 64, 4), {64: 32, 256: 32, 384: 64, 512: 64}),
    ((4096, 1536, 128, 8), {128: 32, 384: 64, 512: 64}),
    ((2048, 1408, 64, 6), {48: 32, 192: 32, 300: 64, 420: 64, 512: 128, 700: 128}),
    ((2048, 768, 128, 8), {256: 32, 384: 32, 512: 64}),
    ((4096, 14336, 8, 2), {16: 32, 128: 32, 192: 128}),
    ((512, 4096, 32, 4), {192: 32}),
    ((512, 2048, 64, 4), {384: 32, 512: 64, 640: 64}),
    ((1024, 2048, 32, 4), {192: 32, 256: 64})])
def test_columns_of_the_int8_gemm(shape, columns):
    assert dict(zip(columns, ask([("gemm", *shape, T, CUS) for T in columns]))) == columns


@pytest.mark.parametrize("shape,columns", [
    ((7168, 2048, 256, 8), {256: 32, 512: 64, 1000: 64, 1900: 64, 2000: 128}),
    ((2048, 1408, 64, 6), {200: 32, 300: 64, 512: 64, 600: 64, 700: 128}),
    ((4096, 14336, 8, 2), {128: 32, 192: 64, 300: 128})])
def test_gate_up_columns_of_the_int8_gemm(shape, columns):
    assert dict(zip(columns, ask([("gate_up", *shape, T, CUS) for T in columns]))) == columns


@pytest.mark.parametrize("middle,wide,row_tiles,takes", [
    (143, 72, 24, 1), (75, 40, 32, 1), (72, 36, 12, 1),   # 900 tokens on 32 of 128 experts; all on the same picks
    (56, 28, 22, 0), (45, 27, 24, 0),                     # the wide items make as many or two thirds of the rounds
    (144, 130, 24, 0), (90, 66, 22, 0),                   # spread, skewed picks
    (7, 5, 128, 0), (14, 10, 256, 0)])
def test_wide_items_of_gate_up(middle, wide, row_tiles, takes):
    assert ask([("wide", middle, wide, row_tiles, 2 * CUS, 0, 0)]) == [takes]


@pytest.mark.parametrize("shape,columns", [
    ((7168, 2048), {96: 32, 768: 32, 1000: 128, 1900: 128, 2000: 128}),
    ((7168, 3072), {512: 32, 640: 32, 1000: 128}),
    ((5120, 1536), {1500: 32, 1900: 128}),
    ((2048, 1408), {96: 32, 1900: 32, 4096: 128}),
    ((7168, 512), {3000: 32, 4096: 128}),
    ((7168, 18432), {96: 32, 128: 32, 512: 128}),
    ((128, 128), {65535: 128}), ((65536, 128), {129: 32, 65535: 128})])   # (no overflow at the ends of the range)
def test_columns_of_a_dense_expert(shape, columns):
    assert dict(zip(columns, ask([("dense", *shape, 0, 0, b, CUS) for b in columns]))) == columns
