"""Addresses of the 32 x 32 MFMA kernel's activation copies, on the CPU: csrc/iq3s_wide_copies.h,
which the kernel copies with, built by the host compiler. Every lane of every copy of every tile
shape stays inside the rows that the tile has, the last tile's missing rows included, and the copies
of the rows that there are cover each byte once."""

from __future__ import annotations

import shutil
import subprocess

import pytest

from conftest import REPO

CSRC = REPO / "mambo_amd" / "csrc"

PROGRAM = r"""
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include "iq3s_wide_copies.h"

static void fail(const char *what, int rows, int waves, int last, int j, int lane)
{
    printf("%s: rows %d waves %d last row %d copy %d lane %d\n", what, rows, waves, last, j, lane);
    exit(1);
}

// A tile of `rows` rows by `waves` waves whose last row is `last`, K blocks of 256 in rows of ld bytes
static void check(int rows, int waves, int last, int blocks, uint64_t ldxv, uint64_t ldxs)
{
    const uint64_t end = last * ldxv + 256u * blocks, send = last * ldxs + 8u * blocks;
    const int b = blocks - 1; // the copies' scalar offset of the last block
    static unsigned char seen[128][16], scales[128][2];
    memset(seen, 0, sizeof seen);
    memset(scales, 0, sizeof scales);
    for (int wave = 0; wave < waves; ++wave)
        for (int lane = 0; lane < 64; ++lane) {
            for (int j = 0; j < rows / 4 / waves; ++j) {
                const uint64_t o = wide_value_offset(wave, lane, waves, j, last, (uint32_t)ldxv) + 256ull * b;
                if (o + 16 > end || o % 16)
                    fail("values past the end", rows, waves, last, j, lane);
                const int row = 4 * (wave + waves * j) + lane / 16, want = row < last ? row : last;
                if (o - 256ull * b < want * ldxv || o - 256ull * b + 16 > want * ldxv + 256)
                    fail("values of another row", rows, waves, last, j, lane);
                if (row <= last)
                    ++seen[row][(o - 256ull * b - row * ldxv) / 16];
                if (row <= last && (int)((o - 256ull * b - row * ldxv) / 16) != (lane % 16 ^ row % 16))
                    fail("chunk in another slot", rows, waves, last, j, lane);
            }
            if (wave < rows / 32) {
                const uint64_t o = wide_scale_offset(wave, lane, last, (uint32_t)ldxs) + 8ull * b;
                if (o + 4 > send || o % 4)
                    fail("scales past the end", rows, waves, last, wave, lane);
                const int row = 32 * wave + lane / 2;
                if (row <= last)
                    ++scales[row][(o - 8ull * b - row * ldxs) / 4];
            }
        }
    for (int r = 0; r <= last; ++r) {
        for (int c = 0; c < 16; ++c)
            if (seen[r][c] != 1)
                fail("values not copied once", rows, waves, last, r, c);
        if (scales[r][0] != 1 || scales[r][1] != 1)
            fail("scales not copied once", rows, waves, last, r, 0);
    }
}

int main()
{
    static const int shapes[][2] = {{64, 2}, {64, 4}, {128, 4}, {128, 8}}; // tokens, waves of a K group
    for (const auto &s : shapes)
        for (int last = 0; last < s[0]; ++last) {
            check(s[0], s[1], last, 4, 1024, 32);
            check(s[0], s[1], last, 11, 11 * 256 + 16, 11 * 8 + 8);
            check(s[0], s[1], last, 32, 100000, 99992);
            check(s[0], s[1], last, 4, (1u << 24) - 16, (1u << 24) - 8); // 256 rows just within 32 bits
        }
    puts("ok");
}
"""


def test_every_copy_stays_inside_the_rows(tmp_path):
    compiler = shutil.which("g++") or shutil.which("clang++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no host C++ compiler")
    source, program = tmp_path / "copies.cpp", tmp_path / "copies"
    source.write_text(PROGRAM)
    subprocess.run([compiler, "-std=c++20", "-O1", f"-I{CSRC}", str(source), "-o", str(program)], check=True)
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0 and done.stdout == "ok\n", done.stdout


def test_the_kernel_copies_with_these_addresses():
    """Only the block is in the copies' scalar offset."""
    kernel = " ".join((CSRC / "iq3s_wide.hip").read_text().split())
    assert "16, vo, 256u * b, 0, 0);" in kernel and "4, soff_stage, 8u * b, 0, 0);" in kernel
    assert "voff[j] = wide_value_offset(wave, lane, W, j, last_row, (uint32_t)ldxv);" in kernel
    assert "soff_stage = wide_scale_offset(srow, lane, last_row, (uint32_t)ldxs);" in kernel
