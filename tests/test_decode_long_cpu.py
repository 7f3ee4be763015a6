"""The tables and cursors of the decoder for long chunks
(csrc/cachegen_decode.h: LongTables, RingCursor, PairCursor), compiled for
the host with g++ and checked against the oracle's decoder on random CDF rows
and byte streams; see tests/decode_long_check.cpp."""

from __future__ import annotations

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++") or not shutil.which("gcc"):
        pytest.skip("needs gcc and g++")
    d = tmp_path_factory.mktemp("declong")
    obj = d / "oracle_cachegen.o"
    exe = d / "decode_long_check"
    subprocess.run(["gcc", "-O2", "-c", os.path.join(REPO, "oracle", "cachegen.c"), "-o", str(obj)], check=True)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    os.path.join(HERE, "decode_long_check.cpp"), str(obj), "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_long_chunk_decoder_matches_oracle(program, seed):
    res = subprocess.run([program, "3000", str(seed)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout + res.stderr
    assert res.stdout.startswith("ok"), res.stdout
