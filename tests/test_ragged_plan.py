"""Chunk arithmetic of the ragged decode plan (csrc/ragged_plan.hpp), compiled for the host."""
import ctypes
import os
import random
import shutil
import subprocess

import pytest

from supersonic_amd import build as B

SHIM = r"""
#include "ragged_plan.hpp"
extern "C" int chunk_of(const int* lens, int B, int Hkv, int target, int min_chunk, int strict) {
    int64_t tot = 0, mx = 0;
    for (int b = 0; b < B; ++b) { tot += lens[b]; mx = lens[b] > mx ? lens[b] : mx; }
    return ssa::ragged_chunk(tot, Hkv, target, min_chunk, strict != 0, [&](int64_t c) {
        int64_t n = 0;
        for (int b = 0; b < B; ++b) { const int64_t s = (lens[b] + c - 1) / c; n += s > 1 ? s : 1; }
        return n * Hkv;
    }, [&]() { return mx; });
}
"""


@pytest.fixture(scope="module")
def chunk_of(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host C++ compiler")
    d = tmp_path_factory.mktemp("ragged")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "shim.so"
    subprocess.run([cxx, "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover", "-shared", "-fPIC", "-I",
                    B.CSRC, str(d / "shim.cpp"), "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))

    def call(lens, hkv, target, min_chunk=128, strict=True):
        return lib.chunk_of((ctypes.c_int * len(lens))(*lens), len(lens), hkv, target, min_chunk, int(strict))
    return call


def items(lens, hkv, ch):
    return hkv * sum(max(1, (n + ch - 1) // ch) for n in lens)


# (sequences, kv heads, length, workgroups): far more (sequence, kv head) pairs than workgroups, where the growth's
# product passes 32 bits (1024 x 4 pairs of 4096 tokens on 256: 2^32) and 64
@pytest.mark.parametrize("B,hkv,n,target", [(1024, 4, 4096, 256), (8, 4, 2048, 1), (8, 4, 32768, 1), (16, 4, 1024, 1),
                                            (16, 2, 2048, 1), (4, 4, 4096, 1), (4096, 4, 4096, 256),
                                            (16384, 1, 65536, 1), (512, 32, 32768, 128)])
@pytest.mark.parametrize("strict", [False, True])
def test_more_pairs_than_workgroups_take_one_split_each(chunk_of, B, hkv, n, target, strict):
    lens = [n] * B
    ch = chunk_of(lens, hkv, target, strict=strict)
    assert ch >= n and items(lens, hkv, ch) == B * hkv


def test_random_batches_get_a_usable_chunk(chunk_of):
    r = random.Random(5)
    for _ in range(3000):
        B, hkv = r.choice([1, 2, 7, 16, 64, 200, 1000]), r.choice([1, 2, 4, 8])
        top = r.choice([1, 17, 300, 4096, 70000])
        lens = [r.randint(0, top) for _ in range(B)]
        target = r.choice([1, 32, 96, 256, 512])
        ch = chunk_of(lens, hkv, target)
        assert ch >= 128
        # everything fits the workgroups, or every sequence has one split
        assert items(lens, hkv, ch) <= max(target, B * hkv)
        if B * hkv <= target:
            assert items(lens, hkv, ch) <= target
