"""The dispatch rules of the decode GEMV (csrc/qgemv_route.h), compiled for the host: which calls of two and three columns
take the folding kernel, and which three-column calls are one launch. Both routes have the same bits, so only speed
depends on the lines checked here; each case is a call just inside and just outside of one."""
import ctypes
import os
import re
import subprocess

import pytest

import codeobj

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen27-engine_amd", "csrc")
SRC = """
#include "qgemv_route.h"
using namespace q27h;
extern "C" int fold(int type, int K, int nc, int tiles) { return fold_pays(type, K, nc, tiles); }
extern "C" int one(int type, int K, int nc) { return one_block(type, K, nc); }
extern "C" int three(int type, int K, int tiles, int fused) { return three_in_one(type, K, tiles, fused != 0); }
"""
IQ3_XXS, IQ3_S, IQ1_M = 18, 21, 29
TYPES = [10, 12, 14, 16, 17, 18, 21, 22, 23, 29]


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    d = tmp_path_factory.mktemp("route")
    (d / "route.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-shared", "-fPIC", "-I", CSRC, "-o", str(d / "route.so"),
                    str(d / "route.cpp")], check=True)
    return ctypes.CDLL(str(d / "route.so"))


@pytest.mark.parametrize("type_,K,nc,inside,outside", [
    (IQ3_S, 16640, 2, 768, 769), (IQ3_S, 24576, 2, 768, 769), (IQ3_S, 24832, 2, 256, 257), (IQ3_S, 32768, 2, 256, 257),
    (IQ3_XXS, 24576, 2, 768, 769), (IQ3_XXS, 24832, 2, 512, 513), (IQ1_M, 24832, 2, 512, 513),
    (IQ1_M, 16640, 3, 1280, 1281), (IQ1_M, 18688, 3, 2048, 2049), (IQ1_M, 24576, 3, 2048, 2049)])
def test_large_workgroups_fold_only_while_resident(route, type_, K, nc, inside, outside):
    assert route.fold(type_, K, nc, 1) and route.fold(type_, K, nc, inside)
    assert not route.fold(type_, K, nc, outside) and not route.fold(type_, K, nc, 1 << 20)


@pytest.mark.parametrize("type_,K,nc", [(IQ3_S, 8448, 2), (IQ3_XXS, 16384, 2), (IQ1_M, 24576, 2), (IQ3_S, 32768, 3),
                                        (IQ3_XXS, 32768, 3), (IQ1_M, 16384, 3), (IQ1_M, 24832, 3)])
def test_folds_at_every_size(route, type_, K, nc):
    for tiles in (1, 768, 2049, 1 << 20):
        assert route.fold(type_, K, nc, tiles)


def test_folds_only_where_the_orders_differ(route):
    for type_ in TYPES:
        for K in range(256, 40961, 256):
            for nc in (1, 2, 3, 4):
                if route.fold(type_, K, nc, 1):
                    assert nc in (2, 3) and type_ in (IQ3_XXS, IQ3_S, IQ1_M) and 8192 < K <= 32768


def test_three_columns_in_one_launch(route):
    for type_ in TYPES:
        for K in range(256, 40961, 256):
            differ = type_ in (IQ3_XXS, IQ3_S, IQ1_M) and 8192 < K <= 32768
            for tiles in (1, 640, 5000):
                assert route.three(type_, K, tiles, 0) == (not differ or route.fold(type_, K, 3, tiles))
                assert route.three(type_, K, tiles, 1) == (not differ and 3 * K <= 40960)


def test_built_kernels_are_those_some_call_takes(route):
    """Every instantiation that a call of some K and number of tiles takes is in the library, and no other."""
    want = set()
    for type_ in TYPES:
        for nc in (1, 2, 3, 4):
            for fused in (0, 1):
                for K in range(256, 40961, 256):
                    if fused and (2 if nc == 3 else nc) * K > 40960:
                        continue
                    for tiles in (1, 1 << 20):
                        cols = [nc] if nc != 3 or route.three(type_, K, tiles, fused) else [2, 1]
                        for c in cols:
                            if not fused and route.fold(type_, K, c, tiles):
                                want.add(f"qgemv_fold_kernelILi{type_}ELi{c}EE")
                            elif route.one(type_, K, c):
                                want.add(f"qgemv_one_kernelILi{type_}ELi{c}ELb{fused}EE")
                            else:
                                want.add(f"qgemv_kernelILi{type_}ELi{c}ELb{int(K <= 8192)}ELb{fused}EE")
    built = {re.search(r"qgemv\w*?_kernelI\w*?EE", n).group(0) for n in codeobj.kernels() if "qgemv" in n}
    assert built == want, (sorted(want - built), sorted(built - want))
