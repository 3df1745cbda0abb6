"""CPU: the map of the prefill launch that starts its heavy streams first gives every item to exactly one workgroup."""
import ctypes
import os
import random
import subprocess

import pytest

from neuralattentionsearch_amd import build

HARNESS = """
#include "nats_balanced_map.h"
#include <vector>
// items that are out of range or given twice, and heavy items that come after a light one
extern "C" long check(uint64_t heavy, int ns, int n_hg, int n_qg) {
  const int total = ns * n_hg * n_qg;
  std::vector<char> seen(total, 0);
  long wrong = 0;
  bool light = false;
  for (int bid = 0; bid < total; ++bid) {
    int ks = -1, hg = -1, rank = -1;
    nats::balanced_item(heavy, ns, n_hg, n_qg, bid, ks, hg, rank);
    if (ks < 0 || ks >= ns || hg < 0 || hg >= n_hg || rank < 0 || rank >= n_qg || seen[(ks * n_hg + hg) * n_qg + rank]++) {
      ++wrong;
      continue;
    }
    const bool h = heavy >> ks & 1;
    wrong += h && light;
    light = light || !h;
  }
  return wrong;
}
"""


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    d = tmp_path_factory.mktemp("balanced_map")
    src, lib = d / "harness.cpp", d / "harness.so"
    src.write_text(HARNESS)
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-fPIC", "-shared", "-fsanitize=undefined", "-fsanitize-undefined-trap-on-error",
                    "-D__host__=", "-D__device__=", "-I", build.CSRC, str(src), "-o", str(lib)], check=True)
    fn = ctypes.CDLL(str(lib)).check
    fn.restype, fn.argtypes = ctypes.c_long, [ctypes.c_uint64] + [ctypes.c_int] * 3
    return fn


def test_few_streams_every_set_of_heavy_ones(check):
    for ns in range(1, 11):
        for heavy in range(1 << ns):
            for n_hg, n_qg in ((1, 1), (1, 7), (2, 5), (3, 16)):
                assert check(heavy, ns, n_hg, n_qg) == 0, (ns, heavy, n_hg, n_qg)


def test_up_to_64_streams(check):
    rng = random.Random(0)
    for ns in (8, 9, 12, 15, 16, 17, 24, 31, 32, 33, 48, 56, 63, 64):
        every = (1 << ns) - 1
        sets = [0, 1, every, every - 1, 1 << (ns - 1), every & 0x0101010101010101, every & 0xff] + [rng.getrandbits(ns) for _ in range(30)]
        for heavy in sets:
            for n_hg, n_qg in ((1, rng.randint(1, 130)), (2, rng.randint(1, 40)), (8, rng.randint(1, 9))):
                assert check(heavy, ns, n_hg, n_qg) == 0, (ns, heavy, n_hg, n_qg)
