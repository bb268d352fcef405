"""The back-off of failed attempts (dmrgpy_amd/csrc/backoff.h), compiled for the
host with g++ (CPU): with every attempt failing, the pauses between them are
1, 2, 4 ... 64, 64; a success in between starts over, and without failures
nothing is passed over."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, os.pardir, "dmrgpy_amd", "csrc")

HARNESS = r"""
#include "backoff.h"
#include <cstdio>
int main() {
  dmrg::Backoff b;
  auto pauses = [&](int attempts) {   // each attempt fails: chances passed over after it
    for (int k = 0; k < attempts; ++k) {
      if (!b.allowed()) { std::printf("refused "); return; }
      b.failed();
      int n = 0;
      while (b.skip > 0) n += !b.allowed();
      std::printf("%d ", n);
    }
  };
  pauses(9);
  b.allowed();
  b.succeeded();
  for (int k = 0; k < 3; ++k) { std::printf("%s", b.allowed() ? "yes " : "no "); b.succeeded(); }
  pauses(3);
  return 0;
}
"""


def test_pauses(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "harness.cpp", tmp_path / "harness"
    src.write_text(HARNESS)
    subprocess.run([gxx, "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split()
    assert out == ["1", "2", "4", "8", "16", "32", "64", "64", "64", "yes", "yes", "yes", "1", "2", "4"]
