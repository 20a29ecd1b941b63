"""The network passes' sharing of the neighbour list (csrc/kernels/nn_items.h),
compiled for the host: every i-sub-cluster of every entry is taken exactly once,
for any number of entries and any number of waves (a launch takes as many per CU
as it likes, on any number of CUs)."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
KERNELS = os.path.join(ROOT, "heddlemd_amd", "csrc", "kernels")

DRIVER = """
#include <vector>
#include "nn_items.h"
extern "C" uint32_t wrong(uint32_t entries, uint32_t n_waves) {
  const HmdNnItems items(entries, HMD_NN_ITEMS);
  std::vector<uint8_t> taken(8u * entries, 0);
  for (uint32_t v = 0; v < n_waves; ++v)
    for (uint32_t w = v; w < items.n; w += n_waves) {
      const uint32_t m = items.mask(w, n_waves);
      if (m == 0u || m > 255u || items.entry(w) >= entries) return ~0u;
      for (uint32_t b = 0; b < 8u; ++b) taken[8u * items.entry(w) + b] += (m >> b) & 1u;
    }
  uint32_t bad = 0;
  for (uint8_t t : taken) bad += t != 1u;
  return bad;
}
"""


@pytest.fixture(scope="module")
def wrong(tmp_path_factory):
    d = tmp_path_factory.mktemp("items")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{KERNELS}", "-o",
                    str(d / "driver.so"), str(d / "driver.cpp")], check=True)
    f = ctypes.CDLL(str(d / "driver.so")).wrong
    f.restype = ctypes.c_uint32
    f.argtypes = [ctypes.c_uint32, ctypes.c_uint32]
    return f


@pytest.mark.parametrize("n_waves", [1, 3, 4, 7, 8, 12, 300, 4 * 255, 4 * 256, 4 * 303,
                                     160 * 255, 160 * 256])
def test_every_sub_cluster_once(wrong, n_waves):
    for entries in (1, 2, 127, 2047, 2048, 2049, 4095, 8191, 8192, 16383, 16384, 53117):
        assert wrong(entries, n_waves) == 0, f"{entries} entries, {n_waves} waves"
