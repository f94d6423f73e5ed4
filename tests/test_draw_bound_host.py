"""The bound that the wavefronts of a sampled draw share, from the kernel's own header compiled for the host."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from subspec_amd import build as build_mod

PROGRAM = r"""
#include "draw_bound.h"
#include <cstdio>
int main() {
  float key;
  while (fread(&key, 4, 1, stdin) == 1) {
    const uint32_t bits = subspec::seen_bits_of(key);
    const float level = subspec::seen_level(bits);
    const uint32_t least = subspec::least_seen_bits(key);
    fwrite(&bits, 4, 1, stdout);
    fwrite(&level, 4, 1, stdout);
    fwrite(&least, 4, 1, stdout);
  }
}
"""


@pytest.fixture(scope="module")
def bound(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc is not installed")
    folder = tmp_path_factory.mktemp("bound")
    src, exe = folder / "bound.cpp", str(folder / "bound")
    src.write_text(PROGRAM)
    subprocess.run([hipcc, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-ffp-contract=off", "-w", "-I", build_mod.CSRC, str(src), "-o", exe],
                   check=True, timeout=300)

    def call(keys):
        out = subprocess.run([exe], input=keys.tobytes(), stdout=subprocess.PIPE, check=True, timeout=60).stdout
        words = np.frombuffer(out, dtype=np.uint32).reshape(-1, 3)
        return words[:, 0].copy(), words[:, 1].copy().view(np.float32), words[:, 2].copy()

    return call


def test_every_key_has_a_bound_below_it_and_in_order(bound):
    """From the smallest subnormal to the largest key a draw can have (p = 1 at the largest u): finite, in the order of the
    keys, never above the key, and within a thousandth of it in log2."""
    rng = np.random.default_rng(0)
    exponents = np.arange(-149, 26, dtype=np.float64)
    keys = np.concatenate([2.0 ** exponents, 2.0 ** rng.uniform(-149, 25, 20000)]).astype(np.float32)
    keys = np.unique(keys[keys > 0])
    bits, level, _ = bound(keys)
    assert np.isfinite(level).all() and (bits > 0).all() and (bits < 0x7f800000).all()
    assert (np.diff(bits.astype(np.int64)) >= 0).all()
    log2 = level.astype(np.float64) / 2 ** 23 + 23
    exact = np.log2(keys.astype(np.float64))
    assert (log2 < exact).all() and (exact - log2 < 1e-3).all()


def test_the_bound_of_a_row_lies_below_the_key_of_its_maximum(bound):
    """Whatever the word of the row's largest element is, from the largest probability to 2^-31 of a flat row; no bound without one."""
    rng = np.random.default_rng(1)
    pmax = np.concatenate([2.0 ** -np.arange(0, 32), 2.0 ** -rng.uniform(0, 31, 2000)]).astype(np.float32)
    worst = (pmax / np.float32(-np.log(0.5 * 2.0 ** -23))).astype(np.float32)        # u = 2^-24, the smallest there is
    least, key = bound(pmax)[2], bound(worst)[0]
    assert (least > 0).all() and (least < key).all()
    assert (least[1:] != least[:-1]).any() and not bound(np.array([0.0, np.nan], np.float32))[2].any()
