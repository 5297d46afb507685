"""The planner autotuner's sweep (csrc/tuning_sweep.h) with made-up timings:
knobs are picked by passes that read them, never by passes that do not (g++
only, no GPU)."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "efficientstructuralgraphclusteringongpus_amd", "csrc")

DRIVER = r"""
#include <stdio.h>
#include <stdlib.h>
#include "tuning_sweep.h"

struct Knobs {
  uint32_t small_max_degree = 1024;
  double small_unit_work = 262144.0, large_unit_work = 8388608.0;
  uint32_t hash_tables = 1, tiny_work = 2048;
};

// counted passes: 100 ms and more for every knob away from the wanted values
int main(int argc, char** argv) {
  const bool filtered = atoi(argv[1]);
  Knobs want;
  want.large_unit_work = atof(argv[2]);
  want.small_max_degree = atoi(argv[3]);
  want.small_unit_work = atof(argv[4]);
  want.tiny_work = atoi(argv[5]);
  int plain = 0, counted = 0;
  auto measure = [&](const Knobs& t, bool filters, double* ms) {
    double slow = 100.0 + (t.large_unit_work != want.large_unit_work) + (t.small_max_degree != want.small_max_degree) +
                  (t.small_unit_work != want.small_unit_work) + (t.tiny_work != want.tiny_work) + 50.0 * !t.hash_tables;
    if (filtered && filters && t.hash_tables)
      *ms = 10.0 - 0.01 * plain++;  // every call a little faster, whatever the knobs
    else
      *ms = slow, ++counted;
    return 0;
  };
  Knobs best;
  double ms = 0, ms_default = 0;
  const int rc = sgc::sweep_tuning(filtered, measure, &best, &ms, &ms_default);
  printf("%d %.1f %u %.1f %u %u %d %d %d\n", rc, best.large_unit_work, best.small_max_degree, best.small_unit_work,
         best.tiny_work, best.hash_tables, ms <= ms_default, plain, counted);
}
"""


@pytest.fixture(scope="module")
def sweep(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not found")
    d = tmp_path_factory.mktemp("sweep")
    (d / "driver.cpp").write_text(DRIVER)
    exe = str(d / "driver")
    subprocess.run([gxx, "-std=c++17", "-Wall", "-Werror", "-I" + CSRC, str(d / "driver.cpp"), "-o", exe], check=True)

    def run(filtered, *want):
        out = subprocess.run([exe, str(int(filtered)), *map(str, want)], check=True, capture_output=True, text=True)
        rc, large, deg, small, tiny, hashes, kept, plain, counted = out.stdout.split()
        assert rc == "0" and hashes == "1" and kept == "1" and int(counted) > 0 and (int(plain) > 0) == filtered
        return float(large), int(deg), float(small), int(tiny)

    return run


@pytest.mark.parametrize("filtered", [False, True])
@pytest.mark.parametrize("want", [(8388608.0, 1024, 262144.0, 2048), (2097152.0, 256, 1048576.0, 0),
                                  (33554432.0, 128, 65536.0, 4096)])
def test_every_knob_is_picked_where_it_acts(sweep, filtered, want):
    assert sweep(filtered, *want) == want
