"""The order in which the workgroups of the attention of runs start, from the kernels' own header, compiled for the host."""
import os
import subprocess

import pytest

from zipage_amd.engine.inputs import plan_prompts, plan_runs
from zipage_amd.engine.sequence import Portion, Sequence

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "zipage_amd", "csrc")
DRIVER = """
#include <cstdio>
#include <cstdlib>
#include "launch_order.h"
int main(int, char** v) {
  const int T = atoi(v[1]), heads = atoi(v[2]), rising = atoi(v[3]);
  for (int z = 0; z < FlowPlace::depth(T, heads); ++z)
    for (int part = 0; part < 8; ++part) {
      const FlowPlace p(T, heads, rising, part, z);
      printf("%d %d %d\\n", part, p.hk, p.tile);
    }
}
"""


@pytest.fixture(scope="module")
def launched(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-D__host__=", "-D__device__=", "-I", CSRC, str(d / "driver.cpp"), "-o", str(d / "driver")], check=True)

    def run(T, heads, rising):
        out = subprocess.run([str(d / "driver"), str(T), str(heads), str(int(rising))], check=True, capture_output=True, text=True).stdout
        return [tuple(map(int, l.split())) for l in out.splitlines()]
    return run


@pytest.mark.parametrize("heads", [1, 2, 3, 4, 6, 8, 12, 16])
@pytest.mark.parametrize("T", [1, 7, 8, 9, 64, 129])
@pytest.mark.parametrize("rising", [False, True])
def test_every_tile_of_every_head_once(launched, heads, T, rising):
    taken = sorted((h, t) for _, h, t in launched(T, heads, rising) if t < T)
    assert taken == [(h, t) for h in range(heads) for t in range(T)]


def _run(*lens):
    portions = []
    for n in lens:
        seq = Sequence([0] * n)
        seq.block_table = list(range(40))
        portions.append(Portion(seq, 0, n))
    return plan_runs(portions, 256, None).tiles


# the plans of whole prompts have their long tiles first, those of a run last
@pytest.mark.parametrize("rising,tiles", [(False, plan_prompts([300, 1000, 40, 2048], [300, 1000, 40, 2048])), (False, plan_prompts([600], [900])),
                                          (True, _run(2048)), (True, _run(130))], ids=["prompts", "cached", "run", "short"])
@pytest.mark.parametrize("heads", [1, 2, 4, 8])
def test_tiles_with_many_keys_start_first(launched, rising, tiles, heads):
    keys = (tiles[:, 1] + tiles[:, 3]).tolist()
    order = launched(len(tiles), heads, rising)
    for part in range(8):
        for head in range(heads):
            started = [keys[t] for p, h, t in order if p == part and h == head and t < len(tiles)]
            assert all(a >= b - 127 for a, b in zip(started, started[1:]))       # tiles are sorted by their first query
