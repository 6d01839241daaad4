"""Workgroup -> query-tile maps (csrc/task_map.h), compiled for the host: every query tile and every key-range part
of a split sink tile is some workgroup's exactly once, and no head holds up an XCD for long."""

import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from sol_attn_amd import _build

CXX = shutil.which("g++")

SOURCE = r"""
#include <algorithm>
#define __host__
#define __device__
using std::max;
using std::min;
#include "task_map.h"
extern "C" int tasks(int ntiles, int front, int split_tiles, int heads, int splits, int head_xcds, int* out, int cap) {
  const int F = (split_tiles * (splits - 1) + front) * heads;
  const unsigned grid = head_xcds ? sol::head_grid(F, heads, ntiles - front, head_xcds)
                                  : sol::balanced_grid(F, heads, ntiles - front);
  if (int(grid) > cap) return -1;
  for (unsigned i = 0; i < grid; ++i) {
    const sol::TileTask t = sol::sol_task(int(i), ntiles, front, split_tiles, heads, splits, head_xcds);
    out[3 * i] = t.bh, out[3 * i + 1] = t.tile, out[3 * i + 2] = t.split;
  }
  return int(grid);
}
"""


@pytest.fixture(scope="module")
def tasks(tmp_path_factory):
    if CXX is None:
        pytest.skip("g++ not installed")
    d = tmp_path_factory.mktemp("map")
    (d / "map.cpp").write_text(SOURCE)
    subprocess.run([CXX, "-O2", "-shared", "-fPIC", "-I", _build.CSRC, str(d / "map.cpp"), "-o", str(d / "map.so")],
                   check=True, timeout=120)
    fn = ctypes.CDLL(str(d / "map.so")).tasks

    def call(ntiles, front, split_tiles, heads, splits, head_xcds):
        cap = heads * (ntiles + split_tiles * splits) + 64
        out = np.empty((cap, 3), np.int32)
        n = fn(ntiles, front, split_tiles, heads, splits, head_xcds, out.ctypes.data_as(ctypes.c_void_p), cap)
        assert n >= 0, "more workgroups than the tasks and a few idle ones"
        return out[:n]
    return call


SHAPES = [(nt, front, split, heads, s)
          for nt in (1, 2, 7, 8, 9, 63, 129) for heads in (1, 3, 7, 8, 9, 16, 24, 29, 504)
          for front, split, s in ((0, 0, 1), (2, 0, 1), (2, 2, 3), (3, 2, 8)) if front <= nt and nt * heads < 20000]


@pytest.mark.parametrize("head_xcds", [0, 1, 2, 4])
def test_every_tile_is_one_workgroups(tasks, head_xcds):
    for nt, front, split, heads, s in SHAPES:
        t = tasks(nt, front, split, heads, s, head_xcds)
        t = t[t[:, 0] >= 0]
        want = heads * (nt - split + split * s)
        assert len(t) == want, (nt, front, split, heads, s)
        assert len(np.unique(t, axis=0)) == want, (nt, front, split, heads, s)
        assert (t[:, 0] < heads).all() and (t[:, 1] >= 0).all() and (t[:, 1] < nt).all()
        assert (t[:, 2] >= 0).all() and (t[:, 2][t[:, 1] >= split] == 0).all() and (t[:, 2] < s).all()


@pytest.mark.parametrize("heads,nt,head_xcds,dense", [
    (16, 297, 4, [0]), (16, 297, 4, range(4)), (16, 297, 4, range(0, 16, 4)),
    (24, 128, 2, range(6)), (32, 64, 1, range(8)), (504, 63, 1, range(0, 504, 24))])
def test_dense_heads_are_shared_out(tasks, heads, nt, head_xcds, dense):
    # Tiles of the dense heads cost 10 times the others': the slowest XCD's work against the average.
    cost = np.ones(heads)
    cost[list(dense)] = 10.0
    t = tasks(nt, 0, 0, heads, 1, head_xcds)
    work = np.zeros(8)
    for x in range(8):
        bh = t[x::8, 0]
        work[x] = cost[bh[bh >= 0]].sum()
    assert work.max() <= 1.75 * work.mean(), work / work.mean()
