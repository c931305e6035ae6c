"""Host check of the Gram's work items (no GPU): rocket_amd/csrc/gram_items.hpp
itself, compiled for the host (gram_items_driver.cpp), must multiply every
128 x 64 block that meets the upper triangle exactly once per slab, from rows
that the item loads at that slab, into that block's place of its partial tile;
a split item must take its slabs in groups of ks; and both kinds of items must
be dealt evenly over the 8 XCDs (id mod 8)."""
import pathlib
import shutil
import subprocess

import numpy as np
import pytest

HERE = pathlib.Path(__file__).parent


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not shutil.which("g++") or not pathlib.Path("/opt/rocm/include/hip/hip_runtime.h").exists():
        pytest.skip("needs g++ and the HIP headers")
    exe = tmp_path_factory.mktemp("gram") / "gram_items_driver"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(HERE / "gram_items_driver.cpp"), "-o", str(exe)], check=True)

    def run(count, ks, S, remap):
        out = subprocess.run([str(exe), str(count), str(ks), str(S), str(int(remap))], check=True,
                             capture_output=True, text=True).stdout.splitlines()
        return [int(v) for v in out[0].split()], np.array([[int(v) for v in ln.split()] for ln in out[1:]])
    return run


@pytest.mark.parametrize("remap", [True, False])
@pytest.mark.parametrize("S", [1, 3, 8, 37, 64])
@pytest.mark.parametrize("count", [1, 120, 128, 129, 300, 384, 600, 800, 1100, 1400])
def test_every_block_and_slab_once(driver, count, S, remap):
    T, split = driver(count, 1, 1, False)[0][:2]
    for ks in {1, split}:
        (_, _, _, xcd_items), rows = driver(count, ks, S, remap)
        ident, u, first, wave, a, b, kqa, kqb, kw, tile, off = rows.T
        assert (first + 0 < S).all() and (kqa == kw).all() and (kqb == kw).all()
        assert (kw[(u < T - 1) | (ks == 1)] == 0).all()        # only the last item takes several slabs
        assert (first[(u == T - 1) & (ks > 1)] % ks == 0).all() and kw.max() < ks
        # the block's place in its partial tile (the triangle's tiles, row by row)
        nt = (count + 255) // 256
        ti, tj = a // 256, b // 256
        assert (tile == ti * nt - ti * (ti - 1) // 2 + (tj - ti)).all()
        assert (off == (a % 256) * 256 + b % 256).all()
        # every block that meets the triangle of the patterns, once per slab
        slab = first + kw
        here = slab < S                                        # past the last slab: not written
        got = sorted(zip(slab[here], a[here], b[here]))
        assert len(set(got)) == len(got)
        need = {(s, i, j) for s in range(S) for i in range(0, count, 128) for j in range(0, count, 64)
                if j + 63 >= i and (i // 128) <= (j // 128)}
        assert need <= set(got)
        assert all(i // 128 <= j // 128 for _, i, j in got)
        if remap:
            assert np.bincount(np.unique(ident) & 7, minlength=8).max() == xcd_items
            per_xcd = np.bincount(np.unique(ident[u < T - (ks > 1)]) & 7, minlength=8)
            assert per_xcd.max() - per_xcd.min() <= T
            per_xcd = np.bincount(np.unique(ident[(u == T - 1) & (ks > 1)]) & 7, minlength=8)
            assert per_xcd.max() - per_xcd.min() <= 1


@pytest.mark.parametrize("count,ks", [(1, 4), (128, 4), (129, 1), (300, 2), (600, 1), (800, 1), (1100, 4), (1300, 2)])
def test_split_fills_the_last_item(driver, count, ks):
    (T, split, _, _), rows = driver(count, ks, 4, False)
    assert split == ks
    last = rows[rows[:, 1] == T - 1]
    if ks > 1:  # its eight waves all work in a full group of slabs
        assert set(last[last[:, 2] == 0][:, 3]) == set(range(8))
