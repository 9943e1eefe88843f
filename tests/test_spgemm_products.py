"""The index arithmetic of SpGEMM's walk over a row's products (csrc/products.hpp), compiled for the host: no place that a
lane reads lies outside the row of B that its entry of A selects, whatever the order of the entries."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "scorch_amd", "csrc")
SLOTS = 4
HARNESS = """
#include "products.hpp"
extern "C" void step(int x, int count, int waves, int wave, int *range, int *read) {
  const scorch::ProductStep s = scorch::product_step(x, count, waves, wave);
  range[0] = s.first, range[1] = s.last;
  for (int u = 0; u < %d; ++u)
    for (int lane = 0; lane < 64; ++lane)
      read[64 * u + lane] = s.first < s.last && s.has(u) ? s.product(u, lane) : -1;
}
""" % SLOTS


@pytest.fixture(scope="module")
def step(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("no host compiler")
    where = tmp_path_factory.mktemp("products")
    (where / "step.cpp").write_text(HARNESS)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(where / "step.cpp"),
                    "-o", str(where / "step.so")], check=True)
    fn = ctypes.CDLL(str(where / "step.so")).step

    def call(x, count, waves, wave):
        bounds, read = np.zeros(2, np.int32), np.zeros(64 * SLOTS, np.int32)
        at = ctypes.POINTER(ctypes.c_int)
        fn(x, count, waves, wave, bounds.ctypes.data_as(at), read.ctypes.data_as(at))
        return bounds[0], bounds[1], read
    return call


def _walk(step, lens, starts, waves):
    """The entries of a batch (numbers of products, first places in B), as the kernels walk them: fill_batch leaves out
    entries without products; the entry of product x of a wavefront is the last one that begins at or before x among those
    that begin before the wavefront's end, which is all that entries_of_products promises."""
    lens, starts = lens[lens > 0], starts[lens > 0]
    first = np.concatenate([[0], np.cumsum(lens)])
    total, first = int(first[-1]), first[:-1]
    made = np.zeros(total, int)
    for x in range(0, total, SLOTS * 64 * waves):
        for wave in range(waves):
            lo, hi, read = step(x, min(SLOTS * 64 * waves, total - x), waves, wave)
            if lo >= hi:
                continue
            assert 0 <= lo < hi <= min(total, lo + SLOTS * 64)
            read_at = np.arange(lo, lo + SLOTS * 64)            # what slot and lane stand for
            begun = first[first < hi]
            entry = np.searchsorted(begun, read_at, side="right") - 1
            loaded = read >= 0
            place = read + starts[entry] - first[entry]
            inside = (place >= starts[entry]) & (place < starts[entry] + lens[entry])
            assert inside[loaded].all(), (x, wave, np.flatnonzero(loaded & ~inside)[:4])
            own = read_at < hi
            assert loaded[own].all() and np.array_equal(read[own], read_at[own])
            made[read_at[own]] += 1
    assert (made == 1).all()


@pytest.mark.parametrize("waves", [4, 8, 16])               # rows to a workgroup of 256 and of 1,024, the sort's of 512
@pytest.mark.parametrize("order", ["ascending", "descending", "shuffled", "repeated", "last row of B in the middle"])
def test_no_lane_reads_outside_its_entrys_row_of_b(step, waves, order):
    rng = np.random.default_rng(waves)
    for _ in range(25):
        rows_of_b = rng.integers(0, rng.choice([2, 5, 40, 300]), 400)
        rows_of_b[-1] = rng.integers(1, 200)
        pos = np.concatenate([[0], np.cumsum(rows_of_b)])
        entries = np.sort(rng.choice(400, rng.integers(1, min(400, 64 * waves)), replace=False))
        if order == "descending":
            entries = entries[::-1]
        elif order == "shuffled":
            entries = rng.permutation(entries)
        elif order == "repeated":
            entries = np.full(entries.size, rng.integers(400))
        elif order.startswith("last row"):
            entries = np.insert(entries, entries.size // 2, 399)
        _walk(step, rows_of_b[entries], pos[entries], waves)


@pytest.mark.parametrize("count", [1, 63, 64, 65, 191, 192, 511, 512, 513, 1024, 1025, 1536, 1537, 2047, 2048])
def test_every_size_of_a_windows_remainder(step, count):
    """One to four slots to a wavefront of the sort's eight, with entries of one product and of a few."""
    for lens in (np.ones(count, int), np.diff(np.unique(np.concatenate([np.arange(0, count, 7), [count]])))):
        _walk(step, np.concatenate([[2048], lens]), np.concatenate([[10_000], 9000 - np.cumsum(lens)]), 8)
