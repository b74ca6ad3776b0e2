"""The k-steps of the ring kernel (``csrc/hip/ring_steps.h``, which the kernel includes), compiled for the host: what they
read of a row and what of it counts."""
import ctypes
import os
import shutil
import subprocess

import pytest

from glassbox_amd import build

SOURCE = """
#include "hip/ring_steps.h"
extern "C" int numbers(int i) { return i == 0 ? gb::RBK : i == 1 ? gb::RING_K : gb::RING_MIN_K; }
extern "C" int steps(int K) { return gb::ring_steps(K); }
extern "C" int step_at(int s, int K, int head) { return gb::ring_step_at(s, K, head != 0); }
extern "C" int dead_half(int K, int head) { return gb::ring_dead_half(K, head != 0); }
extern "C" int has(int height) { return gb::ring_has(height); }
extern "C" int rows(int M, int columns, int K, int i) {
  const gb::RingRows r = gb::ring_rows(M, columns, K);
  return i == 0 ? r.height : i == 1 ? r.tall : r.tiles;
}
"""


@pytest.fixture(scope="module")
def ring(tmp_path_factory):
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host compiler")
    folder = tmp_path_factory.mktemp("ring")
    source, lib = folder / "ring.cpp", folder / "ring.so"
    source.write_text(SOURCE)
    csrc = os.path.join(os.path.dirname(build.__file__), "csrc")
    subprocess.run([cxx, "-std=c++17", "-shared", "-fPIC", "-I", csrc, str(source), "-o", str(lib)], check=True)
    return ctypes.CDLL(str(lib))


def test_every_slice_reads_inside_its_row_and_counts_each_k_once(ring):
    """All products that ``gb_gemm_bf16_grouped`` divides (and undivided ones) up to a k of 1,024: a k-step lies inside the row,
    slices of 32 at the row's head among them, and the halves that count are the slice, each once."""
    step, unit, least = (ring.numbers(i) for i in range(3))
    for K in range(least, 1025, unit):
        for slices in range(1, K // unit + 1):
            k_slice = -(-(K // unit) // slices) * unit if slices > 1 else K
            if (slices - 1) * k_slice >= K:       # refused: a slice without a step
                continue
            for z in range(slices):
                at, size = z * k_slice, min(k_slice, K - z * k_slice)
                seen = []
                for s in range(ring.steps(size)):
                    begin = at + ring.step_at(s, size, int(z == 0))
                    assert 0 <= begin <= K - step, (K, slices, z, s, begin)
                    dead = ring.dead_half(size, int(z == 0)) if s + 1 == ring.steps(size) else -1
                    seen += [begin + i for i in range(step) if i // unit != dead]
                assert seen == list(range(at, at + size)), (K, slices, z)


@pytest.mark.parametrize("columns", [1, 7, 16, 24, 64, 112, 255, 256, 1000])
def test_tiles_hold_every_row_once(ring, columns):
    """The dealing of rows to tiles of two heights: as many rows of 32 as there are, none of them in two tiles, heights that the
    kernel is built for, and 256 wherever the compute units are filled by that."""
    for M in list(range(257, 2100)) + list(range(2100, 9000, 37)) + [30000, 65536, 131072 + 5, 1 << 20]:
        for K in (128, 2048, 14336):
            height, tall, tiles = (ring.rows(M, columns, K, i) for i in range(3))
            assert 5 <= height <= 8 and 1 <= tall <= tiles, (M, K)
            assert tall * height + (tiles - tall) * (height - 1) == -(-M // 32), (M, K)
    for M in (512, 2048, 8192):
        if M // 256 * columns % 256 == 0:
            assert ring.rows(M, columns, 4096, 0) == 8 and ring.rows(M, columns, 4096, 2) == M // 256


def test_rows_too_few_for_any_tile_are_told_from_the_others(ring):
    """A launch refuses a height that no kernel has, in place of launching nothing: up to 128 rows, and none of more."""
    for columns in (1, 16, 300):
        for M in range(1, 1500):
            assert bool(ring.has(ring.rows(M, columns, 2048, 0))) == (M > 128), M


@pytest.mark.parametrize("columns", [1, 3, 7, 24, 112])
def test_the_most_rows_that_a_grid_holds_stay_within_it(ring, columns):
    """A grid's second dimension ends at 65,535: as many tiles of 256 rows are taken, and tiles of fewer rows only as long as they fit."""
    for tiles in list(range(65500, 65536)):
        for M in (256 * tiles, 256 * tiles - 95):
            for K in (128, 2048):
                height, tall, dealt = (ring.rows(M, columns, K, i) for i in range(3))
                assert dealt <= 65535, (M, K)
                assert tall * height + (dealt - tall) * (height - 1) == -(-M // 32), (M, K)


@pytest.mark.parametrize("M,columns,K,heights", [
    (6151, 16, 14336, (7, 13, 30)), (6151, 24, 4096, (7, 7, 31)), (2048, 24, 2048, (7, 4, 10)), (5487, 16, 4096, (6, 12, 32)), (2048, 64, 2048, (8, 8, 8))])
def test_tiles_where_256_rows_leave_units_idle(ring, M, columns, K, heights):
    """The numbers of tiles that were the fastest of those measured."""
    assert tuple(ring.rows(M, columns, K, i) for i in range(3)) == heights
