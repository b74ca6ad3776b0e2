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
