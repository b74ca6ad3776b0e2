"""Which kernel takes a bfloat16 product (``csrc/hip/gemm_bf16.hip``, ``route``): the built library's own answers on either side of the
lines that were measured.  Only sizes go in, so no GPU is needed."""
import ctypes
import os
import re

import pytest

from glassbox_amd import build

KERNELS = ("tiled", "ring", "few", "held", "block", "slices")
EPILOGUES = {"store": 0, "add": 1, "unit": 2, "heads": 3}


@pytest.fixture(scope="module")
def route():
    build.ensure(["gemm_bf16"])
    lib = ctypes.CDLL(os.path.join(os.path.dirname(build.__file__), "_lib", "libgb_gemm_bf16.so"))

    def ask(epilogue, M, N, K, parts=False, workspace=False):
        return KERNELS[lib.gb_gemm_bf16_route(M, N, K, EPILOGUES[epilogue], int(parts), int(workspace))]
    return ask


@pytest.mark.parametrize("epilogue,M,N,K,parts,kernel", [
    # what the held kernel is for: the products of some ten to sixty requests on the shapes of four models
    ("unit", 53, 5120, 960, True, "held"), ("unit", 24, 28672, 4096, True, "held"), ("unit", 20, 16384, 2048, True, "held"),
    ("heads", 24, 6144, 4096, True, "held"), ("heads", 64, 6144, 2048, True, "held"), ("heads", 53, 960, 576, True, "held"),
    ("store", 24, 128256, 4096, False, "held"), ("store", 53, 49152, 960, False, "held"), ("store", 17, 49152, 2048, False, "held"),
    # a short k, where a tile's fixed costs are more than reading the rows again (k of 128 by 4,112 rows of W, 17 rows: 4.4 us, 2.9)
    ("store", 17, 4112, 128, False, "few"), ("store", 64, 2048, 256, False, "few"), ("store", 32, 8192, 320, False, "few"),
    ("heads", 24, 6144, 256, False, "few"), ("unit", 17, 16384, 256, True, "few"),
    # two tiles a workgroup and two column blocks of rows: from a k of 1,280 on
    ("unit", 24, 5120, 960, True, "few"), ("unit", 24, 5120, 1280, True, "held"), ("heads", 17, 4608, 960, False, "few"),
    ("heads", 32, 4608, 1280, False, "held"), ("store", 24, 4112, 1024, False, "few"), ("store", 24, 4112, 1280, False, "held"),
    # 49 rows and more behind a norm: from a shorter one
    ("unit", 64, 5120, 384, True, "few"), ("unit", 64, 5120, 448, True, "held"), ("heads", 49, 4608, 576, True, "few"),
    ("heads", 49, 4608, 640, True, "held")])
def test_products_of_17_to_64_rows_go_to_the_held_kernel_where_it_is_ahead(route, epilogue, M, N, K, parts, kernel):
    assert route(epilogue, M, N, K, parts) == kernel


@pytest.mark.parametrize("epilogue,M,N,K,kernel", [
    # short prompts, turns and mixed steps on the shapes of four models
    ("unit", 131, 16384, 2048, "block"), ("unit", 512, 16384, 2048, "block"), ("unit", 611, 5120, 960, "block"), ("unit", 131, 28672, 4096, "block"),
    ("store", 131, 6144, 2048, "block"), ("store", 512, 6144, 2048, "block"),
    # one workgroup a compute unit either way: the tiled kernel starts sooner (256 x 4,096 x 1,280: 7.8 us, 9.6 in blocks)
    ("store", 256, 4096, 1280, "tiled"), ("add", 512, 512, 2048, "tiled"), ("store", 300, 512, 8192, "tiled"), ("add", 640, 2560, 1280, "tiled"),
    ("add", 1000, 1600, 1280, "block"), ("store", 400, 8192, 1792, "block"), ("store", 256, 3072, 8192, "block"), ("store", 256, 2048, 8192, "tiled"),
    ("store", 65, 6144, 1536, "block"), ("store", 65, 2048, 1536, "tiled"),
    # large tiles that leave units idle or are a second round, or as tall as the tiled kernel's over a short k
    ("unit", 512, 12288, 1280, "tiled"), ("unit", 640, 12288, 1024, "tiled"), ("add", 640, 5120, 1024, "tiled"), ("unit", 512, 8192, 256, "tiled"),
    ("unit", 512, 8192, 1024, "block"),
    # a gated unit of up to 64 rows: few gates and a k below 1,024 stay with the skinny kernel
    ("unit", 33, 4096, 960, "few"), ("unit", 33, 4096, 1024, "block"), ("unit", 33, 8208, 960, "block"), ("unit", 48, 3072, 128, "block"),
    # a vocabulary: 256 x 256 tiles in one round, and up to 64 rows the tiles
    ("store", 300, 32768, 4096, "ring"), ("store", 512, 49152, 3072, "ring"), ("store", 48, 49152, 4096, "tiled"), ("store", 48, 128256, 4096, "block"),
    # rows of W that 8 does not divide, and a k below 1,024
    ("store", 128, 3840, 960, "tiled"), ("store", 128, 9001, 2048, "tiled")])
def test_products_of_some_hundred_rows_go_to_the_block_kernel_where_it_is_ahead(route, epilogue, M, N, K, kernel):
    assert route(epilogue, M, N, K) == kernel


@pytest.mark.parametrize("epilogue,M,N,K,kernel", [
    ("add", 24, 4096, 14336, "slices"), ("add", 131, 2048, 8192, "slices"), ("add", 611, 960, 2560, "slices"), ("add", 2048, 2048, 8192, "slices"),
    # 65 to 128 rows by many rows of W: a long k only (96 x 8,192 x 14,336: 94 us whole, 57 in slices)
    ("add", 96, 8192, 8192, "block"), ("add", 96, 8192, 14336, "slices"), ("store", 100, 6144, 16384, "slices"), ("add", 128, 16384, 28672, "slices"),
    ("add", 24, 576, 1536, "few"), ("store", 131, 6144, 2048, "block"), ("store", 24, 6144, 4096, "held")])
def test_products_with_a_workspace_divide_k_where_that_is_ahead(route, epilogue, M, N, K, kernel):
    assert route(epilogue, M, N, K, workspace=True) == kernel


def test_kernels_of_up_to_16_rows_keep_everything_in_registers():
    """Such a kernel lasts a few microseconds: scratch would be traffic of every lane beside the one pass over W.  Read from what the
    compiler notes beside each kernel of the built library."""
    build.ensure(["gemm_bf16"])
    with open(build.find_current("gemm_bf16"), "rb") as fh:
        notes = re.findall(rb"\.name(?:\xd9.|\xda..)(\w*gemm_few_kernel\w*)\xbb\.private_segment_fixed_size(.)", fh.read(), re.DOTALL)
    assert len(notes) > 100
    assert [name.decode() for name, scratch in notes if scratch != b"\0"] == []
